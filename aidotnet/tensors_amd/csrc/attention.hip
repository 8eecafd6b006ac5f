// Fused scaled-dot-product attention (forward) for gfx950: flash-style, one pass over K/V
// tiles streamed through LDS, QK^T and PV on MFMA, online softmax in fp32 registers.
//
// Replaces, behind the reference's GPU-backend slot, FlashAttentionV2 / FlashAttention /
// ScaledDotProductAttention (src/AiDotNet.Tensors/Engines/DirectGpu/HIP/HipBackend.cs:6118-6302,
// kernel strings Kernels/HipAttentionKernels.cs:33-232); value semantics are the CPU engine's
// (src/AiDotNet.Tensors/Engines/CpuEngine.cs:29146-29288, 27695-27881).
//
// Formulation (per workgroup: 128 query rows of one (batch, head); per wave: 32 query rows):
//   S^T = K_tile * Q^T    MFMA rows = keys, cols = queries.  Lane l then holds query (l % 32)
//                          and 16 keys per 32-key sub-tile, so the row max / sum of a query are
//                          an in-lane reduction plus ONE cross-lane exchange (lane ^ 32), and the
//                          rescale factor of the output accumulator is a per-lane scalar.
//   O^T += V_tile^T * P^T  MFMA rows = head-dim, cols = queries.  P^T in accumulator layout is
//                          already the B-operand fragment (each lane owns the keys it needs), no
//                          shuffles; V is transposed on its way into LDS ([d][key], keys of one
//                          16-group stored in fragment order so a lane's 8 keys are 16 contiguous
//                          bytes).
// K/V tiles are double-buffered in LDS: global loads of tile j+1 are issued before the MFMAs of
// tile j and stored after them, one barrier per tile.
#include "attention_common.hpp"

namespace aidn {

// Per tile and wave the general form of 16-bit head dimension 64 is bound by what it issues (64 keys: 16 MFMAs of 32 cycles beside some 300 other
// instructions, a lone wave one in 5 cycles): loads of a whole tile by a uniform base and fixed lane offsets, one multiply-add per logit, masks
// against one bound a lane.  Against 64-bit addresses a load, a multiplication and a subtraction a logit, two tests an element, bf16 us: B8 H32
// S2048 causal 218 -> 195, B16 H12 S512 29.8 -> 23.7, B8 H12 S512 causal 14.3 -> 12.9.  (A third stage of LDS gained nothing: 19.9 / 20.3.)
// DMA (fp32, plain / causal, aligned contiguous K/V): the K and V tiles go global -> LDS directly, unpadded [key][d] rows with
// XOR-swizzled 16-byte chunks (K: c ^ (key & 15) for the b128 fragment reads; V: c ^ (((key >> 2) & 1) << 3), read as the
// A operand of O^T += V^T P^T with 32-bit LDS reads, the two lane halves -- keys 4 apart -- in different bank halves).  This
// removes the register -> LDS store path (and the V transpose in registers) of the general form.
// KM (DMA form): a keep-mask of the keys shared by the heads and queries of a batch (mask_mode 3).  A tile's mask is one ballot, tested
// per element by a constant bit and only where the tile is mixed; a tile without a visible key is not computed.  A padded batch (bf16 B8
// H12 S512 d64, lengths 256 .. 512) took 85.6 us with the mask as a [B,H,S,S] tensor on the general form, 23.0 this way.
// KG: how many waves share a query row's keys (launch_attn): a workgroup holds 128 / KG rows, a wave takes BC / KG keys of every tile for
// its 32 rows, and the KG unnormalised results of a row are merged through LDS behind the last tile.
template <typename T, typename OutT, int DP, int BC, bool FULL, int MINB, bool DMA = false, bool KM = false, int KG = 1>
__global__ __launch_bounds__(256, MINB) void attn_fwd_kernel(const AttnArgs a)
{
    static_assert(!KM || DMA, "the key mask of a tile is formed beside direct-to-LDS loads");
    static_assert(!DMA || (!FULL && (DP == 64 || (Elem<T>::BYTES == 4 && DP == 128) || (Elem<T>::BYTES == 2 && DP == 256))),
                  "DMA form: head dimension 64 (or fp32 128 / 16-bit 256), plain / causal");
    static_assert(!KM || BC <= 64, "a tile's key mask is one ballot");
    typedef typename Raw2<T>::type raw_t;
    constexpr int E = Elem<T>::PER16, EB = Elem<T>::BYTES;
    constexpr int WQ = 4 / KG;                 // waves over the query rows; the KG waves of a row group share the keys of a tile
    constexpr int NT = 256, BR = 32 * WQ;
    constexpr int KS = Mma32<T>::KS;
    constexpr int DSTEPS = DP / KS;            // fragment steps over the head dim (QK^T)
    constexpr int KPITCH = DP * EB + 16;       // K tile [key][d] row pitch, bytes
    constexpr int VPITCH = BC * EB + 16;       // V^T tile [d][key] row pitch, bytes
    constexpr int KBYTES = DMA ? BC * DP * EB : BC * KPITCH, VBYTES = DMA ? BC * DP * EB : DP * VPITCH;
    constexpr int KT = BC / 32 / KG;           // 32-key sub-tiles per tile and wave
    static_assert(KT >= 1, "every key group has a sub-tile of its own");
    // The two groups of a 16-bit 128-key tile take its 32-key blocks in turn and each block moves the exponent reference: the same keys to a group and
    // the same probabilities that are exactly one as on 64-key tiles, so the same error (64 keys to a reference: 3 - 6 % more).  For half as many
    // barriers (bf16 causal n 480 S2525 33.1 -> 28.8 us, n 528 S1355 20.7 -> 18.7, n 264 S674 13.4 -> 12.6)
    constexpr bool TURNS = EB == 2 && DP == 64 && !FULL && BC == 128 && KG == 2;
    constexpr int KSTEP = TURNS ? 64 : 32;     // keys from one sub-tile of a wave to the next
    constexpr int KG0 = TURNS ? 32 : KT * 32;  // and from a group's first key to the next group's
    constexpr int REF = TURNS ? 1 : KT;        // sub-tiles to one exponent reference
    constexpr int DT = DP / 32;                // 32-row tiles of O^T
    constexpr int PSTEPS = 32 / KS;            // PV fragment steps per key sub-tile
    constexpr int CPR = DP / E;                // 16-byte chunks per K row
    constexpr int NKC = BC * CPR;              // K chunks per tile
    constexpr int UK = (NKC + NT - 1) / NT;
    constexpr int NVU = (BC / 4) * CPR;        // V units: 4 keys x E head-dim elements
    constexpr int UV = (NVU + NT - 1) / NT;

    extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
    unsigned char* Ks = smem;                  // [2][KBYTES]
    unsigned char* Vs = smem + 2 * KBYTES;     // [2][VBYTES]

    const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
    const int l32 = lane & 31, h = lane >> 5;

    int bh, qt;
    attn_block(a, bh, qt);
    const int b = bh / a.H, hd = bh - b * a.H;
    const int kvh = hd / (a.H / a.Hkv);
    const int q0 = qt * BR;
    // this wave's row group and key group (a constant with one group: the compiler does not know that wave < 4)
    const int wq = KG == 1 ? wave : wave % WQ, kg = KG == 1 ? 0 : wave / WQ;
    const int qi = q0 + wq * 32 + l32;         // this lane's query row
    const bool vec = a.vec_in != 0;

    const raw_t* __restrict__ Q = (const raw_t*)a.q + b * a.qs[0] + hd * a.qs[1];
    const raw_t* __restrict__ K = (const raw_t*)a.k + b * a.ks[0] + kvh * a.ks[1];
    const raw_t* __restrict__ V = (const raw_t*)a.v + b * a.vs[0] + kvh * a.vs[1];
    const int* __restrict__ bt = a.bt ? a.bt + b * a.bt_bs : nullptr;

    // ---- Q fragments (B operand of S^T): row qi, 16-byte chunk (2 s + h).  Up to head dimension 128 they stay in registers for
    // the whole kernel; at 256 (where O alone takes 128 registers and the kernel would spill) every tile fetches them again: the
    // query tile is 128 KiB at most and stays in the CU's cache.
    constexpr bool QREG = DP <= 128;
    auto load_q = [&](int s) -> u32x4 {
        int d0 = (2 * s + h) * E;
        return (qi < a.Sq) ? ld16<T>(Q + (long long)qi * a.qs[2] + d0, a.D - d0, vec) : u32x4{0u, 0u, 0u, 0u};
    };
    u32x4 qf[QREG ? DSTEPS : 1];
    if constexpr (QREG) {
#pragma unroll
        for (int s = 0; s < DSTEPS; s++) qf[s] = load_q(s);
    }

    // ---- number of K/V tiles this query tile needs
    int ntiles = (a.Sk + BC - 1) / BC;
    if (a.causal) {
        long long lastkey = (long long)q0 + BR - 1 + a.qoff;      // largest unmasked key of the tile's last row
        if (lastkey < 0) ntiles = 0;
        else { long long nt = lastkey / BC + 1; if (nt < ntiles) ntiles = (int)nt; }
    }
    // a share of them (ranges of the keys; from here on ntiles is where it ends)
    constexpr bool RANGES = EB == 2 && DP == 64 && !FULL;
    int first = 0;
    if (RANGES && a.nsplit > 1) {
        const int per = (ntiles + a.nsplit - 1) / a.nsplit;
        first = min((int)blockIdx.y * per, ntiles);
        ntiles = min(ntiles, first + per);
    }

    u32x4 rk[UK];
    u32x4 rv[UV * 4];

    auto load_tile = [&](int kv0) {
#pragma unroll
        for (int i = 0; i < UK; i++) {
            int u = t + i * NT;
            int row = u / CPR, ch = u - row * CPR;
            int key = kv0 + row, d0 = ch * E;
            u32x4 v = {0u, 0u, 0u, 0u};
            if ((NKC % NT == 0 || u < NKC) && key < a.Sk) v = ld16<T>(K + paged_row(bt, a.bsz, key) * a.ks[2] + d0, a.D - d0, vec);
            rk[i] = v;
        }
#pragma unroll
        for (int i = 0; i < UV; i++) {
            int u = t + i * NT;
            int kb = u % (BC / 4), db = u / (BC / 4);
            int d0 = db * E;
#pragma unroll
            for (int r = 0; r < 4; r++) {
                int key = kv0 + kb * 4 + r;
                u32x4 v = {0u, 0u, 0u, 0u};
                if ((NVU % NT == 0 || u < NVU) && key < a.Sk) v = ld16<T>(V + paged_row(bt, a.bsz, key) * a.vs[2] + d0, a.D - d0, vec);
                rv[i * 4 + r] = v;
            }
        }
    };

    auto store_tile = [&](int stage) {
        unsigned char* ks = Ks + stage * KBYTES;
        unsigned char* vs = Vs + stage * VBYTES;
#pragma unroll
        for (int i = 0; i < UK; i++) {
            int u = t + i * NT;
            int row = u / CPR, ch = u - row * CPR;
            if (NKC % NT == 0 || u < NKC) *(u32x4*)(ks + row * KPITCH + ch * 16) = rk[i];
        }
#pragma unroll
        for (int i = 0; i < UV; i++) {
            int u = t + i * NT;
            int kb = u % (BC / 4), db = u / (BC / 4);
            if (NVU % NT == 0 || u < NVU) {
                if constexpr (E == 8) {
                    // 4 keys x 8 d  ->  8 rows (d) of 4 keys (8 bytes).  Keys of a 16-group are stored
                    // in fragment order: 4-key blocks (0,1,2,3) at block positions (0,2,1,3).
                    int blk = kb & 3;
                    int pblk = ((blk & 1) << 1) | (blk >> 1);
                    int kpos = (kb >> 2) * 16 + pblk * 4;              // in elements
#pragma unroll
                    for (int c = 0; c < 8; c++) {
                        uint32_t a0 = rv[i * 4 + 0][c >> 1], a1 = rv[i * 4 + 1][c >> 1];
                        uint32_t a2 = rv[i * 4 + 2][c >> 1], a3 = rv[i * 4 + 3][c >> 1];
                        u32x2 o;
                        if (c & 1) { o[0] = __builtin_amdgcn_perm(a1, a0, 0x07060302u); o[1] = __builtin_amdgcn_perm(a3, a2, 0x07060302u); }
                        else       { o[0] = __builtin_amdgcn_perm(a1, a0, 0x05040100u); o[1] = __builtin_amdgcn_perm(a3, a2, 0x05040100u); }
                        *(u32x2*)(vs + (db * 8 + c) * VPITCH + kpos * 2) = o;
                    }
                } else {
                    // 4 keys x 4 d -> 4 rows (d) of 4 keys (16 bytes), natural key order
#pragma unroll
                    for (int c = 0; c < 4; c++) {
                        u32x4 o = {rv[i * 4 + 0][c], rv[i * 4 + 1][c], rv[i * 4 + 2][c], rv[i * 4 + 3][c]};
                        *(u32x4*)(vs + (db * 4 + c) * VPITCH + kb * 16) = o;
                    }
                }
            }
        }
    };

    f32x16 oacc[DT];
#pragma unroll
    for (int i = 0; i < DT; i++)
#pragma unroll
        for (int r = 0; r < 16; r++) oacc[i][r] = 0.0f;
    float m_run = -INFINITY;     // running max of the log2-domain logits of query qi (same in lanes l and l^32)
    float l_run = 0.0f;          // this lane's share of the running sum

    const int wq_min = q0 + wq * 32, wq_max = wq_min + 31;
    const float sl2 = a.scale * LOG2E;

    // DMA form: this wave's loads of a tile are K and V wave-loads 4 wave .. 4 wave + 3 (4 keys x 256 bytes each); rows past
    // the end of the sequence repeat the last key (masked below)
    const uint32_t lds0 = (uint32_t)(uintptr_t)((__attribute__((address_space(3))) void*)smem);
    const int wave_s = __builtin_amdgcn_readfirstlane(wave);
    // swizzles of the DMA form (chunk position of 16-byte chunk c of key row `key`):
    //   fp32 (256- / 512-byte rows): K  c ^ (key & 15);         V  c ^ (((key >> 2) & 1) << 3)   (32-bit reads, lane halves 4 keys apart)
    //   16-bit, 128-byte rows:       K  c ^ ((key >> 1) & 7);   V  c ^ (((key >> 1) & 1) << 2)   (transposing reads of 4 consecutive keys)
    //   16-bit, 512-byte rows:       K  c ^ (key & 15);         V  c ^ ((key & 3) << 2)
    constexpr bool WIDE16 = EB == 2 && DP * EB > 128;
    auto k_swz = [](int key) -> int { return (EB == 4 || WIDE16) ? (key & 15) : ((key >> 1) & 7); };
    auto v_swz = [](int key) -> int { return EB == 4 ? (((key >> 2) & 1) << 3) : WIDE16 ? ((key & 3) << 2) : (((key >> 1) & 1) << 2); };
    int rows = 0;                  // paged cache: pool rows of this wave's keys, one tile per lane
    constexpr int ROWB = DP * EB;                          // 256 / 128 bytes per key row
    constexpr int KPL = 1024 / ROWB;                       // keys per 1 KiB wave-load
    constexpr int LPW = DMA ? BC / KPL / 4 : 1;            // wave-loads per wave and tile (K and V each)
    constexpr int CPRW = ROWB / 16;                        // chunks per row
    constexpr int NK = KPL * LPW;                          // keys per wave and tile
    constexpr int NO = LPW < 16 / KPL ? LPW : 16 / KPL;    // loads until the swizzle repeats
    const int ld_key = lane / CPRW, ld_pos = lane % CPRW;
    constexpr bool FIXED = DMA && DP <= 128;               // (at 256 the offsets do not fit the registers)
    uint32_t koff[NO], voff[NO];
    if constexpr (FIXED) {
#pragma unroll
        for (int i = 0; i < NO; i++) {
            const int key = NK * wave + KPL * i + ld_key;
            koff[i] = (uint32_t)(ld_key * (int)a.ks[2] + (ld_pos ^ k_swz(key)) * E) * EB;
            voff[i] = (uint32_t)(ld_key * (int)a.vs[2] + (ld_pos ^ v_swz(key)) * E) * EB;
        }
    }
    auto issue_tile = [&](int tile, int stage) {
        // first row of the wave's keys and the last one to load, relative to it
        int row0 = tile * BC + NK * wave_s, left = a.Sk - 1 - row0;
        if (bt) {
            const int last_group = (a.Sk - 1) / NK * NK;
            if (((tile - first) & 63) == 0) rows = paged_tile_rows(bt, a.bsz, a.dbsz, NK * wave_s, BC, tile, lane, last_group);
            left = a.Sk - 1 - min(row0, last_group);
            row0 = __builtin_amdgcn_readlane(rows, (tile - first) & 63);
        }
        if (FIXED && left >= NK - 1) {
            // whole: a uniform base and lane offsets that stay (the swizzle repeats with 16 keys)
            const unsigned char* kb = (const unsigned char*)(K + (long long)row0 * a.ks[2]);
            const unsigned char* vb = (const unsigned char*)(V + (long long)row0 * a.vs[2]);
#pragma unroll
            for (int i = 0; i < LPW; i++) {
                attn_dma16_base(kb + (long long)(KPL * i) * a.ks[2] * EB, koff[i % NO], lds0 + stage * KBYTES + (LPW * wave_s + i) * 1024);
                attn_dma16_base(vb + (long long)(KPL * i) * a.vs[2] * EB, voff[i % NO], lds0 + 2 * KBYTES + stage * VBYTES + (LPW * wave_s + i) * 1024);
            }
            return;
        }
#pragma unroll
        for (int i = 0; i < LPW; i++) {
            const int key = KPL * (LPW * wave + i) + ld_key;               // key inside the tile
            const long long gkey = row0 + min(KPL * i + ld_key, left);
            attn_dma16(K + gkey * a.ks[2] + (ld_pos ^ k_swz(key)) * E, lds0 + stage * KBYTES + (LPW * wave_s + i) * 1024);
            attn_dma16(V + gkey * a.vs[2] + (ld_pos ^ v_swz(key)) * E,
                       lds0 + 2 * KBYTES + stage * VBYTES + (LPW * wave_s + i) * 1024);
        }
    };
    // KM: visible keys of the current tile (keys past the end are not), the same in every wave
    const unsigned char* __restrict__ kmask = KM ? (const unsigned char*)a.mask + (long long)b * a.Sk : nullptr;
    auto tile_keys = [&](int kv0, unsigned keep) -> uint64_t {
        return __builtin_amdgcn_ballot_w64(lane < BC && kv0 + lane < a.Sk && keep != 0);
    };
    uint64_t kbits = ~0ull;
    if constexpr (DMA) {
        if (first < ntiles) issue_tile(first, first & 1);
        if constexpr (KM) kbits = tile_keys(first * BC, kmask[min(first * BC + lane, a.Sk - 1)]);
        __builtin_amdgcn_s_waitcnt(0);
    } else {
        if (first < ntiles) {
            load_tile(first * BC);
            store_tile(first & 1);
        }
    }
    __syncthreads();

    for (int j = first; j < ntiles; j++) {
        const int stage = j & 1;
        const int kv0 = j * BC;
        const int kw0 = kv0 + kg * KG0;          // first key of this wave's sub-tiles
        unsigned next_keep = 0;        // (read with the next tile's loads, looked at when they have landed)
        if constexpr (KM) next_keep = kmask[min(kv0 + BC + lane, a.Sk - 1)];
        if constexpr (DMA) { if (j + 1 < ntiles) issue_tile(j + 1, stage ^ 1); }
        else if (j + 1 < ntiles) load_tile(kv0 + BC);

        // a wave whose 32 rows are all above the causal diagonal of its keys, or past the last row or key, only helps with the copies
        const bool active = wq_min < a.Sq && kw0 < a.Sk && !(a.causal && (long long)kw0 > (long long)wq_max + a.qoff) && (!KM || kbits != 0);
        if (active) {
            const int kr0 = kg * KG0;            // this wave's first key inside the tile
            const unsigned char* ks = Ks + stage * KBYTES + (kr0 + l32) * KPITCH + h * 16;
            const unsigned char* vs = Vs + stage * VBYTES + l32 * VPITCH + kr0 * EB + h * 16;

            // general form: a mask of the keys alone as one ballot per tile too (a third kind of mask in the test of every element cost the
            // calls with planes and biases up to 5 %)
            unsigned keep = 1;
            if constexpr (FULL) { if (a.mask_mode == 3) keep = ((const unsigned char*)a.mask)[(long long)b * a.Sk + min(kv0 + lane, a.Sk - 1)]; }

            f32x16 st[KT];
#pragma unroll
            for (int kt = 0; kt < KT; kt++)
#pragma unroll
                for (int r = 0; r < 16; r++) st[kt][r] = 0.0f;
            // fp32: the two MFMA phases run at a raised wave priority, ahead of the other workgroup's softmax on the SIMD (1-3 %
            // measured; the 16-bit instances lose with it)
            if constexpr (EB == 4) __builtin_amdgcn_s_setprio(2);
            constexpr int QA = 4;                 // Q fragments fetched ahead when they are not resident
            u32x4 qring[QREG ? 1 : QA];
            if constexpr (!QREG) {
#pragma unroll
                for (int s = 0; s < QA; s++) qring[s] = load_q(s);
            }
#pragma unroll
            for (int s = 0; s < DSTEPS; s++) {
                u32x4 qs;
                if constexpr (QREG) qs = qf[s];
                else {
                    qs = qring[s % QA];
                    if (s + QA < DSTEPS) qring[s % QA] = load_q(s + QA);
                }
#pragma unroll
                for (int kt = 0; kt < KT; kt++) {
                    u32x4 kf;
                    if constexpr (DMA) kf = *(const u32x4*)(Ks + stage * KBYTES + (kr0 + kt * KSTEP + l32) * (DP * EB) + (((2 * s + h) ^ k_swz(l32)) << 4));
                    else kf = *(const u32x4*)(ks + kt * KSTEP * KPITCH + s * 32);
                    Mma32<T>::run(st[kt], kf, qs);
                }
            }
            if constexpr (EB == 4) __builtin_amdgcn_s_setprio(0);

            // ---- logits in the log2 domain, masks
            const bool need_mask = (kw0 + (KT - 1) * KSTEP + 32 > a.Sk) || (a.causal && (long long)kw0 + (KT - 1) * KSTEP + 31 > (long long)wq_min + a.qoff);
            if constexpr (FULL) kbits = __builtin_amdgcn_ballot_w64(keep != 0);      // (keys past the end are masked below)
            const bool mixed = (KM || FULL) && (BC == 64 ? kbits != ~0ull : (uint32_t)kbits != ~0u);
            if constexpr (FULL) {
                // one pass over the tile per option, out-of-range elements on clamped addresses: with the options tested per element every
                // load waited for itself (fp32 B4 H4 235 x 1436 d64 causal with a mask plane 237 us, 123 this way; B6 H16 309 x 552 d64 with a bias
                // 176 / 96; B12 H32 398 x 293 d64, a full chip, 284 / 274)
#pragma unroll
                for (int kt = 0; kt < KT; kt++)
#pragma unroll
                    for (int r = 0; r < 16; r++) st[kt][r] *= a.scale;
                if (a.softcap > 0.0f) {
#pragma unroll
                    for (int kt = 0; kt < KT; kt++) {
                        if constexpr (DP == 256 && Elem<T>::BYTES == 2) {      // (out of registers: 11 of them would go to scratch memory)
#pragma unroll
                            for (int r = 0; r < 16; r++) {
                                st[kt][r] = a.softcap * tanhf(st[kt][r] / a.softcap);
                                __builtin_amdgcn_sched_barrier(0);
                            }
                        } else soft_cap<16>(st[kt], a.softcap);
                    }
                }
                // (rows and keys are formed anew, the keys for each pass, and few loads are asked for at a time where registers are short)
                int qr = min(qi, a.Sq - 1), key0 = kw0 + 4 * h;
                asm volatile("" : "+v"(qr));
                const int last = a.Sk - 1;
                constexpr int FEW = DP == 256 ? 2 : DP == 128 ? 4 : 16;
                auto groups = [&](auto f) {
#pragma unroll
                    for (int kt = 0; kt < KT; kt++)
#pragma unroll
                        for (int r0 = 0; r0 < 16; r0 += FEW) {
                            if (kw0 + kt * 32 + acc_row(r0, 0) >= a.Sk) continue;              // (past the end for every lane: masked below)
#pragma unroll
                            for (int r = r0; r < r0 + FEW; r++) f(kt, r, min(key0 + kt * 32 + acc_row(r, 0), last));
                            if (FEW < 16) __builtin_amdgcn_sched_barrier(0);
                        }
                };
                if (a.bias) {
                    asm volatile("" : "+v"(key0));
                    const float* __restrict__ row = a.bias + b * a.bias_bs + ((long long)hd * a.Sq + qr) * a.Sk;
                    groups([&](int kt, int r, int key) { st[kt][r] += row[key]; });
                }
                if (a.mask_mode == 1 || a.mask_mode == 2) {
                    asm volatile("" : "+v"(key0));
                    const float* __restrict__ row = a.mask + ((a.mask_mode == 2 ? (long long)bh * a.Sq : 0LL) + qr) * a.Sk;
                    groups([&](int kt, int r, int key) { if (row[key] == 0.0f) st[kt][r] = -INFINITY; });
                }
            }
            // (the factor is positive: the -inf of a masked key stays one)
            const float factor = FULL ? LOG2E : sl2 != 0.0f ? fabsf(sl2) : 1.0f;
            if constexpr (!FULL) {
                if (sl2 <= 0.0f) {
                    const float sign = sl2 < 0.0f ? -1.0f : 0.0f;
#pragma unroll
                    for (int kt = 0; kt < KT; kt++)
#pragma unroll
                        for (int r = 0; r < 16; r++) st[kt][r] *= sign;
                }
            }
            if (need_mask) {
                // the query's last visible key, relative to the lane's first (formed here, not kept through the loop)
                int first = __lane_id();
                asm volatile("" : "+v"(first));
                const int row = first & 31;
                first = -4 * (first >> 5);
                int seen = a.Sk - 1 - kw0 + first;
                if (a.causal) seen = min(seen, (int)max(min((long long)wq_min + a.qoff - kw0, 1LL << 20), -(1LL << 20)) + row + first);
#pragma unroll
                for (int kt = 0; kt < KT; kt++)
#pragma unroll
                    for (int r = 0; r < 16; r++) if (kt * KSTEP + acc_row(r, 0) > seen) st[kt][r] = -INFINITY;
            }
            if constexpr (KM || FULL) {
                if (mixed) {
#pragma unroll
                    for (int kt = 0; kt < KT; kt++) {
                        const uint32_t kept = (uint32_t)(kbits >> (kr0 + 32 * kt)) >> (4 * h);       // bit acc_row(r, 0): the key of element r
#pragma unroll
                        for (int r = 0; r < 16; r++) if (!(kept >> acc_row(r, 0) & 1u)) st[kt][r] = -INFINITY;
                    }
                }
            }
#pragma unroll
            for (int k0 = 0; k0 < KT; k0 += REF) {
                float mloc = -INFINITY;
#pragma unroll
                for (int kt = k0; kt < k0 + REF; kt++)
#pragma unroll
                    for (int r = 0; r < 16; r++) mloc = fmaxf(mloc, st[kt][r]);
                mloc = max_with_partner32(mloc) * factor;
                const float m_new = fmaxf(m_run, mloc);
                const float m_use = (m_new == -INFINITY) ? 0.0f : m_new;
                const float alpha = __builtin_amdgcn_exp2f(m_run - m_use);
                m_run = m_new;

                float psum = 0.0f;
#pragma unroll
                for (int kt = k0; kt < k0 + REF; kt++)
#pragma unroll
                    for (int r = 0; r < 16; r++) {
                        float p = __builtin_amdgcn_exp2f(fmaf(st[kt][r], factor, -m_use));
                        st[kt][r] = p;
                        psum += p;
                    }
                l_run = l_run * alpha + psum;
                // alpha == 1 in every lane (no row maximum moved) is the common case once a few tiles have been seen
                if (__builtin_amdgcn_ballot_w64(alpha != 1.0f) != 0ull) {
#pragma unroll
                    for (int i = 0; i < DT; i++)
#pragma unroll
                        for (int r = 0; r < 16; r++) oacc[i][r] *= alpha;
                }

                // ---- O^T += V^T * P^T
                if constexpr (EB == 4) __builtin_amdgcn_s_setprio(2);
#pragma unroll
                for (int kt = k0; kt < k0 + REF; kt++) {
#pragma unroll
                    for (int ps = 0; ps < PSTEPS; ps++) {
                        u32x4 pf;
                        if constexpr (E == 8) {
#pragma unroll
                            for (int w = 0; w < 4; w++) pf[w] = pack2_p<T>(st[kt][8 * ps + 2 * w], st[kt][8 * ps + 2 * w + 1]);
                        } else {
#pragma unroll
                            for (int w = 0; w < 4; w++) pf[w] = as_u32(st[kt][4 * ps + w]);
                        }
#pragma unroll
                        for (int i = 0; i < DT; i++) {
                            u32x4 vf;
                            if constexpr (DMA && EB == 4) {
                                // V[key = 32 kt + 8 ps + 4 h + q][d = 32 i + l32]; (key >> 2) & 1 == h
                                const int d = i * 32 + l32;
                                const unsigned char* vp = Vs + stage * VBYTES + (kr0 + kt * 32 + 8 * ps + 4 * h) * (DP * 4) + ((((d >> 2) ^ (h << 3)) << 4) + (d & 3) * 4);
#pragma unroll
                                for (int q = 0; q < 4; q++) vf[q] = *(const uint32_t*)(vp + q * (DP * 4));
                            } else if constexpr (DMA) {
                                // 16-bit: the lane's eight k-slots are keys 16 ps + 4 h + (0..3) and 16 ps + 8 + 4 h + (0..3) (the order of
                                // the accumulator rows its P values come from); one transposing read per group of four: in a
                                // 16-lane group lane j addresses key (base + j / 4), 8 bytes at head-dim 4 (j % 4) of the 16-wide block
                                const int jl = lane & 15;
                                const int chunk = (i * 32 + 16 * ((lane >> 4) & 1) + 4 * (jl & 3)) >> 3;
#pragma unroll
                                for (int q = 0; q < 2; q++) {
                                    const int row = kr0 + kt * KSTEP + 16 * ps + 8 * q + 4 * h + (jl >> 2);
                                    u32x2 w = __builtin_bit_cast(u32x2, __builtin_amdgcn_ds_read_tr16_b64_v4i16(
                                        (__attribute__((address_space(3))) s16x4a*)(Vs + stage * VBYTES + row * (DP * 2) + ((chunk ^ v_swz(row)) << 4) + (jl & 1) * 8)));
                                    vf[2 * q] = w[0];
                                    vf[2 * q + 1] = w[1];
                                }
                            } else {
                                vf = *(const u32x4*)(vs + i * 32 * VPITCH + kt * KSTEP * EB + ps * 32);
                            }
                            Mma32<T>::run(oacc[i], vf, pf);
                        }
                    }
                }
            }
            if constexpr (EB == 4) __builtin_amdgcn_s_setprio(0);
        }
        if constexpr (DMA) __builtin_amdgcn_s_waitcnt(0);      // this wave's loads of tile j + 1 have landed
        else if (j + 1 < ntiles) store_tile(stage ^ 1);
        if constexpr (KM) kbits = tile_keys(kv0 + BC, next_keep);
        __syncthreads();
    }

    // ---- key groups: the waves of groups 1 .. KG - 1 leave (O, m, l) in the idle tile memory and group 0 merges them.  The areas of
    // row group wq are the ones its own output staging below overwrites.
    if constexpr (KG > 1) {
        constexpr int AREA = DT * 16 * 64;                          // floats of one wave's O
        static_assert((KG - 1) * WQ * (AREA + 128) * 4 <= 2 * (KBYTES + VBYTES), "the partial results fit the tile memory");
        static_assert(KG == 2 || WQ == 1, "a row group's partial results lie where that row group stages its output");
        float* O1 = (float*)smem + wq * (KG - 1) * AREA;
        float* ML = (float*)smem + (KG - 1) * WQ * AREA + wq * (KG - 1) * 128;
        if (kg > 0) {
            f32x4* dst = (f32x4*)(O1 + (kg - 1) * AREA);
#pragma unroll
            for (int i = 0; i < DT; i++)
#pragma unroll
                for (int g = 0; g < 4; g++)
                    dst[(i * 4 + g) * 64 + lane] = f32x4{oacc[i][4 * g], oacc[i][4 * g + 1], oacc[i][4 * g + 2], oacc[i][4 * g + 3]};
            ML[(kg - 1) * 128 + lane] = m_run;
            ML[(kg - 1) * 128 + 64 + lane] = l_run;
        }
        __syncthreads();
        if (kg > 0) return;
#pragma unroll
        for (int u = 0; u < KG - 1; u++) {
            const float m1 = ML[u * 128 + lane], l1 = ML[u * 128 + 64 + lane];
            const float m_new = fmaxf(m_run, m1);
            const float m_use = (m_new == -INFINITY) ? 0.0f : m_new;
            const float w0 = __builtin_amdgcn_exp2f(m_run - m_use), w1 = __builtin_amdgcn_exp2f(m1 - m_use);
            m_run = m_new;
            l_run = l_run * w0 + l1 * w1;
            const f32x4* src = (const f32x4*)(O1 + u * AREA);
#pragma unroll
            for (int i = 0; i < DT; i++)
#pragma unroll
                for (int g = 0; g < 4; g++) {
                    const f32x4 v = src[(i * 4 + g) * 64 + lane];
#pragma unroll
                    for (int e = 0; e < 4; e++) oacc[i][4 * g + e] = oacc[i][4 * g + e] * w0 + v[e] * w1;
                }
        }
    }

    // ---- normalise and store: lane holds query qi, head-dim elements i*32 + 8 g + 4 h + (0..3)
    const float l_tot = l_run + shfl_xor_f(l_run, 32);
    if constexpr (RANGES) {
        if (a.part) {
            // a key range: (m, l, O) for the merge, whole rows at a time through the (idle) tile memory
            unsigned char* stg = smem + wq * (32 * DP * 4);
            const int row0 = q0 + wq * 32, nrow = min(32, a.Sq - row0);
            if (nrow <= 0) return;
#pragma unroll
            for (int i = 0; i < DT; i++)
#pragma unroll
                for (int g = 0; g < 4; g++)
                    *(f32x4*)(stg + l32 * (DP * 4) + (((8 * i + 2 * g + h) ^ (l32 & 15)) << 4)) =
                        f32x4{oacc[i][4 * g + 0], oacc[i][4 * g + 1], oacc[i][4 * g + 2], oacc[i][4 * g + 3]};
            float* __restrict__ P = a.part + (((long long)bh * a.Sq + row0) * a.nsplit + blockIdx.y) * (2 + DP);
            const long long pitch = (long long)a.nsplit * (2 + DP);
            if (h == 0 && l32 < nrow) *(f32x2p*)(P + l32 * pitch) = f32x2p{m_run, l_tot};
            for (int r = h; r < nrow; r += 2)                           // a row to each half of the wave, a pair of elements to a lane
                *(f32x2p*)(P + r * pitch + 2 + 2 * l32) = *(const f32x2p*)(stg + r * (DP * 4) + (((l32 >> 1) ^ (r & 15)) << 4) + 8 * (l32 & 1));
            return;
        }
    }
    const float inv = l_tot > 0.0f ? 1.0f / l_tot : 0.0f;
    if constexpr (DMA && Elem<OutT>::BYTES == 4 && DP <= 128) {
        if (a.vec_out && a.D == DP) {
            // fp32 O through the (idle) tile memory, as in the fast kernel: staged per wave as [32 rows][DP * 4 bytes] (chunk c of row
            // r at position c ^ r) and written back as whole rows with non-temporal stores; a lane otherwise writes 16-byte pieces
            // of one row, 64 partial lines per instruction.  Every wave left the last tile at the barrier that ends the loop.
            constexpr int CH = DP / 4;                   // 16-byte chunks of a row
            constexpr int RPI = 64 / CH;                 // rows per store instruction
            unsigned char* stg = smem + wq * (32 * DP * 4);
#pragma unroll
            for (int i = 0; i < DT; i++)
#pragma unroll
                for (int g = 0; g < 4; g++)
                    *(f32x4*)(stg + l32 * (DP * 4) + (((8 * i + 2 * g + h) ^ (l32 & (CH - 1))) << 4)) =
                        f32x4{oacc[i][4 * g + 0] * inv, oacc[i][4 * g + 1] * inv, oacc[i][4 * g + 2] * inv, oacc[i][4 * g + 3] * inv};
            if (a.lse && h == 0 && qi < a.Sq)
                a.lse[(long long)bh * a.Sq + qi] = l_tot > 0.0f ? (m_run + __builtin_amdgcn_logf(l_tot)) * LN2 : -INFINITY;
            const int c = lane % CH;
#pragma unroll
            for (int q = 0; q < 32 / RPI; q++) {
                const int r = RPI * q + lane / CH;
                const int row = q0 + wq * 32 + r;
                const f32x4 v = *(const f32x4*)(stg + r * (DP * 4) + ((c ^ (r & (CH - 1))) << 4));
                f32x4* dst = (f32x4*)((float*)a.o + b * a.os[0] + hd * a.os[1] + (long long)row * a.os[2] + c * 4);
                if (row < a.Sq) __builtin_nontemporal_store(v, dst);
            }
            return;
        }
    }
    if (qi < a.Sq) {
        typedef typename Raw2<OutT>::type out_t;
        out_t* __restrict__ O = (out_t*)a.o + b * a.os[0] + hd * a.os[1] + (long long)qi * a.os[2];
#pragma unroll
        for (int i = 0; i < DT; i++) {
#pragma unroll
            for (int g = 0; g < 4; g++) {
                const int d0 = i * 32 + 8 * g + 4 * h;
                float v0 = oacc[i][4 * g + 0] * inv, v1 = oacc[i][4 * g + 1] * inv;
                float v2 = oacc[i][4 * g + 2] * inv, v3 = oacc[i][4 * g + 3] * inv;
                if constexpr (Elem<OutT>::BYTES == 4) {
                    if (a.vec_out && d0 + 4 <= a.D) {
                        *(f32x4*)(O + d0) = f32x4{v0, v1, v2, v3};
                    } else {
                        if (d0 + 0 < a.D) O[d0 + 0] = as_u32(v0);
                        if (d0 + 1 < a.D) O[d0 + 1] = as_u32(v1);
                        if (d0 + 2 < a.D) O[d0 + 2] = as_u32(v2);
                        if (d0 + 3 < a.D) O[d0 + 3] = as_u32(v3);
                    }
                } else {
                    uint32_t w0 = Elem<OutT>::narrow(v0) | (Elem<OutT>::narrow(v1) << 16);
                    uint32_t w1 = Elem<OutT>::narrow(v2) | (Elem<OutT>::narrow(v3) << 16);
                    if (a.vec_out && d0 + 4 <= a.D) {
                        *(u32x2*)(O + d0) = u32x2{w0, w1};
                    } else {
                        if (d0 + 0 < a.D) O[d0 + 0] = (out_t)(w0 & 0xFFFFu);
                        if (d0 + 1 < a.D) O[d0 + 1] = (out_t)(w0 >> 16);
                        if (d0 + 2 < a.D) O[d0 + 2] = (out_t)(w1 & 0xFFFFu);
                        if (d0 + 3 < a.D) O[d0 + 3] = (out_t)(w1 >> 16);
                    }
                }
            }
        }
        if (a.lse && h == 0)
            a.lse[(long long)bh * a.Sq + qi] = l_tot > 0.0f ? (m_run + __builtin_amdgcn_logf(l_tot)) * LN2 : -INFINITY;
    }
}

// ---------------------------------------------------------------------------------------------
// Fast path: 16-bit inputs, head dim 128, 16-byte aligned rows, no bias / mask / soft-cap.
// Same formulation as above (S^T = K Q^T, O^T += V^T P^T), but K and V tiles go global -> LDS with the
// gfx950 direct load (no staging registers, no ds_write, no register transposes) and V^T fragments are
// produced by the transposing LDS read:
//   K tile [64 keys][256 B]: 16-byte chunk c of key k at chunk position c ^ (k & 15)        (b128 reads)
//   V tile [64 keys][256 B]: 16-byte chunk c of key k at chunk position c ^ ((k & 3) << 2)  (tr16 reads)
// Softmax: the scale is folded into one FMA per logit (p = exp2(s * c - m)); the running max used for
// the exponent is only raised when the true max has grown by more than 8 (log2 units), so the O
// accumulator is rescaled rarely and P never exceeds 2^8 -- exact mathematics, LSE = m + log2(l) holds
// for any reference point m.


// Heads whose query tiles are interleaved (heaviest first) in the causal workgroup order of one XCD: 4 heads x 1 MiB of K and V
// (S = 2048, d = 128, 16-bit) is what one XCD's 4 MiB L2 holds, and four heads' tiles are enough to balance the CUs.
#define ATTN_HEAD_GROUP 4
// Depth of the register ring that prefetches MFMA operand fragments from LDS inside a tile; must divide 8.
#define AIDN_ATTN_RING 4
// PAGED: K and V are pools behind a block table (block size a multiple of 16); a wave's 16 keys of a tile then lie in one block, and all
// that changes is where the uniform base of its loads comes from (paged_tile_rows).  A 512-query chunk after 3584 keys (bf16, 32 / 8
// heads) took 347 us on the general kernel, whose loads go through registers and which cannot split the keys of its 128 query tiles; here
// 54 us with the merge of its four key ranges (the kernel alone 49; bound by what the vector unit issues beside the MFMAs: which heads share
// K and V, and the order of the blocks, make no difference).
// KM: a keep-mask of the keys shared by the heads and queries of a batch (mask_mode 3), one ballot per tile as in the kernel above.
template <typename T, typename OutT, int D = 128, bool PAGED = false, bool KM = false>
__global__ __launch_bounds__(256, D == 128 ? 2 : 1) void attn_fwd_dl_kernel(const AttnArgs a)
{
    typedef uint16_t raw_t;
    static_assert(D == 128 || D == 256, "head dimension 128 (two workgroups per CU) or 256 (one)");
    constexpr int BC = 64, BR = 128;
    constexpr int ROWB = 2 * D;                     // bytes of a K or V row in a tile
    constexpr int KBYTES = BC * ROWB, VBYTES = BC * ROWB;
    constexpr int DSTEPS = D / 16, DT = D / 32;
    constexpr int CH = ROWB / 16;                   // 16-byte chunks per row
    constexpr int KPL = 1024 / ROWB;                // keys per wave-load (64 lanes x 16 bytes)
    constexpr int NL = 16 / KPL;                    // wave-loads per wave and tile (a wave loads 16 keys of K and 16 of V)
    // how far a row's maximum may run ahead of the exponent reference before O and the row sum are rescaled.  Behind a block table and
    // under a key mask not at all, as in the general kernel that served those calls before: the largest probability of a row is then 1,
    // which the 16-bit operand of the P V product holds exactly, where one that lags rounds it like any other (relative error against
    // float64, 512 queries after 3584 keys bf16: 1.45e-3 against 1.62e-3, general kernel 1.53e-3; f16 154 + 130: 1.68e-4, 1.97e-4, 1.74e-4).
    // The rescales cost 8 %: that call 54 us, contiguous keys with a lag of 8 50.
    constexpr float SLACK = PAGED || KM ? 0.0f : 8.0f;

    extern __shared__ __attribute__((aligned(1024))) unsigned char smem[];

    const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
    const int l32 = lane & 31, h = lane >> 5;
    int bh, qt, split = 0;
    {
        int nblk = gridDim.x, pid = blockIdx.x;
        int per = nblk >> 3, rem = nblk & 7;
        int xcd = pid & 7, idx = pid >> 3;
        int logical = (xcd < rem ? xcd * (per + 1) : rem * (per + 1) + (xcd - rem) * per) + idx;
        bh = logical / a.qtiles;
        qt = a.qtiles - 1 - (logical - bh * a.qtiles);
        if (a.nsplit > 1) {
            // the key ranges of a query tile are neighbours; late (heavy, under a causal mask) query tiles first
            const int per_head = a.qtiles * a.nsplit;
            bh = logical / per_head;
            const int r = logical - bh * per_head;
            qt = a.qtiles - 1 - r / a.nsplit;
            split = r % a.nsplit;
        } else if (a.paired) {
            // XCD-contiguous heads, qtiles / 2 workgroups per head: first the late (heavy) tile of the pair, then the early one
            const int units = a.qtiles >> 1;
            bh = logical / units;
            qt = a.qtiles - 1 - (logical - bh * units);
        } else if (a.causal) {
            // take the heads in groups of ATTN_HEAD_GROUP and hand out the query tiles of a group heaviest first across its heads
            // (all heads at once runs as fast but re-fetches K and V 3.3 times from beyond the L2; head by head leaves a heavy
            // tile for the very end).  When every XCD owns whole heads the groups are formed inside the XCD's own heads.
            const bool whole = rem == 0 && per % a.qtiles == 0;
            const int heads = whole ? per / a.qtiles : nblk / a.qtiles;
            const int at = whole ? idx : logical;
            const int gsz = heads < ATTN_HEAD_GROUP ? heads : ATTN_HEAD_GROUP;
            const int per_group = gsz * a.qtiles;
            const int grp = at / per_group, in = at - grp * per_group;
            const int first = grp * gsz;
            const int cur = heads - first < gsz ? heads - first : gsz;   // the last group may be short
            qt = a.qtiles - 1 - in / cur;
            bh = (whole ? xcd * heads : 0) + first + in % cur;
        }
    }
    const int npass = a.paired ? 2 : 1;
    for (int pass = 0; pass < npass; pass++) {
    if (pass == 1) qt = a.qtiles - 1 - qt;
    const int b = bh / a.H, hd = bh - b * a.H;
    const int kvh = hd / (a.H / a.Hkv);
    const int q0 = qt * BR;
    const int qi = q0 + wave * 32 + l32;

    const raw_t* __restrict__ Q = (const raw_t*)a.q + b * a.qs[0] + hd * a.qs[1];
    const raw_t* __restrict__ K = (const raw_t*)a.k + b * a.ks[0] + kvh * a.ks[1];
    const raw_t* __restrict__ V = (const raw_t*)a.v + b * a.vs[0] + kvh * a.vs[1];
    // keys this workgroup sees: all of them, or its split's range (which may be empty)
    int Sk = a.Sk;
    long long qoff = a.qoff;                 // causal: query i sees keys j <= i + qoff (j counted from the first key of the range)
    int kbeg = 0;
    if (a.nsplit > 1) {
        kbeg = split * a.chunk;
        if constexpr (!PAGED) {
            K += (long long)kbeg * a.ks[2];
            V += (long long)kbeg * a.vs[2];
        }
        Sk = max(0, min(a.chunk, a.Sk - kbeg));
        qoff -= kbeg;
    }

    u32x4 qf[DSTEPS];
#pragma unroll
    for (int s = 0; s < DSTEPS; s++) {
        u32x4 z = {0u, 0u, 0u, 0u};
        qf[s] = (qi < a.Sq) ? *(const u32x4*)(Q + (long long)qi * a.qs[2] + (2 * s + h) * 8) : z;
    }

    int ntiles = (Sk + BC - 1) / BC;
    if (a.causal) {
        long long lastkey = (long long)q0 + BR - 1 + qoff;
        if (lastkey < 0) ntiles = 0;
        else { long long nt = lastkey / BC + 1; if (nt < ntiles) ntiles = (int)nt; }
    }

    // LDS: K ring [2][KBYTES] then V ring [2][VBYTES].  This wave's DMA per tile: NL wave-loads of K and NL of V, each KPL keys
    // x ROWB bytes (4 x 256 at head dimension 128, 2 x 512 at 256); lane -> (key = KPL * load + lane / CH, chunk position = lane % CH).
    // For a tile that lies fully inside the sequence the source address is a scalar base (tile, wave, load) plus
    // a per-lane byte offset fixed for the whole kernel, so issuing a load costs no vector arithmetic.
    const uint32_t lds0 = (uint32_t)(uintptr_t)((__attribute__((address_space(3))) void*)smem);
    const int wave_s = __builtin_amdgcn_readfirstlane(wave);
    const int ld_key = lane / CH, ld_pos = lane % CH;
    const long long k_row_bytes = a.ks[2] * 2, v_row_bytes = a.vs[2] * 2;
    // (the swizzle of a lane's chunk depends on its key inside the wave's 16: load i, lane key ld_key -> key KPL i + ld_key; for V only
    // on the key's two low bits, which at 4 keys per load are ld_key for every load and at 2 keys per load alternate with the load)
    uint32_t k_lane_off[NL], v_lane_off[2];
#pragma unroll
    for (int i = 0; i < NL; i++) k_lane_off[i] = (uint32_t)(ld_key * k_row_bytes) + ((ld_pos ^ (KPL * i + ld_key)) << 4);
#pragma unroll
    for (int i = 0; i < 2; i++) v_lane_off[i] = (uint32_t)(ld_key * v_row_bytes) + ((ld_pos ^ (((KPL * i + ld_key) & 3) << 2)) << 4);
    // the row of the wave's first key of a tile, and for the last tile the rows that exist from there on
    int rows = 0;
    auto tile_row = [&](int tile) -> int {
        if constexpr (!PAGED) return tile * BC + 16 * wave_s;
        return __builtin_amdgcn_readlane(rows, tile & 63);
    };
    auto rows_left = [&](int tile) -> int {             // (a group of keys that lies past the end repeats the last group / the last row)
        const int g = tile * BC + 16 * wave_s;
        return Sk - 1 - (PAGED ? min(g, (Sk - 1) & ~15) : g);
    };
    auto next_rows = [&](int tile) {                     // ahead of the loads of a tile
        if constexpr (PAGED)
            if ((tile & 63) == 0) rows = paged_tile_rows(a.bt + b * a.bt_bs, a.bsz, a.dbsz, kbeg + 16 * wave_s, BC, tile, lane, (a.Sk - 1) & ~15);
    };
    auto issue_k = [&](int tile) {
        const uint32_t dst = lds0 + (tile & 1) * KBYTES + wave_s * (16 * ROWB);
        if (tile * BC + BC <= Sk) {
            const unsigned char* src = (const unsigned char*)K + (long long)tile_row(tile) * k_row_bytes;
            if (a.stream) {
#pragma unroll
                for (int i = 0; i < NL; i++) attn_dma16_base_stream(src + KPL * i * k_row_bytes, k_lane_off[i], dst + i * 1024);
            } else {
#pragma unroll
                for (int i = 0; i < NL; i++) attn_dma16_base(src + KPL * i * k_row_bytes, k_lane_off[i], dst + i * 1024);
            }
        } else {
            const long long row0 = tile_row(tile);
            const int left = rows_left(tile);
#pragma unroll
            for (int i = 0; i < NL; i++) {
                int key = KPL * (wave * NL + i) + ld_key;          // key inside the tile
                const long long gkey = row0 + min(KPL * i + ld_key, left);      // clamp: rows past the end are masked later
                attn_dma16(K + gkey * a.ks[2] + (ld_pos ^ (key & 15)) * 8, dst + i * 1024);
            }
        }
    };
    auto issue_v = [&](int tile) {
        const uint32_t dst = lds0 + 2 * KBYTES + (tile & 1) * VBYTES + wave_s * (16 * ROWB);
        if (tile * BC + BC <= Sk) {
            const unsigned char* src = (const unsigned char*)V + (long long)tile_row(tile) * v_row_bytes;
            if (a.stream) {
#pragma unroll
                for (int i = 0; i < NL; i++) attn_dma16_base_stream(src + KPL * i * v_row_bytes, v_lane_off[i & 1], dst + i * 1024);
            } else {
#pragma unroll
                for (int i = 0; i < NL; i++) attn_dma16_base(src + KPL * i * v_row_bytes, v_lane_off[i & 1], dst + i * 1024);
            }
        } else {
            const long long row0 = tile_row(tile);
            const int left = rows_left(tile);
#pragma unroll
            for (int i = 0; i < NL; i++) {
                int key = KPL * (wave * NL + i) + ld_key;
                const long long gkey = row0 + min(KPL * i + ld_key, left);
                attn_dma16(V + gkey * a.vs[2] + (ld_pos ^ ((key & 3) << 2)) * 8, dst + i * 1024);
            }
        }
    };

    f32x16 oacc[DT];
#pragma unroll
    for (int i = 0; i < DT; i++)
#pragma unroll
        for (int r = 0; r < 16; r++) oacc[i][r] = 0.0f;
    float m_ref = -INFINITY;     // reference point of the exponent (log2 domain); same in lanes l and l ^ 32
    float l_run = 0.0f;

    const int wq_min = q0 + wave * 32, wq_max = wq_min + 31;
    const float sl2 = a.scale * LOG2E;
    // tiles this wave computes: under a causal mask a prefix of the workgroup's tiles
    int nact = wq_min < a.Sq ? ntiles : 0;      // a wave without query rows only takes part in the loads
    if (a.causal) {
        long long lk = (long long)wq_max + qoff;
        if (lk < 0) nact = 0;
        else { long long nt = lk / BC + 1; if (nt < nact) nact = (int)nt; }
    }

    // Fragment addressing.  K (b128 reads): lane reads key l32 (+ 32 per sub-tile), chunk (2 s + h) ^ (key & 15).
    // V^T (transposing reads): in a 16-lane group lane j addresses key (base + j / 4), 8 bytes at head-dim
    // 4 (j % 4) of the 16-wide block; chunk position (c + 4 dt) ^ ((key & 3) << 2).
    const int jl = lane & 15;
    const uint32_t k_lane = l32 * ROWB + ((h ^ (l32 & 15)) << 4);
    const uint32_t v_lane = (4 * h + (jl >> 2)) * ROWB + ((16 * ((lane >> 4) & 1) + 4 * (jl & 3)) >> 3) * 16 + (jl & 1) * 8
                          + ((jl >> 2) << 6);

    // last key a query may see (sequence end and causal diagonal folded into one 32-bit bound); klim carries the
    // lane's accumulator row offset 4 h so that the per-element test is against a constant
    auto key_limit = [&](int q) -> int {
        long long lim = Sk - 1;
        if (a.causal) { long long c = (long long)q + qoff; if (c < lim) lim = c; }
        return (int)(lim < -1 ? -1 : lim);
    };
    const int klim = key_limit(qi) - 4 * h;
    const int wave_klim = __builtin_amdgcn_readfirstlane(key_limit(wq_min));

    // KM: visible keys of the current tile, the same in every wave
    const unsigned char* __restrict__ kmask = KM ? (const unsigned char*)a.mask + (long long)b * a.Sk + kbeg : nullptr;
    auto tile_keys = [&](int kv0, unsigned keep) -> uint64_t { return __builtin_amdgcn_ballot_w64(kv0 + lane < Sk && keep != 0); };
    uint64_t kbits = ~0ull;
    if (ntiles > 0) { next_rows(0); issue_k(0); issue_v(0); }
    if constexpr (KM) { if (ntiles > 0) kbits = tile_keys(0, kmask[min(lane, Sk - 1)]); }
    __builtin_amdgcn_s_waitcnt(0);
    __syncthreads();

    // raise the exponent reference only when a row max has moved by more than SLACK (or on first use)
    auto rescale = [&](float m_old) {
        const float alpha = (m_ref == -INFINITY) ? 1.0f : __builtin_amdgcn_exp2f(m_old - m_ref);
        l_run *= alpha;
#pragma unroll
        for (int i = 0; i < DT; i++) {
            // (head dimension 256: the accumulators live in accumulation registers, which the multiply cannot read.  The two
            // opaque statements pin them there on both sides of it, so that the copies to and from vector registers are made
            // here, on this rare path, and not once per tile on the common one.)
            if constexpr (D == 256) asm volatile("" : "+a"(oacc[i]));
#pragma unroll
            for (int r = 0; r < 16; r++) oacc[i][r] *= alpha;
            if constexpr (D == 256) asm volatile("" : "+a"(oacc[i]));
        }
    };
    auto lazy_rescale = [&](float mloc) {
        if (__builtin_amdgcn_ballot_w64(mloc > m_ref + SLACK) != 0ull) {
            const float m_old = m_ref;
            if (mloc > m_ref + SLACK) m_ref = mloc;
            rescale(m_old);
        }
    };
    // p = exp2(s * c - m) of two scores, rounded and packed; the row sum accumulates the rounded values (the
    // same numbers the P V product uses) with one dot instruction per pair
    auto exp_pair = [&](float s0, float s1, float m_use, uint32_t& packed, float& sum) {
        float p0 = __builtin_amdgcn_exp2f(fmaf(s0, sl2, -m_use));
        float p1 = __builtin_amdgcn_exp2f(fmaf(s1, sl2, -m_use));
        packed = pack2_p<T>(p0, p1);
        sum = add_pair<T>(packed, sum);
    };

    // Per tile (64 keys = two 32-key sub-tiles) the work of a wave is pipelined so that the exponentials sit in
    // the shadow of the matrix pipe:   S0 = QK(sub 0) | S1 = QK(sub 1) with exp(S0) | PV(sub 0) with exp(S1) | PV(sub 1)
    // invariant per-lane read addresses; ring stage, sub-tile and key block enter as immediate offsets
    // (the swizzle occupies address bits 4-7: a step or d-block index beyond them -- bit 8, head dimension 256 -- is a plain offset)
    uint32_t k_ad[8], v_ad[4];
#pragma unroll
    for (int s = 0; s < 8; s++) k_ad[s] = (lds0 + k_lane) ^ (uint32_t)(s << 5);
#pragma unroll
    for (int i = 0; i < 4; i++) v_ad[i] = (lds0 + 2 * KBYTES + v_lane) ^ (uint32_t)(i << 6);

    auto tile_body = [&](const int j, auto stage_c) {
        constexpr int stage = decltype(stage_c)::value;
        // Loads of the next tile: when this wave computes and the next tile lies fully inside the sequence they are
        // issued one per MFMA inside the first phase below (a vector-memory instruction holds the wave's issue slot for
        // some tens of cycles; there it is covered by the running MFMA).  Otherwise all at once here.
        const bool computes = j < nact && (!KM || kbits != 0);
        const bool spread = !a.stream && computes && j + 1 < ntiles && (j + 1) * BC + BC <= Sk;
        unsigned next_keep = 0;
        if constexpr (KM) next_keep = kmask[min(j * BC + BC + lane, Sk - 1)];
        if (j + 1 < ntiles) next_rows(j + 1);
        if (j + 1 < ntiles && !spread) { issue_k(j + 1); issue_v(j + 1); }
        if (computes) {
            const int kv0 = j * BC;
            const bool need_mask = kv0 + BC - 1 > wave_klim || (KM && kbits != ~0ull);
            const int rel_lim = klim - kv0;                   // keys of this tile with index > rel_lim are masked
            auto mask_sub = [&](int kt, f32x16& st) {
#pragma unroll
                for (int r = 0; r < 16; r++)
                    if (kt * 32 + 8 * (r >> 2) + (r & 3) > rel_lim) st[r] = -INFINITY;
                if constexpr (KM) {
                    const uint32_t kept = (uint32_t)(kbits >> (32 * kt)) >> (4 * h);
#pragma unroll
                    for (int r = 0; r < 16; r++)
                        if (!(kept >> (8 * (r >> 2) + (r & 3)) & 1u)) st[r] = -INFINITY;
                }
            };
            auto sub_max = [&](const f32x16& st) -> float {
                float m = -INFINITY;
#pragma unroll
                for (int r = 0; r < 16; r++) m = fmaxf(m, st[r]);
                return max_with_partner32(m) * sl2;            // scale > 0: max commutes with the scaling
            };

            // Fragment addresses: the swizzle is an XOR on address bits that only the lane's chunk index occupies,
            // so one base per tile and lane serves every step (XOR with a constant, then an immediate offset).
            auto k_frag = [&](int kt, int s) -> u32x4 {
                return *(const __attribute__((address_space(3))) u32x4*)(k_ad[s & 7] + (s >> 3) * 256 + stage * KBYTES + kt * 32 * ROWB);
            };
            auto v_frag8 = [&](int kt, int s) -> u32x4 {          // s = DT * (16-key half) + head-dim block
                const uint32_t ad = v_ad[(s % DT) & 3] + ((s % DT) >> 2) * 256 + stage * VBYTES + (32 * kt + 16 * (s / DT)) * ROWB;
                u32x2 w0 = __builtin_bit_cast(u32x2, __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) s16x4a*)ad));
                u32x2 w1 = __builtin_bit_cast(u32x2, __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) s16x4a*)(ad + 8 * ROWB)));
                return u32x4{w0[0], w0[1], w1[0], w1[1]};
            };

            // LDS fragment reads run R ahead of the MFMAs that consume them (fr[] is an R-deep ring; an idle LDS read takes
            // about 90 cycles, three MFMAs); sched_barrier pins that order and the MFMA / exp interleave.
            // ---- S0 = K[0:32] Q^T
            f32x16 s0, s1;
#pragma unroll
            for (int r = 0; r < 16; r++) { s0[r] = 0.0f; s1[r] = 0.0f; }
            constexpr int R = AIDN_ATTN_RING;       // (head dimension 256, one wave per SIMD: 2 and 4 measure the same, 8 costs registers and 5-15 %)
            static_assert(DSTEPS % R == 0 && DSTEPS == 2 * DT, "the fragment ring is indexed s % R over DSTEPS steps in every phase");
            constexpr int EV = DSTEPS / 8;          // steps per pair of exponentials (eight pairs per 32-key sub-tile)
            u32x4 fr[R];
#pragma unroll
            for (int s = 0; s < R; s++) fr[s] = k_frag(0, s);
            // the phases that issue nothing but MFMAs (this one and the last) run at a raised wave priority: the matrix pipe then
            // takes them ahead of the other wave's instructions on the SIMD, whose exponentials fill the gaps (1-2 % measured)
            __builtin_amdgcn_s_setprio(2);
            if (spread) {
                const unsigned char* ksrc = (const unsigned char*)K + (long long)tile_row(j + 1) * k_row_bytes;
                const unsigned char* vsrc = (const unsigned char*)V + (long long)tile_row(j + 1) * v_row_bytes;
                const uint32_t kdst = lds0 + (stage ^ 1) * KBYTES + wave_s * (16 * ROWB);
                const uint32_t vdst = lds0 + 2 * KBYTES + (stage ^ 1) * VBYTES + wave_s * (16 * ROWB);
#pragma unroll
                for (int s = 0; s < DSTEPS; s++) {
                    Mma32<T>::run(s0, fr[s % R], qf[s]);
                    fr[s % R] = s + R < DSTEPS ? k_frag(0, s + R) : k_frag(1, s + R - DSTEPS);
                    if (s < NL) attn_dma16_base(ksrc + KPL * s * k_row_bytes, k_lane_off[s], kdst + s * 1024);
                    else attn_dma16_base(vsrc + KPL * (s - NL) * v_row_bytes, v_lane_off[(s - NL) & 1], vdst + (s - NL) * 1024);
                    __builtin_amdgcn_sched_barrier(0);
                }
            } else {
#pragma unroll
                for (int s = 0; s < DSTEPS; s++) {
                    Mma32<T>::run(s0, fr[s % R], qf[s]);
                    fr[s % R] = s + R < DSTEPS ? k_frag(0, s + R) : k_frag(1, s + R - DSTEPS);
                    __builtin_amdgcn_sched_barrier(0);
                }
            }
            __builtin_amdgcn_s_setprio(0);
            if (need_mask) mask_sub(0, s0);
            lazy_rescale(sub_max(s0));
            float m_use = (m_ref == -INFINITY) ? 0.0f : m_ref;

            // ---- S1 = K[32:64] Q^T interleaved with P0 = exp(S0)
            u32x4 p0f[2], p1f[2];
            float psum = 0.0f;
#pragma unroll
            for (int s = 0; s < DSTEPS; s++) {
                Mma32<T>::run(s1, fr[s % R], qf[s]);
                fr[s % R] = s + R < DSTEPS ? k_frag(1, s + R) : v_frag8(0, s + R - DSTEPS);
                if (s % EV == 0) {
                    const int e = s / EV;
                    uint32_t pk;
                    exp_pair(s0[2 * e], s0[2 * e + 1], m_use, pk, psum);
                    asm volatile("" : "+v"(pk), "+v"(psum));       // keeps the exponentials here, between the MFMAs
                    p0f[e >> 2][e & 3] = pk;
                }
                __builtin_amdgcn_sched_barrier(0);
            }
            if (need_mask) mask_sub(1, s1);
            // ---- O^T += V[0:32]^T P0^T interleaved with P1 = exp(S1).  P1 is formed against the reference that S1 asks for at once; what is
            // accumulated against the older one, P0 V among it, is rescaled behind this phase.  (Formed against the old reference and a
            // second time when S1 raised it, 512 queries after 3584 keys took 56 us in this kernel; so, and with the partials through LDS, 49.)
            const float mloc1 = sub_max(s1);
            const bool raised = __builtin_amdgcn_ballot_w64(mloc1 > m_ref + SLACK) != 0ull;
            const float m_old = m_ref;
            if (mloc1 > m_ref + SLACK) m_ref = mloc1;
            m_use = (m_ref == -INFINITY) ? 0.0f : m_ref;
            float psum1 = 0.0f;
#pragma unroll
            for (int s = 0; s < 2 * DT; s++) {
                Mma32<T>::run(oacc[s % DT], fr[s % R], p0f[s / DT]);
                fr[s % R] = s + R < 2 * DT ? v_frag8(0, s + R) : v_frag8(1, s + R - 2 * DT);
                if (s % EV == 0) {
                    const int e = s / EV;
                    uint32_t pk;
                    exp_pair(s1[2 * e], s1[2 * e + 1], m_use, pk, psum1);
                    asm volatile("" : "+v"(pk), "+v"(psum1));
                    p1f[e >> 2][e & 3] = pk;
                }
                __builtin_amdgcn_sched_barrier(0);
            }
            l_run += psum;
            if (raised) rescale(m_old);
            l_run += psum1;

            // ---- O^T += V[32:64]^T P1^T
            __builtin_amdgcn_s_setprio(2);
#pragma unroll
            for (int s = 0; s < 2 * DT; s++) {
                Mma32<T>::run(oacc[s % DT], fr[s % R], p1f[s / DT]);
                if (s + R < 2 * DT) fr[s % R] = v_frag8(1, s + R);
            }
            __builtin_amdgcn_s_setprio(0);
        }
        __builtin_amdgcn_s_waitcnt(0);      // this wave's DMA of tile j+1 has landed ...
        if constexpr (KM) kbits = tile_keys(j * BC + BC, next_keep);
        __syncthreads();                    // ... everyone's has, and everyone is done with tile j
    };
    for (int j = 0; j < ntiles; j += 2) {
        tile_body(j, std::integral_constant<int, 0>{});
        if (j + 1 < ntiles) tile_body(j + 1, std::integral_constant<int, 1>{});
    }

    const float l_tot = sum_with_partner32(l_run);
    const float inv = l_tot > 0.0f ? 1.0f / l_tot : 0.0f;
    if (a.part) {
        // partial of a key range, unnormalised, for the merge: [2 + D] floats a row, whole rows at a time through LDS as below (the tile
        // memory is idle).  From the registers a store instruction touched 8 bytes in each of 64 places: contiguous 512 queries after 3584
        // keys, four ranges, 53.5 us with the merge, so 50.
        constexpr int OROWB = 4 * D;
        const int nrow = min(32, a.Sq - q0 - wave * 32);
        if (nrow <= 0) return;                                             // (one pass: a key range is never paired)
        unsigned char* stg = smem + wave * (32 * OROWB);
#pragma unroll
        for (int i = 0; i < DT; i++)
#pragma unroll
            for (int g = 0; g < 4; g++)
                *(f32x4*)(stg + l32 * OROWB + (((8 * i + 2 * g + h) ^ l32) << 4)) =
                    f32x4{oacc[i][4 * g + 0], oacc[i][4 * g + 1], oacc[i][4 * g + 2], oacc[i][4 * g + 3]};
        float* __restrict__ P = a.part + (((long long)bh * a.Sq + q0 + wave * 32) * a.nsplit + split) * (D + 2);
        const long long pitch = (long long)a.nsplit * (D + 2);
        if (h == 0 && qi < a.Sq) *(f32x2p*)(P + l32 * pitch) = f32x2p{m_ref, l_tot};
        int ln = lane;
        asm volatile("" : "+v"(ln));
#pragma unroll 4
        for (int r = 0; r < nrow; r++)
#pragma unroll
            for (int u = 0; u < D / 128; u++) {
                const int d2 = ln + 64 * u;                                // this lane's pair of elements
                *(f32x2p*)(P + r * pitch + 2 + 2 * d2) = *(const f32x2p*)(stg + r * OROWB + (((d2 >> 1) ^ r) << 4) + 8 * (d2 & 1));
            }
    } else
    if (Elem<OutT>::BYTES == 4 && a.vec_out && a.stage_out) {
        // fp32 O through LDS: the lane holds 16-byte pieces of ONE row (64 rows per store instruction, each a partial line);
        // staged per wave as [32 rows][4 D bytes] (chunk c of row r at position c ^ r, conflict-free both ways) and written back
        // as whole rows, 1024 bytes per instruction (two rows at head dimension 128, one at 256).  The tile memory is idle here:
        // every wave left the last tile at the barrier that ends the loop; the barrier below keeps the next pass's loads off the
        // staged rows.
        constexpr int OROWB = 4 * D, OCH = OROWB / 16, RPI = 64 / OCH;
        unsigned char* stg = smem + wave * (32 * OROWB);
#pragma unroll
        for (int i = 0; i < DT; i++)
#pragma unroll
            for (int g = 0; g < 4; g++) {
                const int c = 8 * i + 2 * g + h;
                *(f32x4*)(stg + l32 * OROWB + ((c ^ l32) << 4)) =
                    f32x4{oacc[i][4 * g + 0] * inv, oacc[i][4 * g + 1] * inv, oacc[i][4 * g + 2] * inv, oacc[i][4 * g + 3] * inv};
            }
        if (a.lse && h == 0 && qi < a.Sq)
            a.lse[(long long)bh * a.Sq + qi] = l_tot > 0.0f ? (m_ref + __builtin_amdgcn_logf(l_tot)) * LN2 : -INFINITY;
        // (the lane index is taken through an opaque copy: the row addresses below are then formed here, not ahead of the tile loop)
        int ln = lane;
        asm volatile("" : "+v"(ln));
        const int c = ln % OCH;
#pragma unroll
        for (int q = 0; q < 32 / RPI; q++) {
            const int r = RPI * q + ln / OCH;
            const int row = q0 + wave * 32 + r;
            const f32x4 v = *(const f32x4*)(stg + r * OROWB + ((c ^ r) << 4));
            f32x4* dst = (f32x4*)((float*)a.o + b * a.os[0] + hd * a.os[1] + (long long)row * a.os[2] + c * 4);
            // non-temporal: O is written once and would otherwise displace K and V tiles that other workgroups re-read
            // (alternated in one process: causal B4 H32 S2048 835 -> 879 TFLOP/s, unmasked 973 -> 999, never slower)
            if (row < a.Sq) __builtin_nontemporal_store(v, dst);
        }
        if (npass > 1) __syncthreads();
    } else
    if (qi < a.Sq) {
        typedef typename Raw2<OutT>::type out_t;
        out_t* __restrict__ O = (out_t*)a.o + b * a.os[0] + hd * a.os[1] + (long long)qi * a.os[2];
#pragma unroll
        for (int i = 0; i < DT; i++) {
#pragma unroll
            for (int g = 0; g < 4; g++) {
                const int d0 = i * 32 + 8 * g + 4 * h;
                float v0 = oacc[i][4 * g + 0] * inv, v1 = oacc[i][4 * g + 1] * inv;
                float v2 = oacc[i][4 * g + 2] * inv, v3 = oacc[i][4 * g + 3] * inv;
                if constexpr (Elem<OutT>::BYTES == 4) {
                    if (a.vec_out) *(f32x4*)(O + d0) = f32x4{v0, v1, v2, v3};
                    else { O[d0] = as_u32(v0); O[d0 + 1] = as_u32(v1); O[d0 + 2] = as_u32(v2); O[d0 + 3] = as_u32(v3); }
                } else {
                    uint32_t w0 = Elem<OutT>::narrow(v0) | (Elem<OutT>::narrow(v1) << 16);
                    uint32_t w1 = Elem<OutT>::narrow(v2) | (Elem<OutT>::narrow(v3) << 16);
                    if (a.vec_out) *(u32x2*)(O + d0) = u32x2{w0, w1};
                    else { O[d0] = (out_t)(w0 & 0xFFFFu); O[d0 + 1] = (out_t)(w0 >> 16); O[d0 + 2] = (out_t)(w1 & 0xFFFFu); O[d0 + 3] = (out_t)(w1 >> 16); }
                }
            }
        }
        if (a.lse && h == 0)
            a.lse[(long long)bh * a.Sq + qi] = l_tot > 0.0f ? (m_ref + __builtin_amdgcn_logf(l_tot)) * LN2 : -INFINITY;
    }
    }   // pass
}

// Merge of the key-range partials of the fast kernel and of the split one (part: [row][nsplit][2 + D], D up to 128), WPR waves per query row.  With a
// workgroup of 128 threads per row (weights through LDS, then the rows) 16384 rows of four ranges took 16.2 us, this way 8.8 (34 MB).
template <typename OutT, int WPR, bool KEEP_NAN>
__global__ __launch_bounds__(256) void attn_split_merge_kernel(const AttnArgs a, int rows)
{
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
    const int row = blockIdx.x * (4 / WPR) + wave / WPR;                                   // (b * H + hd) * Sq + qi
    if (row >= rows) return;
    const int bh = row / a.Sq, qi = row - bh * a.Sq;
    const int b = bh / a.H, hd = bh - b * a.H;
    f32x2p o[1];
    const float lse = merge_partials<1, WPR, KEEP_NAN>(a.part + (long long)row * a.nsplit * (2 + a.D), a.nsplit, a.D, a.D, wave % WPR, lane, o);
    if (wave % WPR != 0) return;
    if (lane == 0 && a.lse) a.lse[row] = lse;
    if (2 * lane >= a.D) return;
    typedef typename Raw2<OutT>::type out_t;
    out_t* O = (out_t*)a.o + b * a.os[0] + hd * a.os[1] + (long long)qi * a.os[2] + 2 * lane;
    if constexpr (Elem<OutT>::BYTES == 4) {
        if (a.vec_out) *(f32x2p*)O = o[0];
        else { O[0] = as_u32(o[0][0]); O[1] = as_u32(o[0][1]); }
    } else {
        const uint32_t w = Elem<OutT>::narrow(o[0][0]) | (Elem<OutT>::narrow(o[0][1]) << 16);
        if (a.vec_out) *(uint32_t*)O = w;
        else { O[0] = (out_t)(w & 0xFFFFu); O[1] = (out_t)(w >> 16); }
    }
}
template <typename OutT, bool KEEP_NAN>
static hipError_t launch_merge(const AttnArgs& a, hipStream_t stream)
{
    const long long rows = (long long)a.B * a.H * a.Sq;
    if (rows > 0x7FFFFFFFLL) return hipErrorInvalidValue;
    if (merge_waves_per_row(a.nsplit) == 1) hipLaunchKernelGGL((attn_split_merge_kernel<OutT, 1, KEEP_NAN>), dim3((unsigned)((rows + 3) / 4)), dim3(256), 0, stream, a, (int)rows);
    else hipLaunchKernelGGL((attn_split_merge_kernel<OutT, 4, KEEP_NAN>), dim3((unsigned)rows), dim3(256), 0, stream, a, (int)rows);
    return hipGetLastError();
}

template <typename T, typename OutT, int D = 128, bool PAGED = false, bool KM = false>
static hipError_t launch_attn_dl(AttnArgs a, hipStream_t stream)
{
    auto kern = attn_fwd_dl_kernel<T, OutT, D, PAGED, KM>;
    constexpr int smem = 2 * (64 * 2 * D + 64 * 2 * D);      // K and V tiles, two stages each (64 KB; 128 KB at head dimension 256)
    static unsigned long long attr_done = 0;
    if (hipError_t e = ensure_dynamic_smem((const void*)kern, smem, &attr_done)) return e;
    a.qtiles = (a.Sq + 127) / 128;
    a.stage_out = 1;
    if (D != 128 && a.nsplit > 1) return hipErrorInvalidValue;      // (the merge pass of the key ranges is written for 128)
    if (a.nsplit > 1) {
        // few query tiles over a long key sequence: every tile's keys are cut into ranges that run side by side; a merge pass follows
        a.paired = 0;
        const long long nblk = (long long)a.qtiles * a.B * a.H * a.nsplit;
        if (nblk > 0x7FFFFFFFLL || (long long)a.B * a.H * a.Sq > 0x7FFFFFFFLL) return hipErrorInvalidValue;
        hipLaunchKernelGGL(kern, dim3((unsigned)nblk), dim3(256), smem, stream, a);
        if (hipError_t e = hipGetLastError()) return e;
        return launch_merge<OutT, false>(a, stream);
    }
    // causal self-attention with an even number of query tiles: pair tile i with tile qtiles-1-i, so every workgroup has the same work
    a.paired = (a.causal && a.qoff == 0 && a.Sq == a.Sk && a.qtiles >= 2 && a.qtiles % 2 == 0) ? 1 : 0;
    long long nblk = (long long)(a.paired ? a.qtiles / 2 : a.qtiles) * a.B * a.H;
    if (nblk > 0x7FFFFFFFLL) return hipErrorInvalidValue;
    hipLaunchKernelGGL(kern, dim3((unsigned)nblk), dim3(256), smem, stream, a);
    return hipGetLastError();
}

// Grouped decode (one query row per head, H / Hkv >= 2 query heads per K/V head, 16-bit, head dimension 128, contiguous aligned
// cache): the query heads of a K/V head are the rows of one query tile of the fast kernel, so a K/V row is fetched once for the
// whole group instead of once per query head.  One workgroup per (batch, K/V head, split); with several splits the partials go
// to `part` ([B*H][nsplit][130] floats: m, l, O) for the decode merge pass, with one split the kernel writes O and LSE itself.
bool attn_group_decode_applies(int kind, const AttnParams& p)
{
    if (kind == 0 || p.D != 128 || p.Sq != 1 || p.Hkv <= 0 || p.H % p.Hkv != 0 || p.block_table || !p.allow_fast_path) return false;
    const int G = p.H / p.Hkv;
    if (G < 2 || G > 128 || !(p.scale > 0.0f)) return false;
    auto al = [](const void* ptr, long long s0, long long s1, long long s2) {
        return ((uintptr_t)ptr & 15u) == 0 && (s0 * 2) % 16 == 0 && (s1 * 2) % 16 == 0 && (s2 * 2) % 16 == 0;
    };
    if (!al(p.q, p.qs[0], p.qs[1], 0) || !al(p.k, p.ks[0], p.ks[1], p.ks[2]) || !al(p.v, p.vs[0], p.vs[1], p.vs[2])) return false;
    const int oeb = p.out16 ? 2 : 4;
    if (((uintptr_t)p.o & 15u) != 0 || (p.os[0] * oeb) % 16 != 0 || (p.os[1] * oeb) % 16 != 0) return false;
    return p.ks[2] > 0 && p.ks[2] < (1LL << 28) && p.vs[2] > 0 && p.vs[2] < (1LL << 28);
}

// sk: keys every query sees (the causal offset already applied); nsplit ranges of `chunk` keys (a multiple of 64)
hipError_t attn_group_decode(hipStream_t stream, int kind, const AttnParams& p, int sk, int nsplit, int chunk, float* part)
{
    const int G = p.H / p.Hkv;
    AttnArgs a;
    a.paired = 0; a.hgroup = 0;
    a.q = p.q; a.k = p.k; a.v = p.v; a.o = p.o; a.lse = p.lse; a.bias = nullptr; a.mask = nullptr;
    a.B = p.B; a.H = p.Hkv; a.Hkv = p.Hkv; a.Sq = G; a.Sk = sk; a.D = p.D;
    a.scale = p.scale; a.causal = 0; a.qoff = 0; a.softcap = 0.0f; a.mask_mode = 0; a.bias_bs = 0;
    a.qs[0] = p.qs[0]; a.qs[1] = p.qs[1] * G; a.qs[2] = p.qs[1];        // a query row is a query head
    a.os[0] = p.os[0]; a.os[1] = p.os[1] * G; a.os[2] = p.os[1];
    for (int i = 0; i < 3; i++) { a.ks[i] = p.ks[i]; a.vs[i] = p.vs[i]; }
    a.vec_in = 1; a.vec_out = 1;
    a.bt = nullptr; a.bsz = 0; a.bt_bs = 0;
    a.nsplit = nsplit; a.chunk = chunk; a.part = nsplit > 1 ? part : nullptr; a.stream = 1; a.stage_out = 0;
    a.qtiles = 1;
    const long long nblk = (long long)p.B * p.Hkv * nsplit;
    if (nblk > 0x7FFFFFFFLL || sk <= 0) return hipErrorInvalidValue;
    constexpr int smem = 2 * (64 * 256 + 64 * 256);
    auto go = [&](auto kern) -> hipError_t {
        static unsigned long long attr_done = 0;
        if (hipError_t e = ensure_dynamic_smem((const void*)kern, smem, &attr_done)) return e;
        hipLaunchKernelGGL(kern, dim3((unsigned)nblk), dim3(256), smem, stream, a);
        return hipGetLastError();
    };
    if (kind == 1) return p.out16 ? go(attn_fwd_dl_kernel<f16_t, f16_t>) : go(attn_fwd_dl_kernel<f16_t, float>);
    return p.out16 ? go(attn_fwd_dl_kernel<bf16_t, bf16_t>) : go(attn_fwd_dl_kernel<bf16_t, float>);
}

// Normalised probabilities P[b,h,i,j] = exp(logit - LSE[b,h,i]) for callers that ask for the attention-weights tensor (the
// optional output of ScaledDotProductAttention, src/AiDotNet.Tensors/Engines/DirectGpu/IDirectGpuBackend.cs:1421-1424), after
// the attention kernel has left the log-sum-exp of every row.
// Bound: the store of P (4 bytes per logit) and, in fp32, the matrix pipe that forms the logits a second time.  A workgroup makes
// a 64 x 128 tile of P, each of its four waves 32 queries x 64 keys: rows = queries, columns = keys, so that a lane's column is a key
// and every store instruction writes two whole 128-byte lines.  Q and K rows go global -> LDS directly, 128 bytes of the head
// dimension at a time in two stages (48 KB: three workgroups share a CU, one's stores run under another's products); fragments read
// from global memory instead touch 32 rows per load instruction, which the address unit serves at a quarter of the rate (36-38 us where
// this form takes 30).  Tiles above the causal diagonal are only cleared.
// B4 H12 S512 d64 fp32 causal, 50 MB of P: one scalar dot product per logit took 2377 us, this takes 30.
// FAST: rows in whole 16-byte chunks and D a multiple of the fragment step; other operands take guarded loads without LDS.
// FULL: bias, mask or soft-cap.
template <typename T, bool FAST, bool FULL>
__global__ __launch_bounds__(256) void attn_weights_kernel(const AttnArgs a, float* __restrict__ w, int qtiles, int ktiles)
{
    typedef typename Raw2<T>::type raw_t;
    constexpr int E = Elem<T>::PER16, KS = Mma32<T>::KS, BQ = 64, BK = 128;
    const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
    const int l32 = lane & 31, h = lane >> 5;
    // XCD-contiguous order: the tiles of one head share an L2; the key tiles of a query tile are neighbours
    int bh, q0, k0;
    {
        const int nblk = gridDim.x, pid = blockIdx.x, per = nblk >> 3, rem = nblk & 7, xcd = pid & 7, idx = pid >> 3;
        const int logical = (xcd < rem ? xcd * (per + 1) : rem * (per + 1) + (xcd - rem) * per) + idx;
        const int row_tile = logical / ktiles;
        k0 = (logical - row_tile * ktiles) * BK;
        bh = row_tile / qtiles;
        q0 = (row_tile - bh * qtiles) * BQ;
    }
    const int b = bh / a.H, hd = bh - b * a.H;
    float* __restrict__ W = w + (long long)bh * a.Sq * a.Sk;
    if (a.causal && (long long)k0 > (long long)q0 + BQ - 1 + a.qoff) {
        const int nk = min(BK, a.Sk - k0);
        for (int r = wave; r < BQ && q0 + r < a.Sq; r += 4)
            for (int c = lane; c < nk; c += 64) W[(long long)(q0 + r) * a.Sk + k0 + c] = 0.0f;
        return;
    }
    const int qw = q0 + 32 * (wave >> 1), kw = k0 + 64 * (wave & 1);      // this wave's 32 x 64 part
    const raw_t* __restrict__ Q = (const raw_t*)a.q + b * a.qs[0] + hd * a.qs[1];
    const raw_t* __restrict__ K = (const raw_t*)a.k + b * a.ks[0] + (hd / (a.H / a.Hkv)) * a.ks[1];
    f32x16 s[2];
#pragma unroll
    for (int j = 0; j < 2; j++)
#pragma unroll
        for (int r = 0; r < 16; r++) s[j][r] = 0.0f;
    // (asked for here, ahead of the products: inside the row loop below every row would wait for its own load)
    float lse[16];
#pragma unroll
    for (int r = 0; r < 16; r++) lse[r] = a.lse[(long long)bh * a.Sq + min(qw + acc_row(r, h), a.Sq - 1)];
    // (rows past the end are clamped loads whose products are never stored)
    const int steps = (a.D + KS - 1) / KS;
    if constexpr (FAST) {
        // wave-load i of the tile is eight rows of 128 bytes: 0 .. 7 are Q rows, 8 .. 23 K rows; 16-byte chunk c of row r at chunk
        // position c ^ ((r >> 1) & 7) (conflict-free fragment reads)
        constexpr int STAGE = (BQ + BK) * 128;
        __shared__ __attribute__((aligned(1024))) unsigned char smem[2 * STAGE];
        const uint32_t lds0 = (uint32_t)(uintptr_t)((__attribute__((address_space(3))) void*)smem);
        const int wave_s = __builtin_amdgcn_readfirstlane(wave);
        const raw_t* src[6];
        int chunk[6];
#pragma unroll
        for (int i = 0; i < 6; i++) {
            const int row = 8 * (6 * wave_s + i) + (lane >> 3);
            src[i] = row < BQ ? Q + (long long)min(q0 + row, a.Sq - 1) * a.qs[2] : K + (long long)min(k0 + row - BQ, a.Sk - 1) * a.ks[2];
            chunk[i] = (lane & 7) ^ ((row >> 1) & 7);
        }
        const int last_chunk = a.D / E - 1;
        auto issue = [&](int part) {
#pragma unroll
            for (int i = 0; i < 6; i++)      // (chunks past the head dimension repeat the last one; no step reads them)
                attn_dma16(src[i] + min(8 * part + chunk[i], last_chunk) * E, lds0 + (part & 1) * STAGE + (6 * wave_s + i) * 1024);
        };
        const int parts = (steps + 3) / 4;
        issue(0);
        if (parts > 1) issue(1);
        const int sw = (l32 >> 1) & 7;
        for (int part = 0; part < parts; part++) {
            // (loads complete in issue order: with the next part's six outstanding this part has landed)
            if (part + 1 < parts) asm volatile("s_waitcnt vmcnt(6)" ::: "memory");
            else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
            __syncthreads();
            const unsigned char* qs = smem + (part & 1) * STAGE + (qw - q0 + l32) * 128;
            const unsigned char* ks = smem + (part & 1) * STAGE + (BQ + kw - k0 + l32) * 128;
#pragma unroll
            for (int i = 0; i < 4; i++) {
                if (4 * part + i < steps) {
                    const int at = ((2 * i + h) ^ sw) << 4;
                    const u32x4 qf = *(const u32x4*)(qs + at), kf = *(const u32x4*)(ks + at), kf2 = *(const u32x4*)(ks + 32 * 128 + at);
                    Mma32<T>::run(s[0], qf, kf);
                    Mma32<T>::run(s[1], qf, kf2);
                }
            }
            if (part + 2 < parts) {
                __syncthreads();             // everyone has left the stage that is filled again
                issue(part + 2);
            }
        }
    } else {
        const bool vec = a.vec_in != 0;
        Q += (long long)min(qw + l32, a.Sq - 1) * a.qs[2];
        const raw_t* __restrict__ K2 = K + (long long)min(kw + 32 + l32, a.Sk - 1) * a.ks[2];
        K += (long long)min(kw + l32, a.Sk - 1) * a.ks[2];
        for (int i = 0; i < steps; i++) {
            const int d0 = (2 * i + h) * E;
            const u32x4 qf = ld16<T>(Q + d0, a.D - d0, vec), kf = ld16<T>(K + d0, a.D - d0, vec), kf2 = ld16<T>(K2 + d0, a.D - d0, vec);
            Mma32<T>::run(s[0], qf, kf);
            Mma32<T>::run(s[1], qf, kf2);
        }
    }
    // logits in place, one pass over the tile per option (a test per element would make the epilogue five thousand instructions
    // of branches, which then bound the kernel), out-of-range elements on clamped addresses
    const int keys[2] = {kw + l32, kw + 32 + l32};
#pragma unroll
    for (int j = 0; j < 2; j++)
#pragma unroll
        for (int r = 0; r < 16; r++) s[j][r] *= a.scale;
    if constexpr (FULL) {
        if (a.softcap > 0.0f) {
#pragma unroll
            for (int j = 0; j < 2; j++) soft_cap<16>(s[j], a.softcap);
        }
        if (a.bias) {
            const float* __restrict__ Bi = a.bias + b * a.bias_bs + (long long)hd * a.Sq * a.Sk;
#pragma unroll
            for (int j = 0; j < 2; j++)
#pragma unroll
                for (int r = 0; r < 16; r++) s[j][r] += Bi[(long long)min(qw + acc_row(r, h), a.Sq - 1) * a.Sk + min(keys[j], a.Sk - 1)];
        }
        if (a.mask_mode == 3) {
            const unsigned char* __restrict__ Mk = (const unsigned char*)a.mask + (long long)b * a.Sk;
#pragma unroll
            for (int j = 0; j < 2; j++) {
                const bool hidden = Mk[min(keys[j], a.Sk - 1)] == 0;
#pragma unroll
                for (int r = 0; r < 16; r++) s[j][r] = hidden ? -INFINITY : s[j][r];
            }
        } else if (a.mask_mode != 0) {
            const float* __restrict__ Mk = a.mask + (a.mask_mode == 2 ? (long long)bh * a.Sq * a.Sk : 0LL);
#pragma unroll
            for (int j = 0; j < 2; j++)
#pragma unroll
                for (int r = 0; r < 16; r++)
                    if (Mk[(long long)min(qw + acc_row(r, h), a.Sq - 1) * a.Sk + min(keys[j], a.Sk - 1)] == 0.0f) s[j][r] = -INFINITY;
        }
    }
    if (a.causal && (long long)kw + 63 > (long long)qw + a.qoff) {
#pragma unroll
        for (int j = 0; j < 2; j++)
#pragma unroll
            for (int r = 0; r < 16; r++)
                if ((long long)keys[j] > (long long)qw + acc_row(r, h) + a.qoff) s[j][r] = -INFINITY;
    }
    // a row without any visible key (log-sum-exp -inf) has no probabilities
#pragma unroll
    for (int j = 0; j < 2; j++)
#pragma unroll
        for (int r = 0; r < 16; r++) s[j][r] = lse[r] == -INFINITY ? 0.0f : __expf(s[j][r] - lse[r]);
    float* __restrict__ out = W + (long long)qw * a.Sk + keys[0];
    if (qw + 32 <= a.Sq && kw + 64 <= a.Sk) {
#pragma unroll
        for (int r = 0; r < 16; r++) {
            float* p = out + (long long)acc_row(r, h) * a.Sk;
            p[0] = s[0][r];
            p[32] = s[1][r];
        }
    } else {
#pragma unroll
        for (int r = 0; r < 16; r++) {
            float* p = out + (long long)acc_row(r, h) * a.Sk;
            if (qw + acc_row(r, h) < a.Sq) {
                if (keys[0] < a.Sk) p[0] = s[0][r];
                if (keys[1] < a.Sk) p[32] = s[1][r];
            }
        }
    }
}

// ------------------------------------------------------------------ host side
template <typename T, typename OutT, int DP, int BC, bool FULL, int MINB, bool DMA = false, bool KM = false, int KG = 1>
static hipError_t launch_attn_kg(AttnArgs a, hipStream_t stream)
{
    constexpr int BR = 128 / KG;
    auto kern = attn_fwd_kernel<T, OutT, DP, BC, FULL, MINB, DMA, KM, KG>;
    constexpr int EB = Elem<T>::BYTES;
    constexpr int smem = DMA ? 4 * BC * DP * EB : 2 * (BC * (DP * EB + 16) + DP * (BC * EB + 16));
    static unsigned long long attr_done = 0;
    if (hipError_t e = ensure_dynamic_smem((const void*)kern, smem, &attr_done)) return e;
    a.qtiles = (a.Sq + BR - 1) / BR;
    long long nblk = (long long)a.qtiles * a.B * a.H;
    if (nblk > 0x7FFFFFFFLL) return hipErrorInvalidValue;
    // causal order: up to 768 workgroups the balanced placement of a grid that is (nearly) resident at once (measured equal or
    // better than the grouped order up to that size); beyond, groups of at least 16 heads and at least 128 workgroups
    a.hgroup = !a.causal || a.nsplit > 1 ? 0 : nblk <= 768 ? -1 : (a.qtiles >= 8 ? 16 : (128 + a.qtiles - 1) / a.qtiles);
    hipLaunchKernelGGL(kern, dim3((unsigned)nblk, (unsigned)a.nsplit), dim3(256), smem, stream, a);
    return hipGetLastError();
}

// How many waves share the keys of a query row's tiles (KG).  With one (128 query rows per workgroup, 32 per wave) a grid that does not
// fill the chip takes as long as its longest wave: fp32 B4 H12 S512 d64 causal is 192 workgroups whose last ones run eight tiles of 64
// MFMAs of 64 cycles with nothing else on their SIMDs, 44 us -- as long as twice the batch.  Two waves per 32 rows (64-row workgroups,
// each wave half of every tile, merged through LDS at the end): 27 us; B1 H12 S1024 81 -> 48, and 32 with four.  Once the chip is full
// the same matrix work only pays for more tile loads and merges (B16 H12 S512 83 -> 89 us).  The lines, as workgroups of the finer
// grid on 256 CUs, from a sweep over 58 shapes (time with one / two key groups in us at the last size on either side):
//   64-key tiles, two workgroups per CU, head dimension up to 64: 768 (fp32 plain S512 74 / 67, causal S4096 308 / 253; 960: 54 / 54, S900
//     89 / 118); short causal fp32 sequences 640, beyond which the halved workgroups' starts and merges cost what they balance (S512 44.0 / 44.2);
//     16-bit causal 1024 (S500 19.3 / 14.8, S1900 46 / 35; plain 20.4 / 21.1; 1536: 21 / 28)
//   up to 128: 512, all resident at once (16-bit d80 plain 28.1 / 26.5; 768: 32.8 / 46.4)
//   fp32 above 64: 64-key tiles need 128 KiB, one workgroup per CU: 256 (plain d128 151 / 88; 384: 66 / 83), causal 384 (64 / 42)
//   four groups on 128-key tiles (head dimension 64, dense K and V, no mask): 256, causal 384, from 192 keys on (two / four groups: plain
//     B4 H8 S256 16.0 / 12.2, causal B1 H32 S300 18.8 / 16.3; plain at 304 32 / 40, 64 keys 7.9 / 8.8)
// Beyond 64 queries, where the finer grid has more workgroups, short sequences do not repay the merge by balance but only by a round of
// workgroups saved (240 shapes of 12 - 300 keys; up to 64 queries the second group takes waves that would idle, and the lines above hold):
//   one 64-key tile, plain or causal: up to 256, and up to 512 (head dimension 32, of whose workgroups a CU holds more: 768) where the 128-row
//     grid needs a second workgroup per CU (fp32 Sq 130 n 480 14.7 / 11.1, bf16 Sq 131 n 429 7.1 / 6.9, d32 Sq 256 n 628 10.7 / 10.1; but fp32
//     Sq 69 n 286 9.7 / 10.8, n 618 13.8 / 16.5, bf16 Sq 105 n 848 7.2 / 8.9); masks and biases up to 512 (Sq 310 n 400 12.3 / 10.7), at
//     head dimension 32 as above
//   up to 256 keys, fp32 plain: not at n 257 - 512 on a 128-row grid of up to 256 (S 115 n 360 14.7 / 15.5)
//   16-bit causal beyond 768: a 128-row grid of more than 512, or long rows (S 300 n 1000 14.0 / 11.9; but S 232 n 944 10.5 / 11.5)
//   fp32 above 64: up to 32 keys the second group has none (Sk 12 10.6 / 12.8); causal 384 only where the row tiles differ in length
//     (Sq 204 n 288 44 / 35; but Sq 62, Sk 12 n 352 16 / 26)
// These lines do not depend on how the tiles are loaded, so the direct-to-LDS and the register-staged forms add up the same way.
// 16-bit head dimension 64 with direct loads goes further, two workgroups of four groups to a CU (us on two groups and 64-key tiles / so):
//   four groups over long rows up to 512 plain (from 320 keys on: S910 n 464 16.5 / 14.3, 1940 on 3042 n 488 39.5 / 29.4, S406 n 312 10.2 / 10.0; S271 n 288
//     8.7 / 9.2) and 640 causal (from 1024 keys on: S2145 n 544 29.8 / 20.1; S471 n 720 10.7 / 13.9, S1355 n 1032 20.7 / 25.4); also behind a block table
//     whose blocks hold a wave's 32 keys
//   beyond, causal, two groups on 128-key tiles up to 512 (S471 n 384 10.7 / 10.0, S834 n 448 14.7 / 13.4, S1534 n 384 22.7 / 19.6) and over long rows 576
//     (S1355 n 528 20.7 / 18.6; S530 n 544 11.5 / 13.2)
// More groups also make more of the probabilities exactly one.  Fewer than all these lines give, as one group from n 257 plain and 641 causal on, are 3 - 9 %
// further from float64 (S200 plain f16 1.51e-4, on two groups where four are now 1.64e-4; S251 causal bf16 1.035e-3 / 1.088e-3), padded layers 0.3 - 0.8 %,
// and slower (S1191 plain n 304 22.2 on two, 26.7 on one; S1964 causal n 744 28.4 / 40.7).
template <typename T, typename OutT, int DP, int BC, bool FULL, int MINB, bool DMA = false, bool KM = false>
static hipError_t launch_attn(const AttnArgs& a, hipStream_t stream)
{
    constexpr bool WIDE32 = Elem<T>::BYTES == 4 && BC == 32 && DP == 128;
    if constexpr ((BC == 64 && MINB == 2) || WIDE32) {
        auto grid = [&](int rows) { return (long long)((a.Sq + rows - 1) / rows) * a.B * a.H; };
        if constexpr (!FULL && !KM && DP == 64) {
            constexpr bool HALF = Elem<T>::BYTES == 2 && DMA;
            const long long four = !a.causal ? (HALF && a.Sk >= 320 ? 512 : 256) : HALF && a.Sk >= 1024 ? 640 : 384;
            if ((!a.bt || (HALF && a.bsz % 32 == 0)) && a.Sk >= 192 && grid(32) <= four) return launch_attn_kg<T, OutT, DP, 128, FULL, HALF ? 2 : 1, DMA, KM, 4>(a, stream);
            if constexpr (HALF) {
                if ((!a.bt || a.bsz % 32 == 0) && a.causal && a.Sk >= 192 && grid(64) <= (a.Sk >= 1024 ? 576 : 512)) return launch_attn_kg<T, OutT, DP, 128, FULL, 2, DMA, KM, 2>(a, stream);
            }
        }
        long long line;
        if constexpr (WIDE32) line = a.Sk <= 32 ? 0 : a.causal && a.Sq > 64 && a.Sk > 128 ? 384 : 256;
        else if (grid(64) > grid(128) && a.Sk <= 64 && !(FULL && DP == 32)) line = FULL ? 512 : grid(128) <= 256 ? 256 : DP == 32 ? 768 : 512;
        else if (Elem<T>::BYTES == 4 && !FULL && !a.causal && a.Sk <= 256 && grid(64) > grid(128) && grid(128) <= 256) line = 256;
        else if constexpr (DP > 64) line = 512;
        else if constexpr (Elem<T>::BYTES == 2) line = !FULL && a.causal && (a.Sk >= 448 || grid(128) > 512) ? 1024 : 768;
        else line = a.causal && a.Sk < 1024 ? 640 : 768;
        if (grid(64) <= line) return launch_attn_kg<T, OutT, DP, 64, FULL, WIDE32 ? 1 : 2, DMA, KM, 2>(a, stream);
    }
    return launch_attn_kg<T, OutT, DP, BC, FULL, MINB, DMA, KM>(a, stream);
}

template <typename T>
static hipError_t launch_weights(const AttnArgs& a, float* w, hipStream_t stream)
{
    const int qtiles = (a.Sq + 63) / 64, ktiles = (a.Sk + 127) / 128;
    const long long nblk = (long long)qtiles * ktiles * a.B * a.H;
    if (nblk > 0x7FFFFFFFLL) return hipErrorInvalidValue;
    auto go = [&](auto kern) { hipLaunchKernelGGL(kern, dim3((unsigned)nblk), dim3(256), 0, stream, a, w, qtiles, ktiles); };
    const bool full = a.bias != nullptr || a.mask_mode != 0 || a.softcap > 0.0f;
    if (a.vec_in && a.D % Mma32<T>::KS == 0) full ? go(attn_weights_kernel<T, true, true>) : go(attn_weights_kernel<T, true, false>);
    else full ? go(attn_weights_kernel<T, false, true>) : go(attn_weights_kernel<T, false, false>);
    return hipGetLastError();
}

template <typename T, typename OutT, int BC>
static hipError_t dispatch_attn_d(const AttnArgs& a, bool full, hipStream_t stream)
{
    const int D = a.D;
    if (D <= 32)  return full ? launch_attn<T, OutT, 32, BC, true, 2>(a, stream)  : launch_attn<T, OutT, 32, BC, false, 2>(a, stream);
    if (D <= 64)  return full ? launch_attn<T, OutT, 64, BC, true, 2>(a, stream)  : launch_attn<T, OutT, 64, BC, false, 2>(a, stream);
    if (D <= 128) return full ? launch_attn<T, OutT, 128, BC, true, 2>(a, stream) : launch_attn<T, OutT, 128, BC, false, 2>(a, stream);
    if (D <= 256) {
        // 16-bit, plain / causal, more than two workgroups per CU: 32-key tiles, so that two workgroups share a CU (10-30 % over
        // one workgroup of 64-key tiles; smaller grids lose with it).  The other instances spill at two workgroups per CU.
        if constexpr (Elem<T>::BYTES == 2) {
            if (!full && (long long)((a.Sq + 127) / 128) * a.B * a.H > 512) return launch_attn<T, OutT, 256, 32, false, 2>(a, stream);
        }
        return full ? launch_attn<T, OutT, 256, BC, true, 1>(a, stream) : launch_attn<T, OutT, 256, BC, false, 1>(a, stream);
    }
    return hipErrorInvalidValue;
}


static bool attn_aligned16(const void* ptr, const long long* s, int bytes)
{
    return ((uintptr_t)ptr & 15u) == 0 && (s[0] * bytes) % 16 == 0 && (s[1] * bytes) % 16 == 0 && (s[2] * bytes) % 16 == 0;
}

// the fast kernel: 16-bit, head dimension 128, aligned rows, plain (optionally causal) attention
static bool attn_dl_applies(int kind, const AttnParams& p)
{
    if (kind == 0 || p.D != 128 || !(p.scale > 0.0f) || !p.allow_fast_path) return false;
    // (behind a block table: blocks of a multiple of 16 keys, fp32 output, which is what the paged entry points return)
    if (p.block_table && (!paged_block_fits(p.block_table, p.block_size) || p.out16)) return false;
    if (p.bias != nullptr || (p.mask && p.mask_mode != 0 && (p.mask_mode != 3 || p.block_table)) || p.softcap > 0.0f) return false;
    if (!(attn_aligned16(p.q, p.qs, 2) && attn_aligned16(p.k, p.ks, 2) && attn_aligned16(p.v, p.vs, 2))) return false;
    // the kernel addresses the K/V rows of a 4-key load group with unsigned 32-bit byte offsets
    return p.ks[2] > 0 && p.ks[2] < (1LL << 28) && p.vs[2] > 0 && p.vs[2] < (1LL << 28);
}

// Key ranges per query tile for the fast kernel (1 = none): when the query tiles alone leave most CUs idle and the key
// sequence is long (chunked prefill against a long cache, a few speculative tokens), ranges of at least 512 keys up to about two
// workgroups per CU.  *chunk = keys per range (a multiple of 64).
static int attn_dl_splits(const AttnParams& p, int* chunk)
{
    const long long base = (long long)((p.Sq + 127) / 128) * p.B * p.H;
    int sk = p.Sk;
    if (p.causal) {                              // keys nobody sees do not count
        const long long lim = (long long)p.Sq + p.qoff;
        if (lim < sk) sk = (int)(lim < 0 ? 0 : lim);
    }
    *chunk = 0;
    if (base >= 256 || sk < 1024 || p.weights) return 1;
    int ns = (int)((512 + base - 1) / base);
    if (ns > sk / 512) ns = sk / 512;
    if (ns > 32) ns = 32;
    if (ns < 2) return 1;
    int c = (sk + ns - 1) / ns;
    c = (c + 63) / 64 * 64;
    ns = (sk + c - 1) / c;
    *chunk = c;
    return ns >= 2 ? ns : 1;
}

// 16-bit, head dimension 64, at most half of the CUs with a workgroup of 64 queries: shares of each query tile's keys run as workgroups of their
// own (1 = none).  A workgroup takes 4.5 us and 1.15 for 128 keys there, the second launch 4 and the partials as in attn_split_ranges; a call costs its
// caller 11.7 us, with two launches 14 (us in one / cut: 189 queries on 3984 keys, 16 heads 31.3 / 18.7, 614 on 3138, 12 heads 25.7 / 24.0; self-attention
// H2 S4000 31.3 / 27.5, causal 30.9 / 25.4, H1 S3595 28.0 / 17.6, but H4 S2000 18.5 / 20.2; left whole: 40 queries on 1024 keys, 16 heads 12.0).
static int attn_half64_ranges(int kind, const AttnParams& p)
{
    if (kind == 0 || p.D != 64 || p.bias || p.softcap > 0.0f || (p.mask && p.mask_mode != 0)) return 1;
    const long long keys = p.causal ? std::min((long long)p.Sk, std::max(0LL, (long long)p.Sq + p.qoff)) : p.Sk;
    const long long grid = (long long)((p.Sq + 63) / 64) * p.B * p.H, tiles = (keys + 127) / 128;
    if (grid > 128) return 1;
    const double part_us = (double)p.B * p.H * p.Sq * (2 + p.D) * 8.0 / 4e6;
    int best = 1;
    double least = std::max(11.7, 4.5 + 1.15 * tiles) - 0.3;
    for (int ns = 2; ns <= std::min(std::min(256 / grid, tiles), 32LL); ns++) {
        const double us = std::max(14.0, 8.5 + 1.15 * (double)((tiles + ns - 1) / ns) + part_us * ns);
        if (us < least) { least = us; best = ns; }
    }
    return best;
}

static AttnArgs attn_args(int kind, const AttnParams& p)
{
    AttnArgs a;
    a.paired = 0;
    a.hgroup = 0;
    a.nsplit = 1; a.chunk = 0; a.part = nullptr; a.stream = 0; a.stage_out = 0;
    a.q = p.q; a.k = p.k; a.v = p.v; a.o = p.o; a.lse = p.lse; a.bias = p.bias; a.mask = p.mask;
    a.B = p.B; a.H = p.H; a.Hkv = p.Hkv; a.Sq = p.Sq; a.Sk = p.Sk; a.D = p.D;
    a.scale = p.scale; a.causal = p.causal; a.qoff = p.qoff; a.softcap = p.softcap; a.mask_mode = p.mask ? p.mask_mode : 0;
    a.bias_bs = p.bias_bs;
    for (int i = 0; i < 3; i++) { a.qs[i] = p.qs[i]; a.ks[i] = p.ks[i]; a.vs[i] = p.vs[i]; a.os[i] = p.os[i]; }
    a.qtiles = 0;
    a.bt = p.block_table; a.bsz = p.block_size; a.bt_bs = p.block_table_stride;
    a.dbsz = make_fastdiv((uint32_t)(p.block_table ? p.block_size : 1));
    const int eb = kind == 0 ? 4 : 2, e = 16 / eb;
    const int oeb = (kind == 0 || !p.out16) ? 4 : 2;
    auto al = [](const void* ptr, const long long* s, int bytes) {
        return ((uintptr_t)ptr & 15u) == 0 && (s[0] * bytes) % 16 == 0 && (s[1] * bytes) % 16 == 0 && (s[2] * bytes) % 16 == 0;
    };
    a.vec_in = (p.D % e == 0) && al(p.q, p.qs, eb) && al(p.k, p.ks, eb) && al(p.v, p.vs, eb);
    a.vec_out = (p.D % 4 == 0) && al(p.o, p.os, oeb);
    return a;
}

size_t attn_fwd_workspace_bytes(int kind, const AttnParams& p)
{
    int chunk, ns = 1;
    if (kind == 0) {
        const AttnArgs a = attn_args(kind, p);
        if (p.allow_fast_path && attn_split_applies(a)) ns = attn_split_ranges(a);
    } else if (attn_dl_applies(kind, p)) ns = attn_dl_splits(p, &chunk);
    else ns = attn_half64_ranges(kind, p);
    return ns > 1 ? (size_t)p.B * p.H * p.Sq * ns * (2 + p.D) * sizeof(float) : 0;
}

// kind: 0 fp32, 1 fp16, 2 bf16
hipError_t attn_fwd(hipStream_t stream, int kind, const AttnParams& p)
{
    const bool g_attn_allow_dl = p.allow_fast_path != 0;      // 0 (test hook of the context): every shape takes the general kernel
    if (p.block_table && p.weights) return hipErrorInvalidValue;      // the weights output does not follow a block table
    AttnArgs a = attn_args(kind, p);
    const bool full = p.bias != nullptr || a.mask_mode != 0 || p.softcap > 0.0f;
    // a mask of the keys alone is followed by the direct-to-LDS instances at head dimensions 64 and 128 as well
    const bool km = a.mask_mode == 3 && !p.block_table && (p.D == 64 || p.D == 128);
    // the direct-to-LDS kernels address K/V rows of a load group with unsigned 32-bit byte offsets
    const bool rows32 = p.ks[2] > 0 && p.ks[2] < (1LL << 28) && p.vs[2] > 0 && p.vs[2] < (1LL << 28);
    // the direct-to-LDS instances: plain / causal, 16-byte aligned rows, contiguous or in blocks of a multiple of 16 keys
    const bool dma = p.bias == nullptr && !(p.softcap > 0.0f) && (a.mask_mode == 0 || km) && a.vec_in && paged_block_fits(p.block_table, p.block_size) && g_attn_allow_dl && rows32;
    hipError_t err;
    // fast path: 16-bit, head dim 128, aligned rows, plain (optionally causal) attention
    const bool dl = attn_dl_applies(kind, p);
    // fp32 on the fp16 matrix pipe (attention_split.hip), but for two 128-key tiles of head dimension 64 on a grid that leaves CUs idle: four waves to
    // a row's keys on the fp32 pipe take less there (us a launch, split / so: H4 S256 12.5 / 12.0, H16 S200 12.9 / 12.3, B2 H16 S256 13.1 / 12.2;
    // S150 11.1 / 13.2 and S300 13.9 / 15.3 the other way; the probabilities' pass is faster split)
    const long long grid32 = (long long)((a.Sq + 31) / 32) * a.B * a.H;
    const bool groups32 = !full && a.vec_in && p.D == 64 && !p.block_table && !p.weights && p.Sk >= 192 && p.Sk <= 256 && p.Sq > 64 && grid32 <= (p.causal ? 384 : 256);
    const bool split = kind == 0 && p.allow_fast_path && !groups32 && attn_split_applies(a);
    if (dl && p.workspace) {
        int chunk;
        const int ns = attn_dl_splits(p, &chunk);
        if (ns > 1 && p.workspace_bytes >= (size_t)p.B * p.H * p.Sq * ns * 130 * sizeof(float)) {
            a.nsplit = ns; a.chunk = chunk; a.part = (float*)p.workspace;
        }
    }
    const int ns64 = attn_half64_ranges(kind, p);
    if ((split || ns64 > 1) && p.workspace) {
        const int ns = split ? attn_split_ranges(a) : ns64;
        if (ns > 1 && p.workspace_bytes >= (size_t)p.B * p.H * p.Sq * ns * (2 + p.D) * sizeof(float)) { a.nsplit = ns; a.part = (float*)p.workspace; }
    }
    // Unsplit prefill has two kernels.  The software-pipelined one is the faster (894 against 840 TFLOP/s on causal B4 H32 S2048 fp16,
    // 1035 against 983 without the mask, 312 against 292 at S 128) except where a sequence ends inside a 64-key tile and the passes
    // are short: the partial tile is then a larger share of a pass, and the pipelined kernel walks it in plain steps (509 against
    // 530 at S 1100).  allow_fast_path 2 / 3 (test hooks) pin the choice.
    bool pipelined = false;
    if (dl && a.nsplit == 1 && a.mask_mode == 0 && attn_prefill_applies(a)) {      // (dense arrays: its tile loads count on rows 256 bytes apart)
        pipelined = p.allow_fast_path == 3 || (p.allow_fast_path == 1 && (p.Sk % 64 == 0 || p.Sk >= 2048));
    }
    if (pipelined) err = launch_attn_prefill(kind, p.out16, a, stream);
    else
    if (dl && p.block_table) err = kind == 1 ? launch_attn_dl<f16_t, float, 128, true>(a, stream) : launch_attn_dl<bf16_t, float, 128, true>(a, stream);
    else
    if (dl && km) {
        if (kind == 1) err = p.out16 ? launch_attn_dl<f16_t, f16_t, 128, false, true>(a, stream) : launch_attn_dl<f16_t, float, 128, false, true>(a, stream);
        else err = p.out16 ? launch_attn_dl<bf16_t, bf16_t, 128, false, true>(a, stream) : launch_attn_dl<bf16_t, float, 128, false, true>(a, stream);
    } else
    if (dl) {
        if (kind == 1) err = p.out16 ? launch_attn_dl<f16_t, f16_t>(a, stream) : launch_attn_dl<f16_t, float>(a, stream);
        else err = p.out16 ? launch_attn_dl<bf16_t, bf16_t>(a, stream) : launch_attn_dl<bf16_t, float>(a, stream);
    } else
    if (split) {
        err = launch_attn_split(a, full, stream);
        if (err == hipSuccess && a.nsplit > 1) err = launch_merge<float, true>(a, stream);
    }
    else
    if (kind == 0) {
        // fp32: 64-key tiles while two workgroups still fit the LDS of a CU (head dimension up to 64), else 32-key tiles
        if (p.D == 64 && dma && km) err = launch_attn<float, float, 64, 64, false, 2, true, true>(a, stream);
        else if (p.D == 64 && dma) err = launch_attn<float, float, 64, 64, false, 2, true>(a, stream);
        else if (p.D <= 64) err = full ? (p.D <= 32 ? launch_attn<float, float, 32, 64, true, 2>(a, stream) : launch_attn<float, float, 64, 64, true, 2>(a, stream))
                                  : (p.D <= 32 ? launch_attn<float, float, 32, 64, false, 2>(a, stream) : launch_attn<float, float, 64, 64, false, 2>(a, stream));
        else err = dispatch_attn_d<float, float, 32>(a, full, stream);
    }
    else if (p.D == 256 && dma && !p.block_table && rows32 && p.scale > 0.0f && p.allow_fast_path != 2) {
        // head dimension 256, plain / causal, aligned rows: the phase-structured kernel at that width (64-key tiles of 512-byte rows,
        // one workgroup per CU); allow_fast_path 2 (test hook) pins the older form below
        if (kind == 1) err = p.out16 ? launch_attn_dl<f16_t, f16_t, 256>(a, stream) : launch_attn_dl<f16_t, float, 256>(a, stream);
        else err = p.out16 ? launch_attn_dl<bf16_t, bf16_t, 256>(a, stream) : launch_attn_dl<bf16_t, float, 256>(a, stream);
    }
    else if (p.D == 256 && dma) {
        // head dimension 256, plain / causal, aligned contiguous K/V: the direct-to-LDS form on 32-key tiles (Q streamed)
        if (kind == 1) err = p.out16 ? launch_attn<f16_t, f16_t, 256, 32, false, 2, true>(a, stream) : launch_attn<f16_t, float, 256, 32, false, 2, true>(a, stream);
        else err = p.out16 ? launch_attn<bf16_t, bf16_t, 256, 32, false, 2, true>(a, stream) : launch_attn<bf16_t, float, 256, 32, false, 2, true>(a, stream);
    }
    else if (p.D == 64 && dma && km) {
        if (kind == 1) err = p.out16 ? launch_attn<f16_t, f16_t, 64, 64, false, 2, true, true>(a, stream) : launch_attn<f16_t, float, 64, 64, false, 2, true, true>(a, stream);
        else err = p.out16 ? launch_attn<bf16_t, bf16_t, 64, 64, false, 2, true, true>(a, stream) : launch_attn<bf16_t, float, 64, 64, false, 2, true, true>(a, stream);
    }
    else if (p.D == 64 && dma) {
        // head dimension 64, plain / causal, aligned contiguous K/V: the direct-to-LDS form of the general kernel
        if (kind == 1) err = p.out16 ? launch_attn<f16_t, f16_t, 64, 64, false, 2, true>(a, stream) : launch_attn<f16_t, float, 64, 64, false, 2, true>(a, stream);
        else err = p.out16 ? launch_attn<bf16_t, bf16_t, 64, 64, false, 2, true>(a, stream) : launch_attn<bf16_t, float, 64, 64, false, 2, true>(a, stream);
    }
    else if (kind == 1) err = p.out16 ? dispatch_attn_d<f16_t, f16_t, 64>(a, full, stream) : dispatch_attn_d<f16_t, float, 64>(a, full, stream);
    else err = p.out16 ? dispatch_attn_d<bf16_t, bf16_t, 64>(a, full, stream) : dispatch_attn_d<bf16_t, float, 64>(a, full, stream);
    if (err != hipSuccess) return err;
    if (ns64 > 1 && a.nsplit > 1) {
        err = !p.out16 ? launch_merge<float, true>(a, stream) : kind == 1 ? launch_merge<f16_t, true>(a, stream) : launch_merge<bf16_t, true>(a, stream);
        if (err != hipSuccess) return err;
    }
    if (p.weights) {
        a.lse = p.lse;
        err = split ? launch_attn_weights_split(a, p.weights, stream)
              : kind == 0 ? launch_weights<float>(a, p.weights, stream) : kind == 1 ? launch_weights<f16_t>(a, p.weights, stream)
                                                                                  : launch_weights<bf16_t>(a, p.weights, stream);
    }
    return err;
}

}  // namespace aidn
