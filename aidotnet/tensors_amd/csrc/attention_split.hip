// fp32 attention on the fp16 matrix pipe.  Q, K, V and the probabilities are scaled by powers of two and held as two fp16 values each,
// x = h + m (h = fp16(x), m = fp16(x - h): 22 to 23 of the 24 bits, no value further off than 2^-25 of a unit), and three of the four products
// are formed, m h, h m, h h; what is left out, m m, is 2^-24 of a product at most.  Sums are fp32.
//
// Why fp16 and not bf16: three bf16 values hold every fp32 value whatever its size, but cost six products and 5.5 vector instructions a value where
// two fp16 values cost three and 3 (one v_fma_mix_f32 takes the scale and the half of the packed word as they are), and the vector pipe is what
// bounds the kernel (B8 H12 S512 d64 causal 37.8 us, 24 this way; the fp32 pipe 44).
//
// Scales.  Each row of Q has its own (its largest magnitude becomes 2^12 .. 2^13), K and V one per workgroup from its first tile (2^10 and 2^11:
// later tiles may be 32 and 16 times larger).  Probabilities are formed against the next whole number above the row maximum, times 2^4, so that
// their exponents are near zero where fp32 is fine (times 2^14 they were off by up to 3e-7), and split times 2^14: a row whose weight lies on a key
// with next to nothing in V is the sum of its smallest probabilities, and what the split cuts of those, 2^-39 of the largest, does not show in it
// (2^-29 did: V of 2e-3 at the key of the weight, 2^-14 at the others, 1e-5 of O).  What the split does not hold is computed again on the fp32
// pipe, by workgroup: results that are not finite (infinities, NaN, values beyond the first tile's scale), and those whose scale was set by values
// far larger than what they are formed from (below).
//
// Error against float64, fp32 pipe / here, 2-norm: O of B8 H12 S512 causal d32 2.45e-7 / 1.72e-7, d64 2.77e-7 / 2.03e-7, d128 3.41e-7 / 2.34e-7, plain d64
// 4.08e-7 / 3.25e-7, S80 causal d64 1.87e-7 / 1.56e-7, padded B4 d64 3.68e-7 / 2.88e-7, soft-cap 4.15e-7 / 3.35e-7; probabilities of B4 H12 S512 d64 causal
// 3.23e-7 / 2.70e-7; log-sum-exp d64 causal 5.03e-8 / 4.10e-8.  Over 100 drawn shapes no output is further off than the fp32 pipe has it.
#include "attention_common.hpp"
#include <algorithm>

namespace aidn {

constexpr float P_EXP = 4.0f;        // probabilities are formed and summed times 2^4
constexpr int P_SPLIT = 10;          // and split times 2^10 more

// Power of two (its exponent) that brings a magnitude into [2^to, 2^(to + 1)); 2^8 for zero: behind a first tile of zeros values from 2^-10 to 2^7
// have their bits
__device__ __forceinline__ int exponent_to(float magnitude, int to)
{
    const int e = (int)(as_u32(magnitude) >> 23);
    return magnitude == 0.0f ? 8 : min(max(to + 127 - e, -126), 126);
}
__device__ __forceinline__ float power2(int e) { return as_f32((uint32_t)(e + 127) << 23); }
// Factor 2^e of the logits of a row.  Below 2^-100 they are zero in any case (2^36 units at most); the factor itself stays above zero, so that the
// -inf of a masked key does
__device__ __forceinline__ float logit_factor(float scale, int e) { return fmaxf(__builtin_ldexpf(scale, e), 0x1p-100f); }

__device__ __forceinline__ uint32_t f16_pair(float a, float b)
{
    typedef float f32x2 __attribute__((ext_vector_type(2)));
    typedef _Float16 f16x2 __attribute__((ext_vector_type(2)));
    uint32_t u = __builtin_bit_cast(uint32_t, __builtin_convertvector((f32x2{a, b}), f16x2));
    asm("" : "+v"(u));               // (opaque: the compiler otherwise converts the low half a second time by itself)
    return u;
}
// a s, b s as h + m: one multiply-add per value takes the half of the packed word as it is.  UNIFORM: s is the same in every lane
template <bool UNIFORM>
__device__ __forceinline__ void split2(float a, float b, float s, uint32_t (&p)[2])
{
    p[0] = f16_pair(a * s, b * s);
    float x, y;
    if constexpr (UNIFORM) {
        asm("v_fma_mix_f32 %0, %1, %2, -%3 op_sel_hi:[0,0,1]" : "=v"(x) : "v"(a), "s"(s), "v"(p[0]));
        asm("v_fma_mix_f32 %0, %1, %2, -%3 op_sel:[0,0,1] op_sel_hi:[0,0,1]" : "=v"(y) : "v"(b), "s"(s), "v"(p[0]));
    } else {
        asm("v_fma_mix_f32 %0, %1, %2, -%3 op_sel_hi:[0,0,1]" : "=v"(x) : "v"(a), "v"(s), "v"(p[0]));
        asm("v_fma_mix_f32 %0, %1, %2, -%3 op_sel:[0,0,1] op_sel_hi:[0,0,1]" : "=v"(y) : "v"(b), "v"(s), "v"(p[0]));
    }
    p[1] = f16_pair(x, y);
}
__device__ __forceinline__ float wave_max(float v)
{
    auto step = [&](auto ctrl) { v = fmaxf(v, as_f32((uint32_t)__builtin_amdgcn_mov_dpp((int)as_u32(v), decltype(ctrl)::value, 0xF, 0xF, true))); };
    step(std::integral_constant<int, 0xB1>{});          // lanes 1 and 2 apart, then the mirrors of 8 and 16 lanes
    step(std::integral_constant<int, 0x4E>{});
    step(std::integral_constant<int, 0x141>{});
    step(std::integral_constant<int, 0x140>{});
    return max_with_partner32(max_with_partner16(v));
}

// eight values to a chunk of either plane
template <bool UNIFORM>
__device__ __forceinline__ void split8(const u32x4 (&r)[2], float s, u32x4 (&w)[2])
{
#pragma unroll
    for (int e = 0; e < 4; e++) {
        uint32_t p[2];
        split2<UNIFORM>(as_f32(r[e >> 1][2 * (e & 1)]), as_f32(r[e >> 1][2 * (e & 1) + 1]), s, p);
        w[0][e] = p[0];
        w[1][e] = p[1];
    }
}
__device__ __forceinline__ float largest(const u32x4 (&r)[2])
{
    float m = 0.0f;
#pragma unroll
    for (int e = 0; e < 8; e++) m = fmaxf(m, fabsf(as_f32(r[e >> 2][e & 3])));
    return m;
}
// Q operand: lane (l32, h) holds values 16 s + 8 h .. + 7 of row l32, the row scaled to its own largest magnitude; returns that exponent
template <int DS>
__device__ __forceinline__ int split_q(const float* __restrict__ row, bool exists, int D, int h, u32x4 (&qf)[DS][2])
{
    u32x4 r[DS][2];
    float most = 0.0f;
#pragma unroll
    for (int s = 0; s < DS; s++) {
        const int d0 = 16 * s + 8 * h;
        r[s][0] = r[s][1] = u32x4{0u, 0u, 0u, 0u};
        if (exists && d0 < D) {
            r[s][0] = *(const u32x4*)(row + d0);
            r[s][1] = *(const u32x4*)(row + d0 + 4);
        }
        most = fmaxf(most, largest(r[s]));
    }
    most = max_with_partner32(most);
    const int e = most == 0.0f ? 126 : exponent_to(most, 12);      // (logits of a row of zeros are not coarse)
#pragma unroll
    for (int s = 0; s < DS; s++) split8<false>(r[s], power2(e), qf[s]);
    return e;
}
// Byte offset of 16-byte chunk `ch` (eight values) of row `key` of a plane with rows of RB bytes.  K is read as 16 rows of one chunk at a time,
// V as four chunks of 4 rows; PER rows until the bank repeats
template <int RB> constexpr int PER = RB == 256 ? 1 : RB == 128 ? 2 : 4;
template <int RB> __device__ __forceinline__ int k_at(int key, int ch) { return key * RB + ((ch ^ ((key / PER<RB>) & (16 / PER<RB> - 1))) << 4); }
template <int RB> __device__ __forceinline__ int v_at(int key, int ch) { return key * RB + ((ch ^ (((key / PER<RB>) & (4 / PER<RB> - 1)) << 2)) << 4); }

// LDS: the planes of a tile of K and of V, or behind the last tile the results of all key groups but the first, then 16 rows of each wave
constexpr int split_lds(int DP, int BC, int NW, int KG)
{
    const int tiles = 8 * BC * DP, merge = (KG - 1) * (NW / KG) * (DP * 32 + 128) * 4, rows = NW / KG * 16 * DP * 4;
    return tiles > merge ? (tiles > rows ? tiles : rows) : (merge > rows ? merge : rows);
}

// One workgroup: NW waves of 32 query rows each, KG of them on the same rows and different keys of a tile.
//
// S^T = K Q^T and O^T += V^T P^T as in attn_fwd_kernel, on v_mfma_f32_32x32x16_f16: a lane holds one query, its row maximum is an in-lane reduction and
// one exchange, and P is the second product's operand as it stands.  K and V are loaded to registers a tile ahead, split there and kept in LDS as
// planes of [key][d] rows, single: V of a tile is written beside the first product and K of the next one beside the second, a barrier behind
// either.  (Both twice in LDS with one barrier a tile: 24.4 -> 27.8 us, the loads then land a phase later.)
//
// Bound by issue: per 64 keys (d64) a wave issues about 400 vector instructions, 48 MFMAs and 70 LDS operations, and matrix and vector work of the
// two waves of a SIMD overlap only in part (counted: vector pipe 63 % of a full CU's cycles, matrix pipe 44 %; no LDS bank conflicts).  Against the
// fp32 pipe, us: B8 H12 S512 d64 causal 44 / 24, plain 69 / 32; B2 H16 S2048 causal d64 165 / 71, d128 310 / 131; B8 H16 S512 d32 48 / 23; bias, masks
// and soft-cap alike (B4 H12 S512 d64 padded 40 / 24, soft-cap 62 / 36).
template <int DP, int BC, int NW, int KG, bool OPT, bool PAGED>
__global__ __launch_bounds__(64 * NW, 2) void attn_split_kernel(const AttnArgs a)
{
    constexpr int NT = 64 * NW, WQ = NW / KG, BR = 32 * WQ;
    constexpr int RB = 2 * DP, PL = BC * RB;      // bytes of a row of a plane, of a plane
    constexpr int KT = BC / 32 / KG;              // 32-key sub-tiles of a wave in a tile
    constexpr int DS = DP / 16, DT = DP / 32;     // 16-wide steps and 32-wide blocks of the head dimension
    constexpr int CPR = DP / 8;                   // chunks of eight values of a row
    constexpr int U = BC * CPR / NT;              // chunks of K (and of V) that a thread stages per tile
    constexpr int RPU = NT / CPR;                 // rows between a thread's chunks
    constexpr int AHEAD = !OPT;       // fragments are read a step ahead where the registers hold two sets
    static_assert(BC * CPR % NT == 0 && KT > 0 && (RPU % 16 == 0 || U == 1), "whole chunks to a thread, at one place of rows that share a swizzle");

    extern __shared__ __attribute__((aligned(1024))) unsigned char smem[];
    unsigned char* Ks = smem;                     // [2][BC][DP] fp16
    unsigned char* Vs = smem + 2 * PL;            // [2][BC][DP] fp16

    int t = threadIdx.x;
    const int wave = __builtin_amdgcn_readfirstlane(t >> 6);
    int lane = t & 63, l32 = lane & 31, h = lane >> 5;
    int bh, qt;
    attn_block(a, bh, qt);
    const int b = bh / a.H, hd = bh - b * a.H;
    const int kvh = hd / (a.H / a.Hkv);
    const int wq = wave % WQ, kg = wave / WQ;
    const int q0 = qt * BR + wq * 32;             // first query row of this wave
    const float* __restrict__ Q = (const float*)a.q + b * a.qs[0] + hd * a.qs[1];
    const float* __restrict__ K = (const float*)a.k + b * a.ks[0] + kvh * a.ks[1];
    const float* __restrict__ V = (const float*)a.v + b * a.vs[0] + kvh * a.vs[1];
    const int* __restrict__ bt = PAGED ? a.bt + b * a.bt_bs : nullptr;

    int ntiles = (a.Sk + BC - 1) / BC;
    if (a.causal) {
        const long long lastkey = (long long)qt * BR + BR - 1 + a.qoff;
        if (lastkey < 0) ntiles = 0;
        else { const long long nt = lastkey / BC + 1; if (nt < ntiles) ntiles = (int)nt; }
    }
    // this workgroup's share of them (from here on ntiles is where it ends)
    constexpr bool RANGES = !OPT || DP <= 64;     // (the others are out of registers: 12 of them would go to scratch memory)
    int first = 0;
    if (RANGES && a.nsplit > 1) {
        const int per = (ntiles + a.nsplit - 1) / a.nsplit;
        first = min((int)blockIdx.y * per, ntiles);
        ntiles = min(ntiles, first + per);
    }

    // ---- staging: thread t takes chunk t % CPR of keys t / CPR + i RPU
    u32x4 rk[U][2], rv[U][2];
    const int col = min(8 * (t % CPR), a.D - 8);   // (chunks past the head dimension repeat the last one: they meet zeros of Q, or are not stored)
    // what is asked for next: byte offsets of the rows, which follow the tiles and stop at the last row; paged, rows of the pool, looked up a
    // tile ahead
    uint32_t kat[U], vat[U], klast = 0, vlast = 0;
    auto rows_of = [&](int tile) {
#pragma unroll
        for (int i = 0; i < U; i++) {
            const int key = min(tile * BC + t / CPR + i * RPU, a.Sk - 1), blk = (int)fastdiv((uint32_t)key, a.dbsz);
            kat[i] = bt[blk] * a.bsz + (key - blk * a.bsz);
        }
    };
    auto load = [&](const float* __restrict__ src, uint32_t rs, uint32_t (&at)[U], uint32_t last, u32x4 (&v)[U][2]) {
#pragma unroll
        for (int i = 0; i < U; i++) {
            const unsigned char* p;
            if constexpr (PAGED) p = (const unsigned char*)(src + (uint64_t)at[i] * rs + col);
            else p = (const unsigned char*)src + at[i];
            v[i][0] = *(const u32x4*)p;
            v[i][1] = *(const u32x4*)(p + 16);
            if constexpr (!PAGED) at[i] = min(at[i] + 4u * BC * rs, last);
        }
    };
    float ksc = 1.0f, vsc = 1.0f;
    auto store_k = [&](int i) {
        u32x4 w[2];
        split8<true>(rk[i], ksc, w);
#pragma unroll
        for (int s = 0; s < 2; s++) *(u32x4*)(Ks + s * PL + i * RPU * RB + k_at<RB>(t / CPR, t % CPR)) = w[s];
    };
    auto store_v = [&](int i) {
        u32x4 w[2];
        split8<true>(rv[i], vsc, w);
#pragma unroll
        for (int s = 0; s < 2; s++) *(u32x4*)(Vs + s * PL + i * RPU * RB + v_at<RB>(t / CPR, t % CPR)) = w[s];
    };
    const uint32_t krs = (uint32_t)a.ks[2], vrs = (uint32_t)a.vs[2];
    if (first < ntiles) {
        if constexpr (PAGED) rows_of(first);
        else {
            klast = 4u * ((uint32_t)(a.Sk - 1) * krs + col);
            vlast = 4u * ((uint32_t)(a.Sk - 1) * vrs + col);
#pragma unroll
            for (int i = 0; i < U; i++) {
                kat[i] = min(4u * ((uint32_t)(first * BC + t / CPR + i * RPU) * krs + col), klast);
                vat[i] = min(4u * ((uint32_t)(first * BC + t / CPR + i * RPU) * vrs + col), vlast);
            }
        }
        load(K, krs, kat, klast, rk);
        load(V, vrs, PAGED ? kat : vat, vlast, rv);
        if constexpr (PAGED) rows_of(first + 1);
    }

    u32x4 qf[DS][2];
    int logit_exp = -split_q(Q + (long long)min(q0 + l32, a.Sq - 1) * a.qs[2], q0 + l32 < a.Sq, a.D, h, qf);      // logits are 2^logit_exp Q' K'
    // ---- K and V: one power of two each, from the first tile
    int vexp = 0, oexp = 0;                        // O is formed times 2^oexp
    if (first < ntiles) {
        float km = 0.0f, vm = 0.0f;
#pragma unroll
        for (int i = 0; i < U; i++) {
            km = fmaxf(km, largest(rk[i]));
            vm = fmaxf(vm, largest(rv[i]));
        }
        km = wave_max(km);
        vm = wave_max(vm);
        float* red = (float*)Vs;
        if (lane == 0) { red[wave] = km; red[NW + wave] = vm; }
        __syncthreads();
        km = vm = 0.0f;
#pragma unroll
        for (int w = 0; w < NW; w++) { km = fmaxf(km, red[w]); vm = fmaxf(vm, red[NW + w]); }
        const int kexp = __builtin_amdgcn_readfirstlane(exponent_to(km, 10));
        vexp = __builtin_amdgcn_readfirstlane(exponent_to(vm, 11));
        ksc = power2(kexp);
        vsc = power2(vexp);
        oexp = vexp + P_SPLIT;
        logit_exp -= kexp;
#pragma unroll
        for (int i = 0; i < U; i++) store_k(i);
        __syncthreads();                           // (the maxima have been read before V is written over them)
    }

    f32x16 oacc[DT];
    float m_run, l_run;
    auto clear = [&]() {
        m_run = -INFINITY;
        l_run = 0.0f;
#pragma unroll
        for (int i = 0; i < DT; i++)
#pragma unroll
            for (int r = 0; r < 16; r++) oacc[i][r] = 0.0f;
    };
    clear();

    float to_log2 = logit_factor(OPT ? a.scale : a.scale * LOG2E, logit_exp);       // OPT: the logit itself
    // What the split cuts of Q' and K' (2^-25 of a value) shows in a logit as about 2^-12 of a unit of Q' K'.  Where that is more than 2^-25 of an
    // exponent the row's largest logit, near which all of its weight lies, has to be that far from zero itself (2^13 units), or it is computed
    // again: large values that meet zeros, keys out of the row's sight, or far lower logits can have set the scale
    const bool coarse = to_log2 > 0x1p-13f;
    float pexp = P_EXP;
    // logits of NB 32-key sub-tiles from key k0 on (st[kt][r]: key k0 + 32 kt + acc_row(r, h), query q0 + l32) to probabilities times 2^pexp against
    // the new running maximum; returns what the sums so far are to be multiplied with.  Bit i of `kept`: key k0 + i is visible (OPT)
    auto softmax = [&](auto& st, int k0, uint64_t kept) -> float {
        constexpr int NB = sizeof(st) / sizeof(st[0]);
        float factor = to_log2;
        if constexpr (OPT) {
            const int key0 = k0 + 4 * h;
            int qr = __lane_id();
            asm volatile("" : "+v"(qr));
            qr = min(q0 + (qr & 31), a.Sq - 1);
            factor = LOG2E;
#pragma unroll
            for (int kt = 0; kt < NB; kt++)
#pragma unroll
                for (int r = 0; r < 16; r++) st[kt][r] *= to_log2;
            if (a.softcap > 0.0f) {
#pragma unroll
                for (int kt = 0; kt < NB; kt++) soft_cap<16>(st[kt], a.softcap);
            }
            if (a.bias) {
                const float* __restrict__ row = a.bias + b * a.bias_bs + ((long long)hd * a.Sq + qr) * a.Sk;
#pragma unroll
                for (int kt = 0; kt < NB; kt++)
#pragma unroll
                    for (int r = 0; r < 16; r++) {
                        st[kt][r] += row[min(key0 + 32 * kt + acc_row(r, 0), a.Sk - 1)];
                        if (r % 4 == 3) __builtin_amdgcn_sched_barrier(0);
                    }
            }
            if (a.mask_mode == 1 || a.mask_mode == 2) {
                const float* __restrict__ row = a.mask + ((a.mask_mode == 2 ? (long long)bh * a.Sq : 0LL) + qr) * a.Sk;
#pragma unroll
                for (int kt = 0; kt < NB; kt++)
#pragma unroll
                    for (int r = 0; r < 16; r++) {
                        if (row[min(key0 + 32 * kt + acc_row(r, 0), a.Sk - 1)] == 0.0f) st[kt][r] = -INFINITY;
                        if (r % 4 == 3) __builtin_amdgcn_sched_barrier(0);
                    }
            }
        }
        if (k0 + 32 * NB > a.Sk || (a.causal && (long long)k0 + 32 * NB - 1 > (long long)q0 + a.qoff)) {
            // (formed here, not kept through the loop)
            int at = __lane_id();
            asm volatile("" : "+v"(at));
            const int first = -4 * (at >> 5);
            at = min(at & 31, a.Sq - 1 - q0);          // (rows past the last one see what it sees: they stand beside it in the tests below)
            // the query's last visible key, relative to the lane's first
            int seen = a.Sk - 1 - k0 + first;
            if (a.causal) seen = min(seen, (int)max(min((long long)q0 + a.qoff - k0, 1LL << 20), -(1LL << 20)) + at + first);
#pragma unroll
            for (int kt = 0; kt < NB; kt++)
#pragma unroll
                for (int r = 0; r < 16; r++) if (32 * kt + acc_row(r, 0) > seen) st[kt][r] = -INFINITY;
        }
        if constexpr (OPT) {
            if (kept != ~0ull) {
                int half = __lane_id();
                asm volatile("" : "+v"(half));
                half >>= 5;
#pragma unroll
                for (int kt = 0; kt < NB; kt++) {
                    const uint32_t bits = (uint32_t)(kept >> (32 * kt)) >> (4 * half);
#pragma unroll
                    for (int r = 0; r < 16; r++) if (!(bits >> acc_row(r, 0) & 1u)) st[kt][r] = -INFINITY;
                }
            }
        }
        float mloc = -INFINITY;
#pragma unroll
        for (int kt = 0; kt < NB; kt++)
#pragma unroll
            for (int r = 0; r < 16; r++) mloc = fmaxf(mloc, st[kt][r]);
        // (the reference is the next whole number: what is subtracted and what the sums are rescaled with are then exact)
        const float m_new = fmaxf(m_run, ceilf(max_with_partner32(mloc) * factor));
        const float m_use = m_new == -INFINITY ? 0.0f : m_new;
        const float alpha = __builtin_amdgcn_exp2f(m_run - m_use);
        const float down = pexp - m_use;
        m_run = m_new;
        float psum = 0.0f;
#pragma unroll
        for (int kt = 0; kt < NB; kt++)
#pragma unroll
            for (int r = 0; r < 16; r++) {
                const float p = __builtin_amdgcn_exp2f(fmaf(st[kt][r], factor, down));
                st[kt][r] = p;
                psum += p;
            }
        l_run = l_run * alpha + psum;
        return alpha;
    };

    auto visible = [&](int k0, int n) -> uint64_t {        // keep-mask of the keys: bit i of the result is key k0 + i
        int ln = __lane_id();
        asm volatile("" : "+v"(ln));
        return __builtin_amdgcn_ballot_w64(ln < n && k0 + ln < a.Sk && ((const unsigned char*)a.mask)[(long long)b * a.Sk + min(k0 + ln, a.Sk - 1)] != 0);
    };

    const int q_last = q0 + 31;
    const unsigned char* kbase = Ks + (kg * KT * 32) * RB;
    const unsigned char* vbase = Vs + (kg * KT * 32) * RB;
    const int jl = lane & 15, vkey = 4 * h + (jl >> 2), vch = 2 * ((lane >> 4) & 1) + ((jl & 3) >> 1), vcol = 8 * (jl & 1);      // transposing reads
    for (int j = first; j < ntiles; j++) {
        const int kw0 = j * BC + kg * KT * 32;                      // this wave's first key
        load(K, krs, kat, klast, rk);                                 // (past the last tile rows are repeated)
        uint64_t kept = ~0ull;
        if constexpr (OPT) { if (a.mask_mode == 3) kept = visible(kw0, KT * 32) | (KT == 1 ? ~0ull << 32 : 0ull); }
        const bool none = OPT && (KT == 1 ? (uint32_t)kept == 0 : kept == 0);
        const bool active = q0 < a.Sq && kw0 < a.Sk && !(a.causal && (long long)kw0 > (long long)q_last + a.qoff) && !none;
        f32x16 st[KT];
        // ---- S^T = K Q^T, beside it V to LDS
        if (active) {
#pragma unroll
            for (int kt = 0; kt < KT; kt++)
#pragma unroll
                for (int r = 0; r < 16; r++) st[kt][r] = 0.0f;
            f16x8 k[AHEAD + 1][KT][2];
            auto read_k = [&](int s) {
#pragma unroll
                for (int kt = 0; kt < KT; kt++)
#pragma unroll
                    for (int p = 0; p < 2; p++) k[s & AHEAD][kt][p] = *(const f16x8*)(kbase + p * PL + kt * 32 * RB + k_at<RB>(l32, 2 * s + h));
            };
            if (AHEAD) read_k(0);
#pragma unroll
            for (int s = 0; s < DS; s++) {
                if (s + AHEAD < DS) read_k(s + AHEAD);
                auto add = [&](int x, int y) {
#pragma unroll
                    for (int kt = 0; kt < KT; kt++) st[kt] = __builtin_amdgcn_mfma_f32_32x32x16_f16(k[s & AHEAD][kt][x], __builtin_bit_cast(f16x8, qf[s][y]), st[kt], 0, 0, 0);
                };
                add(1, 0); add(0, 1); add(0, 0);
                if (s < U) store_v(s);
                if (OPT && DP > 64) __builtin_amdgcn_sched_barrier(0);
            }
            static_assert(U <= DS && U <= 2 * KT, "a chunk beside every step");
        } else {
#pragma unroll
            for (int i = 0; i < U; i++) store_v(i);
        }
        load(V, vrs, PAGED ? kat : vat, vlast, rv);
        if constexpr (PAGED) rows_of(j + 2);
        __syncthreads();
        // ---- O^T += V^T P^T, beside it the next K to LDS
        if (active) {
            const float alpha = softmax(st, kw0, kept);
            if (__builtin_amdgcn_ballot_w64(alpha != 1.0f) != 0) {
#pragma unroll
                for (int i = 0; i < DT; i++)
#pragma unroll
                    for (int r = 0; r < 16; r++) oacc[i][r] *= alpha;
            }
            constexpr int G = DT < 2 || DP > 64 || !AHEAD ? 1 : 2, STEPS = 2 * KT * (DT / G);      // blocks of the head dimension side by side; 16 keys to a step
            u32x4 pf[2 * KT][2];
            f16x8 v[AHEAD + 1][G][2];
            auto split_p = [&](int ps) {
#pragma unroll
                for (int e = 0; e < 4; e++) {
                    uint32_t p[2];
                    split2<true>(st[ps >> 1][8 * (ps & 1) + 2 * e], st[ps >> 1][8 * (ps & 1) + 2 * e + 1], power2(P_SPLIT), p);
                    pf[ps][0][e] = p[0];
                    pf[ps][1][e] = p[1];
                }
            };
            auto read_v = [&](int u) {
                const int i0 = u / (2 * KT) * G, ps = u % (2 * KT);
#pragma unroll
                for (int i = 0; i < G; i++)
#pragma unroll
                    for (int p = 0; p < 2; p++) {
                        u32x4 w;
#pragma unroll
                        for (int q = 0; q < 2; q++) {
                            const u32x2 x = __builtin_bit_cast(u32x2, __builtin_amdgcn_ds_read_tr16_b64_v4i16(
                                (__attribute__((address_space(3))) s16x4a*)(vbase + p * PL + (16 * ps + 8 * q) * RB + v_at<RB>(vkey, 4 * (i0 + i) + vch) + vcol)));
                            w[2 * q] = x[0];
                            w[2 * q + 1] = x[1];
                        }
                        v[u & AHEAD][i][p] = __builtin_bit_cast(f16x8, w);
                    }
            };
            if (AHEAD) read_v(0);
            split_p(0);
#pragma unroll
            for (int u = 0; u < STEPS; u++) {
                const int i0 = u / (2 * KT) * G, ps = u % (2 * KT);
                if (u + AHEAD < STEPS) read_v(u + AHEAD);
                if (u + 1 < 2 * KT) split_p(u + 1);
                auto add = [&](int x, int y) {
#pragma unroll
                    for (int i = 0; i < G; i++)
                        oacc[i0 + i] = __builtin_amdgcn_mfma_f32_32x32x16_f16(v[u & AHEAD][i][x], __builtin_bit_cast(f16x8, pf[ps][y]), oacc[i0 + i], 0, 0, 0);
                };
                add(1, 0); add(0, 1); add(0, 0);
                if (u < U) store_k(u);
                if (OPT && DP > 64) __builtin_amdgcn_sched_barrier(0);
            }
        } else {
#pragma unroll
            for (int i = 0; i < U; i++) store_k(i);
        }
        __syncthreads();
    }

    // (what follows is addressed from here: nothing of it is kept through the loop)
    lane = __lane_id();
    asm volatile("" : "+v"(lane));
    t = 64 * wave + lane;
    l32 = lane & 31;
    h = lane >> 5;
    // ---- the waves of key groups 1 .. KG - 1 leave (O, m, l) in LDS, group 0 merges them
    auto merge_groups = [&]() {
        if constexpr (KG > 1) {
            constexpr int AREA = DT * 16 * 64;                          // floats of one wave's O
            float* O1 = (float*)smem + wq * (KG - 1) * AREA;
            float* ML = (float*)smem + (KG - 1) * WQ * AREA + wq * (KG - 1) * 128;
            __syncthreads();
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
            if (kg == 0) {
#pragma unroll
                for (int u = 0; u < KG - 1; u++) {
                    const float m1 = ML[u * 128 + lane], l1 = ML[u * 128 + 64 + lane];
                    const float m_new = fmaxf(m_run, m1), m_use = m_new == -INFINITY ? 0.0f : m_new;
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
            __syncthreads();
        }
    };
    merge_groups();
    // ---- does the split hold these results?  Group 0 has them
    float m_sum, l_sum;                            // the row's reference and sum as they leave
    {
        const float l = kg == 0 ? sum_with_partner32(l_run) : 0.0f;               // (the products run over the keys of both halves)
        m_sum = m_run;
        l_sum = l * __builtin_amdgcn_exp2f(-P_EXP);
        const bool row = l > 0.0f;
        float poison = l * 0.0f, top = 0.0f;
        bool own = poison == poison;               // the sum is held, whatever the results are
#pragma unroll
        for (int i = 0; i < DT; i++)
#pragma unroll
            for (int r = 0; r < 16; r++) {
                poison = fmaf(oacc[i][r], 0.0f, poison);
                top = fmaxf(top, fabsf(oacc[i][r]));
            }
        bool bad = kg == 0 && poison != poison;    // infinities, NaN, values beyond the scale of the first tile
        // (m_run is rounded up to a whole number; with a bias or a cap it is not the logit's)
        if (coarse && row && ((OPT && (a.bias || a.softcap > 0.0f)) || fabsf(m_run) - 1.0f < 0x1p13f * (OPT ? LOG2E : 1.0f) * to_log2)) {
            bad = true;
            own = false;
        }
        // V' is cut at 2^-25 units, and its largest value in the first tile is 2^11 or more.  A row of O that nowhere reaches one unit may be made of
        // values that the scale has left too few bits of: those that set it can be hidden from the row, or weigh nothing in it
        const bool dim = row && q0 + l32 < a.Sq && max_with_partner32(top) < l * (1 << P_SPLIT);
        // ... and so may a column without a value of 2^-5 units in any row
        const float witness = row ? l * (0x1p-5f * (1 << P_SPLIT)) : INFINITY;
        uint32_t fewest = ~0u;                     // (rows that reach it, a bit each: zero where some column has none)
#pragma unroll
        for (int i = 0; i < DT; i++)
#pragma unroll
            for (int r = 0; r < 16; r++) {
                const uint64_t w = __builtin_amdgcn_ballot_w64(fabsf(oacc[i][r]) >= witness);
                fewest = min(fewest, min((uint32_t)w, (uint32_t)(w >> 32)));
            }
        const bool blank = fewest == 0 && __builtin_amdgcn_ballot_w64(row) != 0;
        __shared__ int flags[NW];
        auto any_wave = [&](int x) {               // (with less to keep in registers than __syncthreads_or, which wants the thread's y and z)
            if (lane == 0) flags[wave] = x;
            __syncthreads();
            int any = 0;
#pragma unroll
            for (int w = 0; w < NW; w++) any |= flags[w];
            __syncthreads();
            return __builtin_amdgcn_readfirstlane(any);
        };
        constexpr int BAD = 1, DIM = 2, BLANK = 4;
        const int found = any_wave((__builtin_amdgcn_ballot_w64(bad) != 0 ? BAD : 0) | (__builtin_amdgcn_ballot_w64(dim) != 0 ? DIM : 0) | (blank ? BLANK : 0));
        bool again = (found & BAD) != 0;
        if (found != 0 && !again) {
            // The split holds them all the same where every value of such a column is zero or has its bits (half a unit), and for such rows where
            // V is zero.  Which rows see which values is not asked: a hidden one may cost a needless second computation
            uint32_t* cols = (uint32_t*)smem;
            if (t < DT) cols[t] = (found & DIM) != 0 ? ~0u : 0u;
            __syncthreads();
            if (blank) {
#pragma unroll
                for (int i = 0; i < DT; i++) {
                    uint32_t none = 0;             // bit d: no row reaches it in column 32 i + d
#pragma unroll
                    for (int r = 0; r < 16; r++) {
                        const uint64_t w = __builtin_amdgcn_ballot_w64(fabsf(oacc[i][r]) >= witness);
                        none |= ((uint32_t)w == 0 ? 1u << acc_row(r, 0) : 0u) | ((uint32_t)(w >> 32) == 0 ? 1u << acc_row(r, 1) : 0u);
                    }
                    if (lane == 0) atomicOr(cols + i, none);
                }
            }
            __syncthreads();
            const int keys = min(ntiles * BC, a.Sk), d0 = 4 * (t % (DP / 4));
            const uint32_t mine = cols[d0 / 32] >> (d0 % 32) & 15u;
            int small = 0;
            if (d0 < a.D && mine != 0) {
                f32x4 least = {INFINITY, INFINITY, INFINITY, INFINITY};           // magnitude that is not zero
#pragma unroll 8
                for (int key = first * BC + t / (DP / 4); key < keys; key += NT / (DP / 4)) {
                    const f32x4 x = *(const f32x4*)(V + paged_row(bt, a.bsz, key) * a.vs[2] + d0);
#pragma unroll
                    for (int e = 0; e < 4; e++) least[e] = fminf(least[e], x[e] == 0.0f ? INFINITY : fabsf(x[e]));
                }
#pragma unroll
                for (int e = 0; e < 4; e++) small |= (int)((mine >> e & 1u) != 0 && least[e] < ((found & DIM) != 0 ? INFINITY : 0.5f / vsc));
            }
            again = any_wave(__builtin_amdgcn_ballot_w64(small != 0) != 0 ? 1 : 0) != 0;
        }
        if (again) {
            // again on the fp32 pipe, rows straight from memory
            clear();
            oexp = 0;
            pexp = 0.0f;                           // (V at the end of the range: nothing above one is to meet it)
            to_log2 = OPT ? a.scale : a.scale * LOG2E;
#pragma unroll 1
            for (int k0 = first * BC + kg * KT * 32; k0 < ntiles * BC; k0 += k0 % (KT * 32) + 32 < KT * 32 ? 32 : BC - (KT - 1) * 32) {
                if (q0 >= a.Sq || k0 >= a.Sk || (a.causal && (long long)k0 > (long long)q_last + a.qoff)) continue;
                uint64_t kept = ~0ull;
                if constexpr (OPT) { if (a.mask_mode == 3) kept = visible(k0, 32) | ~0ull << 32; }
                if (OPT && (uint32_t)kept == 0) continue;
                f32x16 s2[1];
#pragma unroll
                for (int r = 0; r < 16; r++) s2[0][r] = 0.0f;
                const float* kp = K + paged_row(bt, a.bsz, min(k0 + l32, a.Sk - 1)) * a.ks[2] + 4 * h;
                const float* qp = Q + (long long)min(q0 + l32, a.Sq - 1) * a.qs[2] + 4 * h;
#pragma unroll 1
                for (int d = 0; d < a.D; d += 8) Mma32<float>::run(s2[0], *(const u32x4*)(kp + d), *(const u32x4*)(qp + d));
                const float alpha = softmax(s2, k0, kept);
                const float* vp[16];
#pragma unroll
                for (int r = 0; r < 16; r++) vp[r] = V + paged_row(bt, a.bsz, min(k0 + acc_row(r, h), a.Sk - 1)) * a.vs[2];
#pragma unroll
                for (int i = 0; i < DT; i++) {
#pragma unroll
                    for (int r = 0; r < 16; r++) oacc[i][r] *= alpha;
#pragma unroll
                    for (int r = 0; r < 16; r++) {
                        float x = vp[r][min(32 * i + l32, a.D - 1)];
                        if (k0 + acc_row(r, h) >= a.Sk) x = 0.0f;              // (an infinite last row is not repeated)
                        oacc[i] = __builtin_amdgcn_mfma_f32_32x32x2f32(x, s2[0][r], oacc[i], 0, 0, 0);
                    }
                    __builtin_amdgcn_sched_barrier(0);
                }
            }
            merge_groups();
            // A sum that the split holds is kept where the results are not, or another row's: the pass behind this one forms its probabilities, and
            // on the pipe that the sum was formed on (apart, over V with a column of 1e-12 they were 2 - 5 times as far off as both passes on the
            // fp32 pipe have them, 3.6e-5 over logits of deviation 64)
            if (!own) {
                m_sum = m_run;
                l_sum = sum_with_partner32(l_run);
            }
        }
    }
    if (kg > 0) return;

    // ---- normalise and store: lane holds query q0 + l32, head-dim elements 32 i + 8 g + 4 h + (0..3)
    const int qi = q0 + l32;
    const float l = sum_with_partner32(l_run);
    // through LDS (16 rows at a time for each wave: chunk c of row r at position c ^ r) and written as whole rows
    auto by_rows = [&](auto value, auto store) {
        constexpr int CH = DP / 4, RPI = 64 / CH;
        unsigned char* stg = smem + wq * (16 * DP * 4);
        const int c = lane % CH;
#pragma unroll
        for (int half = 0; half < 2; half++) {
            if ((l32 >> 4) == half) {
#pragma unroll
                for (int i = 0; i < DT; i++)
#pragma unroll
                    for (int g = 0; g < 4; g++)
                        *(f32x4*)(stg + (l32 & 15) * (DP * 4) + (((8 * i + 2 * g + h) ^ (l32 & (CH - 1) & 15)) << 4)) =
                            f32x4{value(oacc[i][4 * g]), value(oacc[i][4 * g + 1]), value(oacc[i][4 * g + 2]), value(oacc[i][4 * g + 3])};
            }
            __builtin_amdgcn_wave_barrier();
#pragma unroll
            for (int q = 0; q < 16 / RPI; q++) {
                const int r = RPI * q + lane / CH, row = q0 + 16 * half + r;
                const f32x4 v = *(const f32x4*)(stg + r * (DP * 4) + ((c ^ (r & (CH - 1) & 15)) << 4));
                if (row < a.Sq) store(row, 4 * c, v);
            }
            __builtin_amdgcn_wave_barrier();
        }
    };
    if (RANGES && a.part) {
        // a key range: (m, l, O) for the merge.  Everything is scaled by a power of two that brings l below 2^-5 (2^0 where V is small), so that
        // the sum over up to 32 ranges does not leave the range of fp32 where the result does not; m takes that power and stays exact, being whole
        float* __restrict__ P = a.part + ((long long)bh * a.Sq * a.nsplit + blockIdx.y) * (2 + a.D);
        const long long pitch = (long long)a.nsplit * (2 + a.D);
        const float inv = l > 0.0f ? l_sum / l : __builtin_amdgcn_exp2f(-pexp);       // (results to the sum that leaves: a power of two where that is theirs)
        const int e = __builtin_amdgcn_frexp_expf(l_sum) + (oexp > P_SPLIT ? 0 : 5);
        if (h == 0 && qi < a.Sq) *(f32x2p*)(P + qi * pitch) = f32x2p{m_sum + (float)e, __builtin_amdgcn_ldexpf(l_sum, -e)};
        by_rows([&](float x) { return __builtin_amdgcn_ldexpf(x * inv, -oexp - e); },
                [&](int row, int d0, f32x4 v) {
                    if (d0 >= a.D) return;
                    float* __restrict__ p = P + row * pitch + 2 + d0;                  // (8-byte aligned)
                    *(f32x2p*)p = f32x2p{v[0], v[1]};
                    *(f32x2p*)(p + 2) = f32x2p{v[2], v[3]};
                });
        return;
    }
    const float inv = l > 0.0f ? 1.0f / l : 0.0f;
    auto result = [&](float x) { return __builtin_amdgcn_ldexpf(x * inv, -oexp); };       // (in this order: 2^-oexp / l may lie below the normal numbers)
    if (a.lse && h == 0 && qi < a.Sq) a.lse[(long long)bh * a.Sq + qi] = l_sum > 0.0f ? log_sum(m_sum, l_sum) : -INFINITY;
    float* __restrict__ O = (float*)a.o + b * a.os[0] + hd * a.os[1];
    if (a.vec_out && a.D == DP) {
        by_rows(result,
                [&](int row, int d0, f32x4 v) { __builtin_nontemporal_store(v, (f32x4*)(O + (long long)row * a.os[2] + d0)); });
    } else if (qi < a.Sq) {
        float* __restrict__ p = O + (long long)qi * a.os[2];
#pragma unroll
        for (int i = 0; i < DT; i++)
#pragma unroll
            for (int g = 0; g < 4; g++) {
                const int d0 = 32 * i + 8 * g + 4 * h;
                if (a.vec_out) { if (d0 < a.D) *(f32x4*)(p + d0) = f32x4{result(oacc[i][4 * g]), result(oacc[i][4 * g + 1]), result(oacc[i][4 * g + 2]), result(oacc[i][4 * g + 3])}; }
                else {
#pragma unroll
                    for (int e = 0; e < 4; e++) if (d0 + e < a.D) p[d0 + e] = result(oacc[i][4 * g + e]);
                }
            }
    }
}

template <int DP, int BC, int NW, int KG, bool OPT, bool PAGED>
static hipError_t launch_split_as(AttnArgs a, hipStream_t stream)
{
    constexpr int BR = 32 * NW / KG, smem = split_lds(DP, BC, NW, KG);
    auto kern = attn_split_kernel<DP, BC, NW, KG, OPT, PAGED>;
    static unsigned long long attr_done = 0;
    if (hipError_t e = ensure_dynamic_smem((const void*)kern, smem, &attr_done)) return e;
    a.qtiles = (a.Sq + BR - 1) / BR;
    const long long nblk = (long long)a.qtiles * a.B * a.H;
    if (nblk > 0x7FFFFFFFLL) return hipErrorInvalidValue;
    a.hgroup = !a.causal || a.nsplit > 1 ? 0 : nblk <= 768 ? -1 : (a.qtiles >= 8 ? 16 : (128 + a.qtiles - 1) / a.qtiles);
    hipLaunchKernelGGL(kern, dim3((unsigned)nblk, (unsigned)a.nsplit), dim3(64 * NW), smem, stream, a);
    return hipGetLastError();
}

// keys that some query sees
static long long seen_keys(const AttnArgs& a) { return a.causal ? std::min((long long)a.Sk, (long long)a.Sq + a.qoff) : a.Sk; }

// fp32, rows on the 16-byte grid, head dimension up to 128 in whole chunks of eight, a head's K and V within 4 GB (contiguous).  At head
// dimensions 33 .. 64 up to 64 keys stay on the fp32 pipe: one tile of them costs less than the splitting beside it (us: B1 H8 S52 7.9 / 8.6, B15 H32
// S27 8.5 / 9.8; 71 keys 10.0 / 9.0; d128 S62 12.1 / 12.2).  Below that width few keys stay there for the sake of the results: what the split cuts,
// 1.2e-7 of a row of one key, shows where neither the products nor the sums are long enough to round as much (error of O against float64 in units
// of 1e-7, split / fp32 pipe, causal: d8 S256 1.56 / 1.47, 400 1.63 / 1.63; d16 S128 1.43 / 1.37, 200 1.49 / 1.50; d24 S80 1.46 / 1.42, 128 1.52 / 1.56;
// d32 S32 1.31 / 1.23, 56 1.37 / 1.39; plain: d8 S64 1.71 / 1.61, 81 1.77 / 1.71; d16 S20 1.48 / 1.45, 32 1.56 / 1.67).  It costs up to a half there:
// B64 H16 S64 d16 plain 9.5 / 14.3 us, S27 B15 H32 d32 causal 7.5 / 7.0
bool attn_split_applies(const AttnArgs& a)
{
    auto fits = [&](long long row) { return row > 0 && row < (1LL << 30) && (a.bt || row * a.Sk < (1LL << 30)); };
    if (a.bt && (a.bias || a.mask_mode != 0 || a.softcap > 0.0f)) return false;
    if (a.D <= 64 && seen_keys(a) <= (a.D > 32 ? 64 : a.causal ? 4096 / a.D - 80 : 1024 / a.D)) return false;
    return a.vec_in && a.D % 8 == 0 && a.D <= 128 && a.scale > 0.0f && a.scale < 0x1p20f && fits(a.ks[2]) && fits(a.vs[2]);
}

// Waves and key groups.  A wave alone on its SIMD issues half as fast as two do together, so grids that do not fill the chip take workgroups of
// fewer rows whose waves share the keys; full grids lose by it (every workgroup splits the K and V that it reads).  From 128 drawn shapes, us with
// 128 rows / 64 rows in two key groups / 64 rows of eight waves in four:
//   d64: four groups up to 256 workgroups from 448 keys on (S1024 H12 36 / 28 / 25; S300 H16 16.2 / 13.9 / 14.5)
//        two groups up to 64 queries, causal up to 640 workgroups (B4 H12 S512 21.5 / 18.7; 576: 28.8 / 26.5; 768: 24.8 / 29.7), plain up to 256
//        (264: 44.4 / 46.0) and where the coarser grid just needs a second workgroup per CU (280 of 128 rows 31.4 / 25.8)
//   d32: two groups up to 768 (648: 16.4 / 14.6; 2520: 97 / 109), four as above (S1525 H12 33 / 27 / 21)
//   d65 .. 128: 64-key tiles of eight waves in two groups up to 256 from 224 keys on (S1024 H8 65 / 54; B2 H16 S512 37.7 / 33.5; 288: 27 / 36; S152 19.0 / 20.3),
//        else 32-key tiles
template <bool OPT, bool PAGED>
static hipError_t launch_split_opt(const AttnArgs& a, hipStream_t stream)
{
    auto grid = [&](int rows) { return (long long)((a.Sq + rows - 1) / rows) * a.B * a.H; };
    if (a.D <= 32) {
        if (grid(64) <= 256 && seen_keys(a) >= 448) return launch_split_as<32, 128, 8, 4, OPT, PAGED>(a, stream);
        return a.Sq <= 64 || grid(64) <= 768 ? launch_split_as<32, 64, 4, 2, OPT, PAGED>(a, stream) : launch_split_as<32, 64, 4, 1, OPT, PAGED>(a, stream);
    }
    if (a.D <= 64) {
        if (grid(64) <= 256 && seen_keys(a) >= 448) return launch_split_as<64, 128, 8, 4, OPT, PAGED>(a, stream);
        const bool fine = a.Sq <= 64 || (a.causal ? grid(64) <= 640 : grid(64) <= 256 || (grid(128) > 256 && grid(64) <= 512));
        return fine ? launch_split_as<64, 64, 4, 2, OPT, PAGED>(a, stream) : launch_split_as<64, 64, 4, 1, OPT, PAGED>(a, stream);
    }
    return grid(128) <= 256 && seen_keys(a) >= 224 ? launch_split_as<128, 64, 8, 2, OPT, PAGED>(a, stream) : launch_split_as<128, 32, 4, 1, OPT, PAGED>(a, stream);
}
// Ranges of the keys that run as workgroups of their own and are merged by a pass behind (1 = none), where the query tiles leave at least half of
// the CUs without one.  A workgroup on a CU of its own takes 2.4 us a tile of 64 keys beyond head dimension 64, 1.7 and 1.0 a tile of 128 up to 64
// and 32; the second launch is 4, the partials are written and read at 4 TB/s (us a call, in one / cut: 8 heads of 40 queries d128
// 256 keys 20.2 / 16.4, 1024 47.9 / 17.6, 2048 84.4 / 19.4; d64 1024 22.7 / 14.7, 2048 36.2 / 15.1; plain self-attention d128 H8 S1000 52.8 / 36.3, H16 S1000
// 53.0 / 48.2, H16 S500 33.0 / 30.7, d64 H4 S2000 37.1 / 30.8, H8 S1000 23.2 / 23.2; in two ranges d128 H32 S390 29.9 / 34.5, d64 H8 S800 20.9 / 22.3, d32 14.3 / 16.1).
int attn_split_ranges(const AttnArgs& a)
{
    const bool wide = a.D > 64;
    const int rows = wide ? 128 : 64, tile = wide ? 64 : 128;
    const long long grid = (long long)((a.Sq + rows - 1) / rows) * a.B * a.H, keys = seen_keys(a);
    if (grid > 128 || keys < (wide ? 224 : 448) || (wide && (a.bias || a.mask_mode != 0 || a.softcap > 0.0f))) return 1;
    const long long tiles = (keys + tile - 1) / tile, most = std::min(std::min(256 / grid, tiles), 32LL);
    const double tile_us = wide ? 2.4 : a.D > 32 ? 1.7 : 1.0, part_us = (double)a.B * a.H * a.Sq * (2 + a.D) * 8.0 / 4e6;
    int best = 1;
    double gain = 0.5;
    for (int ns = 2; ns <= most; ns++) {
        const double g = tile_us * (double)(tiles - (tiles + ns - 1) / ns) - 4.0 - part_us * ns;
        if (g > gain) { gain = g; best = ns; }
    }
    return best;
}
hipError_t launch_attn_split(const AttnArgs& a, bool options, hipStream_t stream)
{
    if (a.bt) return launch_split_opt<false, true>(a, stream);
    return options ? launch_split_opt<true, false>(a, stream) : launch_split_opt<false, false>(a, stream);
}

// ---------------------------------------------------------------------------------------------
// The probabilities that ScaledDotProductAttention returns, from the log-sum-exp of the pass above.  One workgroup: 128 query rows (four waves of
// 32) and `tiles` tiles of 64 keys.  S = Q K^T with the queries as rows, so that a lane holds one key of 16 rows and a store covers whole lines.
template <int DP, bool OPT>
__global__ __launch_bounds__(256, 2) void attn_weights_split_kernel(const AttnArgs a, float* __restrict__ w, int ktiles, int chunks, int tiles)
{
    constexpr int BK = 64, RB = 2 * DP, PL = BK * RB, DS = DP / 16, CPR = DP / 8, U = BK * CPR / 256, RPU = 256 / CPR;
    __shared__ __attribute__((aligned(1024))) unsigned char Ks[4 * PL];      // two stages of [2][64][DP] fp16
    __shared__ __attribute__((aligned(16))) float rows[2][128], red[4];                                   // of each query: factor of its logits, its log-sum-exp
    constexpr int SROW = BK + 4;                                             // (16 bytes on: the rows of a store's four pieces on other banks)
    constexpr bool STAGE = !OPT && DP <= 64;                                 // (elsewhere it would cost a workgroup per CU)
    __shared__ __attribute__((aligned(16))) float stage[STAGE ? 4 : 1][STAGE ? 16 * SROW : 4];
    const int t = threadIdx.x, lane = t & 63, wave = __builtin_amdgcn_readfirstlane(t >> 6), l32 = lane & 31, h = lane >> 5;
    // XCD-contiguous order: the tiles of one head share an L2
    int bh, qt, chunk;
    {
        const int nblk = gridDim.x, pid = blockIdx.x, per = nblk >> 3, rem = nblk & 7, xcd = pid & 7, idx = pid >> 3;
        const int logical = (xcd < rem ? xcd * (per + 1) : rem * (per + 1) + (xcd - rem) * per) + idx;
        chunk = logical % chunks;
        qt = logical / chunks % a.qtiles;
        bh = logical / chunks / a.qtiles;
    }
    const int b = bh / a.H, hd = bh - b * a.H, q0 = qt * 128 + wave * 32;
    const float* __restrict__ Q = (const float*)a.q + b * a.qs[0] + hd * a.qs[1];
    const float* __restrict__ K = (const float*)a.k + b * a.ks[0] + (hd / (a.H / a.Hkv)) * a.ks[1];
    float* __restrict__ W = w + (long long)bh * a.Sq * a.Sk;
    const int first = chunk * tiles, end = min(first + tiles, ktiles);
    // tiles from `seen` on lie above the causal diagonal of all 128 rows
    int seen = end;
    if (a.causal) {
        const long long last = (long long)qt * 128 + 127 + a.qoff;
        seen = last < 0 ? first : (int)min((long long)end, max((long long)first, last / BK + 1));
    }
    auto zeros = [&](int k0, int k1) {             // columns k0 .. k1 - 1 of this wave's rows
        for (int r = lane >> 4; r < 32 && q0 + r < a.Sq; r += 4)
            for (int c = k0 + 4 * (lane & 15); c < k1; c += 64) {
                float* __restrict__ out = W + (long long)(q0 + r) * a.Sk + c;
                if (c + 4 <= k1) __builtin_nontemporal_store((u32x4_a4){0u, 0u, 0u, 0u}, (u32x4_a4*)out);
                else for (int e = 0; c + e < k1; e++) out[e] = 0.0f;
            }
    };
    if (seen < end) zeros(seen * BK, min(end * BK, a.Sk));
    if (seen == first) return;

    const uint32_t krs = (uint32_t)a.ks[2];
    const int col = min(8 * (t % CPR), a.D - 8);
    const uint32_t klast = 4u * ((uint32_t)(a.Sk - 1) * krs + col);
    uint32_t kat[U];
    u32x4 rk[U][2];
    auto load = [&]() {
#pragma unroll
        for (int i = 0; i < U; i++) {
            const unsigned char* p = (const unsigned char*)K + kat[i];
            rk[i][0] = *(const u32x4*)p;
            rk[i][1] = *(const u32x4*)(p + 16);
            kat[i] = min(kat[i] + 4u * BK * krs, klast);
        }
    };
#pragma unroll
    for (int i = 0; i < U; i++) kat[i] = min(4u * ((uint32_t)(first * BK + t / CPR + i * RPU) * krs + col), klast);
    load();
    const float lse = a.lse[(long long)bh * a.Sq + min(q0 + l32, a.Sq - 1)];
    u32x4 qf[DS][2];
    int logit_exp = -split_q(Q + (long long)min(q0 + l32, a.Sq - 1) * a.qs[2], q0 + l32 < a.Sq, a.D, h, qf);
    float km = 0.0f;
#pragma unroll
    for (int i = 0; i < U; i++) km = fmaxf(km, largest(rk[i]));
    km = wave_max(km);
    if (lane == 0) red[wave] = km;
    __syncthreads();
    km = fmaxf(fmaxf(red[0], red[1]), fmaxf(red[2], red[3]));
    const int kexp = __builtin_amdgcn_readfirstlane(exponent_to(km, 10));
    const float ksc = power2(kexp);
    logit_exp -= kexp;
    const float to_logit = logit_factor(OPT ? a.scale : a.scale * LOG2E, logit_exp);
    // (such rows are formed on the fp32 pipe, as above, and as above not where their largest logits, here the log-sum-exp, are far from zero: with the
    // two passes on different pipes a probability of one was off by the logits' error of either, 7e-4 - 2e-3 over logits of thousands)
    const float unit = OPT ? to_logit * LOG2E : to_logit;
    const bool coarse = unit > 0x1p-13f && ((OPT && (a.bias || a.softcap > 0.0f)) || fabsf(lse) * LOG2E - 1.0f < 0x1p13f * unit);
    const uint32_t coarse_rows = (uint32_t)__builtin_amdgcn_ballot_w64(coarse);
    if (h == 0) { rows[0][32 * wave + l32] = !coarse ? to_logit : OPT ? a.scale : a.scale * LOG2E; rows[1][32 * wave + l32] = lse == -INFINITY ? INFINITY : lse * LOG2E; }
    __builtin_amdgcn_wave_barrier();
    for (int j = first; j < seen; j++) {
        unsigned char* ks = Ks + (j & 1) * 2 * PL;
#pragma unroll
        for (int i = 0; i < U; i++) {
            u32x4 p[2];
            split8<true>(rk[i], ksc, p);
            *(u32x4*)(ks + i * RPU * RB + k_at<RB>(t / CPR, t % CPR)) = p[0];
            *(u32x4*)(ks + PL + i * RPU * RB + k_at<RB>(t / CPR, t % CPR)) = p[1];
        }
        __syncthreads();
        load();                                    // (past the last tile rows are repeated)
        const int k0 = j * BK;
        if (q0 >= a.Sq) continue;
        if (a.causal && (long long)k0 > (long long)q0 + 31 + a.qoff) { zeros(k0, min(k0 + BK, a.Sk)); continue; }
        f32x16 s[2];
#pragma unroll
        for (int i = 0; i < 2; i++)
#pragma unroll
            for (int r = 0; r < 16; r++) s[i][r] = 0.0f;
#pragma unroll
        for (int d = 0; d < DS; d++) {
            f16x8 k[2][2];
#pragma unroll
            for (int i = 0; i < 2; i++)
#pragma unroll
                for (int p = 0; p < 2; p++) k[i][p] = *(const f16x8*)(ks + p * PL + i * 32 * RB + k_at<RB>(l32, 2 * d + h));
            auto add = [&](int x, int y) {
#pragma unroll
                for (int i = 0; i < 2; i++) s[i] = __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(f16x8, qf[d][y]), k[i][x], s[i], 0, 0, 0);
            };
            add(1, 0); add(0, 1); add(0, 0);
        }
        float poison = 0.0f;
#pragma unroll
        for (int i = 0; i < 2; i++)
#pragma unroll
            for (int r = 0; r < 16; r++) poison = fmaf(s[i][r], 0.0f, poison);
        const bool exact = __builtin_amdgcn_ballot_w64(poison != poison) != 0;
        const uint32_t again = exact ? ~0u : coarse_rows;
        if (again != 0) {
            // (the other rows stay as they are: zeros are added to them)
            int ln = __lane_id();
            asm volatile("" : "+v"(ln));           // (which rows is formed here, not kept)
            const uint32_t mine = (again >> (ln & 31) & 1u) != 0 ? ~0u : 0u, those = again >> (4 * (ln >> 5));
#pragma unroll
            for (int i = 0; i < 2; i++) {
#pragma unroll
                for (int r = 0; r < 16; r++) s[i][r] = (those >> acc_row(r, 0) & 1u) != 0 ? 0.0f : s[i][r];
                const float* kp = K + (long long)min(k0 + 32 * i + (ln & 31), a.Sk - 1) * a.ks[2] + 4 * (ln >> 5);
                const float* qp = Q + (long long)min(q0 + (ln & 31), a.Sq - 1) * a.qs[2] + 4 * (ln >> 5);
#pragma unroll 1
                for (int d = 0; d < a.D; d += 8) Mma32<float>::run(s[i], *(const u32x4*)(qp + d) & mine, *(const u32x4*)(kp + d));
            }
        }
        int keys[2] = {k0 + l32, k0 + 32 + l32}, h = lane >> 5;
        asm volatile("" : "+v"(h));                // (rows are formed anew for every tile, not kept beside the fragments)
        __builtin_amdgcn_sched_barrier(0);
        u32x4 factors[4], sums[4];                 // of rows 8 g + 4 h .. + 3
#pragma unroll
        for (int g = 0; g < 4; g++) {
            factors[g] = *(const u32x4*)&rows[0][32 * wave + 8 * g + 4 * h];
            sums[g] = *(const u32x4*)&rows[1][32 * wave + 8 * g + 4 * h];
        }
        // logits in place, one pass over the tile per option, out-of-range elements on clamped addresses
        if constexpr (OPT) {
#pragma unroll
            for (int r = 0; r < 16; r++) {
                const float f = exact ? a.scale : as_f32(factors[r >> 2][r & 3]);
#pragma unroll
                for (int i = 0; i < 2; i++) s[i][r] *= f;
            }
            if (a.softcap > 0.0f) {
#pragma unroll
                for (int i = 0; i < 2; i++) soft_cap<16>(s[i], a.softcap);
            }
            if (a.bias) {
                const float* __restrict__ Bi = a.bias + b * a.bias_bs + (long long)hd * a.Sq * a.Sk;
#pragma unroll
                for (int i = 0; i < 2; i++)
#pragma unroll
                    for (int r = 0; r < 16; r++) {
                        s[i][r] += Bi[(long long)min(q0 + acc_row(r, h), a.Sq - 1) * a.Sk + min(keys[i], a.Sk - 1)];
                        if (r % 4 == 3) __builtin_amdgcn_sched_barrier(0);
                    }
            }
            if (a.mask_mode == 3) {
                const unsigned char* __restrict__ Mk = (const unsigned char*)a.mask + (long long)b * a.Sk;
#pragma unroll
                for (int i = 0; i < 2; i++) {
                    const bool hidden = Mk[min(keys[i], a.Sk - 1)] == 0;
#pragma unroll
                    for (int r = 0; r < 16; r++) s[i][r] = hidden ? -INFINITY : s[i][r];
                }
            } else if (a.mask_mode != 0) {
                const float* __restrict__ Mk = a.mask + (a.mask_mode == 2 ? (long long)bh * a.Sq * a.Sk : 0LL);
#pragma unroll
                for (int i = 0; i < 2; i++)
#pragma unroll
                    for (int r = 0; r < 16; r++) {
                        if (Mk[(long long)min(q0 + acc_row(r, h), a.Sq - 1) * a.Sk + min(keys[i], a.Sk - 1)] == 0.0f) s[i][r] = -INFINITY;
                        if (r % 4 == 3) __builtin_amdgcn_sched_barrier(0);
                    }
            }
        }
        if (a.causal && (long long)k0 + 63 > (long long)q0 + a.qoff) {
#pragma unroll
            for (int i = 0; i < 2; i++)
#pragma unroll
                for (int r = 0; r < 16; r++) if ((long long)keys[i] > (long long)q0 + acc_row(r, h) + a.qoff) s[i][r] = -INFINITY;
        }
        // (a row without any visible key has no probabilities: its log-sum-exp counts as infinite)
        auto probability = [&](int i, int r) {
            const float f = OPT ? LOG2E : exact ? a.scale * LOG2E : as_f32(factors[r >> 2][r & 3]);
            return __builtin_amdgcn_exp2f(fmaf(s[i][r], f, -as_f32(sums[r >> 2][r & 3])));
        };
        if constexpr (STAGE) {
            // 16 rows at a time through LDS, so that a store is four whole pieces of a row, past the caches
            float* mine = stage[wave];
#pragma unroll
            for (int half = 0; half < 2; half++) {
#pragma unroll
                for (int r = 8 * half; r < 8 * half + 8; r++)
#pragma unroll
                    for (int i = 0; i < 2; i++) mine[(acc_row(r, h) - 16 * half) * SROW + 32 * i + l32] = probability(i, r);
                __builtin_amdgcn_wave_barrier();
#pragma unroll
                for (int u = 0; u < 4; u++) {
                    const int r = 4 * u + (lane >> 4), c = 4 * (lane & 15), row = q0 + 16 * half + r;
                    const u32x4 v = *(const u32x4*)(mine + r * SROW + c);
                    float* __restrict__ out = W + (long long)row * a.Sk + k0 + c;
                    if (row < a.Sq) {
                        if (k0 + c + 4 <= a.Sk) __builtin_nontemporal_store((u32x4_a4)v, (u32x4_a4*)out);
                        else {
#pragma unroll
                            for (int e = 0; e < 4; e++) if (k0 + c + e < a.Sk) out[e] = as_f32(v[e]);
                        }
                    }
                }
                __builtin_amdgcn_wave_barrier();
            }
        } else {
            const bool whole = q0 + 32 <= a.Sq && k0 + BK <= a.Sk;
#pragma unroll
            for (int r = 0; r < 16; r++) {
                float* __restrict__ out = W + (long long)(q0 + acc_row(r, h)) * a.Sk;
#pragma unroll
                for (int i = 0; i < 2; i++) {
                    const float p = probability(i, r);
                    if (whole || (q0 + acc_row(r, h) < a.Sq && keys[i] < a.Sk)) __builtin_nontemporal_store(p, out + keys[i]);
                }
            }
        }
    }
}

template <int DP>
static hipError_t launch_weights_split_as(AttnArgs a, float* w, hipStream_t stream)
{
    a.qtiles = (a.Sq + 127) / 128;
    const int ktiles = (a.Sk + 63) / 64;
    const long long rows = (long long)a.qtiles * a.B * a.H;
    // Key tiles to a workgroup: two where that makes a grid of several rounds (fp32 B8 H16 S1000 d64 with attention 319 us, 296 this way;
    // B2 H16/4 700 x 900 d128 causal 98, 91), else as many as leave two workgroups per CU (B4 H12 S512 d64 causal, of which two tiles each make
    // 768: 40, 36)
    const int split = (int)std::max(1LL, std::min((long long)ktiles, 512 / rows));
    const int tiles = rows * ktiles >= 2048 ? 2 : (ktiles + split - 1) / split;
    const int chunks = (ktiles + tiles - 1) / tiles;
    if (rows * chunks > 0x7FFFFFFFLL) return hipErrorInvalidValue;
    auto go = [&](auto kern) { hipLaunchKernelGGL(kern, dim3((unsigned)(rows * chunks)), dim3(256), 0, stream, a, w, ktiles, chunks, tiles); };
    if (a.bias || a.mask_mode != 0 || a.softcap > 0.0f) go(attn_weights_split_kernel<DP, true>);
    else go(attn_weights_split_kernel<DP, false>);
    return hipGetLastError();
}
hipError_t launch_attn_weights_split(const AttnArgs& a, float* w, hipStream_t stream)
{
    return a.D <= 32 ? launch_weights_split_as<32>(a, w, stream) : a.D <= 64 ? launch_weights_split_as<64>(a, w, stream) : launch_weights_split_as<128>(a, w, stream);
}

}  // namespace aidn
