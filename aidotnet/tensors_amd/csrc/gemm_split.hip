// fp32 products on the bf16 matrix pipe.  Every operand value is split into three bf16 values, x = h + m + l (h = bf16(x), m = bf16(x - h),
// l = x - h - m, exact for |x| >= 2^-110), and the six products whose weight is at least 2^-18 of the largest are formed: h h, h m, m h,
// m m, h l, l h.  What is left out (m l, l m, l l) is at most 2^-24 of a product; the fp32 pipe, whose products are exact, rounds its sum
// after every second of them, this one after every sixth of 32.  From four terms on the error is the smaller one; a sum that one term rules
// (a row with a single value in it, no power of two) keeps the error of its product, up to 2.6 x 2^-24 where that pipe rounds once.
#include "gemm_common.hpp"

namespace aidn {

// One BM x 64 CPT tile of C: four waves, 2 x 2, K in tiles of 32.  PB: bf16 values per element of B, 3, or 2 for fp16 weights (11 bits).
//
//   A  a thread loads 8 consecutive k of BM / 64 rows; LDS plane [k / 8][row][8 k]
//   B  a thread loads 8 k-rows of CPT consecutive columns, so that its values pair up along k without a transpose; LDS plane
//      [k / 8][column % CPT][column / CPT][8 k], and a lane of the 16 x 16 x 32 MFMA ends with CPT consecutive columns of a row of C
//
// Rows are swizzled by 2 (k / 8): writes (eight lanes on two rows of four chunks, or eight rows of one) and fragment reads are free of
// bank conflicts (counted: none).  One LDS stage (37 / 49 / 61 KB) and two or three workgroups per CU: one's loads, splitting and LDS
// writes run under the other's MFMAs.  The six products of 32 k are summed smallest first from zero and join the accumulators in one
// fp32 addition.
//
// Bound by the matrix pipe (half of its cycles at two workgroups per CU) and the vector pipe beside it: 5.5 instructions split a value,
// a third of what a wave issues; a CU's clock under this load is 1.8 GHz.  Four waves that only load and split beside four that only
// multiply came out equal (4096^3 683 / 677 us).  Against the fp32 pipe, us: 4096^3 920 / 680, 4096 x 3072 x 768 with GELU 149.5 / 105.9,
// 2048 x 12288 x 1024 416 / 260, 2368 x 64 x 16181 998 / 70; fp16 weights (five products) 1991 x 2849 x 4800 1149 / 307, 50 x 192 x 5888
// 246 / 16.  Error against float64, |error| / |result| over 140 shapes: 0.21 - 0.45 of the fp32 pipe's (4096 x 3072 x 768 5.0e-7 / 1.05e-7).
//
// Where the split is not exact enough a result is computed again on the fp32 pipe: one that is not finite (infinities and values that round
// to one do not survive a split), and one whose row or column holds a value below 2^-110 (which a split cuts at 2^-134) where the largest
// possible sum of what is cut, K 2^-134 times the other operand's largest magnitude, exceeds 2^-30 of it.  A result's own row and column
// decide that and nothing beside them, and zeros decide nothing.  us, 4096 x 3072 x 768 / 2048 x 2048 x 4096: normal values 109 / 200, every
// seventh row zero 110 / 206, one NaN 186 / 268, A of probabilities down to 0 (every tile's operands looked at again) 125 / 360; the fp32 pipe
// 157 / 258 for all of them; with whole tiles computed again, by one load at a time, and the second look taken for zeros too 109 / 202, 134 / 257,
// 1690 / 2950, 102 / 2980.
// EDGES: 0 whole tiles, 1 ragged M or N, 2 a remainder of K too.
template <int BM, int CPT, int PB, int EDGES>
__global__ __launch_bounds__(256, BM == 64 ? 3 : 2) void gemm_split_kernel(const GemmArgs g)
{
    constexpr int BN = 64 * CPT, TI = BM / 32, TJ = 2 * CPT, UA = BM / 64;
    constexpr int APL = BM * 64, BPL = BN * 64;                   // bytes of one plane
    static_assert(CPT == 2 || EDGES == 0, "edges: two columns to a thread");
    constexpr bool B16 = PB == 2, EDGE = EDGES > 0, REST = EDGES > 1;
    typedef typename std::conditional<B16, uint16_t, float>::type b_t;
    extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
    unsigned char* As = smem;
    unsigned char* Bs = smem + 3 * APL;
    const int t = threadIdx.x, lane = t & 63, wave = __builtin_amdgcn_readfirstlane(t >> 6), l16 = lane & 15, gq = lane >> 4;
    const int wm = wave >> 1, wn = wave & 1;
    int tm, tn;
    tile_of_block(blockIdx.x, gridDim.x, g.tiles_m, g.tiles_n, tm, tn);
    const int m0 = tm * BM, n0 = tn * BN;
    const long long bz = blockIdx.z;
    const int K = g.k_total ? min(g.K, g.k_total - (int)bz * g.K) : g.K;
    const float* __restrict__ A = (const float*)g.A + bz * g.sA;
    const b_t* __restrict__ B = (const b_t*)batch_b<sizeof(b_t)>(g, bz);

    // K in tiles of 32; a remainder is a tile of its own, taken first, so that the loads of all others are alike.  NSET sets of
    // registers: tiles travel two ahead where the registers allow it
    constexpr int NSET = CPT == 2 ? 2 : 1;
    const int tiles = K / 32;
    // uniform bases that follow the tiles, lane offsets (bytes) that stay
    const unsigned char* abase = (const unsigned char*)(A + (long long)m0 * g.lda);
    uint32_t aoff[UA];
#pragma unroll
    for (int i = 0; i < UA; i++) {
        const int u = t + 256 * i;
        aoff[i] = 4u * (uint32_t)(min(u >> 2, g.M - 1 - m0) * g.lda + 8 * (u & 3));
    }
    const int bcol = n0 + lane * CPT, past = EDGE ? max(bcol - (g.N - CPT), 0) : 0;      // columns past the end repeat the last one (never stored)
    const int bwave = 8 * wave;
    const unsigned char* bbase = (const unsigned char*)(B + (long long)bwave * g.ldb);
    const uint32_t boff = (uint32_t)sizeof(b_t) * (uint32_t)(bcol - past);
    auto b_at = [&](const unsigned char* row, int c) { return *(const b_t*)(row + boff + c * sizeof(b_t)); };
    u32x4 ra[2][UA][2];                                           // (the second look uses both everywhere)
    b_t rb[2][8][CPT];
    int loaded = 0;
    auto load = [&](auto set) {
        constexpr int S = decltype(set)::value;
#pragma unroll
        for (int i = 0; i < UA; i++) {
            ra[S][i][0] = *(const u32x4_a4*)(abase + aoff[i]);
            ra[S][i][1] = *(const u32x4_a4*)(abase + aoff[i] + 16);
        }
#pragma unroll
        for (int r = 0; r < 8; r++)
#pragma unroll
            for (int c = 0; c < CPT; c++) rb[S][r][c] = b_at(bbase + (long long)r * g.ldb * sizeof(b_t), c);
        // (past the last tile it is read again: a branch around loads would make every wait a wait for all of them)
        const int step = ++loaded < tiles ? 32 : 0;
        abase += 4 * step;
        bbase += (long long)step * g.ldb * sizeof(b_t);
    };
    auto load_remainder = [&]() {                                 // element by element, zeros past the end
        const int k0 = tiles * 32;
#pragma unroll
        for (int i = 0; i < UA; i++) {
            const int k = k0 + 8 * ((t + 256 * i) & 3);
#pragma unroll
            for (int e = 0; e < 8; e++) {
                const float x = *(const float*)(abase + aoff[i] + 4 * (min(k + e, K - 1) - (k - k0)));
                ra[0][i][e >> 2][e & 3] = k + e < K ? as_u32(x) : 0u;
            }
        }
#pragma unroll
        for (int r = 0; r < 8; r++) {
            const int k = k0 + bwave + r;
            const unsigned char* row = (const unsigned char*)(B + (long long)min(k, K - 1) * g.ldb);
#pragma unroll
            for (int c = 0; c < CPT; c++) { const b_t x = b_at(row, c); rb[0][r][c] = k < K ? x : (b_t)0; }
        }
    };
    // the smallest magnitude but zero that this thread staged, if below 2^-110: bits doubled (no sign) less one (zero wraps to the largest).
    // What a tile holds is first compared as it is, zeros included, half an instruction a value; the exact form follows where that was small
    uint32_t tiny = 0xFFFFFFFFu;
    auto nonzero = [](float x) { return 2u * as_u32(x) - 1u; };
    auto stage = [&](auto set) {
        constexpr int S = decltype(set)::value;
        float least = INFINITY;
#pragma unroll
        for (int i = 0; i < UA; i++)
#pragma unroll
            for (int e = 0; e < 8; e++) least = fminf(least, fabsf(as_f32(ra[S][i][e >> 2][e & 3])));
        if (least < 0x1p-110f) {
#pragma unroll
            for (int i = 0; i < UA; i++)
#pragma unroll
                for (int e = 0; e < 8; e++) tiny = min(tiny, nonzero(as_f32(ra[S][i][e >> 2][e & 3])));
        }
        if constexpr (!B16) {
            least = INFINITY;
#pragma unroll
            for (int r = 0; r < 8; r++)
#pragma unroll
                for (int c = 0; c < CPT; c++) least = fminf(least, fabsf(rb[S][r][c]));
            if (least < 0x1p-110f) {
#pragma unroll
                for (int r = 0; r < 8; r++)
#pragma unroll
                    for (int c = 0; c < CPT; c++) tiny = min(tiny, nonzero(rb[S][r][c]));
            }
        }
#pragma unroll
        for (int i = 0; i < UA; i++) {
            const int u = t + 256 * i, row = u >> 2, kg = u & 3;
            u32x4 w[3];
#pragma unroll
            for (int e = 0; e < 4; e++) {
                const float x = as_f32(ra[S][i][e >> 1][2 * (e & 1)]), y = as_f32(ra[S][i][e >> 1][2 * (e & 1) + 1]);
                uint32_t p[3];
                split_pair(x, y, p);
#pragma unroll
                for (int s = 0; s < 3; s++) w[s][e] = p[s];
            }
#pragma unroll
            for (int s = 0; s < 3; s++) *(u32x4*)(As + s * APL + kg * (BM * 16) + (row ^ (2 * kg)) * 16) = w[s];
        }
#pragma unroll
        for (int c = 0; c < CPT; c++) {
            u32x4 w[PB];
#pragma unroll
            for (int e = 0; e < 4; e++) {
                float x, y;
                auto pick = [&](int r) {
                    b_t v = rb[S][r][c];
                    if constexpr (EDGE) { if (c == 0 && past > 0) v = rb[S][r][1]; }
                    return v;
                };
                const b_t bx = pick(2 * e), by = pick(2 * e + 1);
                if constexpr (B16) { x = f16_bits_to_float(bx); y = f16_bits_to_float(by); }
                else { x = bx; y = by; }
                uint32_t p[PB];
                split_pair(x, y, p);
#pragma unroll
                for (int s = 0; s < PB; s++) w[s][e] = p[s];
            }
#pragma unroll
            for (int s = 0; s < PB; s++) *(u32x4*)(Bs + s * BPL + wave * (BN * 16) + ((c * 64 + lane) ^ (2 * wave)) * 16) = w[s];
        }
    };

    f32x4 acc[TI][TJ];                                            // block (i, j): rows 16 i, columns j / 2 + CPT (16 (j & 1) + lane % 16)
#pragma unroll
    for (int i = 0; i < TI; i++)
#pragma unroll
        for (int j = 0; j < TJ; j++) acc[i][j] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
    const unsigned char* ab = As + gq * (BM * 16) + ((wm * (BM / 2) + l16) ^ (2 * gq)) * 16;
    const unsigned char* bb = Bs + gq * (BN * 16) + ((wn * 32 + l16) ^ (2 * gq)) * 16;
    auto multiply = [&]() {
        constexpr int NB = BM == 128 || PB == 2 ? 2 : 1;           // (a second set of B fragments where the registers hold it)
        bf16x8 a[TI][3], b[NB][PB];
        auto read_b = [&](int j) {
#pragma unroll
            for (int s = 0; s < PB; s++) b[j % NB][s] = *(const bf16x8*)(bb + s * BPL + (j >> 1) * 1024 + (j & 1) * 256);
        };
        read_b(0);
#pragma unroll
        for (int s = 2; s >= 0; s--)                              // (in the order of their first use)
#pragma unroll
            for (int i = 0; i < TI; i++) a[i][s] = *(const bf16x8*)(ab + s * APL + i * 256);
#pragma unroll
        for (int j = 0; j < TJ; j++) {
            if (NB == 1 ? j > 0 : j + 1 < TJ) read_b(NB == 1 ? j : j + 1);
            f32x4 sum[TI];
#pragma unroll
            for (int i = 0; i < TI; i++) sum[i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[i][2], b[j % NB][0], (f32x4{0.0f, 0.0f, 0.0f, 0.0f}), 0, 0, 0);
            auto add = [&](int x, int y) {
#pragma unroll
                for (int i = 0; i < TI; i++) sum[i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[i][x], b[j % NB][y], sum[i], 0, 0, 0);
            };
            if constexpr (PB == 3) add(0, PB - 1);
            add(1, 1);
            add(0, 1);
            add(1, 0);
            add(0, 0);
#pragma unroll
            for (int i = 0; i < TI; i++) acc[i][j] += sum[i];
        }
    };
    constexpr std::integral_constant<int, 0> first;
    constexpr std::integral_constant<int, NSET - 1> second;
    if constexpr (REST) {
        if (K % 32 != 0) {
            load_remainder();
            stage(first);
            __syncthreads();
            multiply();
            __syncthreads();                                      // everyone has read the tile
        }
    }
    if (!REST || tiles > 0) {
        load(first);
        if constexpr (NSET == 2) load(second);
        for (int it = 0;; it += NSET) {
            stage(first);
            __builtin_amdgcn_sched_barrier(0);                    // (loads moved up into the staging need a second set of registers)
            load(first);
            __builtin_amdgcn_sched_barrier(0);
            __syncthreads();
            multiply();
            if (it + 1 >= tiles) break;
            __syncthreads();
            if constexpr (NSET == 2) {
                stage(second);
                __builtin_amdgcn_sched_barrier(0);
                load(second);
                __builtin_amdgcn_sched_barrier(0);
                __syncthreads();
                multiply();
                if (it + 2 >= tiles) break;
                __syncthreads();
            }
        }
    }

    // ---- is the split exact enough here?
    constexpr uint32_t CUT_BELOW = 2u * (17u << 23) - 1u;         // 2^-110
    float poison = 0.0f;
#pragma unroll
    for (int i = 0; i < TI; i++)
#pragma unroll
        for (int j = 0; j < TJ; j++)
#pragma unroll
            for (int r = 0; r < 4; r++) poison = fmaf(acc[i][j][r], 0.0f, poison);        // NaN once a value is infinite or NaN
    const bool lossy = tiny < CUT_BELOW;
    int ln = __lane_id();
    asm volatile("" : "+v"(ln));                                  // (what follows is addressed from here: nothing of it is kept through the loop above)
    if (__syncthreads_or(lossy | (poison != poison))) {
        const int th = 64 * wave + ln, row16 = ln & 15, quad = ln >> 4;
        // of the tile's rows, then columns: 1 if it holds a value below 2^-110, and its largest magnitude times K 2^-104
        float* low = (float*)smem;
        float* high = low + BM + BN;
        const bool look = __syncthreads_or(lossy);
        for (int q = th; q < BM + BN; q += 256) { low[q] = 0.0f; high[q] = 0.0f; }
        __syncthreads();
        if (look) {
            uint32_t lo_a[UA], lo_b[CPT];
            float hi_a[UA], hi_b[CPT];
#pragma unroll
            for (int i = 0; i < UA; i++) { lo_a[i] = 0xFFFFFFFFu; hi_a[i] = 0.0f; }
#pragma unroll
            for (int c = 0; c < CPT; c++) { lo_b[c] = 0xFFFFFFFFu; hi_b[c] = 0.0f; }
            auto look_at = [&](auto set) {
                constexpr int S = decltype(set)::value;
#pragma unroll
                for (int i = 0; i < UA; i++)
#pragma unroll
                    for (int e = 0; e < 8; e++) {
                        const float x = as_f32(ra[S][i][e >> 2][e & 3]);
                        lo_a[i] = min(lo_a[i], nonzero(x)); hi_a[i] = fmaxf(hi_a[i], fabsf(x));
                    }
#pragma unroll
                for (int r = 0; r < 8; r++)
#pragma unroll
                    for (int c = 0; c < CPT; c++) {
                        if constexpr (B16) hi_b[c] = fmaxf(hi_b[c], fabsf(f16_bits_to_float(rb[S][r][c])));
                        else { lo_b[c] = min(lo_b[c], nonzero(rb[S][r][c])); hi_b[c] = fmaxf(hi_b[c], fabsf(rb[S][r][c])); }
                    }
            };
            const int back = tiles > 0 ? 32 * (tiles - 1) : 0;    // where the loads have left the pointers
            abase -= 4 * back;
            bbase -= (long long)back * g.ldb * sizeof(b_t);
            if constexpr (REST) {
                if (K % 32 != 0) { load_remainder(); look_at(first); }
            }
            if (tiles > 0) {
                loaded = 0;
                load(first);
#pragma unroll 1
                for (int it = 0; it < tiles; it += 2) {           // (past the last tile it is looked at again)
                    load(std::integral_constant<int, 1>{});
                    __builtin_amdgcn_sched_barrier(0);
                    look_at(first);
                    __builtin_amdgcn_sched_barrier(0);
                    load(first);
                    __builtin_amdgcn_sched_barrier(0);
                    look_at(std::integral_constant<int, 1>{});
                }
            }
            const float scale = (float)K * 0x1p-104f;
            auto mark = [&](int q, uint32_t lo, float hi) {
                if (q < 0) return;                                // (a column of the tile before)
                if (lo < CUT_BELOW) low[q] = 1.0f;
                atomicMax((uint32_t*)&high[q], as_u32(hi * scale));          // (not negative: ordered like its bits)
            };
#pragma unroll
            for (int i = 0; i < UA; i++) mark((th + 256 * i) >> 2, lo_a[i], hi_a[i]);
#pragma unroll
            for (int c = 0; c < CPT; c++) {
                const int q = ln * CPT - past + c;
                mark(q < 0 ? -1 : BM + q, lo_b[c], hi_b[c]);
            }
            __syncthreads();
        }
        // which results the split does not hold: a bit per column block and row of the block, a word per row block; and the blocks of this wave
        uint32_t want[TI], blocks = 0;
        float column_low[TJ], column_high[TJ];
#pragma unroll
        for (int j = 0; j < TJ; j++) {
            const int q = BM + (wn * 32 + 16 * (j & 1) + row16) * CPT + (j >> 1);
            column_low[j] = low[q]; column_high[j] = high[q];
        }
        static_for<0, TI, 1>([&](auto ic) {
            constexpr int i = decltype(ic)::value;
            uint32_t w = 0;
#pragma unroll
            for (int r = 0; r < 4; r++) {
                const int q = wm * (BM / 2) + 16 * i + 4 * quad + r;
                const float row_low = low[q], row_high = high[q];
#pragma unroll
                for (int j = 0; j < TJ; j++) {
                    const float v = fabsf(acc[i][j][r]);
                    w |= !(v < INFINITY) | (v < fmaf(row_low, column_high[j], column_low[j] * row_high)) ? 1u << (4 * j + r) : 0u;
                }
            }
            asm volatile("" : "+v"(w));                           // (formed here, row block by row block: the tests of all of them do not fit the registers)
            want[i] = w;
#pragma unroll
            for (int j = 0; j < TJ; j++) blocks |= __ballot(w >> (4 * j) & 15u) ? 1u << (TJ * i + j) : 0u;
        });
        // those blocks again on the fp32 pipe, one after the other, RK k at a time, the next RK in flight: lane (quad, row16) holds k = 4 quad .. 4 quad + 3
        // of every 16, of its row and of its column, one of them to an instruction
        constexpr int RK = CPT == 3 ? 32 : 64;                    // (what the registers hold beside the accumulators)
        static_for<0, TI, 1>([&](auto ic) {
            constexpr int i = decltype(ic)::value;                // (a loop of its own for each: one over all blocks copies every accumulator, which do not fit twice)
#pragma unroll 1
            for (int bj = 0; bj < TJ; bj++) {
                if (!(blocks >> (TJ * i + bj) & 1)) continue;
                int at = ln;
                asm volatile("" : "+v"(at));
                const int row16 = at & 15, quad = at >> 4;
                const float* x = A + (long long)min(m0 + wm * (BM / 2) + 16 * i + row16, g.M - 1) * g.lda + 4 * quad;
                const int column = min(n0 + (wn * 32 + 16 * (bj & 1) + row16) * CPT + (bj >> 1), g.N - 1);
                const b_t* y = B + (long long)(4 * quad) * g.ldb + column;
                f32x4 sum = {0.0f, 0.0f, 0.0f, 0.0f}, va[2][RK / 16];
                b_t vb[2][RK / 16][4];
                auto fetch = [&](int s, int k) {
#pragma unroll
                    for (int q = 0; q < RK / 16; q++) {
                        va[s][q] = __builtin_bit_cast(f32x4, *(const u32x4_a4*)(x + (k + 16 * q)));
#pragma unroll
                        for (int e = 0; e < 4; e++) vb[s][q][e] = y[(long long)(k + 16 * q + e) * g.ldb];
                    }
                };
                auto multiply16 = [&](const f32x4& a, const b_t (&b)[4]) {
#pragma unroll
                    for (int e = 0; e < 4; e++) {
                        float v;
                        if constexpr (B16) v = f16_bits_to_float(b[e]);
                        else v = b[e];
                        sum = __builtin_amdgcn_mfma_f32_16x16x4f32(a[e], v, sum, 0, 0, 0);
                    }
                };
                auto multiply_all = [&](int s) {
#pragma unroll
                    for (int q = 0; q < RK / 16; q++) multiply16(va[s][q], vb[s][q]);
                };
                const int whole = K / RK * RK;
                if (whole > 0) fetch(0, 0);
#pragma unroll 1
                for (int k = 0; k < whole; k += 2 * RK) {
                    fetch(1, min(k + RK, whole - RK));
                    multiply_all(0);
                    if (k + RK >= whole) break;
                    fetch(0, min(k + 2 * RK, whole - RK));
                    multiply_all(1);
                }
#pragma unroll 1
                for (int k0 = whole; (REST || RK > 32) && k0 < K; k0 += 16) {
#pragma unroll
                    for (int e = 0; e < 4; e++) {
                        const int k = k0 + e, last = K - 1 - 4 * quad;      // (x and y start at k = 4 quad, which may be past the end)
                        const float v = x[min(k, last)];
                        const b_t w = y[(long long)min(k, last) * g.ldb];
                        va[0][0][e] = k <= last ? v : 0.0f; vb[0][0][e] = k <= last ? w : (b_t)0;
                    }
                    multiply16(va[0][0], vb[0][0]);
                }
                asm volatile("" : "+v"(want[i]));
                static_for<0, TJ, 1>([&](auto jc) {
                    constexpr int j = decltype(jc)::value;
                    uint32_t here = bj == j ? 15u << (4 * j) : 0u;
                    asm volatile("" : "+s"(here));                    // (selected and not branched to)
#pragma unroll
                    for (int r = 0; r < 4; r++) acc[i][j][r] = want[i] & here & 1u << (4 * j + r) ? sum[r] : acc[i][j][r];
                });
            }
        });
    }

    // ---- epilogue: rows 4 (lane / 16) + r of a block, CPT consecutive columns to a lane
    float* __restrict__ C = (float*)g.C + bz * g.sC;
    const bool rows_cut = EDGE && m0 + BM > g.M, cut = EDGE && n0 + BN > g.N;
    static_for<0, TI, 1>([&](auto ic) {
        constexpr int i = decltype(ic)::value;
        const int row0 = m0 + wm * (BM / 2) + 16 * i + 4 * (ln >> 4);
        static_for<0, 2, 1>([&](auto hc) {
            constexpr int h = decltype(hc)::value;
            const int col = n0 + (wn * 32 + 16 * h + (ln & 15)) * CPT;
            float v[4][CPT];
#pragma unroll
            for (int r = 0; r < 4; r++)
#pragma unroll
                for (int c = 0; c < CPT; c++) v[r][c] = g.alpha * acc[i][2 * c + h][r];
            if (g.beta != 0.0f) {
#pragma unroll
                for (int r = 0; r < 4; r++)
#pragma unroll
                    for (int c = 0; c < CPT; c++) v[r][c] += g.beta * C[(long long)min(row0 + r, g.M - 1) * g.ldc + min(col + c, g.N - 1)];
            }
            if (g.bias) {
#pragma unroll
                for (int c = 0; c < CPT; c++) {
                    const float b = g.bias[min(col + c, g.N - 1)];
#pragma unroll
                    for (int r = 0; r < 4; r++) v[r][c] += b;
                }
            }
            if (g.act)
                with_activation(g.act, g.act_param, [&](auto fn) {
#pragma unroll
                    for (int r = 0; r < 4; r++)
#pragma unroll
                        for (int c = 0; c < CPT; c++) v[r][c] = fn(v[r][c]);
                });
#pragma unroll
            for (int r = 0; r < 4; r++) {
                float* p = C + (long long)(row0 + r) * g.ldc + col;
                if (rows_cut && row0 + r >= g.M) continue;
                if (cut) {
#pragma unroll
                    for (int c = 0; c < CPT; c++) if (col + c < g.N) p[c] = v[r][c];
                } else {
#pragma unroll
                    for (int c = 0; c < CPT; c++) p[c] = v[r][c];
                }
            }
        });
    });
}

template <int BM, int CPT, int PB, int EDGES>
static hipError_t launch_split_as(GemmArgs g, int batch, hipStream_t stream)
{
    constexpr int smem = 64 * (3 * BM + PB * 64 * CPT);
    auto kern = gemm_split_kernel<BM, CPT, PB, EDGES>;
    static unsigned long long attr_done = 0;
    if (hipError_t e = ensure_dynamic_smem((const void*)kern, smem, &attr_done)) return e;
    g.tiles_m = (g.M + BM - 1) / BM;
    g.tiles_n = (g.N + 64 * CPT - 1) / (64 * CPT);
    hipLaunchKernelGGL(kern, dim3((unsigned)(g.tiles_m * g.tiles_n), 1, (unsigned)batch), dim3(256), smem, stream, g);
    return hipGetLastError();
}
template <int BM, int CPT, int PB>
static hipError_t launch_split_tile(const GemmArgs& g, int batch, hipStream_t stream)
{
    const bool rest = g.K % 32 != 0 || g.k_total % 32 != 0, ragged = g.M % BM != 0 || g.N % (64 * CPT) != 0;
    if constexpr (CPT == 2) {
        if (rest) return launch_split_as<BM, CPT, PB, 2>(g, batch, stream);
        if (ragged) return launch_split_as<BM, CPT, PB, 1>(g, batch, stream);
    } else if (rest || ragged) return hipErrorInvalidValue;       // (such instances of the widest tile do not fit the registers)
    return launch_split_as<BM, CPT, PB, 0>(g, batch, stream);
}
hipError_t launch_gemm_split(const GemmArgs& g, int batch, hipStream_t stream, int tile, bool b16)
{
    if (tile == 192) return b16 ? hipErrorInvalidValue : launch_split_tile<128, 3, 3>(g, batch, stream);
    if (tile == 128) return b16 ? launch_split_tile<128, 2, 2>(g, batch, stream) : launch_split_tile<128, 2, 3>(g, batch, stream);
    if (tile == 64) return b16 ? launch_split_tile<64, 2, 2>(g, batch, stream) : launch_split_tile<64, 2, 3>(g, batch, stream);
    return hipErrorInvalidValue;
}

}  // namespace aidn
