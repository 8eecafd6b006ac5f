// fp32 products on the bf16 matrix pipe.  Every operand value is split into three bf16 values, x = h + m + l (h = bf16(x), m = bf16(x - h),
// l = x - h - m, exact for |x| >= 2^-110), and the six products whose weight is at least 2^-18 of the largest are formed: h h, h m, m h,
// m m, h l, l h.  What is left out is below 2^-26 of the product; the fp32 pipe rounds its sum after every second product, this one after
// every sixth of 32.
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
// multiply came out equal (4096^3 683 / 677 us).  Against the fp32 pipe, us: 4096^3 920 / 680, 4096 x 3072 x 768 with GELU 150 / 105,
// 2048 x 12288 x 1024 416 / 260, 2368 x 64 x 16181 998 / 70; fp16 weights (five products) 1991 x 2849 x 4800 1149 / 307, 50 x 192 x 5888
// 246 / 16.  Error against float64, |error| / |result| over 140 shapes: 0.21 - 0.45 of the fp32 pipe's (4096 x 3072 x 768 5.0e-7 / 1.05e-7).
//
// Where the split is not exact enough the tile is computed again on the fp32 pipe: a result that is not finite (infinities and values
// that round to one do not survive a split), or an operand value below 2^-110, which a split cuts at 2^-134, beside one above 2^30 or a
// result below 2^-60 (otherwise what is cut is less than 2^-40 of the smallest result).
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
    const int t = threadIdx.x, lane = t & 63, wave = t >> 6, l16 = lane & 15, gq = lane >> 4;
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
    const int bwave = __builtin_amdgcn_readfirstlane(8 * wave);
    const unsigned char* bbase = (const unsigned char*)(B + (long long)bwave * g.ldb);
    const uint32_t boff = (uint32_t)sizeof(b_t) * (uint32_t)(bcol - past);
    auto b_at = [&](const unsigned char* row, int c) { return *(const b_t*)(row + boff + c * sizeof(b_t)); };
    u32x4 ra[NSET][UA][2];
    b_t rb[NSET][8][CPT];
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
    float big = 0.0f;                                             // the largest magnitude this thread staged
    auto stage = [&](auto set) {
        constexpr int S = decltype(set)::value;
#pragma unroll
        for (int i = 0; i < UA; i++) {
            const int u = t + 256 * i, row = u >> 2, kg = u & 3;
            u32x4 w[3];
#pragma unroll
            for (int e = 0; e < 4; e++) {
                const float x = as_f32(ra[S][i][e >> 1][2 * (e & 1)]), y = as_f32(ra[S][i][e >> 1][2 * (e & 1) + 1]);
                big = fmaxf(fmaxf(big, fabsf(x)), fabsf(y));
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
                else { x = bx; y = by; big = fmaxf(fmaxf(big, fabsf(x)), fabsf(y)); }
                uint32_t p[PB];
                split_pair(x, y, p);
#pragma unroll
                for (int s = 0; s < PB; s++) w[s][e] = p[s];
            }
#pragma unroll
            for (int s = 0; s < PB; s++) *(u32x4*)(Bs + s * BPL + wave * (BN * 16) + ((c * 64 + lane) ^ (2 * wave)) * 16) = w[s];
        }
        asm volatile("" : "+v"(big));                             // (formed here: moved behind the loads it keeps the old values alive)
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
    float poison = 0.0f, least = INFINITY;
#pragma unroll
    for (int i = 0; i < TI; i++)
#pragma unroll
        for (int j = 0; j < TJ; j++)
#pragma unroll
            for (int r = 0; r < 4; r++) {
                poison = fmaf(acc[i][j][r], 0.0f, poison);        // NaN once a value is infinite or NaN
                least = fminf(least, fabsf(acc[i][j][r]));
            }
    int redo = poison != poison;
    if (__syncthreads_or(redo | (big > 0x1p30f) | (least < 0x1p-60f))) {
        if (!__syncthreads_or(redo)) {                            // (no infinity:) does an operand value lose bits?
            float tiny = 1.0f;
            auto look = [&](float x) { tiny = x != 0.0f ? fminf(tiny, fabsf(x)) : tiny; };
            auto look_all = [&]() {
#pragma unroll
                for (int i = 0; i < UA; i++)
#pragma unroll
                    for (int e = 0; e < 8; e++) look(as_f32(ra[0][i][e >> 2][e & 3]));
                if constexpr (!B16) {
#pragma unroll
                    for (int r = 0; r < 8; r++)
#pragma unroll
                        for (int c = 0; c < CPT; c++) look(rb[0][r][c]);
                }
            };
            const int back = tiles > 0 ? 32 * (tiles - 1) : 0;    // where the loads have left the pointers
            abase -= 4 * back;
            bbase -= (long long)back * g.ldb * sizeof(b_t);
            if constexpr (REST) {
                if (K % 32 != 0) { load_remainder(); look_all(); }
            }
            loaded = 0;
#pragma unroll 1
            for (int it = 0; it < tiles; it++) { load(first); look_all(); }
            redo = tiny < 0x1p-110f;
        }
        if (__syncthreads_or(redo)) {
            static_for<0, TI, 1>([&](auto ic) {
                static_for<0, TJ, 1>([&](auto jc) {
                    constexpr int i = decltype(ic)::value, j = decltype(jc)::value;
                    const float* x = A + (long long)min(m0 + wm * (BM / 2) + 16 * i + l16, g.M - 1) * g.lda;
                    const b_t* y = B + min(n0 + (wn * 32 + 16 * (j & 1) + l16) * CPT + (j >> 1), g.N - 1);
                    f32x4 s = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll 1
                    for (int k = gq; k - gq < K; k += 4) {
                        float va = 0.0f, vb = 0.0f;
                        if (k < K) {
                            va = x[k];
                            if constexpr (B16) vb = f16_bits_to_float(y[(long long)k * g.ldb]);
                            else vb = y[(long long)k * g.ldb];
                        }
                        s = __builtin_amdgcn_mfma_f32_16x16x4f32(va, vb, s, 0, 0, 0);
                    }
                    acc[i][j] = s;
                });
            });
        }
    }

    // ---- epilogue: rows 4 gq + r of a block, CPT consecutive columns to a lane
    float* __restrict__ C = (float*)g.C + bz * g.sC;
    const bool rows_cut = EDGE && m0 + BM > g.M, cut = EDGE && n0 + BN > g.N;
    static_for<0, TI, 1>([&](auto ic) {
        constexpr int i = decltype(ic)::value;
        const int row0 = m0 + wm * (BM / 2) + 16 * i + 4 * gq;
        static_for<0, 2, 1>([&](auto hc) {
            constexpr int h = decltype(hc)::value;
            const int col = n0 + (wn * 32 + 16 * h + l16) * CPT;
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
    if (tile == 192) return b16 ? launch_split_tile<128, 3, 2>(g, batch, stream) : launch_split_tile<128, 3, 3>(g, batch, stream);
    if (tile == 128) return b16 ? launch_split_tile<128, 2, 2>(g, batch, stream) : launch_split_tile<128, 2, 3>(g, batch, stream);
    if (tile == 64) return b16 ? launch_split_tile<64, 2, 2>(g, batch, stream) : launch_split_tile<64, 2, 3>(g, batch, stream);
    return hipErrorInvalidValue;
}

}  // namespace aidn
