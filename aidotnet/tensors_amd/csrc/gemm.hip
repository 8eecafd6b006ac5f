// LDS-staged, double-buffered MFMA GEMM for gfx950: C = alpha * A * op(B) + beta * C,
// row-major, fp32 / fp16 / bf16 inputs with fp32 accumulation.
//
// Replaces, behind the reference's GPU-backend slot, what
// src/AiDotNet.Tensors/Engines/DirectGpu/HIP/HipBackend.cs:1370-1631 (Gemm, MatMulTransposed,
// BatchedGemm) and HipBackend.HalfPrecision.cs:97-150 (Hgemm, GemmFp16In32fOut) do with
// hipBLAS or run-time compiled kernel strings; the arithmetic contract is the CPU path's
// (src/AiDotNet.Tensors/Engines/Simd/SimdGemm.cs:1284-1315, HalfKernels.cs:35-99,
// BFloat16Kernels.cs:144-211): products of the stored values, fp32 accumulation, one
// round-to-nearest-even narrow at the end for 16-bit outputs.
//
// Data movement per workgroup and K-tile of the general kernel (128 bytes of K per row, 256 for the 64 x 64 tile):
//   global --16 B/lane--> registers --(B[K,N]: E x E register transpose)--> LDS [row][k], row pitch
//   = row + 16 bytes of padding (conflict-free ds_read_b128 / ds_write_b128) --> 16-byte MFMA
//   fragments.  Two LDS stages: the next tile's global loads are issued at the top of an iteration and
//   stored to the other stage before its last k-step; one barrier per K-tile.
// The 16-bit 256 x 256 kernel further down loads global -> LDS directly; the skinny (M <= 32, 16-bit) and
// small-M (M <= 8, fp32) kernels are bandwidth-bound split-K streams of B.
#include "gemm_common.hpp"

// This file is compiled three times (the build passes -DAIDN_GEMM_PART=0/1/2) so that its template instances build in
// parallel: part 0 holds the fp32 entry points and everything that exists once, part 1 the fp16 and part 2 the bf16 instances.
#ifndef AIDN_GEMM_PART
#define AIDN_GEMM_PART 0
#endif

namespace aidn {

#if AIDN_GEMM_PART == 0
hipError_t ensure_dynamic_smem(const void* kernel, int bytes, unsigned long long* done_mask)
{
    int dev = 0;
    if (hipError_t e = hipGetDevice(&dev)) return e;
    const unsigned long long bit = 1ULL << (dev & 63);
    if (__atomic_load_n(done_mask, __ATOMIC_ACQUIRE) & bit) return hipSuccess;
    if (hipError_t e = hipFuncSetAttribute(kernel, hipFuncAttributeMaxDynamicSharedMemorySize, bytes)) return e;
    __atomic_fetch_or(done_mask, bit, __ATOMIC_RELEASE);
    return hipSuccess;
}
#endif

// K extent of one tile of the general kernel in 16-byte chunks per row, and the LDS row pitch (one chunk of padding keeps the
// b128 fragment reads conflict-free).  The 64 x 64 tile takes twice the K per barrier: its waves have too little MFMA work
// per tile to hide one barrier every 128 bytes of K.
constexpr int gemm_k_chunks(int bm, int bn) { return bm * bn <= 64 * 64 ? 16 : 8; }
constexpr int gemm_row_pitch(int bm, int bn) { return gemm_k_chunks(bm, bn) * 16 + 16; }
template <typename T> struct Raw;
template <> struct Raw<float> { typedef uint32_t type; };
template <> struct Raw<f16_t> { typedef uint16_t type; };
template <> struct Raw<bf16_t> { typedef uint16_t type; };

// 16 bytes = PER16 consecutive elements starting at p, elements at index >= valid read as 0.
template <typename T>
__device__ __forceinline__ u32x4 load16_guarded(const typename Raw<T>::type* p, int valid)
{
    // a whole chunk: one 16-byte load that is only element-aligned (the hardware takes such loads; rows that start off a 16-byte
    // boundary used to be read element by element, ten times slower)
    typedef u32x4 u32x4_a4 __attribute__((aligned(4)));
    typedef u32x4 u32x4_a2 __attribute__((aligned(2)));
    if (valid >= Elem<T>::PER16) {
        if constexpr (Elem<T>::BYTES == 4) return *(const u32x4_a4*)p;
        else return *(const u32x4_a2*)p;
    }
    u32x4 v = {0u, 0u, 0u, 0u};
    if constexpr (Elem<T>::BYTES == 4) {
#pragma unroll
        for (int e = 0; e < 4; e++) if (e < valid) v[e] = p[e];
    } else {
#pragma unroll
        for (int e = 0; e < 8; e++) if (e < valid) v[e >> 1] |= ((uint32_t)p[e]) << (16 * (e & 1));
    }
    return v;
}

// KS = 2: two groups of WM x WN waves work on the same output tile, each on half of the k-steps of every K-tile, and the
// second group's accumulators are added through LDS at the end (for grids too small to give every SIMD two waves).
// Scheduling pattern for one step of straight-line code: NM MFMAs, each followed by its share of ND LDS reads, NV global
// loads and NW LDS writes (in that order of urgency).
template <int NM, int ND, int NV, int NW>
__device__ __forceinline__ void spread_schedule()
{
    constexpr int TOT = ND + NV + NW;
#pragma unroll
    for (int i = 0; i < NM; i++) {
        __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
#pragma unroll
        for (int o = i * TOT / NM; o < (i + 1) * TOT / NM; o++) {
            if (o < ND) __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
            else if (o < ND + NV) __builtin_amdgcn_sched_group_barrier(0x020, 1, 0);
            else __builtin_amdgcn_sched_group_barrier(0x200, 1, 0);
        }
    }
}

// B16 (fp32 kernels only): B holds fp16 weights [K,N]; they are widened to fp32 on the way into LDS, so the product is that
// of the fp32 A with the exactly widened weights, accumulated in fp32 (weight-only fp16 GEMM).
template <typename T, typename OutT, int BM, int BN, int WM, int WN, bool TRANSB, bool VEC, bool CHECK, int KS = 1, bool B16 = false>
__global__ __launch_bounds__(WM * WN * KS * 64) void gemm_kernel(const GemmArgs g)
{
    static_assert(!B16 || (Elem<T>::BYTES == 4 && !TRANSB), "fp16 weights: fp32 kernel, B stored [K,N]");
    typedef typename Raw<T>::type raw_t;
    constexpr int E = Elem<T>::PER16;
    constexpr int KC = gemm_k_chunks(BM, BN);  // 16-byte chunks of K per tile row
    constexpr int BK = KC * E;                 // elements of K per tile
    constexpr int ROWB = gemm_row_pitch(BM, BN);
    constexpr int NT = WM * WN * KS * 64;
    constexpr int SPG = KC / 2 / KS;                // fragment steps of a K-tile per wave group
    static_assert(KS == 1 || KS == 2, "KS must be 1 or 2");
    constexpr int WTM = BM / WM, WTN = BN / WN;
    constexpr int TM = WTM / 32, TN = WTN / 32;
    constexpr int UA = (BM * KC + NT - 1) / NT;                   // 16-byte chunks of A per thread
    constexpr int UBT = (BN * KC + NT - 1) / NT;                  // same for B stored [N,K]
    constexpr int NBLK = KC * (BN / E);                           // E x E blocks of B stored [K,N]
    constexpr int UBN = (NBLK + NT - 1) / NT;
    static_assert(WTM % 32 == 0 && WTN % 32 == 0, "wave tile must be a multiple of 32x32");

    extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
    unsigned char* As = smem;                          // [2][BM][ROWB]
    unsigned char* Bs = smem + 2 * BM * ROWB;          // [2][BN][ROWB]

    const int t = threadIdx.x;
    const int lane = t & 63, wave = t >> 6;
    const int l32 = lane & 31, h = lane >> 5;
    const int kgrp = wave / (WM * WN), wq = wave - kgrp * (WM * WN);
    const int wm = wq / WN, wn = wq % WN;

    int tile_m, tile_n;
    tile_of_block(blockIdx.x, gridDim.x, g.tiles_m, g.tiles_n, tile_m, tile_n);
    const int m0 = tile_m * BM, n0 = tile_n * BN;
    const long long bz = blockIdx.z;
    const raw_t* __restrict__ A = (const raw_t*)g.A + bz * g.sA;
    const raw_t* __restrict__ B = (const raw_t*)batch_b<sizeof(raw_t)>(g, bz);

    // Global loads run two tiles ahead where the registers allow it (tile t travels in register set t & 1 and has two
    // iterations to arrive from memory: what a small problem with one workgroup per CU needs), otherwise one tile ahead.
    constexpr bool AHEAD2 = BM * BN <= 64 * 64;
    constexpr int NSETS = AHEAD2 ? 2 : 1;
    u32x4 ra2[NSETS][UA];
    u32x4 rb2[NSETS][TRANSB ? UBT : UBN * E];

    auto load_tile = [&](int k0, auto setc) {
        auto& ra = ra2[decltype(setc)::value];
        auto& rb = rb2[decltype(setc)::value];
        // ---- A (and B when stored [N,K]): 16-byte chunks along K
#pragma unroll
        for (int i = 0; i < UA; i++) {
            int u = t + i * NT;
            int row = u / KC, ch = u % KC;
            int gm = m0 + row, gk = k0 + ch * E;
            u32x4 v = {0u, 0u, 0u, 0u};
            if ((BM * KC) % NT == 0 || u < BM * KC) {
                const raw_t* p = A + (long long)(CHECK ? gm : min(gm, g.M - 1)) * g.lda + gk;
                if constexpr (!CHECK) v = *(const u32x4*)p;       // rows past the end repeat the last one (never stored)
                else if (gm < g.M && gk < g.K) {
                    if constexpr (VEC) v = *(const u32x4*)p;
                    else v = load16_guarded<T>(p, g.K - gk);
                }
            }
            ra[i] = v;
        }
        if constexpr (TRANSB) {
#pragma unroll
            for (int i = 0; i < UBT; i++) {
                int u = t + i * NT;
                int row = u / KC, ch = u % KC;
                int gn = n0 + row, gk = k0 + ch * E;
                u32x4 v = {0u, 0u, 0u, 0u};
                if ((BN * KC) % NT == 0 || u < BN * KC) {
                    const raw_t* p = B + (long long)(CHECK ? gn : min(gn, g.N - 1)) * g.ldb + gk;
                    if constexpr (!CHECK) v = *(const u32x4*)p;
                    else if (gn < g.N && gk < g.K) {
                        if constexpr (VEC) v = *(const u32x4*)p;
                        else v = load16_guarded<T>(p, g.K - gk);
                    }
                }
                rb[i] = v;
            }
        } else {
            // ---- B stored [K,N]: E rows of 16 bytes (E consecutive n) per block
#pragma unroll
            for (int i = 0; i < UBN; i++) {
                int u = t + i * NT;
                int kb = u % KC, nb = u / KC;
                int gn = n0 + nb * E;
#pragma unroll
                for (int r = 0; r < E; r++) {
                    int gk = k0 + kb * E + r;
                    u32x4 v = {0u, 0u, 0u, 0u};
                    if (NBLK % NT == 0 || u < NBLK) {
                        if constexpr (B16) {
                            const uint16_t* p = (const uint16_t*)g.B + bz * g.sB + (long long)gk * g.ldb + gn;
                            if (gk < g.K && gn < g.N) {
                                if (VEC && gn + 4 <= g.N) {
                                    u32x2 w = *(const u32x2*)p;
                                    v = u32x4{as_u32(f16_bits_to_float(w[0] & 0xFFFFu)), as_u32(f16_bits_to_float(w[0] >> 16)),
                                              as_u32(f16_bits_to_float(w[1] & 0xFFFFu)), as_u32(f16_bits_to_float(w[1] >> 16))};
                                } else {
#pragma unroll
                                    for (int e = 0; e < 4; e++) if (gn + e < g.N) v[e] = as_u32(f16_bits_to_float(p[e]));
                                }
                            }
                        } else {
                        const raw_t* p = B + (long long)gk * g.ldb + (CHECK ? gn : min(gn, g.N - E));
                        if constexpr (!CHECK) v = *(const u32x4*)p;   // column blocks past the end repeat the last one
                        else if (gk < g.K && gn < g.N) {
                            if constexpr (VEC) v = *(const u32x4*)p;
                            else v = load16_guarded<T>(p, g.N - gn);
                        }
                        }
                    }
                    rb[i * E + r] = v;
                }
            }
        }
    };

    auto store_tile = [&](int stage, auto setc) {
        auto& ra = ra2[decltype(setc)::value];
        auto& rb = rb2[decltype(setc)::value];
        unsigned char* as = As + stage * BM * ROWB;
        unsigned char* bs = Bs + stage * BN * ROWB;
#pragma unroll
        for (int i = 0; i < UA; i++) {
            int u = t + i * NT;
            if ((BM * KC) % NT == 0 || u < BM * KC) *(u32x4*)(as + (u / KC) * ROWB + (u % KC) * 16) = ra[i];
        }
        if constexpr (TRANSB) {
#pragma unroll
            for (int i = 0; i < UBT; i++) {
                int u = t + i * NT;
                if ((BN * KC) % NT == 0 || u < BN * KC) *(u32x4*)(bs + (u / KC) * ROWB + (u % KC) * 16) = rb[i];
            }
        } else {
#pragma unroll
            for (int i = 0; i < UBN; i++) {
                int u = t + i * NT;
                int kb = u % KC, nb = u / KC;
                if (NBLK % NT == 0 || u < NBLK) {
                    if constexpr (E == 8) {
                        u32x4 in[8], out[8];
#pragma unroll
                        for (int r = 0; r < 8; r++) in[r] = rb[i * 8 + r];
                        transpose8x8_b16(in, out);
#pragma unroll
                        for (int c = 0; c < 8; c++) *(u32x4*)(bs + (nb * 8 + c) * ROWB + kb * 16) = out[c];
                    } else {
                        u32x4 in[4], out[4];
#pragma unroll
                        for (int r = 0; r < 4; r++) {
                            in[r] = rb[i * 4 + r];
                            // the renaming moves belong here, not behind the global loads (where they would wait for them)
                            asm volatile("" : "+v"(in[r]));
                        }
                        transpose4x4_b32(in, out);
#pragma unroll
                        for (int c = 0; c < 4; c++) *(u32x4*)(bs + (nb * 4 + c) * ROWB + kb * 16) = out[c];
                    }
                }
            }
        }
    };

    f32x16 acc[TM][TN];
#pragma unroll
    for (int i = 0; i < TM; i++)
#pragma unroll
        for (int j = 0; j < TN; j++)
#pragma unroll
            for (int r = 0; r < 16; r++) acc[i][j][r] = 0.0f;

    const int KT = (g.K + BK - 1) / BK;
    typedef std::integral_constant<int, 0> Set0;
    typedef std::integral_constant<int, 1> Set1;
    load_tile(0, Set0{});
    store_tile(0, Set0{});
    if constexpr (AHEAD2) {
        if (!CHECK || KT > 1) load_tile(min(1, KT - 1) * BK, Set1{});
    }
    __syncthreads();

    // Fragments are double-buffered in registers: the LDS reads of step s+1 are in flight during the MFMAs of step s.
    // Tile kt+1 is published (register -> LDS stores, barrier) BEFORE the last step of tile kt, and its first fragments are
    // read right after the barrier, so the barrier wait and the LDS latency are covered by that step's MFMAs.
    const int frag_off = (wm * WTM + l32) * ROWB + h * 16 + kgrp * SPG * 32;
    const int frag_off_b = (wn * WTN + l32) * ROWB + h * 16 + kgrp * SPG * 32;
    u32x4 fa[2][TM], fb[2][TN];
    auto read_frags = [&](int stage, int step, int buf) {
        const unsigned char* as = As + stage * BM * ROWB + frag_off + step * 32;
        const unsigned char* bs = Bs + stage * BN * ROWB + frag_off_b + step * 32;
#pragma unroll
        for (int i = 0; i < TM; i++) fa[buf][i] = *(const u32x4*)(as + i * 32 * ROWB);
#pragma unroll
        for (int j = 0; j < TN; j++) fb[buf][j] = *(const u32x4*)(bs + j * 32 * ROWB);
    };
    // iteration kt works on LDS stage kt & 1 = SET, requests tile kt+2 into register set SET (free: tile kt was stored one
    // iteration ago) and publishes tile kt+1 from the other set; with one set it requests tile kt+1 and publishes it
    auto iteration = [&](int kt, int SET, auto intoc, auto otherc) {
        typedef decltype(intoc) Into;
        typedef decltype(otherc) Other;
        // The unchecked instance has no branch in the loop body (past the end it fetches the last tile once more and
        // publishes it to the unused stage), so loads, LDS traffic and MFMAs of one iteration can be interleaved freely.
        const bool more = !CHECK || kt + 1 < KT;
        if constexpr (!CHECK) load_tile(min(kt + NSETS, KT - 1) * BK, Into{});
        else if (kt + NSETS < KT) load_tile((kt + NSETS) * BK, Into{});
#pragma unroll
        for (int s = 0; s < SPG; s++) {
            if (s < SPG - 1) read_frags(SET, s + 1, (s + 1) & 1);
            else {
                __builtin_amdgcn_sched_barrier(0);      // keep the MFMAs of the last step below the barrier
                if (more) store_tile(SET ^ 1, Other{});
                __syncthreads();
                if (more) read_frags(SET ^ 1, 0, SPG & 1);
            }
            __builtin_amdgcn_sched_barrier(0);          // fragment reads of the next step are issued before this step's MFMAs
#pragma unroll
            for (int i = 0; i < TM; i++)
#pragma unroll
                for (int j = 0; j < TN; j++) Mma32<T>::run(acc[i][j], fa[s & 1][i], fb[s & 1][j]);
        }
    };
    // Unchecked instance: one iteration is straight-line code, and the order of its instructions is given explicitly: every
    // MFMA is followed by its share of the step's other memory instructions (next fragments, the global loads in the first
    // step, the LDS stores of the next tile in the last step before the barrier), so the matrix pipe never waits behind a
    // burst of them.
    auto mfma_step = [&](int s) {
#pragma unroll
        for (int i = 0; i < TM; i++)
#pragma unroll
            for (int j = 0; j < TN; j++) Mma32<T>::run(acc[i][j], fa[s & 1][i], fb[s & 1][j]);
    };
    auto iteration_il = [&](int kt, int SET, auto intoc, auto otherc) {
        typedef decltype(intoc) Into;
        typedef decltype(otherc) Other;
        constexpr int NM = TM * TN * (E == 4 ? 4 : 1);          // MFMAs per step
        constexpr int NL = UA + (TRANSB ? UBT : UBN * E);       // global loads = LDS stores per tile and thread
        constexpr int NR = TM + TN;                             // fragment reads per step
        load_tile(min(kt + NSETS, KT - 1) * BK, Into{});
#pragma unroll
        for (int s = 0; s < SPG - 1; s++) {
            read_frags(SET, s + 1, (s + 1) & 1);
            if (s == SPG - 2) store_tile(SET ^ 1, Other{});
            mfma_step(s);
            if (s == 0 && s == SPG - 2) spread_schedule<NM, NR, NL, NL>();
            else if (s == 0) spread_schedule<NM, NR, NL, 0>();
            else if (s == SPG - 2) spread_schedule<NM, NR, 0, NL>();
            else spread_schedule<NM, NR, 0, 0>();
            __builtin_amdgcn_sched_barrier(0);
        }
        __syncthreads();
        read_frags(SET ^ 1, 0, SPG & 1);
        mfma_step(SPG - 1);
        spread_schedule<NM, NR, 0, 0>();
        __builtin_amdgcn_sched_barrier(0);
    };
    read_frags(0, 0, 0);
    if constexpr (!CHECK && AHEAD2) {
        for (int kt = 0; kt < KT; kt += 2) {
            iteration_il(kt, 0, Set0{}, Set1{});
            if (kt + 1 < KT) iteration_il(kt + 1, 1, Set1{}, Set0{});
        }
    } else if constexpr (!CHECK) {
        for (int kt = 0; kt < KT; kt++) iteration_il(kt, kt & 1, Set0{}, Set0{});
    } else if constexpr (AHEAD2) {
        for (int kt = 0; kt < KT; kt += 2) {
            iteration(kt, 0, Set0{}, Set1{});
            if (kt + 1 < KT) iteration(kt + 1, 1, Set1{}, Set0{});
        }
    } else {
        for (int kt = 0; kt < KT; kt++) iteration(kt, kt & 1, Set0{}, Set0{});
    }

    if constexpr (KS == 2) {
        // second wave group hands its partial sums over through LDS (the tile stages are free after the last barrier)
        float* xs = (float*)smem;
        if (kgrp == 1) {
#pragma unroll
            for (int i = 0; i < TM; i++)
#pragma unroll
                for (int j = 0; j < TN; j++)
#pragma unroll
                    for (int r = 0; r < 16; r++) xs[((wq * TM + i) * TN + j) * 1024 + r * 64 + lane] = acc[i][j][r];
        }
        __syncthreads();
        if (kgrp == 1) return;
#pragma unroll
        for (int i = 0; i < TM; i++)
#pragma unroll
            for (int j = 0; j < TN; j++)
#pragma unroll
                for (int r = 0; r < 16; r++) acc[i][j][r] += xs[((wq * TM + i) * TN + j) * 1024 + r * 64 + lane];
    }

    // ---- epilogue: lane holds column l32 of each 32x32 tile, 16 rows
    typedef typename Raw<OutT>::type out_t;
    out_t* __restrict__ C = (out_t*)g.C + bz * g.sC;
    const bool use_beta = g.beta != 0.0f;
    const bool fused = g.bias != nullptr || g.act != 0;
    auto store_all = [&](auto fused_c) {
        constexpr bool FUSED = decltype(fused_c)::value;
#pragma unroll
        for (int i = 0; i < TM; i++) {
#pragma unroll
            for (int j = 0; j < TN; j++) {
                const int col = n0 + wn * WTN + j * 32 + l32;
                float bias = 0.0f;
                if constexpr (FUSED) bias = (g.bias && col < g.N) ? g.bias[col] : 0.0f;
                f32x16 v = acc[i][j];
#pragma unroll
                for (int r = 0; r < 16; r++) v[r] *= g.alpha;
                if (use_beta) {                  // (clamped addresses: a guard per element would make every load wait for the one before)
#pragma unroll
                    for (int r = 0; r < 16; r++) {
                        const int row = min(m0 + wm * WTM + i * 32 + acc_row(r, h), g.M - 1);
                        const out_t* p = C + (long long)row * g.ldc + min(col, g.N - 1);
                        if constexpr (Elem<OutT>::BYTES == 4) v[r] += g.beta * as_f32(*p);
                        else v[r] += g.beta * Elem<OutT>::widen(*p);
                    }
                }
                if constexpr (FUSED) {
#pragma unroll
                    for (int r = 0; r < 16; r++) v[r] += bias;
                }
                if constexpr (FUSED)
                    with_activation(g.act, g.act_param, [&](auto fn) {
#pragma unroll
                        for (int r = 0; r < 16; r++) v[r] = fn(v[r]);
                    });
#pragma unroll
                for (int r = 0; r < 16; r++) {
                    const int row = m0 + wm * WTM + i * 32 + acc_row(r, h);
                    if (row < g.M && col < g.N) {
                        out_t* p = C + (long long)row * g.ldc + col;
                        if constexpr (Elem<OutT>::BYTES == 4) *p = as_u32(v[r]);
                        else *p = (out_t)Elem<OutT>::narrow(v[r]);
                    }
                }
            }
        }
    };
    if (fused) store_all(std::true_type{});
    else store_all(std::false_type{});
}

// ---------------------------------------------------------------------------------------------
// Large-tile fast path for 16-bit inputs, B stored [K,N]: 256 x 256 x 64 tile, 8 waves (2 x 4, wave tile
// 128 x 64).  Requires M % 256 == 0, N % 256 == 0, K % 64 == 0 and 16-byte aligned rows.
//   * global -> LDS by the gfx950 direct load (global_load_lds_dwordx4): no staging registers, no
//     ds_write, no register transposes.  One wave-load moves 64 lanes x 16 B into 1 KiB of contiguous LDS,
//     so bank-conflict avoidance is done by choosing WHICH global chunk a lane fetches (XOR swizzle):
//       A tile [256 rows][128 B]: 16-byte chunk c of row r lives at chunk position c ^ ((r >> 1) & 7)
//       B tile [64 k][512 B]    : 16-byte chunk c of row k lives at chunk position c ^ ((k & 3) << 2)
//   * B fragments come out of the [k][n] tile with the transposing LDS read ds_read_b64_tr_b16: within
//     a 16-lane group, lane i receives element (i % 4) of the 8 bytes addressed by lane 4 m + i / 4,
//     for m = 0..3; lanes address B[k0 + j/4][n0 + 4 (j%4)] and receive B[k0 .. k0+3][n0 + i].
//   * the DMA is issued through inline asm: with the builtin the compiler orders every later LDS read
//     that may alias the destination behind s_waitcnt vmcnt(0), which serialises load latency and MFMA.
//     Completion is waited for explicitly (vmcnt(0) + workgroup barrier) before a stage is read.
typedef short s16x4 __attribute__((ext_vector_type(4)));

__device__ __forceinline__ void dma16_to_lds(const void* gptr, void* lds_dst_wave_uniform)
{
    uint32_t l = (uint32_t)(uintptr_t)((__attribute__((address_space(3))) void*)lds_dst_wave_uniform);
    l = __builtin_amdgcn_readfirstlane(l);
    // M0 carries the LDS base of the wave's 1 KiB destination; nothing else in these kernels uses M0
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, off" ::"s"(l), "v"(gptr));
}

// same for data that is read once per launch (a streamed weight matrix): non-temporal, so that it does not displace what the
// caches hold for reuse (a plain read loop reaches 6.0-6.2 TB/s on this part, a non-temporal one 6.9-7.0 TB/s)
__device__ __forceinline__ void dma16_to_lds_stream(const void* gptr, void* lds_dst_wave_uniform)
{
    uint32_t l = (uint32_t)(uintptr_t)((__attribute__((address_space(3))) void*)lds_dst_wave_uniform);
    l = __builtin_amdgcn_readfirstlane(l);
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, off nt" ::"s"(l), "v"(gptr));
}

// same, source = wave-uniform base (scalar register pair) + per-lane unsigned 32-bit byte offset, destination given as the LDS
// byte address
__device__ __forceinline__ void dma16_base(const void* base_uniform, uint32_t lane_off, uint32_t lds_dst)
{
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2" ::"s"(lds_dst), "v"(lane_off), "s"(base_uniform) : "memory");
}

// EDGE: M, N and K need not be multiples of the tile (N and K still multiples of 8): loads of rows / column chunks past the
// end are redirected to the last valid one (their products land in accumulator elements that are never stored), the stores
// are guarded, and in the last, partial K-tile every 16-byte chunk at or past K is fetched from a block of zeros instead.
__device__ __attribute__((aligned(16))) const uint32_t g_zero_chunk[4] = {0u, 0u, 0u, 0u};

// direct global -> LDS load with a full per-lane address (the form for lanes that do not share a base)
__device__ __forceinline__ void dma16_addr(const void* gptr, uint32_t lds_dst)
{
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, off" ::"s"(lds_dst), "v"(gptr) : "memory");
}

// TILE = 256: 8 waves (2 x 4), wave tile 128 x 64, one workgroup per CU.  TILE = 128: 4 waves (2 x 2), wave tile 64 x 64, two
// workgroups per CU (for problems with too few 256 x 256 tiles to occupy the chip).
// TRANSB: B is stored [N,K]; its tile is then loaded and read exactly like the A tile (rows of 128 bytes of K, b128 fragments).
// KSW = 2 (fp32, 64 x 64 tile, whole tiles): eight waves, two groups of four that take half of the k-steps of every K-tile each and are
// summed through LDS at the end (group 0 + group 1, a fixed order).  With about one such tile per CU the four-wave form runs one wave
// per SIMD, which has nothing to switch to while it issues loads or waits at the tile barrier (matrix pipe 69 % busy at 1024^3).
// Args = GemmRopeArgs (16-bit output): the leading columns of C are rotated as they are stored (launch.hpp's RopeEpilogue).
struct GemmRopeArgs : GemmArgs { RopeEpilogue rope; };
template <typename T, typename OutT, bool EDGE = false, int TILE = 256, bool TRANSB = false, int KSW = 1, typename Args = GemmArgs>
__global__ __launch_bounds__((TILE == 256 ? 512 : 256) * KSW, TILE == 256 ? 1 : 2) void gemm_dl_kernel(const Args g)
{
    constexpr int E = Elem<T>::PER16, EB = Elem<T>::BYTES;
    static_assert(TILE == 256 || TILE == 128 || TILE == 64, "tile edge");
    static_assert(KSW == 1 || (KSW == 2 && TILE == 64 && EB == 4 && !EDGE && !TRANSB), "the split form exists for the fp32 64 x 64 tile");
    constexpr int WM = 2, WN = TILE == 256 ? 4 : 2;
    constexpr int BM = TILE, BN = TILE, BK = 128 / EB;          // 128 bytes of K per tile row: 64 halves / 32 floats
    constexpr int WTM = BM / WM, WTN = BN / WN;
    constexpr int TM = WTM / 32, TN = WTN / 32;
    constexpr int BROW = BN * EB;                 // bytes of one k-row of the B tile
    constexpr int ABYTES = BM * 128, BBYTES = BK * BROW, STAGE = ABYTES + BBYTES;
    constexpr int NWAVE = WM * WN * KSW;
    constexpr int LA = BM / 8 / NWAVE, LB = LA;       // 1 KiB wave-loads per wave per tile (4 + 4; 2 + 2 for the 64 x 64 tile, 1 + 1 in its split form)
    constexpr int RPL = 1024 / BROW;              // k-rows of B per wave-load
    constexpr int LPR = 64 / RPL;                 // lanes (16-byte chunks) per B row
    static_assert(BK * BROW / 1024 == LB * NWAVE && BN / 8 == LB * NWAVE && (LA % 2 == 0 || KSW == 2), "B tile = as many wave-loads as the A tile");

    extern __shared__ __attribute__((aligned(1024))) unsigned char smem[];

    const int t = threadIdx.x;
    const int lane = t & 63, wave = t >> 6;                 // wave: index among all waves (partition of the loads)
    const int l32 = lane & 31, h = lane >> 5;
    const int kgrp = KSW == 1 ? 0 : wave / (WM * WN);      // k-step group
    const int wq = KSW == 1 ? wave : wave % (WM * WN);
    const int wm = wq / WN, wn = wq % WN;
    int tile_m, tile_n;
    tile_of_block(blockIdx.x, gridDim.x, g.tiles_m, g.tiles_n, tile_m, tile_n);
    const int m0 = tile_m * BM, n0 = tile_n * BN;
    const long long bz = blockIdx.z;                                         // batch index (strides in elements)
    const unsigned char* __restrict__ A = (const unsigned char*)g.A + bz * g.sA * EB;
    const unsigned char* __restrict__ B = batch_b<EB>(g, bz);

    // Chunk swizzle of the B tile (which 16-byte chunk position of its LDS row a chunk of k-row `row` occupies):
    //   16-bit: c ^ ((row & 3) << 2)  -- the four rows one transposing read touches go to different bank groups (rows of 256
    //           bytes and more; 128-byte rows, which alternate between the bank halves by themselves: c ^ (((row >> 1) & 1) << 2));
    //   fp32:   c ^ (((row >> 2) & 1) << 3)  -- the two lane halves of a b32 fragment read (rows 4 apart) use different bank halves.
    auto b_swz = [](int row) -> int {
        return E == 8 ? (BROW >= 256 ? ((row & 3) << 2) : (((row >> 1) & 1) << 2)) : (((row >> 2) & 1) << 3);
    };

    // Sources of this wave's loads: a wave-uniform base (scalar registers, advanced per tile by scalar adds) plus a per-lane
    // 32-bit byte offset that never changes, so issuing a load costs no vector instruction.  Wave-load w = 4 wave + i covers
    // A rows 8w .. 8w+7 resp. B k-rows RPL w .. RPL w + RPL-1.
    const int wave_s = __builtin_amdgcn_readfirstlane(wave);
    const uint32_t lds0 = (uint32_t)(uintptr_t)((__attribute__((address_space(3))) void*)smem);
    uint32_t a_lane_off[EDGE ? LA : 2], b_lane_off[LB];
#pragma unroll
    for (int par = 0; par < 2; par++) {
        const int ra = lane >> 3, pos_a = lane & 7;           // row inside the wave-load, 16-byte chunk
        // (the swizzle of a row is ((row >> 1) & 7) with row = 8 (LA wave + i) + ra: only the parity of LA wave + i enters)
        if constexpr (!EDGE) a_lane_off[par] = (uint32_t)(ra * g.lda + (pos_a ^ ((4 * par + (ra >> 1)) & 7)) * E) * (uint32_t)EB;
    }
#pragma unroll
    for (int i = 0; i < LB; i++) {
        if constexpr (TRANSB) {
            const int rn = lane >> 3, pos = lane & 7;             // like A: wave-load w covers tile rows (n) 8w .. 8w+7
            int row = 8 * (LB * wave + i) + rn;
            const int sw = (row >> 1) & 7;
            if constexpr (EDGE) row = min(row, g.N - 1 - n0);
            else row = rn;                                        // relative to the wave-load's first row (scalar base)
            b_lane_off[i] = (uint32_t)(row * g.ldb + (pos ^ sw) * E) * (uint32_t)EB;
        } else {
            const int rb = lane / LPR, pos_b = lane % LPR;
            int chunk = pos_b ^ b_swz(RPL * (LB * wave + i) + rb);
            if constexpr (EDGE) chunk = min(chunk, (g.N - n0) / E - 1);      // N % E == 0 and n0 < N: at least one chunk
            b_lane_off[i] = (uint32_t)(rb * g.ldb + chunk * E) * (uint32_t)EB;
        }
    }
    if constexpr (EDGE) {
#pragma unroll
        for (int i = 0; i < LA; i++) {
            const int ra = lane >> 3, pos_a = lane & 7;
            const int row = min(8 * (LA * wave + i) + ra, g.M - 1 - m0);      // source row inside the tile (m0 < M)
            a_lane_off[i] = (uint32_t)(row * g.lda + (pos_a ^ ((4 * (i & 1) + (ra >> 1)) & 7)) * E) * (uint32_t)EB;
        }
    }
    // (EDGE: the A offsets are relative to the tile's first row, since a clamped row may lie before the wave's own rows)
    const unsigned char* a_base = A + (long long)(m0 + (EDGE ? 0 : 8 * LA * wave_s)) * g.lda * EB;
    const unsigned char* b_base = TRANSB ? B + (long long)(n0 + (EDGE ? 0 : 8 * LB * wave_s)) * g.ldb * EB
                                         : B + ((long long)(RPL * LB * wave_s) * g.ldb + n0) * EB;
    // bytes between consecutive wave-loads
    const long long a_step = 8LL * g.lda * EB, b_step = TRANSB ? (EDGE ? 0LL : 8LL * g.ldb * EB) : (long long)RPL * g.ldb * EB;
    const int KT = (g.K + BK - 1) / BK;
    const int ktail = EDGE ? g.K - (KT - 1) * BK : BK;                        // k-rows of the last tile (BK when K % BK == 0)
    auto issue_loads = [&](int kt, int stage) {
        const uint32_t as = lds0 + stage * STAGE + wave_s * (LA * 1024);
        const uint32_t bs = lds0 + stage * STAGE + ABYTES + wave_s * (LB * 1024);
        const unsigned char* a_src = a_base + (long long)kt * 128;
        const unsigned char* b_src = TRANSB ? b_base + (long long)kt * 128 : b_base + (long long)kt * BK * g.ldb * EB;
        if constexpr (EDGE) {
            if (kt == KT - 1 && ktail < BK) {
                // partial last tile: chunks at or past K come from the zero block (a product with zero adds nothing)
#pragma unroll
                for (int i = 0; i < LA; i++) {
                    const int ra = lane >> 3, pos_a = lane & 7;
                    const int chunk = pos_a ^ ((4 * (i & 1) + (ra >> 1)) & 7);               // the chunk this lane fetches
                    const void* src = chunk * E < ktail ? (const void*)(a_src + a_lane_off[i]) : (const void*)g_zero_chunk;
                    dma16_addr(src, as + i * 1024);
                }
#pragma unroll
                for (int i = 0; i < LB; i++) {
                    bool valid;
                    if constexpr (TRANSB) {
                        const int rn = lane >> 3, pos = lane & 7;
                        valid = (pos ^ (((8 * (LB * wave + i) + rn) >> 1) & 7)) * E < ktail;  // the chunk of K this lane fetches
                    } else {
                        valid = RPL * (LB * wave + i) + lane / LPR < ktail;                  // k-row inside the tile
                    }
                    const void* src = valid ? (const void*)(b_src + i * b_step + b_lane_off[i]) : (const void*)g_zero_chunk;
                    dma16_addr(src, bs + i * 1024);
                }
                return;
            }
        }
#pragma unroll
        for (int i = 0; i < LA; i++) {
            if constexpr (EDGE) dma16_base(a_src, a_lane_off[i], as + i * 1024);
            else dma16_base(a_src + i * a_step, a_lane_off[LA % 2 == 0 ? (i & 1) : ((wave + i) & 1)], as + i * 1024);
        }
#pragma unroll
        for (int i = 0; i < LB; i++) dma16_base(b_src + i * b_step, b_lane_off[i], bs + i * 1024);
    };

    // per-lane LDS read offsets
    int a_off[TM], a_sw[TM];
#pragma unroll
    for (int i = 0; i < TM; i++) {
        int row = wm * WTM + i * 32 + l32;
        a_off[i] = row * 128;
        a_sw[i] = ((row >> 1) & 7) ^ (KSW == 2 ? 4 * kgrp : 0);      // group g reads k-steps 2 g and 2 g + 1: chunk (2 (2 g + u) + h) ^ sw
    }
    // 16-bit B fragments (transposing reads): lane j of a 16-lane group addresses k-row (base + j / 4), 8 bytes
    const int jl = lane & 15;
    const int b_rowl = 8 * h + (jl >> 2);                     // + 16 s + 4 q
    const int b_half = (jl & 1) * 8;
    int b_chunk[TN];
#pragma unroll
    for (int j = 0; j < TN; j++) b_chunk[j] = (wn * WTN + j * 32 + 16 * ((lane >> 4) & 1) + 4 * (jl & 3)) >> 3;
    // fp32 B fragments (b32 reads): lane (h, l32) reads column l32 of k-rows 8 s + 4 h + (0..3); (row >> 2) & 1 == h there
    int b_col32[TN];
#pragma unroll
    for (int j = 0; j < TN; j++) {
        const int col = wn * WTN + j * 32 + l32;
        b_col32[j] = (((col >> 2) ^ (h << 3)) << 4) + (col & 3) * 4 + 4 * h * BROW + (KSW == 2 ? 16 * kgrp * BROW : 0);
    }

    int bt_off[TN], bt_sw[TN];                               // B stored [N,K]: like the A fragments
#pragma unroll
    for (int j = 0; j < TN; j++) {
        int row = wn * WTN + j * 32 + l32;
        bt_off[j] = row * 128;
        bt_sw[j] = (row >> 1) & 7;
    }

    auto read_frags = [&](const unsigned char* as, const unsigned char* bs, int s, u32x4 (&fa)[TM], u32x4 (&fb)[TN]) {
#pragma unroll
        for (int i = 0; i < TM; i++) fa[i] = *(const u32x4*)(as + a_off[i] + (((2 * s + h) ^ a_sw[i]) << 4));
#pragma unroll
        for (int j = 0; j < TN; j++) {
            if constexpr (TRANSB) {
                fb[j] = *(const u32x4*)(bs + bt_off[j] + (((2 * s + h) ^ bt_sw[j]) << 4));
            } else if constexpr (E == 4) {
#pragma unroll
                for (int q = 0; q < 4; q++) fb[j][q] = *(const uint32_t*)(bs + (8 * s + q) * BROW + b_col32[j]);
            } else {
#pragma unroll
                for (int q = 0; q < 2; q++) {
                    int row = 16 * s + 4 * q + b_rowl;
                    int pos = b_chunk[j] ^ b_swz(row);
                    s16x4 v = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
                        (__attribute__((address_space(3))) s16x4*)(bs + row * BROW + pos * 16 + b_half));
                    u32x2 w = __builtin_bit_cast(u32x2, v);
                    fb[j][2 * q] = w[0];
                    fb[j][2 * q + 1] = w[1];
                }
            }
        }
    };

    f32x16 acc[TM][TN];
#pragma unroll
    for (int i = 0; i < TM; i++)
#pragma unroll
        for (int j = 0; j < TN; j++)
#pragma unroll
            for (int r = 0; r < 16; r++) acc[i][j][r] = 0.0f;

    issue_loads(0, 0);
    constexpr bool ROPE = std::is_same<Args, GemmRopeArgs>::value;
    static_assert(!ROPE || (TM == 1 && TN == 1), "one block of C to a wave");
    float turn_cos[ROPE ? 16 : 1], turn_sin[ROPE ? 16 : 1];      // (loaded here, they arrive with the first tile)
    if constexpr (ROPE) {
        const RopeEpilogue& rope = g.rope;
        const int col = n0 + wn * WTN + l32, half = rope.head_dim >> 1;
        const int pair = col < rope.cols ? (col % rope.head_dim) >> 1 : 0;
        const long long first = (long long)rope.start_position * half + pair;
        if (rope.seq_len == 1) {                                 // every row at one position, as in a decode step: without sixteen divisions, 0.7 us a launch
            const float c = rope.cosc[first], s = rope.sinc[first];
#pragma unroll
            for (int r = 0; r < 16; r++) { turn_cos[r] = c; turn_sin[r] = s; }
        } else {
#pragma unroll
            for (int r = 0; r < 16; r++) {                       // (rows past the end repeat the last one)
                const long long at = first + (long long)(min(m0 + wm * WTM + acc_row(r, h), g.M - 1) % rope.seq_len) * half;
                turn_cos[r] = rope.cosc[at]; turn_sin[r] = rope.sinc[at];
            }
        }
    }
    __builtin_amdgcn_s_waitcnt(0);
    __syncthreads();
    if constexpr (ROPE) {
#pragma unroll
        for (int r = 0; r < 16; r++) asm volatile("" : "+v"(turn_cos[r]), "+v"(turn_sin[r]));
    }

    // Software pipeline: the fragments of k-step s+1 are read from LDS before the MFMAs of step s are issued, so the
    // LDS latency runs under 8 MFMAs; the barrier that publishes tile kt+1 sits before the MFMAs of the last step, and the
    // first fragments of tile kt+1 are read there too.  sched_barrier pins this order (the scheduler otherwise sinks
    // the reads next to their use to save registers, which exposes the LDS latency every few MFMAs).
    u32x4 fa[2][TM], fb[2][TN];
    read_frags(smem, smem + ABYTES, 0, fa[0], fb[0]);
    for (int kt = 0; kt < KT; kt++) {
        const int stage = kt & 1;
        const unsigned char* as = smem + stage * STAGE;
        const unsigned char* bs = as + ABYTES;
        // the other stage was last read before the barrier inside the previous iteration
        if (kt + 1 < KT) issue_loads(kt + 1, stage ^ 1);
#pragma unroll
        for (int s = 0; s < 4 / KSW; s++) {        // (split form: the group's two k-steps; the fragment bases carry the group's offset)
            if (s < 4 / KSW - 1) {
                read_frags(as, bs, s + 1, fa[(s + 1) & 1], fb[(s + 1) & 1]);
            } else {
                __builtin_amdgcn_s_waitcnt(0);      // this wave's DMA has landed and its LDS reads of this tile are done ...
                __syncthreads();                    // ... and so have everyone else's
                if (kt + 1 < KT) {
                    const unsigned char* an = smem + (stage ^ 1) * STAGE;
                    read_frags(an, an + ABYTES, 0, fa[0], fb[0]);
                }
            }
#pragma unroll
            for (int i = 0; i < TM; i++)
#pragma unroll
                for (int j = 0; j < TN; j++) Mma32<T>::run(acc[i][j], fa[s & 1][i], fb[s & 1][j]);
            // the next step's fragment reads go behind the first half of this step's MFMAs (two each), so the matrix pipe does
            // not wait behind a burst of reads and the last read still has half a step to complete
            constexpr int NMF = TM * TN * (E == 4 ? 4 : 1);             // MFMA instructions per step
            spread_schedule<NMF / 2, TM + (TRANSB ? 1 : E == 4 ? 4 : 2) * TN, 0, 0>();
            __builtin_amdgcn_sched_group_barrier(0x008, NMF - NMF / 2, 0);
            __builtin_amdgcn_sched_barrier(0);
        }
    }

    if constexpr (KSW == 2) {
        // nobody reads the tile ring after the last barrier: group 1 parks its accumulators there, group 0 adds them to its own
        float* red = (float*)smem;
        if (kgrp == 1) {
#pragma unroll
            for (int i = 0; i < TM; i++)
#pragma unroll
                for (int j = 0; j < TN; j++)
#pragma unroll
                    for (int r = 0; r < 16; r++) red[(((wq * TM + i) * TN + j) * 16 + r) * 64 + lane] = acc[i][j][r];
        }
        __syncthreads();
        if (kgrp == 1) return;
#pragma unroll
        for (int i = 0; i < TM; i++)
#pragma unroll
            for (int j = 0; j < TN; j++)
#pragma unroll
                for (int r = 0; r < 16; r++) acc[i][j][r] += red[(((wq * TM + i) * TN + j) * 16 + r) * 64 + lane];
    }
    typedef typename Raw<OutT>::type out_t;
    out_t* __restrict__ C = (out_t*)g.C + bz * g.sC;
    const bool fused = g.bias != nullptr || g.act != 0;
    if (Elem<OutT>::BYTES == 4 && (g.alpha != 1.0f || g.beta != 0.0f)) {
        // C = act(alpha A B + beta C + bias), fp32 output only: the uncommon form, kept apart so the plain stores below stay lean
#pragma unroll 1
        for (int ij = 0; ij < TM * TN; ij++) {
            const int i = ij / TN, j = ij - i * TN;
            const int col = n0 + wn * WTN + j * 32 + l32;
            if (EDGE && col >= (g.c_cols > 0 ? g.c_cols : g.N)) continue;
            const float bias = g.bias ? g.bias[col] : 0.0f;
            f32x16 v = acc[0][0];
#pragma unroll
            for (int ii = 0; ii < TM; ii++)
#pragma unroll
                for (int jj = 0; jj < TN; jj++) if (ii == i && jj == j) v = acc[ii][jj];
#pragma unroll
            for (int r = 0; r < 16; r++) {
                const int row = m0 + wm * WTM + i * 32 + acc_row(r, h);
                if (EDGE && row >= g.M) continue;
                out_t* p = C + (long long)row * g.ldc + col;
                float x = g.alpha * v[r];
                if (g.beta != 0.0f) {
                    if constexpr (Elem<OutT>::BYTES == 4) x += g.beta * as_f32(*p);
                    else x += g.beta * Elem<OutT>::widen(*p);
                }
                if (fused) x = apply_activation(x + bias, g.act, g.act_param);
                if constexpr (Elem<OutT>::BYTES == 4) *p = as_u32(x);
                else *p = (out_t)Elem<OutT>::narrow(x);
            }
        }
        return;
    }
#pragma unroll
    for (int i = 0; i < TM; i++)
#pragma unroll
        for (int j = 0; j < TN; j++) {
            const int col = n0 + wn * WTN + j * 32 + l32;
            const bool col_ok = !EDGE || col < (g.c_cols > 0 ? g.c_cols : g.N);
            if constexpr (ROPE) {
                // the pair is rounded to the output type before it is rotated, as a product followed by the rotation kernel does it; its other
                // half is in the neighbouring lane
                const bool turn = col < g.rope.cols, odd = col & 1;
#pragma unroll
                for (int r = 0; r < 16; r++) {
                    const float mine = Elem<OutT>::widen(Elem<OutT>::narrow(acc[i][j][r]));
                    const float other = as_f32((uint32_t)__builtin_amdgcn_update_dpp(0, (int)as_u32(mine), 0xB1, 0xF, 0xF, true));      // quad_perm 1, 0, 3, 2
                    float even_out, odd_out;
                    rope_rotate(odd ? other : mine, odd ? mine : other, turn_cos[r], turn_sin[r], even_out, odd_out);
                    acc[i][j][r] = turn ? (odd ? odd_out : even_out) : mine;
                }
            }
            if (fused) {                                  // bias and / or activation folded into the store
                const float bias = (g.bias && col_ok) ? g.bias[col] : 0.0f;
#pragma unroll
                for (int r = 0; r < 16; r++) acc[i][j][r] += bias;
                with_activation(g.act, g.act_param, [&](auto fn) {
#pragma unroll
                    for (int r = 0; r < 16; r++) acc[i][j][r] = fn(acc[i][j][r]);
                });
            }
#pragma unroll
            for (int r = 0; r < 16; r++) {
                const int row = m0 + wm * WTM + i * 32 + acc_row(r, h);
                out_t* p = C + (long long)row * g.ldc + col;
                out_t v;
                if constexpr (Elem<OutT>::BYTES == 4) v = as_u32(acc[i][j][r]);
                else v = (out_t)Elem<OutT>::narrow(acc[i][j][r]);
                if (col_ok && (!EDGE || row < g.M)) *p = v;
            }
        }
}

template <typename T, typename OutT, bool EDGE = false, int TILE = 256, bool TRANSB = false, int KSW = 1, typename Args = GemmArgs>
static hipError_t launch_gemm_dl(Args g, int batch, hipStream_t stream)
{
    auto kern = gemm_dl_kernel<T, OutT, EDGE, TILE, TRANSB, KSW, Args>;
    constexpr int smem = 2 * (TILE * 128 + 128 * TILE);         // A tile + B tile (128 bytes of K each), two stages
    static unsigned long long attr_done = 0;
    if (hipError_t e = ensure_dynamic_smem((const void*)kern, smem, &attr_done)) return e;
    g.tiles_m = (g.M + TILE - 1) / TILE;
    g.tiles_n = (g.N + TILE - 1) / TILE;
    hipLaunchKernelGGL(kern, dim3((unsigned)(g.tiles_m * g.tiles_n), 1, (unsigned)batch), dim3((TILE == 256 ? 512 : 256) * KSW), smem, stream, g);
    return hipGetLastError();
}

// ---------------------------------------------------------------------------------------------
// 256 x 256 x 64 direct-to-LDS kernel for 16-bit inputs on v_mfma_f32_16x16x32 (the form the large exact-fit problems take:
// K % 64 == 0, B stored [K,N]; M and N may be ragged, N in whole 16-byte chunks: the rows of A past M and the chunks of B past N are
// clamped loads of the last ones, whose products are never stored).  Same tile, loads and LDS layout as gemm_dl_kernel<.., 256>; what
// differs is the matrix instruction.  Under load this part runs at the clock its power limit allows, and per multiply-add the
// 16 x 16 x 32 instruction moves 20 % fewer register bytes than 32 x 32 x 16 (half the accumulator traffic, twice the
// operand traffic): with random fp16 operands and nothing else running it sustains 1.71 PFLOP/s against 1.52, and this kernel
// 7-10 % more than the 32 x 32 x 16 one on the same box.
//   * wave tile 128 x 64 = 8 x 4 blocks of 16 x 16, 128 accumulator registers; per 32 k: 8 A fragments (ds_read_b128: row
//     16 i + lane % 16, 16-byte chunk lane / 16) and 4 B fragments (two transposing reads each), 32 MFMAs of 16 cycles.
//   * a K-tile is four half-steps of 16 MFMAs (rows 64 hs .. 64 hs + 63 of the wave tile, k32-step s2); the fragments of the
//     next half-step are read one LDS instruction behind each MFMA, the barrier that publishes the next tile sits before the
//     last half-step, whose MFMAs cover the twelve reads of the next tile's first fragments.
//   * the B fragment is the MFMA's first operand, so the accumulators hold C transposed: a lane owns 4 consecutive columns of
//     one row, packs them to 8 bytes, and the wave stages its rows through its 8 KiB of the dead LDS stage so that C leaves as
//     whole 128-byte lines (the 32 x 32 kernel stores 2 bytes per lane and instruction).
//   * MFMA order: one operand changes between consecutive instructions (row-block outer, column-block inner, snaked).
typedef float f32x4_acc __attribute__((ext_vector_type(4)));
template <typename T> struct Mma16;
template <> struct Mma16<f16_t> {
    static __device__ __forceinline__ void run(f32x4_acc& acc, const u32x4& a, const u32x4& b)
    { acc = __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8, a), __builtin_bit_cast(f16x8, b), acc, 0, 0, 0); }
};
template <> struct Mma16<bf16_t> {
    static __device__ __forceinline__ void run(f32x4_acc& acc, const u32x4& a, const u32x4& b)
    { acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), acc, 0, 0, 0); }
};

// TJ = 16-column blocks per wave: the tile is 256 x (64 TJ) -- 256 x 256, 256 x 192 or 256 x 128 -- so that problems whose 256 x 256
// tiles would leave CUs idle in the last round (4096 x 3072: 192 tiles on 256 CUs) get a tile count that fills them.  The B tile
// keeps its 512-byte LDS rows for every TJ (the chunk swizzle needs a power-of-two row); lanes whose swizzled chunk lies past
// the tile's columns fetch a valid chunk again and park it in a position that no fragment read touches.
// HALF: the 128 x 128 tile (TJ = 2): wave tile 64 x 32, B k-rows of 256 bytes, for problems that give fewer than a chip of wider
// tiles (2048^2, 1024 x 4096).  A K-tile is only 256 MFMA cycles per wave here, far less than a memory round trip, so the tile ring
// has four 32 KB stages and is filled three K-tiles ahead (loads complete in issue order: "tile kt+1 has landed" is a count of
// younger loads).
#define DL16_HALF_STAGES 4
// NTS: C is written with non-temporal stores (a compile-time switch: as a run-time branch the two stores are merged by the compiler
// and the hint is lost).
// CUT: N is not a multiple of the tile width (an instance of its own: with the clamps and tests in all of them whole tiles took longer,
// 8192 x 768 x 768 17.2 -> 17.5 us).
// On a page of its own: a launch of one or two rounds begins by fetching up to 70 KB of code, and where that lay within its pages moved an
// attention layer of 8 x 512 x 768, three such launches in a row, by 1.7 % (us, the QKV and output projections at 0x100 and 0xc00 of a page 53.1,
// at 0x400 and 0x800 53.3, at 0x900 and 0xd00 53.6, both at 0 52.7) with every instance added to this file.
template <typename T, typename OutT, int TJ = 4, bool HALF = false, bool NTS = false, int HS = DL16_HALF_STAGES, bool CUT = false>
__global__ __launch_bounds__(512, 1) __attribute__((aligned(4096))) void gemm_dl16_kernel(const GemmArgs g)
{
    static_assert(!HALF || TJ == 2, "the 128-row tile is built for 128 columns");
    constexpr int E = 8, EB = 2;
    constexpr int WN = 4;
    constexpr int BM = HALF ? 128 : 256, BN = 64 * TJ, BK = 64;
    constexpr int WTM = BM / 2, WTN = 16 * TJ;
    constexpr int TI = WTM / 16;                  // 16 x 16 blocks of the wave tile: TI x TJ
    // LDS pitch of a B k-row (16 or 32 chunk positions): 512 bytes, or 256 for the 128-column tiles (with 512-byte rows the 256 x 128
    // tile fetched 256 columns of B per k-row for the 128 it uses: 6-8 % slower on every shape that takes it)
    constexpr int BROW = ((HALF || TJ == 2) ? 128 : 256) * EB;
    constexpr int BCH = BN / E;                   // 16-byte chunks of a k-row that hold tile columns
    constexpr int ABYTES = BM * 128, BBYTES = BK * BROW, STAGE = ABYTES + BBYTES;
    constexpr int LA = BM / 64, LB = BK * BROW / 8192, RPL = 1024 / BROW, LPR = BROW / 16;
    constexpr int OB = Elem<OutT>::BYTES;

    extern __shared__ __attribute__((aligned(1024))) unsigned char smem[];
    const int t = threadIdx.x;
    const int lane = t & 63, wave = t >> 6;
    const int l16 = lane & 15, g4 = lane >> 4;
    const int wm = wave / WN, wn = wave % WN;
    int tile_m, tile_n;
    tile_of_block(blockIdx.x, gridDim.x, g.tiles_m, g.tiles_n, tile_m, tile_n);
    const int m0 = tile_m * BM, n0 = tile_n * BN;
    const long long bz = blockIdx.z;
    const unsigned char* __restrict__ A = (const unsigned char*)g.A + bz * g.sA * EB;
    const unsigned char* __restrict__ B = batch_b<EB>(g, bz);

    // Chunk swizzle of a B k-row (position of 16-byte chunk c in its 512-byte LDS row: c ^ b_swz(row)): the four rows one
    // transposing read touches go to different bank groups, and rows 8 apart -- the two 16-lane groups that share a cycle of
    // that read -- are moved 32 bytes apart.
    auto b_swz = [](int row) -> int { return ((row & 3) << 2) | (((row >> 3) & 1) << 1); };
    const int wave_s = __builtin_amdgcn_readfirstlane(wave);
    const uint32_t lds0 = (uint32_t)(uintptr_t)((__attribute__((address_space(3))) void*)smem);
    // A rows past M (the last tile row of a ragged M) are clamped to row M - 1 and B chunks past N to the last one: valid loads whose
    // products are never stored
    uint32_t a_lane_off[LA], b_lane_off[LB];
#pragma unroll
    for (int i = 0; i < LA; i++) {
        const int ra = lane >> 3, pos_a = lane & 7;
        const int row = min(m0 + 8 * (LA * wave + i) + ra, g.M - 1) - m0;        // relative to the tile's first row, >= 0
        a_lane_off[i] = (uint32_t)(row * g.lda + (pos_a ^ ((4 * (i & 1) + (ra >> 1)) & 7)) * E) * (uint32_t)EB;
    }
#pragma unroll
    for (int i = 0; i < LB; i++) {
        const int rb = lane / LPR, pos_b = lane % LPR;
        int chunk = pos_b ^ b_swz(RPL * (LB * wave + i) + rb);
        if (chunk >= BCH) chunk -= LPR - BCH >= BCH ? BCH : LPR - BCH;    // a valid chunk again (its LDS position is never read)
        if constexpr (CUT) chunk = min(chunk, (g.N - n0) / E - 1);
        b_lane_off[i] = (uint32_t)(rb * g.ldb + chunk * E) * (uint32_t)EB;
    }
    const unsigned char* a_base = A + (long long)m0 * g.lda * EB;
    const unsigned char* b_base = B + ((long long)(RPL * LB * wave_s) * g.ldb + n0) * EB;
    const long long b_step = (long long)RPL * g.ldb * EB;
    // (the instances that take K ranges: fp32 partials)
    const int KT = (OB == 4 && (HALF || TJ == 4) && g.k_total ? min(g.K, g.k_total - (int)bz * g.K) : g.K) / BK;
    auto issue_loads = [&](int kt, int stage) {
        const uint32_t as = lds0 + stage * STAGE + wave_s * (LA * 1024);
        const uint32_t bs = lds0 + stage * STAGE + ABYTES + wave_s * (LB * 1024);
        const unsigned char* a_src = a_base + (long long)kt * 128;
        const unsigned char* b_src = b_base + (long long)kt * BK * g.ldb * EB;
#pragma unroll
        for (int i = 0; i < LA; i++) dma16_base(a_src, a_lane_off[i], as + i * 1024);
#pragma unroll
        for (int i = 0; i < LB; i++) dma16_base(b_src + i * b_step, b_lane_off[i], bs + i * 1024);
    };

    // A fragment of 16-row block i, k32-step s2: row 16 i + l16, chunk 4 s2 + g4, swizzled by (row >> 1) & 7 = (l16 >> 1) & 7
    const int a_row0 = (wm * WTM + l16) * 128;
    const int a_sw = (l16 >> 1) & 7;
    // B fragment of 16-column block j, k32-step s2: two transposing reads (q = 0, 1); the lane addresses k-row
    // 32 s2 + 8 g4 + 4 q + l16 / 4 and the 8 bytes at column 16 j + 4 (l16 % 4), and receives k 8 g4 + 4 q .. + 3 of column 16 j + l16
    const int b_rowl = 8 * g4 + (l16 >> 2);
    const int b_half = (l16 & 1) * 8;
    const int b_chunk0 = wn * (2 * TJ) + ((l16 & 3) >> 1);      // + 2 j

    auto read_a = [&](const unsigned char* as, int s2, int i, u32x4& f) {
        f = *(const u32x4*)(as + a_row0 + i * 2048 + (((4 * s2 + g4) ^ a_sw) << 4));
    };
    auto read_b = [&](const unsigned char* bs, int s2, int j, u32x4& f) {
#pragma unroll
        for (int q = 0; q < 2; q++) {
            const int row = 32 * s2 + 4 * q + b_rowl;
            const int pos = (b_chunk0 + 2 * j) ^ b_swz(row);
            s16x4 v = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
                (__attribute__((address_space(3))) s16x4*)(bs + row * BROW + pos * 16 + b_half));
            u32x2 w = __builtin_bit_cast(u32x2, v);
            f[2 * q] = w[0];
            f[2 * q + 1] = w[1];
        }
    };

    f32x4_acc acc[TI][TJ];
#pragma unroll
    for (int i = 0; i < TI; i++)
#pragma unroll
        for (int j = 0; j < TJ; j++) acc[i][j] = f32x4_acc{0.0f, 0.0f, 0.0f, 0.0f};

    constexpr int NS = HALF ? HS : 2;
    // wait until at most `tiles` of this wave's tile loads (LA + LB instructions each) are outstanding, and for its LDS reads
    auto wait_tiles = [&](int tiles) {
        static_assert(!HALF || (LA + LB == 4 && NS <= 4), "the wait counts below are for four loads per tile and a four-stage ring");
        if (tiles <= 0) asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");
        else if (tiles == 1) asm volatile("s_waitcnt vmcnt(4) lgkmcnt(0)" ::: "memory");
        else asm volatile("s_waitcnt vmcnt(8) lgkmcnt(0)" ::: "memory");
    };
    if constexpr (HALF) {
        for (int kt = 0; kt < NS - 1 && kt < KT; kt++) issue_loads(kt, kt);
        wait_tiles(min(KT - 1, NS - 2));
    } else {
        issue_loads(0, 0);
        __builtin_amdgcn_s_waitcnt(0);
    }
    __syncthreads();

    // fa[p]: the four A fragments of half-step parity p; fb[p]: the four B fragments of k32-step parity p
    u32x4 fa[2][4], fb[2][TJ];
#pragma unroll
    for (int i = 0; i < 4; i++) read_a(smem, 0, i, fa[0][i]);
#pragma unroll
    for (int j = 0; j < TJ; j++) read_b(smem + ABYTES, 0, j, fb[0][j]);

    if constexpr (HALF) {
        // two steps per K-tile (one k32-step each, the whole 64-row wave tile): 8 MFMAs and 8 LDS reads per step
        int stage = 0;
        for (int kt = 0; kt < KT; kt++) {
            const int next = stage + 1 == NS ? 0 : stage + 1;
            const unsigned char* as = smem + stage * STAGE;
            const unsigned char* bs = as + ABYTES;
            const unsigned char* an = smem + next * STAGE;
            // the stage of tile kt-1 was last read before the barrier inside the previous iteration
            if (kt + NS - 1 < KT) issue_loads(kt + NS - 1, stage == 0 ? NS - 1 : stage - 1);
#pragma unroll
            for (int s2 = 0; s2 < 2; s2++) {
                if (s2 == 0) {
#pragma unroll
                    for (int i = 0; i < 4; i++) read_a(as, 1, i, fa[1][i]);
#pragma unroll
                    for (int j = 0; j < TJ; j++) read_b(bs, 1, j, fb[1][j]);
                } else {
                    wait_tiles(min(KT - 2 - kt, NS - 2));   // this wave's part of tile kt+1 has landed (younger tiles may be in flight), its LDS reads of tile kt are done ...
                    __syncthreads();                        // ... and so have everyone else's
                    if (kt + 1 < KT) {
#pragma unroll
                        for (int i = 0; i < 4; i++) read_a(an, 0, i, fa[0][i]);
#pragma unroll
                        for (int j = 0; j < TJ; j++) read_b(an + ABYTES, 0, j, fb[0][j]);
                    }
                }
#pragma unroll
                for (int i = 0; i < 4; i++)
#pragma unroll
                    for (int jj = 0; jj < TJ; jj++) {
                        const int j = (i & 1) ? TJ - 1 - jj : jj;
                        Mma16<T>::run(acc[i][j], fb[s2][j], fa[s2][i]);
                    }
                constexpr int NM = 4 * TJ, RR = 4 + 2 * TJ;
                spread_schedule<RR, RR, 0, 0>();
                if (NM > RR) __builtin_amdgcn_sched_group_barrier(0x008, NM - RR, 0);
                __builtin_amdgcn_sched_barrier(0);
            }
            stage = next;
        }
    } else {
    for (int kt = 0; kt < KT; kt++) {
            const int stage = kt & 1;
            const unsigned char* as = smem + stage * STAGE;
            const unsigned char* bs = as + ABYTES;
            const unsigned char* an = smem + (stage ^ 1) * STAGE;
            // the other stage was last read before the barrier inside the previous iteration
            if (kt + 1 < KT) issue_loads(kt + 1, stage ^ 1);
    #pragma unroll
            for (int u = 0; u < 4; u++) {              // half-step u = 2 s2 + hs
                const int s2 = u >> 1, hs = u & 1;
                if (u == 0) {
    #pragma unroll
                    for (int i = 0; i < 4; i++) read_a(as, 0, 4 + i, fa[1][i]);
                    read_b(bs, 1, 0, fb[1][0]); read_b(bs, 1, 1, fb[1][1]);
                } else if (u == 1) {
    #pragma unroll
                    for (int i = 0; i < 4; i++) read_a(as, 1, i, fa[0][i]);
    #pragma unroll
                    for (int j = 2; j < TJ; j++) read_b(bs, 1, j, fb[1][j]);
                } else if (u == 2) {
    #pragma unroll
                    for (int i = 0; i < 4; i++) read_a(as, 1, 4 + i, fa[1][i]);
                } else {
                    __builtin_amdgcn_s_waitcnt(0);      // this wave's DMA has landed and its LDS reads of this tile are done ...
                    __syncthreads();                    // ... and so have everyone else's
                    if (kt + 1 < KT) {
    #pragma unroll
                        for (int i = 0; i < 4; i++) read_a(an, 0, i, fa[0][i]);
    #pragma unroll
                        for (int j = 0; j < TJ; j++) read_b(an + ABYTES, 0, j, fb[0][j]);
                    }
                }
    #pragma unroll
                for (int i = 0; i < 4; i++)
    #pragma unroll
                    for (int jj = 0; jj < TJ; jj++) {
                        const int j = (i & 1) ? TJ - 1 - jj : jj;
                        Mma16<T>::run(acc[4 * hs + i][j], fb[s2][j], fa[hs][i]);
                    }
                // one LDS read behind each of the first MFMAs, the remaining MFMAs after the reads have been issued
                constexpr int NM = 4 * TJ;                                   // MFMAs per half-step
                constexpr int R0 = 8, R1 = 4 + 2 * (TJ - 2), R2 = 4, R3 = 4 + 2 * TJ;      // LDS reads of the four half-steps
                if (u == 0) { spread_schedule<R0, R0, 0, 0>(); __builtin_amdgcn_sched_group_barrier(0x008, NM - R0, 0); }
                else if (u == 1) { spread_schedule<R1, R1, 0, 0>(); __builtin_amdgcn_sched_group_barrier(0x008, NM - R1, 0); }
                else if (u == 2) { spread_schedule<R2, R2, 0, 0>(); __builtin_amdgcn_sched_group_barrier(0x008, NM - R2, 0); }
                else { spread_schedule<R3, R3, 0, 0>(); __builtin_amdgcn_sched_group_barrier(0x008, NM - R3, 0); }
                __builtin_amdgcn_sched_barrier(0);
            }
        }
    
}

    // ---- epilogue.  acc[i][j]: the lane holds C[row 16 i + l16][columns 16 j + 4 g4 .. + 3].  Staged through the wave's 8 KiB of
    // the last stage (dead after the final barrier), 16-byte chunk c of a staged row at position c ^ ((row >> 1) & 7).
    {
        // (HALF: every stage is dead after the final barrier; the eight waves' 8 KiB take the first two)
        // (the eight waves' 64 KiB may reach past a 48 KiB stage into the other one, which is just as dead; the launch allocates 128 KiB)
        static_assert(HALF || STAGE + 8 * 8192 <= 2 * (256 * 128 + 128 * 256), "C staging must stay inside the allocation");
        unsigned char* stg = smem + (HALF ? 0 : ((KT - 1) & 1) * STAGE) + wave * 8192;
        constexpr int ROWB = WTN * OB;                // bytes of one staged row
        constexpr int CPR = ROWB / 16;                // 16-byte chunks per staged row
        constexpr bool POW2 = (CPR & (CPR - 1)) == 0; // the XOR swizzle of the staged rows needs a power-of-two chunk count
        // (rows of another width, the 96 columns a wave holds of a 192-wide tile, are staged 16 bytes apart from whole rows instead: the
        // pad moves neighbouring rows onto different banks, where unpadded rows cost a fifth of the LDS cycles of that tile in conflicts)
        constexpr int PITCH = POW2 ? ROWB : ROWB + 16;
        constexpr int FIT = 8192 / (16 * PITCH);      // 16-row blocks that fit the wave's 8 KiB
        constexpr int IPR0 = FIT >= 8 ? 8 : FIT >= 4 ? 4 : FIT >= 2 ? 2 : 1;
        constexpr int IPR = IPR0 < TI ? IPR0 : TI;    // blocks per round (divides TI)
        const int sw = POW2 ? ((l16 >> 1) & (CPR - 1) & 7) : 0;
        const bool fused = g.bias != nullptr || g.act != 0;
        f32x4 bias4[TJ];
#pragma unroll
        for (int j = 0; j < TJ; j++) {
            bias4[j] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
            if (g.bias) bias4[j] = *(const f32x4*)(g.bias + (CUT ? min(n0 + wn * WTN + 16 * j + 4 * g4, g.N - 4) : n0 + wn * WTN + 16 * j + 4 * g4));
        }
        unsigned char* Cw = (unsigned char*)g.C + (bz * g.sC + (long long)(m0 + wm * WTM) * g.ldc + n0 + wn * WTN) * OB;
        const bool whole_tile = __builtin_amdgcn_readfirstlane(m0 + BM <= g.M && (!CUT || n0 + BN <= g.N) && g.c_cols == 0);
        static_for<0, TI, IPR>([&](auto ip_const) {
            constexpr int ip = decltype(ip_const)::value;
#pragma unroll
            for (int ii = 0; ii < IPR; ii++) {
                // (a row of blocks at a time: over the whole tile at once the choice outgrows the registers)
                f32x4_acc w[TJ];
#pragma unroll
                for (int j = 0; j < TJ; j++) w[j] = acc[ip + ii][j];
                if (fused)
                    with_activation(g.act, g.act_param, [&](auto fn) {
#pragma unroll
                        for (int j = 0; j < TJ; j++)
#pragma unroll
                            for (int e = 0; e < 4; e++) w[j][e] = fn(w[j][e] + bias4[j][e]);
                    });
#pragma unroll
                for (int j = 0; j < TJ; j++) {
                    const f32x4_acc v = w[j];
                    const int row = ii * 16 + l16;
                    if constexpr (OB == 2) {
                        const uint32_t w0 = Elem<OutT>::narrow(v[0]) | (Elem<OutT>::narrow(v[1]) << 16);
                        const uint32_t w1 = Elem<OutT>::narrow(v[2]) | (Elem<OutT>::narrow(v[3]) << 16);
                        const int chunk = 2 * j + (g4 >> 1);
                        *(u32x2*)(stg + row * PITCH + ((chunk ^ sw) << 4) + (g4 & 1) * 8) = u32x2{w0, w1};
                    } else {
                        const int chunk = 4 * j + g4;
                        *(u32x4*)(stg + row * PITCH + ((chunk ^ sw) << 4)) = u32x4{as_u32(v[0]), as_u32(v[1]), as_u32(v[2]), as_u32(v[3])};
                    }
                }
            }
            // a workgroup whose tile lies inside the matrix (every one but the last tile row or column of a ragged M or N) stores without a
            // test per chunk: with the test the compiler serialises LDS read and store of every chunk, which costs the short-K
            // shapes 3-5 %
            if (whole_tile) {
#pragma unroll
                for (int q = 0; q < IPR * 16 * CPR / 64; q++) {
                    const int u = q * 64 + lane;
                    const int row = u / CPR, c = u % CPR;
                    const u32x4 v = *(const u32x4*)(stg + row * PITCH + ((c ^ (POW2 ? ((row >> 1) & (CPR - 1) & 7) : 0)) << 4));
                    u32x4* dst = (u32x4*)(Cw + (long long)(ip * 16 + row) * g.ldc * OB + c * 16);
                    if constexpr (NTS) __builtin_nontemporal_store(v, dst);
                    else *dst = v;
                }
            } else {
                // (a rolled loop: nothing in it is indexed by q at compile time, and unrolled it grows the epilogue so much that
                // the compiler stops unrolling the loop over ip, whose accumulator indices must be constants)
#pragma unroll 1
                for (int q = 0; q < IPR * 16 * CPR / 64; q++) {
                    const int u = q * 64 + lane;
                    const int row = u / CPR, c = u % CPR;
                    const u32x4 v = *(const u32x4*)(stg + row * PITCH + ((c ^ (POW2 ? ((row >> 1) & (CPR - 1) & 7) : 0)) << 4));
                    u32x4* dst = (u32x4*)(Cw + (long long)(ip * 16 + row) * g.ldc * OB + c * 16);
                    if (m0 + wm * WTM + ip * 16 + row >= g.M) continue;
                    if (g.c_cols > 0) {
                        // rows of C at any element offset: whole chunks by one under-aligned 16-byte store, the chunk that
                        // crosses the last column by elements
                        typedef typename Raw<OutT>::type out_t;
                        typedef u32x4 u32x4_elem __attribute__((aligned(2)));
                        constexpr int PER = 16 / OB;
                        const int col0 = n0 + wn * WTN + c * PER;
                        if (col0 + PER <= g.c_cols) *(u32x4_elem*)dst = v;
                        else {
#pragma unroll
                            for (int e = 0; e < PER; e++)
                                if (col0 + e < g.c_cols) {
                                    if constexpr (OB == 2) ((out_t*)dst)[e] = (out_t)(v[e >> 1] >> ((e & 1) * 16));
                                    else ((out_t*)dst)[e] = v[e];
                                }
                        }
                    } else if (!CUT || n0 + wn * WTN + c * (16 / OB) < g.N) *dst = v;
                }
            }
        });
    }
}

template <typename T, typename OutT, int TJ, bool HALF, int HS, bool CUT>
static hipError_t launch_dl16_as(GemmArgs g, int batch, hipStream_t stream)
{
    constexpr int smem = HALF ? HS * (128 * 128 + 64 * 256) : 2 * (256 * 128 + 128 * 256);
    g.tiles_m = (g.M + (HALF ? 127 : 255)) / (HALF ? 128 : 256);      // the last tile row and column may be partial
    g.tiles_n = (g.N + 64 * TJ - 1) / (64 * TJ);
    const dim3 grid((unsigned)(g.tiles_m * g.tiles_n), 1, (unsigned)batch);
    // Non-temporal stores of C when A, B and C together exceed the 256 MB last-level cache: C then no longer displaces the operand
    // tiles that later workgroups re-read (alternated in one process: fp16 8192^3 1336 -> 1408 TFLOP/s, bf16 1397 -> 1464,
    // 16384 x 8192 x 1024 989 -> 1166, 8192 x 50304 x 768 764 -> 873); a problem that fits the cache is better left to its
    // write-back path (4096 x 3072 x 768 881 -> 770, 8192 x 8192 x 2048 1283 -> 1248 with such stores).
    const long long footprint = ((long long)g.M * g.K * (g.sA == 0 ? 1 : batch) + (long long)g.K * g.N * batch) * 2 + (long long)g.M * g.N * batch * Elem<OutT>::BYTES;
    const bool nts = footprint > (240LL << 20);
    if constexpr (!HALF) {
        if (nts) {
            auto kern = gemm_dl16_kernel<T, OutT, TJ, false, true, HS, CUT>;
            static unsigned long long attr_done_nt = 0;
            if (hipError_t e = ensure_dynamic_smem((const void*)kern, smem, &attr_done_nt)) return e;
            hipLaunchKernelGGL(kern, grid, dim3(512), smem, stream, g);
            return hipGetLastError();
        }
    }
    auto kern = gemm_dl16_kernel<T, OutT, TJ, HALF, false, HS, CUT>;
    static unsigned long long attr_done = 0;
    if (hipError_t e = ensure_dynamic_smem((const void*)kern, smem, &attr_done)) return e;
    hipLaunchKernelGGL(kern, grid, dim3(512), smem, stream, g);
    return hipGetLastError();
}
template <typename T, typename OutT, int TJ = 4, bool HALF = false, int HS = DL16_HALF_STAGES>
static hipError_t launch_gemm_dl16(const GemmArgs& g, int batch, hipStream_t stream)
{
    return g.N % (64 * TJ) == 0 ? launch_dl16_as<T, OutT, TJ, HALF, HS, false>(g, batch, stream) : launch_dl16_as<T, OutT, TJ, HALF, HS, true>(g, batch, stream);
}

// ---------------------------------------------------------------------------------------------
// 16-bit, rows at any element offset (N or K not a multiple of 8, or an operand off the 16-byte grid), B stored [K,N]: BM x 128 tile, 8
// waves (2 x 4, wave tile BM/2 x 32 of 16 x 16 x 32 blocks), K-tiles of 64.  The direct-to-LDS loads want whole 16-byte chunks, so the
// tiles travel through registers: every load is 16 bytes at element alignment and consecutive lanes take consecutive chunks of a row
// (128 bytes of A, 256 of B), two K-tiles ahead, and is written to the LDS layout of gemm_dl16_kernel, from which the fragments are read
// as there (transposing reads for B).  What bounds it is the stream of B for few rows and the load / LDS-write work beyond.
// The general kernel's loads of B are 16 rows of 64 bytes to an instruction, each cache line asked for twice: 64 x 50257 x 768
// takes 43 us there and 17.5 here (84 MB), 212 x 36669 x 704 101 / 27, 512 x 30001 x 4096 232 through padded copies / 157 (ten calls in a
// graph).
// kper > 0: workgroups z take K ranges of kper (a multiple of 64) each and C is their fp32 partials, sum_stride elements apart.
// Bounds: the last K-tile of the matrix is loaded under guards (zeros past K; whole chunks where they fit their row), which costs about 1 us;
// where all rows are whole chunks (operands off the 16-byte grid) tiles of 64 rows take it from clamped addresses instead (20 x 272 x 248 6.8 ->
// 5.8 us, 3 x 7224 x 512 8.9 -> 6.9).  In the others a
// chunk of B that crosses column N reads on into the next row, which exists, and is only multiplied into columns that are not stored.
// Rows of A past M and chunks of B past N are clamped likewise.  N >= 8.
// WHOLE: no chunk crosses the end of a row (N and K multiples of 8).
template <typename T, typename OutT, int BM, bool WHOLE>
__global__ __launch_bounds__(512, 4) void gemm_any16_kernel(const GemmArgs g, int kper, long long sum_stride)
{
    typedef typename Raw<T>::type raw_t;
    typedef u32x4 u32x4_elem __attribute__((aligned(2)));
    constexpr int BN = 128, BK = 64, TI = BM / 32, TJ = 2;
    constexpr int AROW = 128, BROW = 2 * BN;
    constexpr int ABYTES = BM * AROW, STAGE = ABYTES + BK * BROW;
    constexpr int LA = BM / 64, LB = 2;                      // chunks of A and B per thread and tile
    extern __shared__ __attribute__((aligned(1024))) unsigned char smem[];
    const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
    const int l16 = lane & 15, g4 = lane >> 4;
    const int wm = wave >> 2, wn = wave & 3;
    int tile_m, tile_n;
    tile_of_block(blockIdx.x, gridDim.x, g.tiles_m, g.tiles_n, tile_m, tile_n);
    const int m0 = tile_m * BM, n0 = tile_n * BN;
    const int kbeg = kper > 0 ? (int)blockIdx.z * kper : 0;
    const int K = kper > 0 ? min(kper, g.K - kbeg) : g.K;
    const int KT = (K + BK - 1) / BK;

    auto b_swz = [](int row) -> int { return ((row & 3) << 2) | (((row >> 3) & 1) << 1); };
    // this thread's chunks: A rows t / 8 + 64 i, chunk t % 8; B k-rows t / 16 + 32 i, chunk t % 16
    const int ach = t & 7, bch = t & 15;
    // (element offsets from wave-uniform bases that advance with the tile: lda, ldb < 2^21)
    const raw_t* a_base = (const raw_t*)g.A + (long long)m0 * g.lda + kbeg;
    const raw_t* b_base = (const raw_t*)g.B + (long long)kbeg * g.ldb;
    uint32_t pa[LA];
    int a_lds[LA], b_lds[LB];
#pragma unroll
    for (int i = 0; i < LA; i++) {
        const int row = (t >> 3) + 64 * i;
        pa[i] = (uint32_t)((min(m0 + row, g.M - 1) - m0) * g.lda + ach * 8);
        a_lds[i] = row * AROW + ((ach ^ ((row >> 1) & 7)) << 4);
    }
    const int bcol = min(n0 + bch * 8, WHOLE ? g.N - 8 : g.N - 1);
    const uint32_t pb = (uint32_t)((t >> 4) * g.ldb + bcol);
#pragma unroll
    for (int i = 0; i < LB; i++) {
        const int row = (t >> 4) + 32 * i;
        b_lds[i] = ABYTES + row * BROW + ((bch ^ b_swz(row)) << 4);
    }
    u32x4 ra[2][LA], rb[2][LB];
    auto load_plain = [&](int kt, auto set) {
        constexpr int S = decltype(set)::value;
#pragma unroll
        for (int i = 0; i < LA; i++) ra[S][i] = *(const u32x4_elem*)(a_base + kt * BK + pa[i]);
#pragma unroll
        for (int i = 0; i < LB; i++) rb[S][i] = *(const u32x4_elem*)(b_base + (long long)(kt * BK + 32 * i) * g.ldb + pb);
    };
    auto load_any = [&](int kt, auto set) {
        constexpr int S = decltype(set)::value;
        if (kt < KT - 1) { load_plain(kt, set); return; }
        if (kt >= KT) return;
        if constexpr (WHOLE) {
            const int ak = kt * BK + ach * 8, bk = kt * BK + (t >> 4);
#pragma unroll
            for (int i = 0; i < LA; i++) ra[S][i] = *(const u32x4_elem*)(a_base + ((int)pa[i] - ach * 8 + min(ak, K - 8)));
#pragma unroll
            for (int i = 0; i < LB; i++)
                if (i == 0 || kt * BK + 32 * i < K) rb[S][i] = *(const u32x4_elem*)(b_base + (long long)(min(bk + 32 * i, K - 1) - (t >> 4)) * g.ldb + pb);
#pragma unroll
            for (int i = 0; i < LA; i++) ra[S][i] = ak < K ? ra[S][i] : u32x4{0u, 0u, 0u, 0u};
#pragma unroll
            for (int i = 0; i < LB; i++) rb[S][i] = bk + 32 * i < K ? rb[S][i] : u32x4{0u, 0u, 0u, 0u};
            return;
        }
#pragma unroll
        for (int i = 0; i < LA; i++) {
            const int valid = K - (kt * BK + ach * 8);
            ra[S][i] = u32x4{0u, 0u, 0u, 0u};
            if (valid > 0) ra[S][i] = load16_guarded<T>(a_base + kt * BK + pa[i], valid);
        }
#pragma unroll
        for (int i = 0; i < LB; i++) {
            const int k = kt * BK + 32 * i + (t >> 4);
            rb[S][i] = u32x4{0u, 0u, 0u, 0u};
            if (k < K) rb[S][i] = load16_guarded<T>(b_base + (long long)(kt * BK + 32 * i) * g.ldb + pb, g.N - bcol);
        }
    };
    auto store_tile = [&](int stage, auto set) {
        constexpr int S = decltype(set)::value;
        unsigned char* st = smem + stage * STAGE;
#pragma unroll
        for (int i = 0; i < LA; i++) *(u32x4*)(st + a_lds[i]) = ra[S][i];
#pragma unroll
        for (int i = 0; i < LB; i++) *(u32x4*)(st + b_lds[i]) = rb[S][i];
    };

    // fragments: as in gemm_dl16_kernel
    const int a_row0 = (wm * (BM / 2) + l16) * AROW, a_sw = (l16 >> 1) & 7;
    const int b_rowl = 8 * g4 + (l16 >> 2), b_half = (l16 & 1) * 8, b_chunk0 = wn * (2 * TJ) + ((l16 & 3) >> 1);
    f32x4_acc acc[TI][TJ];
#pragma unroll
    for (int i = 0; i < TI; i++)
#pragma unroll
        for (int j = 0; j < TJ; j++) acc[i][j] = f32x4_acc{0.0f, 0.0f, 0.0f, 0.0f};
    auto multiply = [&](int stage) {
        const unsigned char* as = smem + stage * STAGE;
        const unsigned char* bs = as + ABYTES;
#pragma unroll
        for (int s2 = 0; s2 < 2; s2++) {
            u32x4 fa[TI], fb[TJ];
#pragma unroll
            for (int i = 0; i < TI; i++) fa[i] = *(const u32x4*)(as + a_row0 + i * (16 * AROW) + (((4 * s2 + g4) ^ a_sw) << 4));
#pragma unroll
            for (int j = 0; j < TJ; j++)
#pragma unroll
                for (int q = 0; q < 2; q++) {
                    const int row = 32 * s2 + 4 * q + b_rowl;
                    const u32x2 w = __builtin_bit_cast(u32x2, __builtin_amdgcn_ds_read_tr16_b64_v4i16(
                        (__attribute__((address_space(3))) s16x4*)(bs + row * BROW + (((b_chunk0 + 2 * j) ^ b_swz(row)) << 4) + b_half)));
                    fb[j][2 * q] = w[0];
                    fb[j][2 * q + 1] = w[1];
                }
#pragma unroll
            for (int i = 0; i < TI; i++)
#pragma unroll
                for (int j = 0; j < TJ; j++) Mma16<T>::run(acc[i][j], fb[j], fa[i]);
        }
    };
    // iteration kt: tile kt is in stage kt & 1; tile kt + 2 goes into the register set whose tile was stored an iteration ago, tile
    // kt + 1 from the other set into the other stage, which everyone left at the barrier that ended iteration kt - 1
    typedef std::integral_constant<int, 0> Set0;
    typedef std::integral_constant<int, 1> Set1;
    load_any(0, Set0{});
    load_any(1, Set1{});
    store_tile(0, Set0{});
    __syncthreads();
    auto step = [&](int kt, auto plain, auto mine, auto other) {
        constexpr int P = decltype(mine)::value;
        if constexpr (decltype(plain)::value) load_plain(kt + 2, mine);
        else load_any(kt + 2, mine);
        multiply(P);
        if (decltype(plain)::value || kt + 1 < KT) store_tile(P ^ 1, other);
        __syncthreads();
    };
    int kt = 0;
    // (the loop proper loads whole tiles that are not the last one: no branch stands between its loads and their use)
    for (; kt + 4 < KT; kt += 2) {
        step(kt, std::true_type{}, Set0{}, Set1{});
        step(kt + 1, std::true_type{}, Set1{}, Set0{});
    }
    for (; kt < KT; kt += 2) {
        step(kt, std::false_type{}, Set0{}, Set1{});
        if (kt + 1 < KT) step(kt + 1, std::false_type{}, Set1{}, Set0{});
    }

    // epilogue: acc[i][j] holds C[row 16 i + l16][columns 16 j + 4 g4 .. + 3] of the wave tile; staged through the dead stages (16-byte
    // chunk c of row r at position c ^ (r & 15)) so that rows leave in 16-byte stores at element alignment
    constexpr int OB = Elem<OutT>::BYTES, PITCH = BN * OB, CPR = PITCH / 16, PER = 16 / OB;
    static_assert(BM * PITCH <= 2 * STAGE, "C staging must stay inside the tile memory");
    const bool fused = g.bias != nullptr || g.act != 0;
    f32x4_acc bias[TJ];
    if (fused) {
#pragma unroll
        for (int j = 0; j < TJ; j++)
#pragma unroll
            for (int e = 0; e < 4; e++) {
                const int col = n0 + wn * 32 + 16 * j + 4 * g4 + e;
                bias[j][e] = g.bias && col < g.N ? g.bias[col] : 0.0f;
            }
    }
#pragma unroll
    for (int i = 0; i < TI; i++) {
        const int row = wm * (BM / 2) + 16 * i + l16;
        f32x4_acc w[TJ];
#pragma unroll
        for (int j = 0; j < TJ; j++) w[j] = acc[i][j];
        if (fused)
            with_activation(g.act, g.act_param, [&](auto fn) {
#pragma unroll
                for (int j = 0; j < TJ; j++)
#pragma unroll
                    for (int e = 0; e < 4; e++) w[j][e] = fn(w[j][e] + bias[j][e]);
            });
#pragma unroll
        for (int j = 0; j < TJ; j++) {
            const int col = wn * 32 + 16 * j + 4 * g4;
            unsigned char* dst = smem + row * PITCH + ((((col * OB) >> 4) ^ (row & 15)) << 4);
            if constexpr (OB == 2) *(u32x2*)(dst + (g4 & 1) * 8) = u32x2{Elem<OutT>::narrow(w[j][0]) | (Elem<OutT>::narrow(w[j][1]) << 16),
                                                                        Elem<OutT>::narrow(w[j][2]) | (Elem<OutT>::narrow(w[j][3]) << 16)};
            else *(u32x4*)dst = u32x4{as_u32(w[j][0]), as_u32(w[j][1]), as_u32(w[j][2]), as_u32(w[j][3])};
        }
    }
    __syncthreads();
    typedef typename Raw<OutT>::type out_t;
    out_t* C = (out_t*)g.C + (kper > 0 ? (long long)blockIdx.z * sum_stride : 0);
#pragma unroll 4
    for (int u = t; u < BM * CPR; u += 512) {
        const int row = u / CPR, c = u % CPR, col = n0 + c * PER;
        if (m0 + row >= g.M || col >= g.N) continue;
        const u32x4 v = *(const u32x4*)(smem + row * PITCH + ((c ^ (row & 15)) << 4));
        out_t* dst = C + (long long)(m0 + row) * g.ldc + col;
        if (col + PER <= g.N) *(u32x4_elem*)dst = v;
        else
            for (int e = 0; e < g.N - col; e++) dst[e] = (out_t)(OB == 2 ? v[e >> 1] >> ((e & 1) * 16) : v[e]);
    }
}

template <typename T, typename OutT, int BM, bool WHOLE>
static hipError_t launch_any16_as(GemmArgs g, hipStream_t stream, int ks, int kper)
{
    constexpr int smem = 2 * (BM * 128 + 64 * 256);
    auto kern = gemm_any16_kernel<T, OutT, BM, WHOLE>;
    static unsigned long long attr_done = 0;
    if (hipError_t e = ensure_dynamic_smem((const void*)kern, smem, &attr_done)) return e;
    g.tiles_m = (g.M + BM - 1) / BM;
    g.tiles_n = (g.N + 127) / 128;
    hipLaunchKernelGGL(kern, dim3((unsigned)(g.tiles_m * g.tiles_n), 1, (unsigned)ks), dim3(512), smem, stream, g, ks > 1 ? kper : 0, (long long)g.M * g.N);
    return hipGetLastError();
}
template <typename T, typename OutT, int BM>
static hipError_t launch_any16(const GemmArgs& g, hipStream_t stream, int ks = 1, int kper = 0)
{
    if constexpr (BM == 64) {
        if (((g.K | g.N) & 7) == 0) return launch_any16_as<T, OutT, BM, true>(g, stream, ks, kper);
    }
    return launch_any16_as<T, OutT, BM, false>(g, stream, ks, kper);
}

// ---------------------------------------------------------------------------------------------
// Skinny-M path (decode projections): M <= 32, 16-bit, B stored [K,N], N % 8 == 0, K % 64 == 0.
// HBM-bound: B (K x N) is read exactly once.  grid = (ceil(N / 128), KS), about one workgroup per CU: each workgroup streams a
// 128-column slab of B over its K range with the direct global->LDS load through a ring of NS 20 KB stages, filled NS - 1
// K-tiles ahead -- seven stages and one workgroup per CU (120 KB in flight per CU: one memory round trip covers a whole K range of
// up to six tiles, where a two-stage ring paid one round trip per tile), or three stages and two workgroups per CU for wide
// weights (launch_skinny) --, computes a 32 x 128 partial product on MFMA (A rows beyond M are
// clamped duplicates that are never stored) and writes it to an fp32 workspace that skinny_reduce_kernel sums in split order
// (deterministic) and narrows.  Loads complete in issue order, so "tile kt has landed" is a count of younger loads.
//   B tile [64 k][256 B]: chunk c of row k at position c ^ ((k & 3) << 2)   (transposing reads)
//   A tile [32 m][128 B]: chunk c of row m at position c ^ ((m >> 1) & 7)   (b128 reads)
#define SKINNY_STAGES 7
template <typename T, int NS>
__global__ __launch_bounds__(256, NS <= 3 ? 2 : 1) void gemm_skinny_kernel(const GemmArgs g, float* __restrict__ ws, int ksplit, int kper)
{
    typedef uint16_t raw_t;
    constexpr int BK = 64, AHEAD = NS - 1;
    constexpr int ABYTES = 32 * 128, BBYTES = BK * 256, STAGE = ABYTES + BBYTES;
    extern __shared__ __attribute__((aligned(1024))) unsigned char smem[];      // NS stages

    const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
    const int l32 = lane & 31, h = lane >> 5;
    const int n0 = blockIdx.x * 128;
    const int ks = blockIdx.y;
    const int kbeg = ks * kper;
    const int KT = min(kper, g.K - kbeg) / BK;            // the last range may be shorter
    const raw_t* __restrict__ A = (const raw_t*)g.A;
    const raw_t* __restrict__ B = (const raw_t*)g.B;

    // this wave's DMA per K-tile: 4 B wave-loads (k-rows 4w'..4w'+3, w' = 4*wave+i) and A wave-load `wave` (rows 8*wave..)
    const raw_t* pb[4];
#pragma unroll
    for (int i = 0; i < 4; i++) {
        int row = 4 * (wave * 4 + i) + (lane >> 4), pos = lane & 15;
        pb[i] = B + (long long)(kbeg + row) * g.ldb + min(n0 + (pos ^ ((row & 3) << 2)) * 8, g.N - 8);      // (past N: the last chunk, never stored)
    }
    const raw_t* pa;
    {
        int row = 8 * wave + (lane >> 3), pos = lane & 7;
        int grow = min(row, g.M - 1);
        pa = A + (long long)grow * g.lda + kbeg + (pos ^ ((row >> 1) & 7)) * 8;
    }
    auto issue_loads = [&](int kt, int stage) {
        unsigned char* as = smem + stage * STAGE;
        unsigned char* bs = as + ABYTES;
        dma16_to_lds(pa + kt * BK, as + wave * 1024);
#pragma unroll
        for (int i = 0; i < 4; i++) dma16_to_lds_stream(pb[i] + (long long)kt * BK * g.ldb, bs + (wave * 4 + i) * 1024);
    };

    const int a_off = l32 * 128, a_sw = (l32 >> 1) & 7;
    const int jl = lane & 15;
    const int b_rowl = 8 * h + (jl >> 2);
    const int b_half = (jl & 1) * 8;
    const int b_chunk = (wave * 32 + 16 * ((lane >> 4) & 1) + 4 * (jl & 3)) >> 3;

    f32x16 acc;
#pragma unroll
    for (int r = 0; r < 16; r++) acc[r] = 0.0f;

    for (int kt = 0; kt < AHEAD && kt < KT; kt++) issue_loads(kt, kt);
    int stage = 0;
    for (int kt = 0; kt < KT; kt++) {
        // tiles kt+1 .. kt+AHEAD-1 (those that exist) are younger than tile kt: five loads per wave each
        switch (min(KT - 1 - kt, AHEAD - 1)) {
            case 0: asm volatile("s_waitcnt vmcnt(0)" ::: "memory"); break;
            case 1: asm volatile("s_waitcnt vmcnt(5)" ::: "memory"); break;
            case 2: asm volatile("s_waitcnt vmcnt(10)" ::: "memory"); break;
            case 3: asm volatile("s_waitcnt vmcnt(15)" ::: "memory"); break;
            case 4: asm volatile("s_waitcnt vmcnt(20)" ::: "memory"); break;
            default: asm volatile("s_waitcnt vmcnt(25)" ::: "memory"); break;
        }
        __syncthreads();            // everyone's part of tile kt has landed, and everyone has left tile kt-1
        if (kt + AHEAD < KT) issue_loads(kt + AHEAD, stage == 0 ? NS - 1 : stage - 1);      // into the stage tile kt-1 used
        const unsigned char* as = smem + stage * STAGE;
        const unsigned char* bs = as + ABYTES;
#pragma unroll
        for (int s = 0; s < 4; s++) {
            u32x4 fa = *(const u32x4*)(as + a_off + (((2 * s + h) ^ a_sw) << 4));
            u32x4 fb;
#pragma unroll
            for (int q = 0; q < 2; q++) {
                int row = 16 * s + 4 * q + b_rowl;
                int pos = b_chunk ^ ((row & 3) << 2);
                s16x4 v = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
                    (__attribute__((address_space(3))) s16x4*)(bs + row * 256 + pos * 16 + b_half));
                u32x2 w = __builtin_bit_cast(u32x2, v);
                fb[2 * q] = w[0];
                fb[2 * q + 1] = w[1];
            }
            Mma32<T>::run(acc, fa, fb);
        }
        stage = stage + 1 == NS ? 0 : stage + 1;
    }

    const int col = n0 + wave * 32 + l32;
#pragma unroll
    for (int r = 0; r < 16; r++) {
        const int row = acc_row(r, h);
        if (row < g.M && col < g.N) ws[((long long)ks * g.M + row) * g.N + col] = acc[r];
    }
}

template <typename OutT>
__global__ __launch_bounds__(256) void skinny_reduce_kernel(const float* __restrict__ ws, void* __restrict__ Cv, int M, int N, int ksplit,
                                                             const float* __restrict__ bias, int act, float act_param,
                                                             float alpha = 1.0f, float beta = 0.0f)
{
    typedef typename Raw<OutT>::type out_t;
    out_t* C = (out_t*)Cv;
    const long long total = (long long)M * N;
    for (long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x; i < total; i += (long long)gridDim.x * blockDim.x) {
        float s = 0.0f;
        int k = 0;
        for (; k + 8 <= ksplit; k += 8) {              // eight loads in flight, summed in split order
            float t[8];
#pragma unroll
            for (int u = 0; u < 8; u++) t[u] = ws[(long long)(k + u) * total + i];
#pragma unroll
            for (int u = 0; u < 8; u++) s += t[u];
        }
        for (; k < ksplit; k++) s += ws[(long long)k * total + i];
        if constexpr (Elem<OutT>::BYTES == 4) {
            s *= alpha;
            if (beta != 0.0f) s += beta * as_f32(C[i]);
        }
        if (bias) s += bias[i % N];
        s = apply_activation(s, act, act_param);
        if constexpr (Elem<OutT>::BYTES == 4) C[i] = as_u32(s);
        else C[i] = (out_t)Elem<OutT>::narrow(s);
    }
}

// The summing pass with the rotary embedding on top: one thread per column pair (2 j, 2 j + 1) of a row sums both columns in split
// order, rotates the pair when it lies in the first rope.cols columns, and stores both with one rounding.
template <typename OutT>
__global__ __launch_bounds__(256) void skinny_reduce_rope_kernel(const float* __restrict__ ws, uint16_t* __restrict__ C, int M, int N, int ksplit,
                                                                  const RopeEpilogue rope)
{
    typedef float f32x2a __attribute__((ext_vector_type(2)));
    const long long total = (long long)M * N, pairs = total >> 1;
    const int half = rope.head_dim >> 1, row_pairs = N >> 1;
    for (long long p = (long long)blockIdx.x * blockDim.x + threadIdx.x; p < pairs; p += (long long)gridDim.x * blockDim.x) {
        float s0 = 0.0f, s1 = 0.0f;
        for (int k = 0; k < ksplit; k++) {
            const f32x2a t = *(const f32x2a*)(ws + (long long)k * total + 2 * p);
            s0 += t[0]; s1 += t[1];
        }
        const int m = (int)(p / row_pairs), col = 2 * (int)(p - (long long)m * row_pairs);
        if (col < rope.cols) {
            const int i = (col % rope.head_dim) >> 1;
            const long long pos = rope.start_position + m % rope.seq_len;
            // (the pair is rounded to the output type before it is rotated: what a product followed by the rotation kernel computes)
            const float xe = Elem<OutT>::widen(Elem<OutT>::narrow(s0)), xo = Elem<OutT>::widen(Elem<OutT>::narrow(s1));
            rope_rotate(xe, xo, rope.cosc[pos * half + i], rope.sinc[pos * half + i], s0, s1);
        }
        ((uint32_t*)C)[p] = Elem<OutT>::narrow(s0) | (Elem<OutT>::narrow(s1) << 16);
    }
}

// The stream and its summing pass are two launches: from K = 1024 on (768 for up to eight rows) they are faster than the one launch of the
// tiled kernels (us, tiled / here: 8 x 512 x 384 5.0 / 6.7, 8 x 512 x 768 6.8 / 6.6, 32 x 4096 x 768 7.0 / 7.9, 32 x 4096 x 1024 8.2 / 8.3, 8 x 1024 x
// 1536 10.3 / 8.0).  With a ragged last slab (clamped loads) they are taken where the tiled kernels take longer than the 15 us that two
// launches cost their caller anyway (3 x 192 x 6400 32.2 / 6.9, 5 x 5680 x 6272 52 / 20, 17 x 6592 x 2240 21.2 / 11.2, 2 x 4104 x 1536 15.1 / 8.9); the rows of
// such a B share cache lines between slabs, which a streaming load fetches twice, so that more than 256 tiles of 64 columns win over it
// (32 x 12296 x 1536 16.6 / 18.5, 32 x 40008 x 1024 20.7 / 33.0).
static bool skinny_applies(int M, int N, int K)
{
    if (M > 32 || N % 8 != 0 || K % 64 != 0 || N < 128) return false;
    if (N % 128 == 0) return K >= (M <= 8 ? 768 : 1024);
    return K >= (N <= 4096 ? 2560 : M <= 8 || N <= 8192 ? 1536 : 2048) && N <= 16384;
}
static int skinny_slabs(int N) { return (N + 127) / 128; }

// How evenly `tiles` workgroups load the 256 CUs: a CU works through its tiles at about the same rate whether it holds one or
// several at a time, so what counts is the largest number of tiles any CU gets.
static double cu_fill(long long tiles) { return (double)tiles / (double)(((tiles + 255) / 256) * 256); }

// K ranges of the skinny paths: `tiles` K-tiles over `slabs` column slabs, one workgroup per CU at a time.  Returns the K-tiles per
// range (the last range may be shorter); *ks = number of ranges.  Scored as (how evenly slabs x ranges load the 256 CUs) x (the
// share of a workgroup's time that is not its first memory round trip, about three K-tiles' worth).
static int skinny_plan(int slabs, int tiles, int* ks_out, int per_cu = 1, double* score_out = nullptr)
{
    int best_kper = tiles, best_ks = 1;
    double best = -1.0;
    const long long slots = 256LL * per_cu;
    // (two workgroups per CU: one's first round trip runs under the other's stream, so it counts half)
    const double ramp = per_cu == 1 ? 3.0 : 1.5;
    for (int ks = 1; ks <= 32 && ks <= tiles; ks++) {
        const int kper = (tiles + ks - 1) / ks;
        const int kse = (tiles + kper - 1) / kper;
        if (kper < 4 && ks > 1) break;
        const long long wg = (long long)slabs * kse;
        const double fill = (double)wg / (double)(((wg + slots - 1) / slots) * slots);
        const double score = fill * (double)kper / (kper + ramp);
        if (score > best * 1.02) { best = score; best_kper = kper; best_ks = kse; }
    }
    *ks_out = best_ks;
    if (score_out) *score_out = best;
    return best_kper;
}
static int skinny_ksplit(int N, int K) { int ks; skinny_plan(skinny_slabs(N), K / 64, &ks, skinny_slabs(N) > 64 && K <= 4096 ? 2 : 1); return ks; }

// Split-K for 16-bit problems whose 128 x 128 tiles fill less than half the chip over a long K (M <= 512 against a 4096-wide
// weight): K ranges run as the batch dimension of the 128 x 128 kernel into fp32 partials, summed in range order by
// skinny_reduce_kernel (deterministic; bias and activation there).  Returns the number of ranges, 0 = not worth it.  Ranges are whole
// K-tiles and the last may be shorter, so that any K takes as many as suit the tiles (with equal ranges K = 193 x 64 had none: 233 x 528 x
// 12352 100 us / 18, 332 x 2936 x 13888 114 / 48, 129 x 256 x 3904 21 / 12, 2838 x 512 x 4416 39 / 27; 40 drawn sizes of 33 - 512 rows 1.5x).
static int dl16_width(int M, int N, int K, int batch, double* score_out = nullptr);
// Share of a split-K product's time that is the product: the fp32 partials are written and read once per range, 8 bytes per output
// element and range at about 4 TB/s, against 2 K flops per element at about 1.4 PFLOP/s (512 x 8192 x 8192 in four ranges: 49 us of
// product, 33 us of partials)
static double splitk16_partials_factor(int K, int ks) { return 1.0 / (1.0 + 1000.0 * ks / K); }
static int splitk16_ranges(int M, int N, int K, int* kper, int* big_tile = nullptr)
{
    if (big_tile) *big_tile = 0;
    *kper = K;
    if (N % 8 != 0 || K % 64 != 0) return 0;
    const int kt = K / 64;
    // (the last range may be shorter by up to a K-tile per range)
    auto ranges = [&](long long t, int min_k) {
        int ks = (int)(256 / t);
        if (ks > 16) ks = 16;
        while (ks > 1 && K / ks < min_k) ks--;
        const int per = (kt + ks - 1) / ks;
        *kper = 64 * per;
        return (kt + per - 1) / per;
    };
    // (a ragged M or N: the last tile row or column is partial)
    const long long t = (long long)((M + 127) / 128) * ((N + 127) / 128);
    if (t <= 128) {                           // up to half a chip of 128 x 128 tiles
        // (below, the second launch costs what the ranges save: 1000 x 1024 x 1024 8 -> 15 us, 512 x 1024 x 1344 8.9 -> 14.0, 64 x 512 x 1536 9.4 -> 9.8;
        // 128 x 136 x 2112, whose one launch is shorter than what two cost the caller)
        if (K < (N % 128 == 0 || N < 128 ? 1792 : 2560)) return 0;
        // estimates in us: in one launch 0.5 a K-tile and 3; in ranges 0.425 a K-tile, 6.9 for both launches and the sums, and the partials
        // written and read at 3.55 TB/s (fitted on 310 timings of 60 shapes to 5 %; one / two / three / four: 2048 x 512 x 2048 19.3 / 18.5 / 17.8 /
        // 18.0, 1000 x 1024 x 2048 20.0 / 17.8 / 17.5 / 18.2, 512 x 1024 x 1792 16.5 / 15.6 / 15.3 / 15.2; 2048 x 1024 x 2112 19.9 in one, 23.1 in two)
        int best = 1;
        // (fewer than 128 columns: one launch is of 64 x 64 tiles, 0.3 a K-tile; us, one launch / ranges and
        // their sums: 496 x 64 x 8064 39.9 / 13.2, 1433 x 64 x 5120 27.0 / 14.6, 4 x 64 x 3008 25.8 / 9.7, 200 x 96 x 1856 11.6 / 11.0)
        double best_us = (N < 128 ? 0.3 : 0.5) * kt + 3.0;
        for (int ks = 2; ks <= 16 && ks * t <= 256 && K / ks >= 512; ks++) {
            const int per = (kt + ks - 1) / ks, n = (kt + per - 1) / per;
            const double us = 0.425 * per + 6.9 + (double)n * M * N * 8.0 / 3.55e6;
            if (us < best_us) { best_us = us; best = n; *kper = 64 * per; }
        }
        return best >= 2 ? best : 0;
    }
    // Larger problems whose 256 x 256 tiles still fill at most half the chip over a long K (M about 1000 against an 8192-wide
    // weight with K = 28672): narrower tiles would fill the chip but move twice the operand bytes per flop through the L2, which
    // is what bounds them at this K; K ranges of the 256 x 256 tile keep its traffic.
    if (N % 256 != 0) return 0;
    const long long t256 = (long long)((M + 255) / 256) * (N / 256);
    if (t256 > 128 || K < 4096) return 0;
    const int ks = ranges(t256, 2048);
    if (ks < 2 || !big_tile) return 0;
    // against the best single launch, by the scores of the tile choice (CU fill x rate per flop x share of real rows)
    double single = 0.0;
    dl16_width(M, N, K, 1, &single);
    const double split = cu_fill(t256 * ks) * ((double)M / (double)(((M + 255) / 256) * 256)) * splitk16_partials_factor(K, ks);
    if (split <= 1.05 * single) return 0;
    *big_tile = 1;
    return ks;
}

// Rows of a tall 16-bit problem to run as a launch of their own: with N / 256 tile columns that divide the 256 CUs, whole rounds of
// 256 x 256 tiles cover a multiple of 256 * 256 / (N / 256) rows at the full rate; the rows that would start a partly filled round
// (3000 rows against an 8192-wide weight: 1.5 rounds) are better served by whatever suits them alone -- narrower tiles, or K
// ranges of the 256 x 256 tile.  Returns the row count of the first launch, 0 = one launch.  Both estimates are rows / score.
static int msplit16_rows(int M, int N, int K)
{
    if (N % 256 != 0 || K % 64 != 0 || 256 % (N / 256) != 0) return 0;
    const int rows_per_round = 256 / (N / 256) * 256;
    const int first = M / rows_per_round * rows_per_round;
    const int rest = M - first;
    if (first == 0 || rest == 0) return 0;
    auto score = [&](int m) {
        double single = 0.0;
        dl16_width(m, N, K, 1, &single);
        int big = 0, kper;
        const int ks = splitk16_ranges(m, N, K, &kper, &big);
        if (ks && big) {
            const long long t256 = (long long)((m + 255) / 256) * (N / 256);
            const double split = cu_fill(t256 * ks) * ((double)m / (double)(((m + 255) / 256) * 256)) * splitk16_partials_factor(K, ks);
            if (split > single) single = split;
        }
        return single;
    };
    const double whole = score(M), tail = score(rest);
    if (whole <= 0.0 || tail <= 0.0) return 0;
    return (double)first + (double)rest / tail < 0.92 * (double)M / whole ? first : 0;
}

// 16-bit problems whose rows are not 16-byte aligned (N or K not a multiple of 8) would run on 2-byte loads, an order of
// magnitude below the vector-load kernels.  They are copied instead into zero-padded, aligned operands in the workspace
// (K up to a multiple of 64, N up to a multiple of 128, or of 8 for a narrow N), multiplied there by the kernels for aligned
// problems and the columns of C copied back: three extra passes over A, B and C, which a product of this size repays many
// times over.  The zero columns of A meet zero rows of B, so the padded product holds exactly the sums of the plain one.
struct PadPlan {
    int Np, Kp;                                   // padded N and K
    size_t a_off, b_off, c_off, bias_off, inner_off, total;
};
static size_t gemm_16_inner_workspace_bytes(int M, int N, int K)
{
    size_t need = 0;
    if (skinny_applies(M, N, K)) need = (size_t)skinny_ksplit(N, K) * M * N * sizeof(float);
    if (const int first = msplit16_rows(M, N, K)) {
        const size_t a = gemm_16_inner_workspace_bytes(first, N, K), b = gemm_16_inner_workspace_bytes(M - first, N, K);
        if (a > need) need = a;
        if (b > need) need = b;
    }
    int big, kper;
    const int ks = splitk16_ranges(M, N, K, &kper, &big);
    const size_t split = ks ? (size_t)ks * M * N * sizeof(float) : 0;
    return split > need ? split : need;
}
// the padded shapes and the workspace layout for them (no judgement on whether padding pays)
static bool pad16_layout(int M, int N, int K, PadPlan* pl)
{
    const int Np = N >= 512 ? (N + 127) / 128 * 128 : (N + 7) / 8 * 8;
    const int Kp = (K + 63) / 64 * 64;
    auto up = [](size_t b) { return (b + 255) & ~(size_t)255; };
    size_t off = 0;
    pl->Np = Np; pl->Kp = Kp;
    pl->a_off = off; if (Kp != K) off += up((size_t)M * Kp * 2);      // (an A in whole K-tiles is read where it is)
    pl->b_off = off; off += up((size_t)Kp * Np * 2);
    pl->c_off = off; off += up((size_t)M * Np * 4);
    pl->bias_off = off; off += up((size_t)Np * 4);
    pl->inner_off = off; off += gemm_16_inner_workspace_bytes(M, Np, Kp);
    pl->total = off;
    return off <= ((size_t)4 << 30);
}
// gemm_any16_kernel: tile height and K ranges (kper, a multiple of 64; 0 = none).  128 rows where such tiles fill the chip (212 x 36669 x
// 704 28 us against 31 with 64 rows, 2000 x 2001 x 2000 27 / 33), else 64 (1049 x 1216 x 398 7.4 / 9.0) and, with few tiles, K ranges summed by a
// pass of their own.  The estimate (us): a K-tile of 64 rows 0.6 with one workgroup on a CU and 0.95 with two; with ranges 3 for the second
// launch, 0.08 a range and the partials, written and read, at 3 TB/s.  30 x 300 x 9001 87 us in one range, 11 in 29; 100 x 1003 x 5000 57, 13 in
// ten; 16 x 5910 x 1600 21, 11 in five; but 273 x 5224 x 3936 stays whole, 33 us against 37 in two.
static double any16_rounds(long long wgs, double one, double two)
{
    const int last = (int)(wgs % 512);                // (beyond four rounds of 512 the workgroups no longer run in step)
    return wgs >= 2048 ? two * wgs / 512.0 : two * (double)(wgs / 512) + (last == 0 ? 0.0 : last <= 256 ? one : two);
}
static int any16_plan(int M, int N, int K, int* kper, int* ranges)
{
    const long long tn = (N + 127) / 128, t128 = (M + 127) / 128 * tn, t64 = (M + 63) / 64 * tn;
    *kper = 0; *ranges = 1;
    if (M > 64 && t128 >= 256) return 128;
    const int kt = (K + 63) / 64;
    double best = 0.0;
    for (int ks = 1; ks <= 32 && ks <= kt; ks++) {
        const int per = (kt + ks - 1) / ks, n = (kt + per - 1) / per;
        const double us = per * any16_rounds(t64 * n, 0.6, 0.95) + (n > 1 ? 3.0 + 0.08 * n + (double)n * M * N * 8.0 / 3e6 : 0.0);
        if (ks == 1 || us < best) { best = us; *ranges = n; *kper = n > 1 ? 64 * per : 0; }
    }
    return 64;
}

// Up to 16 rows on at most 256 k-rows of at most 16384 columns, with the rows of B aligned and those of A not: the general kernel, which
// reads such a B in whole chunks and starts half as many threads, is as fast or faster (4 x 15424: K 101 4.8 us / 5.3 in place above, 255 6.1 /
// 6.8, 150 6.0 / 5.6; 16 x 15424 x 209 5.9 / 6.3; beyond: 4 x 15424 x 260 7.1 / 6.1, 4 x 32768 x 129 6.1 / 5.4, 32 x 15424 x 209 6.3 and more / 5.5).
static bool general_few_rows(int M, int N, int K) { return M <= 16 && N <= 16384 && K <= 256; }

// Whether the copies repay themselves.  Both ways are estimated in us (fitted on 420 shapes of 100 - 9000 rows, 64 - 66000 columns, K 64 -
// 9000, to 9 and 13 %) and the copies, which served all these shapes before the kernel above, taken up to an estimate 8 % higher: of the
// 420 shapes 8 are then more than 3 % slower than through copies (the worst 6074 x 560 x 3833, 60 -> 70 us), 285 more than 3 % faster.  In
// place: a K-tile takes 0.48 us (64 rows) / 0.75 (128) with one workgroup on a CU and 0.83 / 1.35 with two,
// 15 % less where the rows of A are aligned.  Copied: the passes over the copies at 5.5 TB/s and the aligned kernel at 1.57 PFLOP/s times
// the score of its tiles.  In place / copied, us: 700 x 9001 x 8000 134 / 195, 1677 x 3683 x 3455 79 / 68, 3722 x 1021 x 7711 116 / 95,
// 4096 x 4095 x 4096 154 / 117, 8000 x 5001 x 3001 319 / 240, 2020 x 49751 x 179 118 / 97; three and more K ranges always win in place (372 x
// 2901 x 4904 35 / 64).
static bool pad16_plan(int M, int N, int K, PadPlan* pl)
{
    if (N % 8 == 0 && K % 8 == 0) return false;
    const double mn = (double)M * N, mk = (double)M * K, kn = (double)K * N;
    if (N < 16) {
        // in place these run on the general kernel: an A of whole K-tiles, which is not copied, from 10^10 multiply-adds on (65536 x 12 x
        // 16384 1161 / 388, 200000 x 15 x 8192 3478 / 685)
        return K % 64 == 0 && 0.9e-9 * mn * K > 1e-6 * kn + 8.0 && pad16_layout(M, N, K, pl);
    }
    if (mn * K < 2e9) return false;                   // the launches of the copies alone take as long
    int kper, ranges;
    const bool tall = any16_plan(M, N, K, &kper, &ranges) == 128;
    if (ranges > 2 || !pad16_layout(M, N, K, pl)) return false;
    const long long wgs = (long long)((M + (tall ? 127 : 63)) / (tall ? 128 : 64)) * ((N + 127) / 128) * ranges;
    const double rounds = tall ? any16_rounds(wgs, 0.75, 1.35) : any16_rounds(wgs, 0.48, 0.83);
    const double tiles = kper > 0 ? kper / 64 : (K + 63) / 64;
    const double in_place = 5.5 + rounds * tiles * (K % 8 == 0 ? 0.85 : 1.0) + mn / 1.7e6 + (ranges > 1 ? 3.2 + mn * 16.0 / 3e6 : 0.0);
    double score = 0.0;
    dl16_width(M, pl->Np, pl->Kp, 1, &score);
    const double copied = 13.0 + 4.0 * (kn + (pl->Kp != K ? mk : 0.0) + (pl->Np % 128 ? mn : 0.0)) / 5.5e6 +
                          2.0 * M * (double)pl->Np * pl->Kp / (1.57e9 * score) + mn / 1.55e6;
    return score > 0.0 && copied * (ranges == 1 ? 0.92 : 1.0) < in_place;
}

// dst [rows_dst, cols_dst] (16-byte aligned rows) <- src [rows_src, cols_src] (dense, any alignment), zeros elsewhere; E = element.
// One thread fills one 16-byte chunk of dst from element loads.
template <typename E>
__global__ __launch_bounds__(256) void pad_rows_kernel(const E* __restrict__ src, E* __restrict__ dst, int rows_src, int cols_src,
                                                       int rows_dst, int cols_dst)
{
    constexpr int PER = 16 / (int)sizeof(E);
    typedef E Vec __attribute__((ext_vector_type(PER)));
    const int per_row = cols_dst / PER;
    const long long total = (long long)rows_dst * per_row;
    const long long stride = (long long)gridDim.x * blockDim.x;
    for (long long g = (long long)blockIdx.x * blockDim.x + threadIdx.x; g < total; g += stride) {
        const long long row = g / per_row;
        const int c0 = (int)(g - row * per_row) * PER;
        Vec v;
#pragma unroll
        for (int e = 0; e < PER; e++) v[e] = (row < rows_src && c0 + e < cols_src) ? src[row * cols_src + c0 + e] : (E)0;
        *(Vec*)(dst + row * cols_dst + c0) = v;
    }
}

// The same for 2-byte elements with every access a dword that is contiguous across the wave: one thread per dword of dst
// (columns 2 i, 2 i + 1 of a row).  A source row starts on a dword boundary or 2 bytes past one; in the second case the two
// elements come from the high half of one source dword and the low half of the next.  A dword of the source is only loaded whole
// when both of its elements belong to the array.  grid = (ceil(cols_dst / 512), rows): no division per thread.
#if AIDN_GEMM_PART == 0
__global__ __launch_bounds__(256) void pad_rows16_kernel(const uint16_t* __restrict__ src, uint32_t* __restrict__ dst, int rows_src, int cols_src,
                                                         int rows_dst, int cols_dst)
{
    const int i = blockIdx.x * 256 + threadIdx.x;                    // dword column of dst
    const int per_row = cols_dst >> 1;
    if (i >= per_row) return;
    const uint32_t* base = (const uint32_t*)(((uintptr_t)src) & ~(uintptr_t)3);
    const long long off0 = (((uintptr_t)src) & 2) ? 1 : 0;           // flat element index of src[0] counted from base
    const long long end = off0 + (long long)rows_src * cols_src;     // one past the last element
    auto dword = [&](long long k) -> uint32_t {                      // source dword k: elements 2k (low half) and 2k + 1
        const bool lo = 2 * k >= off0 && 2 * k < end, hi = 2 * k + 1 >= off0 && 2 * k + 1 < end;
        if (lo && hi) return base[k];
        const uint16_t* h = (const uint16_t*)base;
        return (lo ? (uint32_t)h[2 * k] : 0u) | (hi ? (uint32_t)h[2 * k + 1] << 16 : 0u);
    };
    const int col = 2 * i;
    auto one = [&](int row) -> uint32_t {                            // guarded form: any row, any position in the array
        uint32_t v = 0;
        if (row < rows_src && col < cols_src) {
            const long long f = off0 + (long long)row * cols_src + col;
            const long long k = f >> 1;
            if (f & 1) v = (dword(k) >> 16) | (dword(k + 1) << 16);
            else v = dword(k);
            if (col + 1 >= cols_src) v &= 0xFFFFu;
        }
        return v;
    };
    // four rows per step with all eight loads issued before the first use (a row is one dword per thread: the kernel is bound
    // by memory latency unless several rows are in flight); rows whose dwords k and k + 1 lie strictly inside the array only
    const int step = gridDim.y;
    int row = blockIdx.y;
    if (row == 0) { dst[i] = one(0); row += step; }
    const uint32_t keep = col + 1 >= cols_src ? 0xFFFFu : 0xFFFFFFFFu;
    if (col < cols_src && cols_src >= 8) {
        for (; (long long)row + 3LL * step < (long long)rows_src - 1; row += 4 * step) {
            uint32_t d0[4], d1[4];
            long long f[4];
#pragma unroll
            for (int u = 0; u < 4; u++) {
                f[u] = off0 + (long long)(row + u * step) * cols_src + col;
                d0[u] = base[f[u] >> 1];
                d1[u] = base[(f[u] >> 1) + 1];
            }
#pragma unroll
            for (int u = 0; u < 4; u++) {
                const uint32_t v = (f[u] & 1) ? (d0[u] >> 16) | (d1[u] << 16) : d0[u];
                dst[(long long)(row + u * step) * per_row + i] = v & keep;
            }
        }
    }
    for (; row < rows_dst; row += step) dst[(long long)row * per_row + i] = one(row);
}

// 4-byte elements: one thread per element of a dst row, four rows in flight; grid = (ceil(cols_dst / 256), rows).
__global__ __launch_bounds__(256) void pad_rows32_kernel(const uint32_t* __restrict__ src, uint32_t* __restrict__ dst, int rows_src, int cols_src,
                                                         int rows_dst, int cols_dst)
{
    const int i = blockIdx.x * 256 + threadIdx.x;
    if (i >= cols_dst) return;
    const int step = gridDim.y;
    int row = blockIdx.y;
    if (i < cols_src) {
        for (; (long long)row + 3LL * step < rows_src; row += 4 * step) {
            uint32_t d[4];
#pragma unroll
            for (int u = 0; u < 4; u++) d[u] = src[(long long)(row + u * step) * cols_src + i];
#pragma unroll
            for (int u = 0; u < 4; u++) dst[(long long)(row + u * step) * cols_dst + i] = d[u];
        }
    }
    for (; row < rows_dst; row += step) dst[(long long)row * cols_dst + i] = (row < rows_src && i < cols_src) ? src[(long long)row * cols_src + i] : 0u;
}
#endif

// dst [rows, cols] (dense, any row alignment, dst itself 16-byte aligned) <- the first cols columns of src [rows, cols_src]:
// one thread per 16-byte chunk of the flat destination; the last, partial chunk is stored by elements.
template <typename E>
__global__ __launch_bounds__(256) void unpad_rows_kernel(const E* __restrict__ src, E* __restrict__ dst, long long rows, int cols, int cols_src)
{
    constexpr int PER = 16 / (int)sizeof(E);
    typedef E Vec __attribute__((ext_vector_type(PER)));
    const long long total = rows * cols;
    const long long chunks = (total + PER - 1) / PER;
    const long long stride = (long long)gridDim.x * blockDim.x;
    for (long long g = (long long)blockIdx.x * blockDim.x + threadIdx.x; g < chunks; g += stride) {
        const long long f0 = g * PER;
        long long row = f0 / cols;
        int col = (int)(f0 - row * cols);
        Vec v;
#pragma unroll
        for (int e = 0; e < PER; e++) {
            v[e] = f0 + e < total ? src[row * cols_src + col] : (E)0;
            if (++col == cols) { col = 0; row++; }
        }
        if (f0 + PER <= total) *(Vec*)(dst + f0) = v;
        else for (int e = 0; e < PER && f0 + e < total; e++) dst[f0 + e] = v[e];
    }
}

// esize 2 or 4
hipError_t pad_rows(hipStream_t stream, const void* src, void* dst, int rows_src, int cols_src, int rows_dst, int cols_dst, int esize);
hipError_t unpad_rows(hipStream_t stream, const void* src, void* dst, long long rows, int cols, int cols_src, int esize);

#if AIDN_GEMM_PART == 0
static unsigned copy_grid(long long chunks)
{
    const long long wg = (chunks + 255) / 256;
    return (unsigned)(wg > 256 * 16 ? 256 * 16 : wg < 1 ? 1 : wg);
}
hipError_t pad_rows(hipStream_t stream, const void* src, void* dst, int rows_src, int cols_src, int rows_dst, int cols_dst, int esize)
{
    const long long chunks = (long long)rows_dst * (cols_dst / (16 / esize));
    if (esize == 2 && cols_dst >= 256) {
        const unsigned gy = (unsigned)((rows_dst + 7) / 8 < 8192 ? (rows_dst + 7) / 8 : 8192);      // about eight rows per thread
        hipLaunchKernelGGL(pad_rows16_kernel, dim3((unsigned)((cols_dst / 2 + 255) / 256), gy), dim3(256), 0, stream, (const uint16_t*)src, (uint32_t*)dst, rows_src, cols_src, rows_dst, cols_dst);
    } else if (esize == 2) hipLaunchKernelGGL((pad_rows_kernel<uint16_t>), dim3(copy_grid(chunks)), dim3(256), 0, stream, (const uint16_t*)src, (uint16_t*)dst, rows_src, cols_src, rows_dst, cols_dst);
    else if (cols_dst >= 128) {
        const unsigned gy = (unsigned)((rows_dst + 7) / 8 < 8192 ? (rows_dst + 7) / 8 : 8192);
        hipLaunchKernelGGL(pad_rows32_kernel, dim3((unsigned)((cols_dst + 255) / 256), gy), dim3(256), 0, stream, (const uint32_t*)src, (uint32_t*)dst, rows_src, cols_src, rows_dst, cols_dst);
    } else hipLaunchKernelGGL((pad_rows_kernel<uint32_t>), dim3(copy_grid(chunks)), dim3(256), 0, stream, (const uint32_t*)src, (uint32_t*)dst, rows_src, cols_src, rows_dst, cols_dst);
    return hipGetLastError();
}
hipError_t unpad_rows(hipStream_t stream, const void* src, void* dst, long long rows, int cols, int cols_src, int esize)
{
    const long long chunks = (rows * cols + 16 / esize - 1) / (16 / esize);
    if (esize == 2) hipLaunchKernelGGL((unpad_rows_kernel<uint16_t>), dim3(copy_grid(chunks)), dim3(256), 0, stream, (const uint16_t*)src, (uint16_t*)dst, rows, cols, cols_src);
    else hipLaunchKernelGGL((unpad_rows_kernel<uint32_t>), dim3(copy_grid(chunks)), dim3(256), 0, stream, (const uint32_t*)src, (uint32_t*)dst, rows, cols, cols_src);
    return hipGetLastError();
}

// The largest need over the plans gemm_16 may take for these dimensions (the choice also depends on operand alignment; every
// plan checks its own need against the bytes it is handed).
size_t gemm_16_workspace_bytes(int M, int N, int K, bool off_grid)
{
    PadPlan pl;
    const size_t inner = gemm_16_inner_workspace_bytes(M, N, K);
    size_t need = inner;
    if (pad16_plan(M, N, K, &pl) && pl.total > need) need = pl.total;
    if (off_grid || N % 8 != 0 || K % 8 != 0) {
        int kper, ks;
        any16_plan(M, N, K, &kper, &ks);
        if (ks > 1) need = std::max(need, (size_t)ks * M * N * sizeof(float));
    }
    return need;
}
// Pre-packed B (the caller keeps it): B [K,N] zero-padded to [Kp, Np] -- the copy that an unaligned product otherwise makes on every
// call, made once.  An aligned weight is packed the same way (its K and N padded to whole tiles).
size_t gemm_16_packed_b_bytes(int N, int K)
{
    PadPlan pl;
    if (N <= 0 || K <= 0 || !pad16_layout(1, N, K, &pl)) return 0;
    return (size_t)pl.Kp * pl.Np * 2;
}
hipError_t gemm_16_pack_b(hipStream_t stream, const uint16_t* B, int K, int N, void* packed)
{
    PadPlan pl;
    if (!pad16_layout(1, N, K, &pl) || !aligned16(packed)) return hipErrorInvalidValue;
    return pad_rows(stream, B, packed, K, N, pl.Kp, pl.Np, 2);
}
size_t gemm_16_packed_workspace_bytes(int M, int N, int K)
{
    PadPlan pl;
    return pad16_layout(M, N, K, &pl) ? pl.total : 0;
}
#endif

template <typename T, typename OutT>
static hipError_t launch_skinny(const GemmArgs& g, hipStream_t stream, float* ws, const RopeEpilogue* rope = nullptr)
{
    int ks;
    // more than 64 column slabs over a K of at most 4096 (16 x 28672 x 8192 went 77 -> 88 us): the three-stage form, two workgroups per CU (a workgroup's first memory round trip and its last
    // tiles run under the other's stream: 32 x 11008 x 4096 24.5 -> 22.9 us, 32 x 128256 x 4096 193 -> 187 us); with fewer slabs the
    // K ranges of that plan get too short (32 x 4096 x 4096 12.3 -> 14.1 us) and the seven-stage form, one per CU, stays
    const int slabs = skinny_slabs(g.N);
    const bool three = slabs > 64 && g.K <= 4096;
    const int kper = 64 * skinny_plan(slabs, g.K / 64, &ks, three ? 2 : 1);
    if (three) {
        constexpr int smem = 3 * (32 * 128 + 64 * 256);
        static unsigned long long attr_done3 = 0;
        if (hipError_t e0 = ensure_dynamic_smem((const void*)gemm_skinny_kernel<T, 3>, smem, &attr_done3)) return e0;
            hipLaunchKernelGGL((gemm_skinny_kernel<T, 3>), dim3((unsigned)slabs, (unsigned)ks), dim3(256), smem, stream, g, ws, ks, kper);
    } else {
        constexpr int smem = SKINNY_STAGES * (32 * 128 + 64 * 256);
        static unsigned long long attr_done = 0;
        if (hipError_t e0 = ensure_dynamic_smem((const void*)gemm_skinny_kernel<T, SKINNY_STAGES>, smem, &attr_done)) return e0;
        hipLaunchKernelGGL((gemm_skinny_kernel<T, SKINNY_STAGES>), dim3((unsigned)slabs, (unsigned)ks), dim3(256), smem, stream, g, ws, ks, kper);
    }
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
    long long total = (long long)g.M * g.N;
    unsigned grid = (unsigned)((total + 255) / 256);
    if constexpr (!std::is_same<OutT, float>::value) {
        if (rope) {
            grid = (unsigned)((total / 2 + 255) / 256);
            hipLaunchKernelGGL((skinny_reduce_rope_kernel<OutT>), dim3(grid), dim3(256), 0, stream, ws, (uint16_t*)g.C, g.M, g.N, ks, *rope);
            return hipGetLastError();
        }
    }
    hipLaunchKernelGGL((skinny_reduce_kernel<OutT>), dim3(grid), dim3(256), 0, stream, ws, g.C, g.M, g.N, ks, g.bias, g.act, g.act_param,
                       1.0f, 0.0f);
    return hipGetLastError();
}

// ---------------------------------------------------------------------------------------------
// Small-M fp32 path (M <= 8, B stored [K,N] as fp32 or as fp16 weights): the GPU form of the N-parallel small-M GEMM.
// HBM-bound: B is read exactly once and nothing is staged, every lane owns four adjacent columns (one 16-byte load of a
// B row, 8 bytes for fp16 weights) and MR rows of accumulators; the A values of a k-row are the same for the whole wave
// and come through scalar loads.  grid = (ceil(N / 256), ksplit): the four waves of a workgroup take a quarter of the
// workgroup's K range each and are summed through LDS, the K ranges of different workgroups through an fp32 workspace that
// skinny_reduce_kernel sums in split order (deterministic) and finishes with alpha, beta, bias and activation.
template <int MR, bool B16, bool VEC>
__global__ __launch_bounds__(256) void gemm_smallm_kernel(const GemmArgs g, float* __restrict__ ws, int kper)
{
    __shared__ f32x4 red[3][MR][64];
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int n = blockIdx.x * 256 + lane * 4;
    const int ks = blockIdx.y;
    const int kb = ks * kper, ke = min(g.K, kb + kper);
    const int kq = ((ke - kb + 3) >> 2);
    const int k0 = min(ke, kb + wave * kq), k1 = min(ke, k0 + kq);
    const float* __restrict__ A = (const float*)g.A;
    const int nvalid = g.N - n;                       // columns this lane owns: min(4, nvalid), none if <= 0

    auto load_b = [&](int k) -> f32x4 {
        f32x4 r = {0.0f, 0.0f, 0.0f, 0.0f};
        if (nvalid <= 0) return r;
        if constexpr (B16) {
            const uint16_t* p = (const uint16_t*)g.B + (long long)k * g.ldb + n;
            if (VEC) {
                u32x2 w = __builtin_nontemporal_load((const u32x2*)p);
                r[0] = f16_bits_to_float(w[0] & 0xFFFFu); r[1] = f16_bits_to_float(w[0] >> 16);
                r[2] = f16_bits_to_float(w[1] & 0xFFFFu); r[3] = f16_bits_to_float(w[1] >> 16);
            } else if (nvalid >= 4) {
                typedef u32x2 u32x2_a2 __attribute__((aligned(2)));
                const u32x2 w = *(const u32x2_a2*)p;
                r[0] = f16_bits_to_float(w[0] & 0xFFFFu); r[1] = f16_bits_to_float(w[0] >> 16);
                r[2] = f16_bits_to_float(w[1] & 0xFFFFu); r[3] = f16_bits_to_float(w[1] >> 16);
            } else {
#pragma unroll
                for (int e = 0; e < 4; e++) if (e < nvalid) r[e] = f16_bits_to_float(p[e]);
            }
        } else {
            const float* p = (const float*)g.B + (long long)k * g.ldb + n;
            if (VEC) r = __builtin_nontemporal_load((const f32x4*)p);      // B is read once per launch
            else if (nvalid >= 4) {
                // (rows off the 16-byte grid: one load at element alignment instead of four: 1 x 40109 x 1088 45 -> 35 us)
                typedef f32x4 f32x4_a4 __attribute__((aligned(4)));
                r = __builtin_nontemporal_load((const f32x4_a4*)p);
            } else {
#pragma unroll
                for (int e = 0; e < 4; e++) if (e < nvalid) r[e] = p[e];
            }
        }
        return r;
    };

    f32x4 acc[MR];
#pragma unroll
    for (int m = 0; m < MR; m++) acc[m] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
    const float* arow[MR];
#pragma unroll
    for (int m = 0; m < MR; m++) arow[m] = A + (long long)min(m, g.M - 1) * g.lda;

    int k = k0;
    for (; k + 8 <= k1; k += 8) {
        f32x4 b[8];
#pragma unroll
        for (int u = 0; u < 8; u++) b[u] = load_b(k + u);
#pragma unroll
        for (int m = 0; m < MR; m++) {
#pragma unroll
            for (int u = 0; u < 8; u++) {
                const float av = arow[m][k + u];
#pragma unroll
                for (int e = 0; e < 4; e++) acc[m][e] = fmaf(av, b[u][e], acc[m][e]);
            }
        }
    }
    for (; k < k1; k++) {
        const f32x4 b = load_b(k);
#pragma unroll
        for (int m = 0; m < MR; m++) {
            const float av = arow[m][k];
#pragma unroll
            for (int e = 0; e < 4; e++) acc[m][e] = fmaf(av, b[e], acc[m][e]);
        }
    }

    if (wave > 0) {
#pragma unroll
        for (int m = 0; m < MR; m++) red[wave - 1][m][lane] = acc[m];
    }
    __syncthreads();
    if (wave == 0 && nvalid > 0) {
#pragma unroll
        for (int m = 0; m < MR; m++) {
            if (m < g.M) {
                f32x4 v = acc[m];
#pragma unroll
                for (int w = 0; w < 3; w++) {
                    const f32x4 o = red[w][m][lane];
#pragma unroll
                    for (int e = 0; e < 4; e++) v[e] += o[e];
                }
                float* dst = ws + ((long long)ks * g.M + m) * g.N + n;
                if (VEC && (g.N & 3) == 0) *(f32x4*)dst = v;          // (rows of B may be padded beyond an N that is no multiple of 4)
                else {
#pragma unroll
                    for (int e = 0; e < 4; e++) if (e < nvalid) dst[e] = v[e];
                }
            }
        }
    }
}

// The same product in one launch for weights of a few megabytes, where the second launch and the partials cost more than the stream: a
// workgroup of 16 waves owns 64 columns and all of K.  A wave-load is four k-rows of 256 bytes; wave w takes the rows 4 w .. 4 w + 3 of
// every 64, SMALLM1_DEPTH of them in flight, against the rows of A in LDS ([k][MR], read as whole rows); the four k-rows of a wave are
// summed by lane exchanges, the waves through LDS, and the epilogue is applied there.  What bounds it is the memory round trip (times in
// one graph, two launches / one): 8 x 768 x 512 11.2 / 6.3 us, 1 x 768 x 512 7.0 / 3.8, 8 x 1024 x 1024 11.2 / 8.4, 1 x 16384 x 256 9.7 / 3.4; fp16
// weights 8 x 4096 x 512 12.4 / 7.0.
// Beyond a K of 1024 a workgroup's own stream is the longer (8 x 2048 x 2048 11.7 / 13.8, 1 x 768 x 3072 6.2 / 9.1), and wide weights keep
// every CU busy either way (1 x 40109 x 1088 35 / 36).  Up to one workgroup per CU (16384 columns) the form wins at any K (8 x 16384 x 1 4.9 /
// 4.6, x 16 6.2 / 4.9); with more of them a CU pays for starting and summing 16 waves several times over, which only the rows of a K of
// 128 or more repay (8 x 32768 x 128 11.3 / 8.7, but x 64 7.3 / 7.9; 8 x 65536 x 32 7.2 / 13.9; 8 x 262144 x 16 13.3 / 48).
#define SMALLM1_DEPTH 6
static bool smallm1_suits(int N, int K) { return K <= 1024 && (long long)N * K <= (1LL << 22) && (N <= 16384 || K >= 128); }
template <int MR, bool B16>
__global__ __launch_bounds__(1024) void gemm_smallm1_kernel(const GemmArgs g)
{
    extern __shared__ __attribute__((aligned(16))) float sm1[];
    float* red = sm1;                                         // [16 waves][MR][64]; first, so that its 16-byte stores are aligned at any K
    float* As = sm1 + 16 * MR * 64;                           // [K][MR]
    const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
    const int n0 = blockIdx.x * 64, n = n0 + 4 * (lane & 15);
    const int kr = 4 * wave + (lane >> 4);
    const int nvalid = g.N - n;
    auto load_b = [&](int k) -> f32x4 {
        f32x4 r = {0.0f, 0.0f, 0.0f, 0.0f};
        if (nvalid <= 0 || k >= g.K) return r;
        if constexpr (B16) {
            const uint16_t* p = (const uint16_t*)g.B + (long long)k * g.ldb + n;
            typedef u32x2 u32x2_a2 __attribute__((aligned(2)));
            if (nvalid >= 4) {
                const u32x2 w = *(const u32x2_a2*)p;
                r[0] = f16_bits_to_float(w[0] & 0xFFFFu); r[1] = f16_bits_to_float(w[0] >> 16);
                r[2] = f16_bits_to_float(w[1] & 0xFFFFu); r[3] = f16_bits_to_float(w[1] >> 16);
            } else
                for (int e = 0; e < 3; e++) if (e < nvalid) r[e] = f16_bits_to_float(p[e]);
        } else {
            const float* p = (const float*)g.B + (long long)k * g.ldb + n;
            typedef f32x4 f32x4_a4 __attribute__((aligned(4)));
            if (nvalid >= 4) r = *(const f32x4_a4*)p;
            else
                for (int e = 0; e < 3; e++) if (e < nvalid) r[e] = p[e];
        }
        return r;
    };
    f32x4 b[SMALLM1_DEPTH];
#pragma unroll
    for (int u = 0; u < SMALLM1_DEPTH; u++) b[u] = load_b(kr + 64 * u);
    for (int k = t; k < g.K; k += 1024) {
        float a[MR];
#pragma unroll
        for (int m = 0; m < MR; m++) a[m] = ((const float*)g.A)[(long long)min(m, g.M - 1) * g.lda + k];
#pragma unroll
        for (int m = 0; m < MR; m++) As[k * MR + m] = a[m];
    }
    __syncthreads();
    f32x4 acc[MR];
#pragma unroll
    for (int m = 0; m < MR; m++) acc[m] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
    for (int k0 = kr; k0 < g.K; k0 += 64 * SMALLM1_DEPTH) {
        if (k0 != kr) {
#pragma unroll
            for (int u = 0; u < SMALLM1_DEPTH; u++) b[u] = load_b(k0 + 64 * u);
        }
#pragma unroll
        for (int u = 0; u < SMALLM1_DEPTH; u++) {
            const int k = k0 + 64 * u;
            if (k >= g.K) break;
#pragma unroll
            for (int m = 0; m < MR; m++) {
                const float av = As[k * MR + m];
#pragma unroll
                for (int e = 0; e < 4; e++) acc[m][e] = fmaf(av, b[u][e], acc[m][e]);
            }
        }
    }
#pragma unroll
    for (int m = 0; m < MR; m++) {
#pragma unroll
        for (int e = 0; e < 4; e++) acc[m][e] = sum_with_partner32(sum_with_partner16(acc[m][e]));
        if (lane < 16) *(f32x4*)(red + (wave * MR + m) * 64 + 4 * lane) = acc[m];
    }
    __syncthreads();
    if (t >= MR * 64) return;
    const int m = t >> 6, col = n0 + lane;
    if (m >= g.M || col >= g.N) return;
    float v = 0.0f;
#pragma unroll
    for (int w = 0; w < 16; w++) v += red[(w * MR + m) * 64 + lane];
    v *= g.alpha;
    float* c = (float*)g.C + (long long)m * g.ldc + col;
    if (g.beta != 0.0f) v += g.beta * *c;
    if (g.bias) v += g.bias[col];
    *c = apply_activation(v, g.act, g.act_param);
}

// ---------------------------------------------------------------------------------------------
// Skinny-M fp32 path: 9 <= M <= 32, B stored [K,N], N % 128 == 0, K % 32 == 0 -- the fp32 form of gemm_skinny_kernel.
// HBM-bound: B is read exactly once.  grid = (N / 128, KS); a workgroup streams a 128-column slab of B over its K range through
// a ring of NS (three: two workgroups per CU) 20 KB stages (32 k-rows of 512 bytes of B and 32 rows of 128 bytes of A per stage, five
// direct-to-LDS loads per wave and K-tile), each wave multiplies the 32 x 32 block of its 32 columns on the fp32 MFMA (a 64-row
// tile of the general kernel would spend three quarters of its matrix work on padding and run at a quarter of the memory rate)
// and stores the partial product for skinny_reduce_kernel.
//   B tile [32 k][512 B]: chunk c of row k at position c ^ (((k >> 2) & 1) << 3)   (32-bit reads; the lane halves read rows 4 apart)
//   A tile [32 m][128 B]: chunk c of row m at position c ^ ((m >> 1) & 7)          (b128 reads)
// The k index of MFMA step i of 8-k group j is 8 j + 4 h + i for both operands (h = lane half).
#if AIDN_GEMM_PART == 0
template <int NS>
__global__ __launch_bounds__(256, NS <= 3 ? 2 : 1) void gemm_skinny32_kernel(const GemmArgs g, float* __restrict__ ws, int ksplit, int kper)
{
    constexpr int BK = 32, AHEAD = NS - 1;
    constexpr int ABYTES = 32 * 128, BBYTES = BK * 512, STAGE = ABYTES + BBYTES;
    extern __shared__ __attribute__((aligned(1024))) unsigned char smem[];      // NS stages

    const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
    const int l32 = lane & 31, h = lane >> 5;
    const int n0 = blockIdx.x * 128;
    const int ks = blockIdx.y;
    const int kbeg = ks * kper;
    const int KT = min(kper, g.K - kbeg) / BK;            // the last range may be shorter
    const float* __restrict__ A = (const float*)g.A;
    const float* __restrict__ B = (const float*)g.B;

    // this wave's DMA per K-tile: 4 B wave-loads (k-rows 2w', 2w'+1 with w' = 4 wave + i) and A wave-load `wave` (rows 8 wave ..)
    const float* pb[4];
#pragma unroll
    for (int i = 0; i < 4; i++) {
        const int row = 2 * (wave * 4 + i) + (lane >> 5), pos = lane & 31;
        pb[i] = B + (long long)(kbeg + row) * g.ldb + n0 + (pos ^ (((row >> 2) & 1) << 3)) * 4;
    }
    const float* pa;
    {
        const int row = 8 * wave + (lane >> 3), pos = lane & 7;
        const int grow = min(row, g.M - 1);
        pa = A + (long long)grow * g.lda + kbeg + (pos ^ ((row >> 1) & 7)) * 4;
    }
    auto issue_loads = [&](int kt, int stage) {
        unsigned char* as = smem + stage * STAGE;
        unsigned char* bs = as + ABYTES;
        dma16_to_lds(pa + kt * BK, as + wave * 1024);
#pragma unroll
        for (int i = 0; i < 4; i++) dma16_to_lds_stream(pb[i] + (long long)kt * BK * g.ldb, bs + (wave * 4 + i) * 1024);
    };

    const int a_off = l32 * 128, a_sw = (l32 >> 1) & 7;
    const int b_col = wave * 32 + l32;                  // column inside the slab

    f32x16 acc;
#pragma unroll
    for (int r = 0; r < 16; r++) acc[r] = 0.0f;

    for (int kt = 0; kt < AHEAD && kt < KT; kt++) issue_loads(kt, kt);
    int stage = 0;
    for (int kt = 0; kt < KT; kt++) {
        // tiles kt+1 .. kt+AHEAD-1 (those that exist) are younger than tile kt: five loads per wave each
        switch (min(KT - 1 - kt, AHEAD - 1)) {
            case 0: asm volatile("s_waitcnt vmcnt(0)" ::: "memory"); break;
            case 1: asm volatile("s_waitcnt vmcnt(5)" ::: "memory"); break;
            case 2: asm volatile("s_waitcnt vmcnt(10)" ::: "memory"); break;
            case 3: asm volatile("s_waitcnt vmcnt(15)" ::: "memory"); break;
            case 4: asm volatile("s_waitcnt vmcnt(20)" ::: "memory"); break;
            default: asm volatile("s_waitcnt vmcnt(25)" ::: "memory"); break;
        }
        __syncthreads();            // everyone's part of tile kt has landed, and everyone has left tile kt-1
        if (kt + AHEAD < KT) issue_loads(kt + AHEAD, stage == 0 ? NS - 1 : stage - 1);      // into the stage tile kt-1 used
        const unsigned char* as = smem + stage * STAGE;
        const unsigned char* bs = as + ABYTES;
#pragma unroll
        for (int j = 0; j < 4; j++) {
            const u32x4 fa = *(const u32x4*)(as + a_off + (((2 * j + h) ^ a_sw) << 4));
            u32x4 fb;
#pragma unroll
            for (int i = 0; i < 4; i++) {
                const int row = 8 * j + 4 * h + i;          // (row >> 2) & 1 == h
                fb[i] = *(const uint32_t*)(bs + row * 512 + ((((b_col >> 2) ^ (h << 3)) << 4) + (b_col & 3) * 4));
            }
            Mma32<float>::run(acc, fa, fb);
        }
        stage = stage + 1 == NS ? 0 : stage + 1;
    }

    const int col = n0 + b_col;
#pragma unroll
    for (int r = 0; r < 16; r++) {
        const int row = acc_row(r, h);
        if (row < g.M) ws[((long long)ks * g.M + row) * g.N + col] = acc[r];
    }
}
#endif

[[maybe_unused]] static bool skinny32_applies(int M, int N, int K) { return M > 8 && M <= 32 && N % 128 == 0 && K % 32 == 0 && N >= 128; }

// The fp32 skinny kernel runs a three-stage ring, two workgroups per CU: a workgroup's first memory round trip and its last tiles
// run under the other's stream (against seven stages and one per CU: 16 x 8192 x 8192 57.3 -> 48.3 us, 16 x 28672 x 8192 204 -> 171 us,
// 16 x 11008 x 4096 50.3 -> 41.1 us, 16 x 4096 x 4096 20.1 -> 18.4 us).  K-tiles per range; *ks ranges.
#define SKINNY32_STAGES 3
[[maybe_unused]] static int skinny32_plan(int N, int K, int* ks) { return skinny_plan(N / 128, K / 32, ks, 2); }
[[maybe_unused]] static int skinny32_ksplit(int N, int K) { int ks; skinny32_plan(N, K, &ks); return ks; }

// fp32: estimated run time (microseconds) of the direct-to-LDS kernel with `tile` x `tile` tiles when K is cut into `ks` ranges
// that run as batches.  A CU works through its tiles at the same total rate whether it holds one or two at a time, so the time
// is (tiles of the busiest CU) x (MFMA time of one padded tile); per flop the 256 and 128 tiles run at about 0.88 and the 64
// tile at about 0.75 of the fp32 peak (614 GFLOP/s per CU).  K ranges add the pass that sums the fp32 partials.  The estimate
// reproduces what was measured where the choice matters (128 x 50304 x 768: 186 / 93 / 96 us estimated for the three tiles,
// 179 / 93 / 84 measured; 16 x 4096 x 4096 on 64 x 64 tiles: 73 estimated, 77 measured).
[[maybe_unused]] static double f32_time_us(int M, int N, int K, long long batch, int tile, int ks)
{
    const long long wg = (long long)((M + tile - 1) / tile) * ((N + tile - 1) / tile) * batch * ks;
    const double rounds = wg <= 2048 ? (double)((wg + 255) / 256) : (double)wg / 256.0 + 0.5;
    // the 64 x 64 tile comes close to the rate of the larger ones once several workgroups share a CU (3000 x 4096 x 4096: 3008 tiles
    // at 0.88 of the pipe; with operands beyond the caches its doubled traffic per flop costs a few per cent), and 0.75 with one
    // per CU, where a lone wave per SIMD overlaps nothing
    const double eff = tile == 64 ? (wg >= 1024 ? 0.85 : wg >= 512 ? 0.80 : 0.75) : 0.88;
    double tile_us = 2.0 * tile * tile * (double)(K / ks) / (0.614e6 * eff) + 1.5;
    // measured: the 128 x 128 instance with edge handling takes 922 us where the plain one takes 721 us on 768 tiles (M = 2945..3071
    // against 3072, N = K = 4096; one ragged row is enough), 3 % more on 256 tiles (M = 1023) and nothing extra on 1536 tiles.  Two
    // such workgroups share a CU; 512 tiles take 470 us with either instance, and the 256 tiles of the last round are then spread
    // one per CU (+250 us) or packed two per CU on half the chip (+450 us) -- the hardware dispatcher's placement, which came out
    // the second way for the edge instance; the 64 x 64 instance shows no such step
    if (tile == 128 && (M % 128 != 0 || N % 128 != 0)) tile_us *= wg > 512 && wg <= 1024 ? 1.25 : 1.03;
    double t = rounds * tile_us;
    if (ks > 1) t += 3.0 + (double)(ks + 2) * M * N * 4.0 / 3.0e6;
    return t;
}

// fp32 tile edge for a problem that is not split (256 only where the direct-to-LDS kernel may run it)
[[maybe_unused]] static int f32_tile(int M, int N, int K, long long batch, bool allow256)
{
    int best = 128;
    double bt = f32_time_us(M, N, K, batch, 128, 1);
    const double t64 = f32_time_us(M, N, K, batch, 64, 1);
    if (t64 < bt) { bt = t64; best = 64; }
    if (allow256 && f32_time_us(M, N, K, batch, 256, 1) <= bt) best = 256;
    return best;
}

// fp32 split-K: number of K ranges (1 = none) that the estimate prefers for a single product.  Ranges are equal multiples of 32
// of at least 256; a split must beat the unsplit estimate by 15 % to be taken (it costs a second launch and workspace).
[[maybe_unused]] static int splitk32_ranges(int M, int N, int K)
{
    if (K < 1024 || K % 32 != 0) return 1;
    double best = f32_time_us(M, N, K, 1, f32_tile(M, N, K, 1, true), 1) * 0.95;
    int best_ks = 1;
    const int cand[7] = {2, 3, 4, 6, 8, 12, 16};
    for (int i = 0; i < 7; i++) {
        const int ks = cand[i];
        if (K % (ks * 32) != 0 || K / ks < 256) continue;
        const double t = std::min(f32_time_us(M, N, K, 1, 128, ks), f32_time_us(M, N, K, 1, 64, ks));
        if (t < best) { best = t; best_ks = ks; }
    }
    return best_ks;
}

#if AIDN_GEMM_PART == 0
// ---- fp32 products on the bf16 matrix pipe (gemm_split.hip): tile and K ranges by an estimate of the run time in microseconds.
// A WG advances by one K-tile of 32 in us[n - 1] with n of them on a CU and needs `once` for its first loads and its epilogue; the operands
// come at 6.4 TB/s (fp16 weights 4.5), or 2.9 where B lies beyond the last-level cache; ranges add the summing pass, 8 bytes a partial
// element at 5 TB/s.  Fitted on 963 (fp32) and 325 (fp16
// weights) timings of 140 shapes, M 9 - 8192, N 64 - 60000, K 64 - 16384, to 9 and 11 %; the plan it picks is 1 and 2 % behind the best one in the mean.
struct SplitTile { int id, rows, cols, resident; double us[2][3], once[2]; };
static const SplitTile kSplitTiles[3] = {{64, 64, 128, 3, {{1.25, 1.77, 2.30}, {0.97, 1.34, 1.72}}, {0.0, 0.0}},
                                         {128, 128, 128, 2, {{1.89, 2.57, 0.0}, {1.66, 2.10, 0.0}}, {1.7, 0.9}},
                                         {192, 128, 192, 2, {{3.00, 4.17, 0.0}, {0.0, 0.0, 0.0}}, {3.6, 0.0}}};      // (fp32 only)
struct SplitPlan { int tile = 0, ks = 1, kper = 0; double us = 1e30; };
static SplitPlan split_plan(int M, int N, int K, int batch, bool b16, size_t partial_bytes)
{
    SplitPlan best;
    // (from K = 4 on the error is no larger than the fp32 pipe's, whose products are exact and whose sums are rounded: rms over |result| and largest
    // over sum |a b| 2^-24, that pipe / split, K = 1 2.5e-8 / 3.5e-8 and 1.0 / 2.7, K = 3 3.6e-8 / 3.3e-8 and 2.74 / 2.85, K = 4 4.0e-8 / 3.2e-8 and 3.2 / 2.4)
    if (K < 4 || N < 2 || N >= (1 << 21) || K >= (1 << 21)) return best;
    const int kt = (K + 31) / 32;
    // (a B beyond the last-level cache, 54 x 42236 x 1216: 76 us from memory, 64 from the cache)
    const double b_bytes = (b16 ? 2.0 : 4.0) * K * N * batch;
    const double bytes_us = (4.0 * M * K * batch + b_bytes) / (b_bytes > 1.5e8 ? 2.9e6 : b16 ? 4.5e6 : 6.4e6);
    static const int ranges[] = {1, 2, 3, 4, 6, 8, 12, 16, 24, 32};
    for (const SplitTile& s : kSplitTiles) {
        if (s.id == 192 && (b16 || M % 128 != 0 || N % 192 != 0 || K % 32 != 0)) continue;
        const long long tiles = (long long)((M + s.rows - 1) / s.rows) * ((N + s.cols - 1) / s.cols) * batch;
        for (int want : ranges) {
            if (want > 1 && (batch > 1 || kt / want < 2 || tiles * want > 1600)) break;
            const int per = (kt + want - 1) / want, ks = (kt + per - 1) / per;
            if (ks > 1 && (size_t)ks * M * N * sizeof(float) > partial_bytes) break;
            const long long wgs = tiles * ks, slots = 256LL * s.resident;
            double rounds, tile_us;                       // rounds of resident workgroups, and the time of one K-tile in all of them
            if (wgs >= 4 * slots) { rounds = (double)wgs / slots; tile_us = rounds * s.us[b16][s.resident - 1]; }
            else {
                const long long full = wgs / slots, last = (wgs - full * slots + 255) / 256;
                rounds = (double)full + (last ? 1.0 : 0.0);
                tile_us = full * s.us[b16][s.resident - 1] + (last ? s.us[b16][last - 1] : 0.0);
            }
            double us = tile_us * per + rounds * s.once[b16];
            if (us < bytes_us) us = bytes_us;
            us += (b16 ? 5.6 : 5.4) + (ks > 1 ? 3.0 + 8.0 * ks * M * N / 5.0e6 : 0.0);
            if (us < best.us) best = SplitPlan{s.id, ks, ks > 1 ? per * 32 : 0, us};
        }
    }
    return best;
}
// What the kernels on the fp32 pipe need for the same product: the estimate above for rows in whole 16-byte chunks; else (and for fp16
// weights) the general kernel's 64 x 64 tiles at the measured time of 64 k.  They stay ahead on small products, whose few K-tiles they
// walk with twice the K to a barrier (288 x 512 x 192 7.0 us against 10.1, 41 x 2304 x 1536 12.9 / 16.9).
static double fp32_pipe_us(int M, int N, int K, int batch, bool b16, bool* two_launches)
{
    *two_launches = false;
    const bool chunks = K % 4 == 0 && N % 4 == 0;
    if (!b16 && chunks) {
        double us = f32_time_us(M, N, K, batch, f32_tile(M, N, K, batch, true), 1);
        const int ks = batch == 1 ? splitk32_ranges(M, N, K) : 1;
        if (ks > 1) { us = std::min(f32_time_us(M, N, K, 1, 128, ks), f32_time_us(M, N, K, 1, 64, ks)); *two_launches = true; }
        return us + 2.5;
    }
    const long long tiles = (long long)((M + 63) / 64) * ((N + 63) / 64) * batch;
    // (244 x 853 x 1024 0.66 a step, 2317 x 90 x 512 and 605 x 1338 x 12992 1.6 - 1.7; beyond one tile per CU the tiles share it)
    const double step = (b16 ? (chunks ? 2.0 : 3.2) : K % 4 != 0 ? 1.3 : M <= 512 && K <= 1024 ? 0.72 : 1.6) * (tiles > 256 ? 2.0 : 1.0);
    return 5.0 + step * ((K + 63) / 64) * ((tiles + 255) / 256);
}
static SplitPlan split_choice(int M, int N, int K, int batch, bool b16, size_t partial_bytes)
{
    const SplitPlan p = split_plan(M, N, K, batch, b16, partial_bytes);
    bool two;
    const double other = fp32_pipe_us(M, N, K, batch, b16, &two);
    // a call costs its caller about 9.5 us, one of two launches 12, whatever its kernels take (10 x 320 x 640: one launch of 14.5, two of 11)
    auto call = [](double us, bool two_launches) { return std::max(us, two_launches ? 12.0 : 9.5) + 0.05 * us; };
    return 1.08 * call(p.us, p.ks > 1) < call(other, two) ? p : SplitPlan{};
}
static hipError_t run_split(const GemmArgs& g, const SplitPlan& p, int batch, hipStream_t stream, void* workspace, bool b16)
{
    if (p.ks == 1) return launch_gemm_split(g, batch, stream, p.tile, b16);
    GemmArgs gp = g;                                      // the K ranges as batches into fp32 partials, summed in their order
    gp.C = workspace; gp.K = p.kper; gp.k_total = g.K; gp.ldc = g.N; gp.alpha = 1.0f; gp.beta = 0.0f;
    gp.sA = p.kper; gp.sB = (long long)p.kper * g.ldb; gp.sB2 = 0; gp.sC = (long long)g.M * g.N;
    gp.bias = nullptr; gp.act = 0;
    if (hipError_t e = launch_gemm_split(gp, p.ks, stream, p.tile, b16)) return e;
    hipLaunchKernelGGL((skinny_reduce_kernel<float>), dim3((unsigned)(((long long)g.M * g.N + 255) / 256)), dim3(256), 0, stream, (const float*)workspace,
                       g.C, g.M, g.N, p.ks, g.bias, g.act, g.act_param, g.alpha, g.beta);
    return hipGetLastError();
}
#endif

static bool smallm_applies(int M, int N, int K) { return M >= 1 && M <= 8 && (long long)N * K >= 4096; }

// K range of one workgroup: about 1024 workgroups, at least 128 k-rows each (32 per wave), a multiple of 32
static int smallm_kper(int N, int K)
{
    const int colblocks = (N + 255) / 256;
    int ks = (1024 + colblocks - 1) / colblocks;
    int kper = (K + ks - 1) / ks;
    if (kper < 128) kper = 128;
    kper = (kper + 31) / 32 * 32;
    // K ranges that start a multiple of 4 MiB apart put the workgroups of a column block on the same memory channels
    // (1 x 8192 x 8192: 60 us with 256-row ranges, 8 MiB apart, against 43-48 us with any other size)
    for (int tries = 0; tries < 64 && ((long long)kper * N * 4) % (1LL << 22) == 0; tries++) kper += 8;   // (bounded: a very wide N aliases at every multiple of 32)
    return kper;
}

#if AIDN_GEMM_PART == 0
size_t gemm_smallm_workspace_bytes(int M, int N, int K)
{
    if (!smallm_applies(M, N, K) || smallm1_suits(N, K)) return 0;      // (the one-launch form keeps its sums in LDS)
    const int kper = smallm_kper(N, K);
    return (size_t)((K + kper - 1) / kper) * M * N * sizeof(float);
}
// fp32 problems with B [N,K] whose rows are not whole 16-byte chunks (K not a multiple of 4): zero-padded copies of A and B in the
// workspace (K up to a multiple of 32) feed the direct-to-LDS kernel.  Same sums as the plain product: the padding contributes exact
// zeros.  The layout (with N up to a multiple of 4 for B [K,N]) is also that of a packed B.
struct Pad32Plan { int Np, Kp; size_t a_off, b_off, total; };
static bool pad32_layout(int M, int N, int K, int transB, Pad32Plan* pl)
{
    pl->Kp = (K + 31) / 32 * 32;
    pl->Np = transB ? N : (N + 3) / 4 * 4;
    if (pl->Kp >= (1 << 21) || pl->Np >= (1 << 21)) return false;
    auto up = [](size_t b) { return (b + 255) & ~(size_t)255; };
    pl->a_off = 0;
    pl->b_off = up((size_t)M * pl->Kp * 4);
    pl->total = pl->b_off + up((size_t)(transB ? N : pl->Kp) * (transB ? pl->Kp : pl->Np) * 4);
    return pl->total <= ((size_t)4 << 30);
}
static bool pad32_plan(int M, int N, int K, Pad32Plan* pl)       // B [N,K]
{
    if (K % 4 == 0 || N < 16 || (double)M * N * K < (double)(1 << 21)) return false;
    if (M <= 512 && K <= 1024) return false;          // as for 16-bit: the general kernel reads the rows in place
    return pad32_layout(M, N, K, 1, pl);
}

// Pre-packed fp32 B (the caller keeps it): [K,N] zero-padded to [Kp, Np], or [N,K] to [N, Kp] -- the GPU form of the reference's
// cached packed weight operand (SimdGemm.SgemmWithCachedB / PrePackedB): packed once, the product is that of the plain call.
size_t gemm_f32_packed_b_bytes(int N, int K, int transB)
{
    Pad32Plan pl;
    if (N <= 0 || K <= 0 || !pad32_layout(1, N, K, transB, &pl)) return 0;
    return (size_t)(transB ? N : pl.Kp) * (transB ? pl.Kp : pl.Np) * 4;
}
hipError_t gemm_f32_pack_b(hipStream_t stream, const float* B, int K, int N, int transB, void* packed)
{
    Pad32Plan pl;
    if (!pad32_layout(1, N, K, transB, &pl) || !aligned16(packed)) return hipErrorInvalidValue;
    return transB ? pad_rows(stream, B, packed, N, K, N, pl.Kp, 4) : pad_rows(stream, B, packed, K, N, pl.Kp, pl.Np, 4);
}
size_t gemm_f32_packed_workspace_bytes(int M, int N, int K, int transB)
{
    Pad32Plan pl;
    if (!pad32_layout(M, N, K, transB, &pl)) return 0;
    size_t need = pl.b_off;                                           // the padded copy of A, or partials
    if (!transB) {
        if (smallm_applies(M, N, K)) need = std::max(need, gemm_smallm_workspace_bytes(M, N, K));
        const SplitPlan sp = split_choice(M, N, K, 1, false, SIZE_MAX);
        if (sp.ks > 1) need = std::max(need, (size_t)sp.ks * M * N * sizeof(float));
    }
    return need;
}

size_t gemm_f32_f16weight_workspace_bytes(int M, int N, int K)
{
    if (smallm_applies(M, N, K)) return gemm_smallm_workspace_bytes(M, N, K);
    const SplitPlan sp = split_choice(M, N, K, 1, true, SIZE_MAX);
    return sp.ks > 1 ? (size_t)sp.ks * M * N * sizeof(float) : 0;
}

// The largest need over every plan gemm_f32 may take for these dimensions: which one it takes also depends on the alignment of
// the operands, which the sizing does not see, and every plan checks its own need against the bytes it is handed.
size_t gemm_f32_workspace_bytes(int M, int N, int K, int transB)
{
    size_t need = 0;
    auto upto = [&](size_t n) { if (n > need) need = n; };
    if (!transB && smallm_applies(M, N, K) && smallm1_suits(N, K)) return 0;      // taken at any alignment
    Pad32Plan pl;
    if (transB && pad32_plan(M, N, K, &pl)) upto(pl.total);
    if (!transB && !smallm_applies(M, N, K) && !skinny32_applies(M, N, K)) {
        const SplitPlan sp = split_choice(M, N, K, 1, false, SIZE_MAX);
        if (sp.ks > 1) upto((size_t)sp.ks * M * N * sizeof(float));
    }
    if (!transB && smallm_applies(M, N, K)) upto(gemm_smallm_workspace_bytes(M, N, K));
    if (!transB && skinny32_applies(M, N, K)) upto((size_t)skinny32_ksplit(N, K) * M * N * sizeof(float));
    const int ks = splitk32_ranges(M, N, K);
    if (ks > 1) upto((size_t)ks * M * N * sizeof(float));
    return need;
}
#endif

template <bool B16>
static hipError_t launch_smallm(const GemmArgs& g, hipStream_t stream, float* ws)
{
    const int mr = g.M <= 1 ? 1 : g.M <= 2 ? 2 : g.M <= 4 ? 4 : 8;
    if (smallm1_suits(g.N, g.K)) {
        const int bytes = (g.K + 16 * 64) * mr * 4;                       // A and the waves' sums: 64 KiB at most
        const dim3 one((unsigned)((g.N + 63) / 64));
        if (mr == 1) hipLaunchKernelGGL((gemm_smallm1_kernel<1, B16>), one, dim3(1024), bytes, stream, g);
        else if (mr == 2) hipLaunchKernelGGL((gemm_smallm1_kernel<2, B16>), one, dim3(1024), bytes, stream, g);
        else if (mr == 4) hipLaunchKernelGGL((gemm_smallm1_kernel<4, B16>), one, dim3(1024), bytes, stream, g);
        else hipLaunchKernelGGL((gemm_smallm1_kernel<8, B16>), one, dim3(1024), bytes, stream, g);
        return hipGetLastError();
    }
    const int kper = smallm_kper(g.N, g.K);
    const int ks = (g.K + kper - 1) / kper;
    // whole 16-byte loads of B: rows in 16-byte steps that hold every chunk a lane may touch (N a multiple of 4, or rows padded to one)
    const bool vec = (g.N % 4 == 0 || g.ldb >= (g.N + 3) / 4 * 4) && g.ldb % 4 == 0 && (((uintptr_t)g.B) & (B16 ? 7u : 15u)) == 0;
    const dim3 grid((unsigned)((g.N + 255) / 256), (unsigned)ks);
#define AIDN_SMALLM(MR_)                                                                                               \
    do {                                                                                                               \
        if (vec) hipLaunchKernelGGL((gemm_smallm_kernel<MR_, B16, true>), grid, dim3(256), 0, stream, g, ws, kper);     \
        else hipLaunchKernelGGL((gemm_smallm_kernel<MR_, B16, false>), grid, dim3(256), 0, stream, g, ws, kper);        \
    } while (0)
    if (mr == 1) AIDN_SMALLM(1);
    else if (mr == 2) AIDN_SMALLM(2);
    else if (mr == 4) AIDN_SMALLM(4);
    else AIDN_SMALLM(8);
#undef AIDN_SMALLM
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
    const long long total = (long long)g.M * g.N;
    hipLaunchKernelGGL((skinny_reduce_kernel<float>), dim3((unsigned)((total + 255) / 256)), dim3(256), 0, stream, ws, g.C, g.M, g.N, ks,
                       g.bias, g.act, g.act_param, g.alpha, g.beta);
    return hipGetLastError();
}

// ------------------------------------------------------------------ host side
template <typename T, typename OutT, int BM, int BN, int WM, int WN, bool TRANSB, bool VEC, bool CHECK, int KS = 1, bool B16 = false>
static hipError_t launch_gemm(GemmArgs g, int batch, hipStream_t stream)
{
    auto kern = gemm_kernel<T, OutT, BM, BN, WM, WN, TRANSB, VEC, CHECK, KS, B16>;
    constexpr int tiles_smem = 2 * (BM + BN) * gemm_row_pitch(BM, BN), merge_smem = KS == 2 ? BM * BN * 4 : 0;
    constexpr int smem = tiles_smem > merge_smem ? tiles_smem : merge_smem;
    static unsigned long long attr_done = 0;
    if (hipError_t e = ensure_dynamic_smem((const void*)kern, smem, &attr_done)) return e;
    g.tiles_m = (g.M + BM - 1) / BM;
    g.tiles_n = (g.N + BN - 1) / BN;
    dim3 grid((unsigned)(g.tiles_m * g.tiles_n), 1, (unsigned)batch);
    hipLaunchKernelGGL(kern, grid, dim3(WM * WN * KS * 64), smem, stream, g);
    return hipGetLastError();
}



// 128 x 128 or 64 x 64 tile; rel64 = efficiency per flop of the smaller tile relative to the larger one when both load the
// CUs equally well (measured: about 0.85 for fp32, 0.55 for the 16-bit types).
static int choose_tile(long long tiles128, long long tiles64, double rel64)
{
    return cu_fill(tiles128) >= rel64 * cu_fill(tiles64) ? 128 : 64;
}

// what the 16 x 16 x 32 kernel needs beyond whole tiles: 16-byte aligned operand rows, C rows and bias, and the plain product
template <typename OutT>
static bool dl16_applies(const GemmArgs& g)
{
    const int OB = Elem<OutT>::BYTES;
    return g.N % 8 == 0 && aligned16(g.A) && aligned16(g.B) && g.lda % 8 == 0 && g.ldb % 8 == 0 && g.sA % 8 == 0 && g.sB % 8 == 0 && g.sB2 % 8 == 0 &&
           g.lda < (1 << 21) && g.ldb < (1 << 21) &&
           aligned16(g.C) && ((long long)g.ldc * OB) % 16 == 0 && (g.sC * OB) % 16 == 0 && (g.bias == nullptr || aligned16(g.bias)) &&
           g.alpha == 1.0f && g.beta == 0.0f;
}

// Tile width (in 64-column units: 4, 3 or 2) of the 16 x 16 x 32 kernel for a 16-bit problem with K % 64 == 0 (any M and N), or 0
// when the 128 x 128 / 64 x 64 tiles of the 32 x 32 x 16 kernel are expected to finish earlier.
// Every candidate is scored as (how evenly its tiles load the 256 CUs) x (its rate per flop relative to the 256 x 256 tile): a
// narrower tile moves more A bytes per flop (and the 256 x 128 one wastes half of its B loads); the 128 x 128 tile runs at about
// 0.55 and the 64 x 64 tile at about 0.45 of the 256 x 256 rate (2048^3: 128 tiles of 256 x 128 take 36 us, 256 tiles of 128 x 128 29 us).
// A last tile column that N does not fill costs only its padding: before, such an N went to the next width that divides it or to the
// 32 x 32 x 16 kernel with its checks on every K-tile (bf16, us before / now: 1000 x 11008 x 4096 94 / 86, 917 x 15416 x 4416 156 / 113,
// 1158 x 3008 x 1088 20.2 / 13.9, 5236 x 6464 x 6400 469 / 397; 44 drawn sizes 1.07x in the geometric mean).
#define DL16_HALF_EFF 0.7
// The 128 x 128 tile on the two-stage ring runs two workgroups per CU, so that one's first loads and stores run under the other's products:
// the shorter K, the more that counts (rate against the 256 x 256 tile's, us before / with the entry for that K: 7002 x 8112 x 64 44.8 / 33.0,
// 8192 x 14592 x 128 83 / 75, 7002 x 3072 x 256 24.7 / 22.6, 4096 x 10112 x 576, on 256 x 256 tiles, 58.7 / 56.2; at 0.95 8192 x 14592 x 576
// goes 182 -> 203)
static double dl16_half2_eff(int K) { return K <= 128 ? 1.2 : K <= 384 ? 0.95 : K <= 640 ? 0.9 : 0.82; }
static int dl16_width(int M, int N, int K, int batch, double* score_out)
{
    if (score_out) *score_out = 0.0;
    if (K % 64 != 0) return 0;
    // M and N may be ragged (partial last tiles: clamped loads, guarded stores); the rows and columns a tile pads count as waste
    const long long tm256 = (M + 255) / 256, tm128 = (M + 127) / 128, tm64 = (M + 63) / 64;
    const double use256 = (double)M / (double)(tm256 * 256), rows128 = (double)M / (double)(tm128 * 128), rows64 = (double)M / (double)(tm64 * 64);
    const long long tn128 = (N + 127) / 128, tn64 = (N + 63) / 64;
    const double use128 = rows128 * (double)N / (double)(tn128 * 128), use64 = rows64 * (double)N / (double)(tn64 * 64);
    const int widths[3] = {4, 3, 2};
    const double eff[3] = {1.0, 0.94, 0.8};
    int best = 0;
    double best_score = 0.0;
    for (int i = 0; i < 3; i++) {
        const int bn = 64 * widths[i];
        const long long tn = (N + bn - 1) / bn, t = tm256 * tn * batch;
        const double score = cu_fill(t) * eff[i] * use256 * ((double)N / (double)(tn * bn));
        if (score > best_score) { best_score = score; best = widths[i]; }
    }
    const long long t128 = tm128 * tn128 * batch;
    const long long t64 = tm64 * tn64 * batch;
    // the 128 x 128 tile of this kernel (code 1)
    if (DL16_HALF_EFF * cu_fill(t128) * use128 > best_score) { best_score = DL16_HALF_EFF * cu_fill(t128) * use128; best = 1; }
    // the same tile on a two-stage ring, two workgroups per CU (code 5): with more tiles than CUs and a K of at most 6144 one
    // workgroup's first loads, barrier waits and store phase run under the other's MFMAs (8192 x 768 x 3072 50.4 -> 41.8 us,
    // 512 x 12288 x 4096 64.8 -> 54.4 us, 384 x 13824 x 5120 79.8 -> 65.8 us); one tile per CU (2048^3 20.7 -> 27.6 us) and long K
    // (384 x 28672 x 8192 228 -> 265 us) need the deeper ring
    // (beyond one round of 512 resident workgroups only when the last round is nearly full: a workgroup alone on its CU has nothing
    // to hide the two-stage ring's waits behind -- 3000 x 4096 x 4096, 768 tiles: 83 -> 106 us)
    const double fill2 = (double)t128 / (double)(((t128 + 511) / 512) * 512);
    if (t128 > 256 && K <= 6144 && (t128 <= 512 || fill2 >= 0.85)) {
        const double s2 = dl16_half2_eff(K) * (t128 <= 512 ? cu_fill(t128) : fill2) * use128;
        if (s2 > best_score) { best_score = s2; best = 5; }
    }
    // M and N multiples of 64 and N not of 128: the 64 x 64 tile runs without edge handling and wastes nothing where every wider one is cut.
    // Against one round of 128 x 128 tiles it then counts for more, and at K = 128 against two workgroups per CU too (us, cut 128 x 128 / 64 x 64:
    // 512 x 4672 x 512 9.2 / 8.4, 384 x 6976 x 768 11.6 / 11.0, 640 x 3648 x 832 11.2 / 10.7, 1152 x 4032 x 128 7.8 / 7.3; from K = 192 on
    // two workgroups win, 1024 x 6464 x 384 11.7 / 13.0)
    const bool fits64 = M % 64 == 0 && N % 64 == 0 && N % 128 != 0;
    const double eff64 = fits64 && K <= 128 ? 0.76 : fits64 && best == 1 ? 0.53 : 0.45;
    const double s128 = 0.55 * cu_fill(t128) * use128, s64 = eff64 * cu_fill(t64) * use64;
    if (score_out) *score_out = best_score > s128 ? (best_score > s64 ? std::min(best_score, 1.0) : s64) : (s128 > s64 ? s128 : s64);
    if (s128 > best_score || s64 > best_score) return 0;
    return best;
}

// Kernel and tile choice: the 256 x 256 direct-to-LDS kernel for 16-bit B[K,N] problems with at least 128 such tiles,
// otherwise the general kernel with the 128 x 128 or 64 x 64 tile (choose_tile), in its branch-free instance when the
// operands are 16-byte aligned and the K-tile divides K.
template <typename T, typename OutT, bool TRANSB>
static hipError_t dispatch_gemm(const GemmArgs& g, int batch, hipStream_t stream, int force_tile)
{
    constexpr int E = Elem<T>::PER16;
    const bool vec = aligned16(g.A) && aligned16(g.B) && g.lda % E == 0 && g.ldb % E == 0 && g.K % E == 0 &&
                     (TRANSB || g.N % E == 0) && g.sA % E == 0 && g.sB % E == 0 && g.sB2 % E == 0;
    auto tiles = [&](int bm, int bn) { return (long long)((g.M + bm - 1) / bm) * ((g.N + bn - 1) / bn) * batch; };
    int tile = force_tile;
    if (tile == 0) {
        if constexpr (!TRANSB || E == 4) {
            // the direct-to-LDS kernel: rows of A and B in whole 16-byte chunks, leading dimensions within the 32-bit lane
            // offsets of its loads; M, N and K may be ragged
            if (vec && g.lda < (1 << 21) && g.ldb < (1 << 21) && (Elem<OutT>::BYTES == 4 || (g.alpha == 1.0f && g.beta == 0.0f))) {
                // 16-bit: the 256 x 256 tile moves half the bytes per flop of the 128 x 128 one and wins from half a chip of
                // tiles on; fp32 runs both at about the same rate per flop, so there the better CU load decides
                if constexpr (E == 8 && !TRANSB) {
                    if (dl16_applies<OutT>(g)) {
                        const int w = dl16_width(g.M, g.N, g.K, batch);
                        if (w == 4) return launch_gemm_dl16<T, OutT, 4>(g, batch, stream);
                        if (w == 3) return launch_gemm_dl16<T, OutT, 3>(g, batch, stream);
                        if (w == 2) return launch_gemm_dl16<T, OutT, 2>(g, batch, stream);
                        if (w == 1) return launch_gemm_dl16<T, OutT, 2, true>(g, batch, stream);
                        if (w == 5) return launch_gemm_dl16<T, OutT, 2, true, 2>(g, batch, stream);
                    }
                }
                if constexpr (E == 4) {
                    // fp32 runs every tile at about the same rate per flop: the estimated time, padding included, decides
                    const int t = f32_tile(g.M, g.N, g.K, batch, true);
                    tile = t == 256 ? 256 : t == 128 ? 129 : 65;
                } else {
                    const long long t256 = tiles(256, 256), t128 = tiles(128, 128);
                    // (16-bit, ragged or unaligned for the 16 x 16 x 32 kernel: the 256 x 256 tile of this kernel when it scores best)
                    const bool big = t256 >= 128 && cu_fill(t256) >= 0.55 * cu_fill(t128);
                    // otherwise the same kernel with 128 x 128 or 64 x 64 tiles (codes 129, 65), whichever loads the CUs better; per
                    // flop the 64 x 64 instance runs at about 0.8 of the 128 x 128 one
                    if (big) tile = 256;
                    else tile = choose_tile(t128, tiles(64, 64), 0.8) == 128 ? 129 : 65;
                }
            }
        }
        // (at most 64 rows: bound by the stream of B, which more and smaller workgroups keep fuller)
        if (tile == 0) tile = g.M <= 64 ? 64 : E == 4 ? f32_tile(g.M, g.N, g.K, batch, false) : choose_tile(tiles(128, 128), tiles(64, 64), 0.55);
    }
    if constexpr (E == 8 && !TRANSB) {
        if (tile == 192 || tile == 193) {                 // 256 x 192 / 256 x 128 tiles of the 16 x 16 x 32 kernel (whole tiles only)
            const int bn = tile == 192 ? 192 : 128;
            if (!(g.N % bn == 0 && g.K % 64 == 0 && dl16_applies<OutT>(g))) return hipErrorInvalidValue;
            return tile == 192 ? launch_gemm_dl16<T, OutT, 3>(g, batch, stream) : launch_gemm_dl16<T, OutT, 2>(g, batch, stream);
        }
    }
    if constexpr (E == 8 && !TRANSB) {
        if (tile == 131) {                                // the same on the two-stage ring (two workgroups per CU)
            if (!(g.N % 128 == 0 && g.K % 64 == 0 && dl16_applies<OutT>(g))) return hipErrorInvalidValue;
            return launch_gemm_dl16<T, OutT, 2, true, 2>(g, batch, stream);
        }
        if (tile == 130) {                                // 128 x 128 tiles of the 16 x 16 x 32 kernel (whole tiles only)
            if (!(g.N % 128 == 0 && g.K % 64 == 0 && dl16_applies<OutT>(g))) return hipErrorInvalidValue;
            return launch_gemm_dl16<T, OutT, 2, true>(g, batch, stream);
        }
    }
    if (tile == 192 || tile == 193 || tile == 130 || tile == 131) return hipErrorInvalidValue;
    if constexpr (E == 4 || !TRANSB) {
        if (tile == 65) {                                 // 64 x 64 tiles on the direct-to-LDS kernel
            if (!(vec && (TRANSB || g.N >= E) && g.lda < (1 << 21) && g.ldb < (1 << 21))) return hipErrorInvalidValue;
            if (Elem<OutT>::BYTES != 4 && (g.alpha != 1.0f || g.beta != 0.0f)) return hipErrorInvalidValue;
            const bool exact_fit = g.M % 64 == 0 && g.N % 64 == 0 && g.K % (8 * E) == 0 && g.c_cols == 0;
            if constexpr (E == 4 && !TRANSB) {
                // about one tile per CU: the eight-wave form (two k-step groups), so that every SIMD has a second wave to switch to
                if (exact_fit && tiles(64, 64) <= 512) return launch_gemm_dl<T, OutT, false, 64, TRANSB, 2>(g, batch, stream);
            }
            return exact_fit ? launch_gemm_dl<T, OutT, false, 64, TRANSB>(g, batch, stream) : launch_gemm_dl<T, OutT, true, 64, TRANSB>(g, batch, stream);
        }
    }
    if (tile == 65) tile = 64;
    if constexpr (!TRANSB || E == 4) {
        if (tile == 256 || tile == 129) {
            if (!(vec && (TRANSB || g.N >= E) && g.lda < (1 << 21) && g.ldb < (1 << 21))) return hipErrorInvalidValue;
            if (Elem<OutT>::BYTES != 4 && (g.alpha != 1.0f || g.beta != 0.0f)) return hipErrorInvalidValue;
            const int edge = tile == 256 ? 256 : 128;
            const bool exact_fit = g.M % edge == 0 && g.N % edge == 0 && g.K % (8 * E) == 0 && g.c_cols == 0;
            // (bf16 output with ragged edges on the 256 x 256 tile: that one instance does not fit the register file -- the
            // compiler moves accumulators to scratch memory -- so such problems take the 128 x 128 tile)
            constexpr bool kSpills256Edge = std::is_same<T, bf16_t>::value && std::is_same<OutT, bf16_t>::value;
            if constexpr (E == 8 && !TRANSB) {
                // 16-bit, whole tiles: the 16 x 16 x 32 kernel (its stores and bias loads are 16-byte vectors: C rows and the bias
                // must be 16-byte aligned; it computes act(A B + bias), so alpha = 1 and beta = 0)
                if (tile == 256 && exact_fit && dl16_applies<OutT>(g)) return launch_gemm_dl16<T, OutT, 4>(g, batch, stream);
            }
            if (tile == 256 && exact_fit) return launch_gemm_dl<T, OutT, false, 256, TRANSB>(g, batch, stream);
            if constexpr (!kSpills256Edge) {
                if (tile == 256) return launch_gemm_dl<T, OutT, true, 256, TRANSB>(g, batch, stream);
            }
            return exact_fit ? launch_gemm_dl<T, OutT, false, 128, TRANSB>(g, batch, stream) : launch_gemm_dl<T, OutT, true, 128, TRANSB>(g, batch, stream);
        }
    }
    if (tile == 129) tile = 128;
    if (g.c_cols > 0) return hipErrorInvalidValue;        // only the direct-to-LDS kernels above know that C is narrower than N
    // 16-byte aligned operands whose K the K-tile divides take the instance without bounds checks in its loop (no zero fill
    // is needed; rows and column blocks past the end are clamped loads whose products are never stored)
    auto exact = [&](int bt) { return vec && g.N >= E && g.K % (gemm_k_chunks(bt, bt) * E) == 0; };
    if (tile == 128) {
        if (exact(128)) return launch_gemm<T, OutT, 128, 128, 2, 2, TRANSB, true, false>(g, batch, stream);
        if (vec) return launch_gemm<T, OutT, 128, 128, 2, 2, TRANSB, true, true>(g, batch, stream);
        return launch_gemm<T, OutT, 128, 128, 2, 2, TRANSB, false, true>(g, batch, stream);
    }
    if (tile == 64) {
        // at most about one 64 x 64 tile per CU: split every K-tile between two wave groups so each SIMD still holds two waves
        if (vec && tiles(64, 64) <= 320 && g.K >= 4 * 16 * E) {
            if (exact(64)) return launch_gemm<T, OutT, 64, 64, 2, 2, TRANSB, true, false, 2>(g, batch, stream);
            return launch_gemm<T, OutT, 64, 64, 2, 2, TRANSB, true, true, 2>(g, batch, stream);
        }
        if (exact(64)) return launch_gemm<T, OutT, 64, 64, 2, 2, TRANSB, true, false>(g, batch, stream);
        if (vec) return launch_gemm<T, OutT, 64, 64, 2, 2, TRANSB, true, true>(g, batch, stream);
        return launch_gemm<T, OutT, 64, 64, 2, 2, TRANSB, false, true>(g, batch, stream);
    }
    return hipErrorInvalidValue;
}

template <typename E>
[[maybe_unused]] static void set_b3(GemmArgs& g, const E* const (&B)[3])
{
    auto at = [&](int i) { return (long long)((intptr_t)B[i] - (intptr_t)B[0]) / (long long)sizeof(E); };      // (whole elements: the blocks are aligned)
    g.sB = at(1);
    g.sB2 = at(2) - 2 * at(1);
}

// C [M, 3 n] = A [M, K] x [B0 | B1 | B2], the three [K, n] blocks wherever they are (row stride ldb): one launch of three batches that
// share A.  gemm_x3_suits: the tiles of an n-wide product load the chip as well as those of the 3 n-wide one would (n a multiple of 64,
// so that no tile is cut that was not cut before; estimates within 3 %) -- then B need not be copied side by side for it.
#if AIDN_GEMM_PART == 0
bool gemm_x3_suits(int kind, int M, int n, int K)
{
    if (n % 64 != 0) return false;
    if (kind == 0) {
        const SplitPlan s1 = split_choice(M, 3 * n, K, 1, false, 0), s3 = split_choice(M, n, K, 3, false, 0);
        if (s1.tile || s3.tile) return s3.tile && (!s1.tile || s3.us <= 1.03 * s1.us);
        const int t1 = f32_tile(M, 3 * n, K, 1, true), t3 = f32_tile(M, n, K, 3, true);
        return f32_time_us(M, n, K, 3, t3, 1) <= 1.03 * f32_time_us(M, 3 * n, K, 1, t1, 1);
    }
    double s1, s3;
    dl16_width(M, 3 * n, K, 1, &s1);
    dl16_width(M, n, K, 3, &s3);
    return s3 >= 0.97 * s1;
}
hipError_t gemm_f32_x3(hipStream_t stream, const float* A, const float* const (&B)[3], float* C, int M, int n, int K, int ldb, int force_tile)
{
    GemmArgs g{A, B[0], C, M, n, K, K, ldb, 3 * n, 0, 0, n, 1.0f, 0.0f, 0, 0, nullptr, 0, 0.0f};
    set_b3(g, B);
    const SplitPlan sp = force_tile == 0 ? split_choice(M, n, K, 3, false, 0) : SplitPlan{};
    if (sp.tile) return run_split(g, sp, 3, stream, nullptr, false);
    return dispatch_gemm<float, float, false>(g, 3, stream, force_tile);
}
#endif
template <typename T>
static hipError_t gemm_16_x3_typed(hipStream_t stream, const uint16_t* A, const uint16_t* const (&B)[3], uint16_t* C, int M, int n, int K, int ldb, int force_tile)
{
    GemmArgs g{A, B[0], C, M, n, K, K, ldb, 3 * n, 0, 0, n, 1.0f, 0.0f, 0, 0, nullptr, 0, 0.0f};
    set_b3(g, B);
    return dispatch_gemm<T, T, false>(g, 3, stream, force_tile);
}

#if AIDN_GEMM_PART == 0
hipError_t gemm_f32(hipStream_t stream, const float* A, const float* B, float* C, int M, int N, int K,
                    float alpha, float beta, int transB, int batch, long long sA, long long sB, long long sC,
                    int force_tile, const float* bias, int act, float act_param, void* workspace, const float* Bpre,
                    size_t workspace_bytes)
{
    GemmArgs g{A, B, C, M, N, K, K, transB ? K : N, N, sA, sB, sC, alpha, beta, 0, 0, bias, act, act_param};
    if (!workspace) workspace_bytes = 0;
    // every plan below that writes to the workspace first holds its own need against the bytes handed in, and is passed over
    // (down to the tiled kernels, which need none) when they do not suffice
    const bool smallm_fits = smallm_applies(M, N, K) && gemm_smallm_workspace_bytes(M, N, K) <= workspace_bytes;
    if (!Bpre && force_tile == 0 && smallm_fits && !transB && batch == 1)
        return launch_smallm<false>(g, stream, (float*)workspace);
    // Bpre: B already packed by gemm_f32_pack_b (B itself is then not read)
    Pad32Plan pl;
    if (Bpre && !(batch == 1 && aligned16(Bpre) && pad32_layout(M, N, K, transB, &pl))) return hipErrorInvalidValue;
    if (Bpre && !transB) {
        GemmArgs gs = g;
        gs.B = Bpre; gs.ldb = pl.Np;                 // the padded rows; only the first K of them are read
        if (smallm_fits) return launch_smallm<false>(gs, stream, (float*)workspace);
        const SplitPlan sp = split_choice(M, N, K, 1, false, workspace_bytes);
        if (sp.tile) return run_split(gs, sp, 1, stream, workspace, false);
    }
    if (Bpre && !(pl.Kp == K ? aligned16(A) : (workspace && aligned16(workspace) && pl.b_off <= workspace_bytes))) return hipErrorInvalidValue;
    if (!Bpre && force_tile == 0 && !transB) {
        // (M <= 32 on whole slabs: bound by the stream of B, which the skinny kernel below keeps fuller)
        int ks;
        const bool skinny = batch == 1 && workspace && skinny32_applies(M, N, K) && aligned16(A) && aligned16(B) && skinny32_plan(N, K, &ks) > 0 &&
                            (size_t)ks * M * N * sizeof(float) <= workspace_bytes;
        const SplitPlan sp = skinny ? SplitPlan{} : split_choice(M, N, K, batch, false, workspace_bytes);
        if (sp.tile) return run_split(g, sp, batch, stream, workspace, false);
    }
    if (Bpre || (transB && force_tile == 0 && workspace && batch == 1 && aligned16(workspace) && pad32_plan(M, N, K, &pl) && pl.total <= workspace_bytes)) {
        unsigned char* w = (unsigned char*)workspace;
        const float* Ap = A;
        if (pl.Kp != K) {
            if (hipError_t e = pad_rows(stream, A, w + pl.a_off, M, K, M, pl.Kp, 4)) return e;
            Ap = (const float*)(w + pl.a_off);
        }
        const void* Bp = Bpre;
        if (!Bpre) {
            if (hipError_t e = pad_rows(stream, B, w + pl.b_off, N, K, N, pl.Kp, 4)) return e;
            Bp = w + pl.b_off;
        }
        GemmArgs gp{Ap, Bp, C, M, pl.Np, pl.Kp, pl.Kp, transB ? pl.Kp : pl.Np, N, 0, 0, 0, alpha, beta, 0, 0, bias, act, act_param};
        if (pl.Np != N) gp.c_cols = N;
        return transB ? dispatch_gemm<float, float, true>(gp, 1, stream, 0) : dispatch_gemm<float, float, false>(gp, 1, stream, 0);
    }
    int ks32 = 0;
    const int kper32 = (force_tile == 0 && workspace && !transB && batch == 1 && skinny32_applies(M, N, K)) ? 32 * skinny32_plan(N, K, &ks32) : 0;
    if (kper32 && aligned16(A) && aligned16(B) && (size_t)ks32 * M * N * sizeof(float) <= workspace_bytes) {
        const int ks = ks32, kper = kper32;
        constexpr int smem = SKINNY32_STAGES * (32 * 128 + 32 * 512);
        static unsigned long long attr_done = 0;
        if (hipError_t e0 = ensure_dynamic_smem((const void*)gemm_skinny32_kernel<SKINNY32_STAGES>, smem, &attr_done)) return e0;
        hipLaunchKernelGGL(gemm_skinny32_kernel<SKINNY32_STAGES>, dim3((unsigned)(N / 128), (unsigned)ks), dim3(256), smem, stream, g, (float*)workspace, ks, kper);
        if (hipError_t e = hipGetLastError()) return e;
        const long long total = (long long)M * N;
        hipLaunchKernelGGL((skinny_reduce_kernel<float>), dim3((unsigned)((total + 255) / 256)), dim3(256), 0, stream, (const float*)workspace,
                           C, M, N, ks, bias, act, act_param, alpha, beta);
        return hipGetLastError();
    }
    if (force_tile == 0 && workspace && batch == 1) {
        // few tiles over a long K: the K ranges run as batches into fp32 partials, summed in range order (deterministic)
        // by the pass that also applies alpha, beta, bias and activation
        const int ks = splitk32_ranges(M, N, K);
        if (ks > 1 && (size_t)ks * M * N * sizeof(float) <= workspace_bytes) {
            GemmArgs gp = g;
            gp.C = workspace; gp.K = K / ks; gp.ldc = N; gp.alpha = 1.0f; gp.beta = 0.0f;
            gp.sA = K / ks; gp.sB = transB ? (long long)(K / ks) : (long long)(K / ks) * N; gp.sC = (long long)M * N;
            gp.bias = nullptr; gp.act = 0;
            hipError_t e = transB ? dispatch_gemm<float, float, true>(gp, ks, stream, 0) : dispatch_gemm<float, float, false>(gp, ks, stream, 0);
            if (e != hipSuccess) return e;
            const long long total = (long long)M * N;
            hipLaunchKernelGGL((skinny_reduce_kernel<float>), dim3((unsigned)((total + 255) / 256)), dim3(256), 0, stream, (const float*)workspace,
                               C, M, N, ks, bias, act, act_param, alpha, beta);
            return hipGetLastError();
        }
    }
    if (transB) return dispatch_gemm<float, float, true>(g, batch, stream, force_tile);
    return dispatch_gemm<float, float, false>(g, batch, stream, force_tile);
}

// fp32 A [M,K] x fp16 weights B [K,N] -> fp32 C, optional fused epilogue
hipError_t gemm_f32_f16weight(hipStream_t stream, const float* A, const uint16_t* B, float* C, int M, int N, int K,
                              int force_tile, const float* bias, int act, float act_param, void* workspace, size_t workspace_bytes)
{
    GemmArgs g{A, B, C, M, N, K, K, N, N, 0, 0, 0, 1.0f, 0.0f, 0, 0, bias, act, act_param};
    if (!workspace) workspace_bytes = 0;
    if (force_tile == 0 && smallm_applies(M, N, K) && gemm_smallm_workspace_bytes(M, N, K) <= workspace_bytes)
        return launch_smallm<true>(g, stream, (float*)workspace);
    if (force_tile == 0) {
        const SplitPlan sp = split_choice(M, N, K, 1, true, workspace_bytes);
        if (sp.tile) return run_split(g, sp, 1, stream, workspace, true);
    }
    // rows of A in 16-byte steps, rows of the fp16 B in 8-byte steps
    const bool vec = aligned16(A) && K % 4 == 0 && (((uintptr_t)B) & 7u) == 0 && N % 4 == 0;
    auto tiles = [&](int bm, int bn) { return (long long)((M + bm - 1) / bm) * ((N + bn - 1) / bn); };
    int tile = force_tile == 64 || force_tile == 128 ? force_tile : choose_tile(tiles(128, 128), tiles(64, 64), 0.85);
    if (tile == 128) {
        if (vec) return launch_gemm<float, float, 128, 128, 2, 2, false, true, true, 1, true>(g, 1, stream);
        return launch_gemm<float, float, 128, 128, 2, 2, false, false, true, 1, true>(g, 1, stream);
    }
    if (vec) return launch_gemm<float, float, 64, 64, 2, 2, false, true, true, 1, true>(g, 1, stream);
    return launch_gemm<float, float, 64, 64, 2, 2, false, false, true, 1, true>(g, 1, stream);
}

#endif

// The products of the K ranges of splitk16_ranges, as batches into the workspace; *ks = 0: not taken (no ranges, or too little workspace)
template <typename T>
static hipError_t launch_k_ranges16(const GemmArgs& g, hipStream_t stream, void* workspace, size_t workspace_bytes, int* ks)
{
    int big = 0, kper;
    *ks = splitk16_ranges(g.M, g.N, g.K, &kper, &big);
    GemmArgs gp = g;
    gp.C = workspace; gp.K = kper; gp.k_total = g.K; gp.ldc = g.N;
    gp.sA = kper; gp.sB = (long long)kper * g.N; gp.sC = (long long)g.M * g.N;
    gp.bias = nullptr; gp.act = 0;
    if (*ks == 0 || (size_t)*ks * g.M * g.N * sizeof(float) > workspace_bytes || !dl16_applies<float>(gp)) { *ks = 0; return hipSuccess; }
    return big ? launch_gemm_dl16<T, float, 4>(gp, *ks, stream) : launch_gemm_dl16<T, float, 2, true>(gp, *ks, stream);
}

// one 16-bit type per part: T = f16_t in part 1, bf16_t in part 2; out32: C is fp32 (else the same 16-bit type as the inputs)
template <typename T>
static hipError_t gemm_16_typed(hipStream_t stream, const uint16_t* A, const uint16_t* B, void* C, int out32,
                                int M, int N, int K, int force_tile, void* workspace, size_t workspace_bytes, const float* bias, int act,
                                float act_param, const uint16_t* Bpre = nullptr)
{
    // Every plan below that writes to the workspace holds its own need against workspace_bytes first and is passed over when the
    // bytes do not suffice (the tiled kernels at the end need none).
    if (!workspace) workspace_bytes = 0;
    // Bpre: B already packed by gemm_16_pack_b (B itself is then not read); such a call always takes the padded shapes
    PadPlan pl;
    if (Bpre && !(workspace && aligned16(C) && aligned16(workspace) && aligned16(Bpre) && pad16_layout(M, N, K, &pl) && pl.total <= workspace_bytes))
        return hipErrorInvalidValue;
    if (Bpre || (force_tile == 0 && workspace && aligned16(C) && aligned16(workspace) && pad16_plan(M, N, K, &pl) && pl.total <= workspace_bytes)) {
        unsigned char* w = (unsigned char*)workspace;
        const bool padA = pl.Kp != K, padC = pl.Np != N;
        const uint16_t* Ap = A;
        if (padA) {
            if (hipError_t e = pad_rows(stream, A, w + pl.a_off, M, K, M, pl.Kp, 2)) return e;
            Ap = (const uint16_t*)(w + pl.a_off);
        }
        const uint16_t* Bp = Bpre;
        if (!Bpre) {
            if (hipError_t e = pad_rows(stream, B, w + pl.b_off, K, N, pl.Kp, pl.Np, 2)) return e;
            Bp = (const uint16_t*)(w + pl.b_off);
        }
        const float* bp = bias;
        if (bias && padC) {
            if (hipError_t e = pad_rows(stream, bias, w + pl.bias_off, 1, N, 1, pl.Np, 4)) return e;
            bp = (const float*)(w + pl.bias_off);
        }
        if (padC && pl.Np % 128 == 0 && pl.Kp < (1 << 21) && pl.Np < (1 << 21)) {
            // the 16 x 16 x 32 kernel stores the N real columns straight into the caller's C
            GemmArgs gp{Ap, Bp, C, M, pl.Np, pl.Kp, pl.Kp, pl.Np, N, 0, 0, 0, 1.0f, 0.0f, 0, 0, bp, act, act_param};
            gp.c_cols = N;
            const int wd = aligned16(Ap) ? dl16_width(M, pl.Np, pl.Kp, 1) : 0;
            if (wd == 4) return out32 ? launch_gemm_dl16<T, float, 4>(gp, 1, stream) : launch_gemm_dl16<T, T, 4>(gp, 1, stream);
            if (wd == 3) return out32 ? launch_gemm_dl16<T, float, 3>(gp, 1, stream) : launch_gemm_dl16<T, T, 3>(gp, 1, stream);
            if (wd == 2) return out32 ? launch_gemm_dl16<T, float, 2>(gp, 1, stream) : launch_gemm_dl16<T, T, 2>(gp, 1, stream);
            if (wd == 1) return out32 ? launch_gemm_dl16<T, float, 2, true>(gp, 1, stream) : launch_gemm_dl16<T, T, 2, true>(gp, 1, stream);
            if (wd == 5) return out32 ? launch_gemm_dl16<T, float, 2, true, 2>(gp, 1, stream) : launch_gemm_dl16<T, T, 2, true, 2>(gp, 1, stream);
        }
        void* Cp = padC ? (void*)(w + pl.c_off) : C;
        if (hipError_t e = gemm_16_typed<T>(stream, Ap, Bp, Cp, out32, M, pl.Np, pl.Kp, 0,
                                            pl.total > pl.inner_off ? (void*)(w + pl.inner_off) : nullptr,
                                            pl.total > pl.inner_off ? pl.total - pl.inner_off : 0, bp, act, act_param)) return e;
        return padC ? unpad_rows(stream, Cp, C, M, N, pl.Np, out32 ? 4 : 2) : hipSuccess;
    }
    GemmArgs g{A, B, C, M, N, K, K, N, N, 0, 0, 0, 1.0f, 0.0f, 0, 0, bias, act, act_param};
    const bool b_rows = N % 8 == 0 && aligned16(B);                       // rows of B in whole 16-byte chunks
    if (force_tile == 0 && !(b_rows && K % 8 == 0 && aligned16(A)) && !(b_rows && general_few_rows(M, N, K)) && N >= 16 && N < (1 << 21) && K < (1 << 21)) {
        int kper, ks;
        const int bm = any16_plan(M, N, K, &kper, &ks);
        if (ks > 1 && (size_t)ks * M * N * sizeof(float) <= workspace_bytes) {
            GemmArgs gp = g;
            gp.C = workspace; gp.bias = nullptr; gp.act = 0;
            if (hipError_t e = launch_any16<T, float, 64>(gp, stream, ks, kper)) return e;
            const unsigned grid = (unsigned)(((long long)M * N + 255) / 256);
            if (out32) hipLaunchKernelGGL((skinny_reduce_kernel<float>), dim3(grid), dim3(256), 0, stream, (const float*)workspace, C, M, N, ks, bias, act, act_param, 1.0f, 0.0f);
            else hipLaunchKernelGGL((skinny_reduce_kernel<T>), dim3(grid), dim3(256), 0, stream, (const float*)workspace, C, M, N, ks, bias, act, act_param, 1.0f, 0.0f);
            return hipGetLastError();
        }
        if (bm == 64) return out32 ? launch_any16<T, float, 64>(g, stream) : launch_any16<T, T, 64>(g, stream);
        return out32 ? launch_any16<T, float, 128>(g, stream) : launch_any16<T, T, 128>(g, stream);
    }
    if (force_tile == 0 && workspace && skinny_applies(M, N, K) && aligned16(A) && aligned16(B) &&
        (size_t)skinny_ksplit(N, K) * M * N * sizeof(float) <= workspace_bytes) {
        float* ws = (float*)workspace;
        return out32 ? launch_skinny<T, float>(g, stream, ws) : launch_skinny<T, T>(g, stream, ws);
    }
    if (force_tile == 0 && dl16_applies<float>(g)) {
        if (const int first = msplit16_rows(M, N, K)) {
            // the rows of the whole rounds, then the rest (stream order; the two share the workspace one after the other)
            if (hipError_t e = gemm_16_typed<T>(stream, A, B, C, out32, first, N, K, 0, workspace, workspace_bytes, bias, act, act_param)) return e;
            return gemm_16_typed<T>(stream, A + (size_t)first * K, B, (unsigned char*)C + (size_t)first * N * (out32 ? 4 : 2), out32, M - first, N, K, 0,
                                    workspace, workspace_bytes, bias, act, act_param);
        }
    }
    if (force_tile == 0 && workspace) {
        int ks;
        if (hipError_t e = launch_k_ranges16<T>(g, stream, workspace, workspace_bytes, &ks)) return e;
        if (ks) {
            const unsigned grid = (unsigned)(((long long)M * N + 255) / 256);
            if (out32) hipLaunchKernelGGL((skinny_reduce_kernel<float>), dim3(grid), dim3(256), 0, stream, (const float*)workspace, C, M, N, ks, bias, act, act_param, 1.0f, 0.0f);
            else hipLaunchKernelGGL((skinny_reduce_kernel<T>), dim3(grid), dim3(256), 0, stream, (const float*)workspace, C, M, N, ks, bias, act, act_param, 1.0f, 0.0f);
            return hipGetLastError();
        }
    }
    if (out32) return dispatch_gemm<T, float, false>(g, 1, stream, force_tile);
    return dispatch_gemm<T, T, false>(g, 1, stream, force_tile);
}

hipError_t gemm_16_f16(hipStream_t stream, const uint16_t* A, const uint16_t* B, void* C, int out32,
                       int M, int N, int K, int force_tile, void* workspace, size_t workspace_bytes, const float* bias, int act, float act_param, const uint16_t* Bpre);
hipError_t gemm_16_bf16(hipStream_t stream, const uint16_t* A, const uint16_t* B, void* C, int out32,
                        int M, int N, int K, int force_tile, void* workspace, size_t workspace_bytes, const float* bias, int act, float act_param, const uint16_t* Bpre);
hipError_t gemm_16_x3_f16(hipStream_t stream, const uint16_t* A, const uint16_t* const (&B)[3], uint16_t* C, int M, int n, int K, int ldb, int force_tile);
hipError_t gemm_16_x3_bf16(hipStream_t stream, const uint16_t* A, const uint16_t* const (&B)[3], uint16_t* C, int M, int n, int K, int ldb, int force_tile);
hipError_t gemm_16_rope_f16(hipStream_t stream, const uint16_t* A, const uint16_t* B, uint16_t* C, int M, int N, int K, int force_tile,
                            void* workspace, size_t workspace_bytes, const RopeEpilogue& rope);
hipError_t gemm_16_rope_bf16(hipStream_t stream, const uint16_t* A, const uint16_t* B, uint16_t* C, int M, int N, int K, int force_tile,
                             void* workspace, size_t workspace_bytes, const RopeEpilogue& rope);
// Few rows over a K too short for skinny_applies: gemm_16_typed goes to the 64 x 64 direct-to-LDS tile with edge handling (M <= 32 leaves half
// of its rows empty, three quarters of every larger tile's; N up to 16384 is at most one such tile per CU, so no larger one loads the
// chip better), and the rotation rides on its stores: same sums, one launch (us, product and rotation in two launches / here / on the stream's
// summing pass: 1 x 4096 x 512 7.5 / 6.6 / 6.8, 32 x 512 x 384 7.2 / 6.1 / 7.2, 32 x 12288 x 768 12.6 / 11.0 / 11.7; only towards the
// upper end of that K the stream would be ahead: 1 x 2048 x 704 8.4 / 7.4 / 6.9, 32 x 1024 x 960 9.8 / 8.6 / 7.7, where the plain product is not).
// 33 - 64 rows fill that tile better still and take it over any K that has no ranges, where no wider tile is chosen (49 x 512 x 512, product and
// rotation 6.4 + 2.6 us in two launches / 6.5).
static bool rope_on_tile(const GemmArgs& g)
{
    if (!(g.M <= 64 && g.N % 128 == 0 && g.N <= 16384 && g.K % 64 == 0 && !skinny_applies(g.M, g.N, g.K) && aligned16(g.A) && aligned16(g.B))) return false;
    int kper;
    return g.M <= 32 || (splitk16_ranges(g.M, g.N, g.K, &kper) == 0 && dl16_width(g.M, g.N, g.K, 1) == 0);
}
// C = A B, then interleaved RoPE over the leading columns of C (launch.hpp)
template <typename T>
static hipError_t gemm_16_rope_typed(hipStream_t stream, const uint16_t* A, const uint16_t* B, uint16_t* C, int M, int N, int K, int force_tile,
                                     void* workspace, size_t workspace_bytes, const RopeEpilogue& rope)
{
    if (!workspace) workspace_bytes = 0;
    GemmArgs g{A, B, C, M, N, K, K, N, N, 0, 0, 0, 1.0f, 0.0f, 0, 0, nullptr, 0, 0.0f};
    // the plans of gemm_16_typed that sum K ranges in a pass of their own take the rotation into that pass (the second from 33 rows on;
    // 34 x 2048 x 2048, us of the second and third launch before / the one that does both: 2.7 + 2.6 / 3.1)
    if (force_tile == 0 && workspace && skinny_applies(M, N, K) && aligned16(A) && aligned16(B) &&
        (size_t)skinny_ksplit(N, K) * M * N * sizeof(float) <= workspace_bytes) {
        return launch_skinny<T, T>(g, stream, (float*)workspace, &rope);
    }
    if (force_tile == 0 && workspace && aligned16(A) && aligned16(B) && ((uintptr_t)C & 3u) == 0 && !skinny_applies(M, N, K) && msplit16_rows(M, N, K) == 0) {
        int ks;
        if (hipError_t e = launch_k_ranges16<T>(g, stream, workspace, workspace_bytes, &ks)) return e;
        if (ks) {
            const long long pairs = (long long)M * N / 2;
            hipLaunchKernelGGL((skinny_reduce_rope_kernel<T>), dim3((unsigned)((pairs + 255) / 256)), dim3(256), 0, stream, (const float*)workspace, C, M, N, ks, rope);
            return hipGetLastError();
        }
    }
    if (force_tile == 0 && rope.cols > 0 && rope_on_tile(g)) return launch_gemm_dl<T, T, true, 64, false, 1, GemmRopeArgs>(GemmRopeArgs{g, rope}, 1, stream);
    if (hipError_t e = gemm_16_typed<T>(stream, A, B, C, 0, M, N, K, force_tile, workspace, workspace_bytes, nullptr, 0, 0.0f)) return e;
    return rope_cols16(stream, std::is_same<T, f16_t>::value ? 1 : 2, C, rope.cosc, rope.sinc, M, N, rope.cols, rope.head_dim, rope.seq_len, rope.start_position);
}

#if AIDN_GEMM_PART == 1
hipError_t gemm_16_f16(hipStream_t stream, const uint16_t* A, const uint16_t* B, void* C, int out32,
                       int M, int N, int K, int force_tile, void* workspace, size_t workspace_bytes, const float* bias, int act, float act_param, const uint16_t* Bpre)
{ return gemm_16_typed<f16_t>(stream, A, B, C, out32, M, N, K, force_tile, workspace, workspace_bytes, bias, act, act_param, Bpre); }
hipError_t gemm_16_x3_f16(hipStream_t stream, const uint16_t* A, const uint16_t* const (&B)[3], uint16_t* C, int M, int n, int K, int ldb, int force_tile)
{ return gemm_16_x3_typed<f16_t>(stream, A, B, C, M, n, K, ldb, force_tile); }
hipError_t gemm_16_rope_f16(hipStream_t stream, const uint16_t* A, const uint16_t* B, uint16_t* C, int M, int N, int K, int force_tile,
                            void* workspace, size_t workspace_bytes, const RopeEpilogue& rope)
{ return gemm_16_rope_typed<f16_t>(stream, A, B, C, M, N, K, force_tile, workspace, workspace_bytes, rope); }
#elif AIDN_GEMM_PART == 2
hipError_t gemm_16_bf16(hipStream_t stream, const uint16_t* A, const uint16_t* B, void* C, int out32,
                        int M, int N, int K, int force_tile, void* workspace, size_t workspace_bytes, const float* bias, int act, float act_param, const uint16_t* Bpre)
{ return gemm_16_typed<bf16_t>(stream, A, B, C, out32, M, N, K, force_tile, workspace, workspace_bytes, bias, act, act_param, Bpre); }
hipError_t gemm_16_x3_bf16(hipStream_t stream, const uint16_t* A, const uint16_t* const (&B)[3], uint16_t* C, int M, int n, int K, int ldb, int force_tile)
{ return gemm_16_x3_typed<bf16_t>(stream, A, B, C, M, n, K, ldb, force_tile); }
hipError_t gemm_16_rope_bf16(hipStream_t stream, const uint16_t* A, const uint16_t* B, uint16_t* C, int M, int N, int K, int force_tile,
                             void* workspace, size_t workspace_bytes, const RopeEpilogue& rope)
{ return gemm_16_rope_typed<bf16_t>(stream, A, B, C, M, N, K, force_tile, workspace, workspace_bytes, rope); }
#else
// kind: 0 = fp16, 1 = bf16
hipError_t gemm_16(hipStream_t stream, int kind, const uint16_t* A, const uint16_t* B, void* C, int out32,
                   int M, int N, int K, int force_tile, void* workspace, size_t workspace_bytes, const float* bias, int act, float act_param, const uint16_t* Bpre)
{
    if (kind == 0) return gemm_16_f16(stream, A, B, C, out32, M, N, K, force_tile, workspace, workspace_bytes, bias, act, act_param, Bpre);
    return gemm_16_bf16(stream, A, B, C, out32, M, N, K, force_tile, workspace, workspace_bytes, bias, act, act_param, Bpre);
}
hipError_t gemm_16_x3(hipStream_t stream, int kind, const uint16_t* A, const uint16_t* const (&B)[3], uint16_t* C, int M, int n, int K, int ldb, int force_tile)
{
    return kind == 0 ? gemm_16_x3_f16(stream, A, B, C, M, n, K, ldb, force_tile) : gemm_16_x3_bf16(stream, A, B, C, M, n, K, ldb, force_tile);
}
hipError_t gemm_16_rope(hipStream_t stream, int kind, const uint16_t* A, const uint16_t* B, uint16_t* C, int M, int N, int K, int force_tile,
                        void* workspace, size_t workspace_bytes, const RopeEpilogue& rope)
{
    if (kind == 0) return gemm_16_rope_f16(stream, A, B, C, M, N, K, force_tile, workspace, workspace_bytes, rope);
    return gemm_16_rope_bf16(stream, A, B, C, M, N, K, force_tile, workspace, workspace_bytes, rope);
}
#endif

}  // namespace aidn
