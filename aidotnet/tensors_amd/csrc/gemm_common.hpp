// Shared by the GEMM translation units: the kernel argument block, the fused activations, the order in which workgroups walk the tiles.
#pragma once
#include "common.hpp"
#include "launch.hpp"
#include <type_traits>

namespace aidn {

// f(std::integral_constant<int, I>) for I = BEGIN, BEGIN + STEP, ... < END: a loop the compiler cannot leave rolled (register
// arrays indexed by the loop variable need constant indices)
template <int BEGIN, int END, int STEP, typename F>
__device__ __forceinline__ void static_for(F&& f)
{
    if constexpr (BEGIN < END) {
        f(std::integral_constant<int, BEGIN>{});
        static_for<BEGIN + STEP, END, STEP>(f);
    }
}

struct GemmArgs {
    const void* A; const void* B; void* C;
    int M, N, K;
    int lda, ldb, ldc;
    long long sA, sB, sC;   // batch strides in elements
    float alpha, beta;
    int tiles_m, tiles_n;
    // fused epilogue: C = act(alpha * A B + beta * C + bias[col]); bias may be null, act 0 = none
    const float* bias;
    int act;
    float act_param;
    // direct-to-LDS kernels only (the 16 x 16 x 32 one and the instances of the 32 x 32 one with edge handling).  > 0: C has this
    // many columns (fewer than N, the columns past them are padding of B that is computed and dropped) and ldc is any element
    // count, so a row of C may start off a 16-byte boundary
    int c_cols = 0;
    // gemm_split_kernel and the 16-bit K ranges.  > 0: the batches are ranges of one K this long; all but the last hold K elements
    // (here it fills the block to eight bytes: one more word moves the grid's size, which every kernel reads first, to a third cache line of
    // the kernel arguments, 0.2 us a launch)
    int k_total = 0;
    // three products with one A in one launch (three batches): their Bs lie anywhere, B at B, B + sB and B + 2 sB + sB2.  (A stride and not
    // two pointers: choosing one by branches in front of the first load cost every kernel 0.1 - 0.3 us, 9 % of a 1 x 256 x 101 product)
    long long sB2 = 0;
};
static_assert(sizeof(GemmArgs) == 0x78, "the hidden arguments follow in the second cache line");

// B of batch bz, in units of B's elements of EB bytes
template <int EB>
__device__ __forceinline__ const unsigned char* batch_b(const GemmArgs& g, long long bz)
{
    return (const unsigned char*)g.B + (bz * g.sB + (bz == 2 ? g.sB2 : 0LL)) * EB;
}

[[maybe_unused]] static bool aligned16(const void* p) { return (((uintptr_t)p) & 15u) == 0; }

// num / (1 + e^-v): GELU (tanh form: (1 + tanh u) / 2 is the logistic function of 2 u), sigmoid and swish, on the vector pipe's exponential
// (base 2) and reciprocal.  The exponent is split into its nearest whole number, added to the exponent field, and a remainder formed from
// v log2(e) in two parts (LONG: with one rounding, for arguments of any size; GELU's matter near zero, where two do as well).  The quotient is
// corrected by its remainder against 1 + e^-v and what that sum lost, so that the error is that of e^-v and one rounding of the result.
// Numerator and denominator are scaled by 2^-4, which keeps the reciprocal normal down to the v where e^-v overflows; below it is zero.
// Largest errors against float64 in units in the last place, with the library's expf or tanhf and an IEEE division / this way: sigmoid
// 2.6 / 2.6 at -20 to -10, 2.2 / 1.7 to 0, 1.5 / 0.8 above; swish 2.7 / 2.7, 2.1 / 1.7, 1.5 / 0.9; GELU above -0.1 1.8 / 1.2, at -2 to -1 15 / 5.5.
// An epilogue holds nothing but these values and nothing runs beside it on one tile per CU, so their length is time: the fp32 product
// 4096 x 3072 x 768 with GELU took 199 us with the library functions chosen per element and takes 149, bf16 1000 x 11008 x 4096 with swish
// 130 and 112 (107 with an exponential rounded twice and the product with the reciprocal: errors up to 3.5 units, zero below -87).
template <bool LONG>
__device__ __forceinline__ float over_one_plus_exp(float num, float v)
{
#pragma clang fp contract(off)
    constexpr float L2E = 1.44269502f, L2E_LO = 1.92596299e-8f;                          // log2(e) = L2E + L2E_LO
    constexpr float WHOLE = 12582912.0f, ONE = 0x1p-4f;                                  // 1.5 2^23: a sum with it is rounded to a whole number
    float whole, rest;
    if constexpr (LONG) {
        const float t = v * -L2E;
        whole = t + WHOLE;
        rest = fmaf(v, -L2E_LO, fmaf(v, -L2E, -t)) + (t - (whole - WHOLE));
    } else {
        whole = fmaf(v, -L2E, WHOLE);
        rest = fmaf(v, -L2E_LO, fmaf(v, -L2E, WHOLE - whole));
    }
    const float e = __builtin_amdgcn_ldexpf(__builtin_amdgcn_exp2f(rest), __builtin_bit_cast(int, whole) - (__builtin_bit_cast(int, WHOLE) + 4));
    const float d = e + ONE, lost = e - (d - ONE);
    const float n = num * ONE, r = __builtin_amdgcn_rcpf(d);
    float q = n * r;
    q = fmaf(-fmaf(lost, q, fmaf(d, q, -n)), r, q);                                      // (in this order a zero keeps its sign)
    q = v < -88.72f ? num * 0.0f : q;
    return v > 88.0f ? num : q;
}

// Pointwise activations of the fused projection epilogues, numbered like the reference's FusedActivationType
// (src/AiDotNet.Tensors/Engines/FusedActivationType.cs:23-70); the functions are those of its HIP activation kernels
// (src/AiDotNet.Tensors/Engines/DirectGpu/HIP/Kernels/HipActivationKernels.cs:19-70).  NaN stays NaN in all of them.
// f(fn) with fn the activation `act`: the choice is made once around whatever f does with it, never per element (a tile of
// accumulators with a test on each is thousands of branches).  Sigmoid and swish share a body: with one each the 256 x 256 fp32 tile's
// epilogue outgrows what the compiler unrolls, and its accumulators go to scratch memory.
template <typename F>
__device__ __forceinline__ void with_activation(int act, float p, F&& f)
{
    switch (act) {
    case 1: f([](float x) { return x < 0.0f ? 0.0f : x; }); break;                       // ReLU, NaN-preserving form (CpuFusedOperations.cs:1271-1274)
    case 2: f([](float x) { return over_one_plus_exp<false>(x, x * fmaf(0.0713548163f, x * x, 1.5957691216f)); }); break;      // GELU, tanh form: 2 u = 2 0.7978845608 (x + 0.044715 x^3)
    case 3:                                                                               // sigmoid
    case 6: f([act](float x) { return over_one_plus_exp<true>(act == 3 ? 1.0f : x, x); }); break;      // swish
    case 4: f([](float x) { return tanhf(x); }); break;
    case 5: f([p](float x) { return x > 0.0f ? x : p * x; }); break;                      // leaky ReLU, slope p
    default: f([](float x) { return x; }); break;
    }
}
__device__ __forceinline__ float apply_activation(float x, int act, float p)
{
    with_activation(act, p, [&](auto fn) { x = fn(x); });
    return x;
}

constexpr int GROUP_M = 8;   // tile rows walked together so one XCD's L2 sees a compact footprint

// Workgroup id -> (tile row, tile col).  Hardware hands consecutive workgroup ids to the 8
// XCDs round-robin; remap so each XCD owns a contiguous run of logical ids, then walk
// that run in GROUP_M-tall column-major groups.
__device__ __forceinline__ void tile_of_block(int pid, int nblk, int tiles_m, int tiles_n, int& tm, int& tn)
{
    int per = nblk >> 3, rem = nblk & 7;
    int xcd = pid & 7, idx = pid >> 3;
    int logical = (xcd < rem ? xcd * (per + 1) : rem * (per + 1) + (xcd - rem) * per) + idx;
    int width = GROUP_M * tiles_n;
    int group = logical / width;
    int first = group * GROUP_M;
    int gsz = min(tiles_m - first, GROUP_M);
    int in = logical - group * width;
    tm = first + in % gsz;
    tn = in / gsz;
}

// fp32 products on the bf16 matrix pipe (gemm_split.hip): C = act(alpha A B + beta C + bias), B [K,N] of fp32 or (b16) fp16, N >= 2,
// lda and ldb below 2^21, operands at any element.  tile: 64 or 128 rows by 128 columns; 192, fp32 and whole 128 x 192
// tiles over whole K-tiles of 32 only.
hipError_t launch_gemm_split(const GemmArgs& g, int batch, hipStream_t stream, int tile, bool b16);

}  // namespace aidn
