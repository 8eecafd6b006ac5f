// Declarations shared by the attention translation units: the kernel argument block, direct-to-LDS loads, packed
// conversions of probabilities.
#pragma once
#include "common.hpp"
#include "launch.hpp"
#include <type_traits>

namespace aidn {

// Division of a 31-bit unsigned number by a divisor fixed at launch: q = (mulhi(x, m) + x) >> s with s = ceil(log2 d),
// m = floor(2^32 (2^s - d) / d) + 1 (two scalar instructions and a shift where the compiler's general sequence takes about 25).
struct FastDiv { uint32_t m, s; };
inline FastDiv make_fastdiv(uint32_t d)
{
    uint32_t s = 0;
    while ((1ull << s) < d) s++;
    return FastDiv{(uint32_t)((((1ull << s) - d) << 32) / d + 1), s};
}
__device__ __forceinline__ uint32_t fastdiv(uint32_t x, FastDiv f) { return (__umulhi(x, f.m) + x) >> f.s; }

struct AttnArgs {
    const void* q; const void* k; const void* v; void* o;
    float* lse; const float* bias; const float* mask;
    int B, H, Hkv, Sq, Sk, D;
    float scale; int causal; int qoff; float softcap; int mask_mode;
    long long bias_bs;
    long long qs[3], ks[3], vs[3], os[3];
    int qtiles;
    int nvb;       // pipelined prefill kernel: virtual blocks (the grid's workgroups take them in turn)
    int alt_from;  // pipelined prefill kernel: first workgroup of the second half of a resident grid (shares its CU with an earlier one)
    FastDiv dgroup, dunits, dqtiles;      // pipelined prefill kernel: H / Hkv, qtiles / 2, qtiles as divisors
    int hgroup;    // general kernel, causal: > 0 heads per group of the workgroup order of a large grid; < 0 the placement of a small one
    // fp32 on the fp16 pipe: workgroup (x, y) of the grid takes the y-th of nsplit equal shares of its query tile's keys, part as below with D in the place of 128
    // fast kernel, grouped decode: the workgroup's key range is split `split` of nsplit (chunk keys each) and, when part is not
    // null, it stores its unnormalised partial (m, l, O[128]) at part + ((b H_q + head) nsplit + split) * 130 for the merge pass
    int nsplit, chunk; float* part;
    int stream;    // fast kernel: K and V are read once per launch (grouped decode): non-temporal loads
    int stage_out; // fast kernel: fp32 O goes through LDS and is written as whole rows
    int paired;    // fast kernel, causal: a workgroup runs query tile qtiles-1-i and then tile i of a head (equal work for every workgroup)
    int vec_in;    // q/k/v rows are 16-byte aligned and D is a multiple of the 16-byte element count
    int vec_out;
    const int* bt; int bsz; long long bt_bs;   // block table of a paged K/V cache (null = contiguous), block size, batch stride
    FastDiv dbsz;  // direct-to-LDS kernels on a paged cache: the block size as a divisor
};

// Workgroup -> (batch*head, query tile): XCD-contiguous so the q-tiles of one head share an L2;
// late (heavy, under a causal mask) query tiles first.
__device__ __forceinline__ void attn_block(const AttnArgs& a, int& bh, int& qt)
{
    int nblk = gridDim.x, pid = blockIdx.x;
    int per = nblk >> 3, rem = nblk & 7;
    int xcd = pid & 7, idx = pid >> 3;
    int logical = (xcd < rem ? xcd * (per + 1) : rem * (per + 1) + (xcd - rem) * per) + idx;
    bh = logical / a.qtiles;
    qt = a.qtiles - 1 - (logical - bh * a.qtiles);
    if (a.causal && a.hgroup < 0) {
        // A grid that is resident all at once (at most three workgroups per CU) is not balanced by the order of
        // dispatch: hand the query tiles out heaviest first across ALL heads, so the workgroups that end up sharing a
        // CU are a heavy one and, later in the id order, a light one.
        // (the first 256 ids, one per CU, in ascending weight, so that the ids after them -- which land on the same
        // CUs in the same order -- pair the lightest of the first round with the heaviest of the second; reversed by eights, so that
        // where 8 divides the number of heads all query tiles of a head stay on one XCD, 1-4 % against reversing one by one)
        const int nbh = nblk / a.qtiles;
        const int rank = (nblk > 256 && pid < 256) ? 255 - (pid | 7) + (pid & 7) : pid;
        qt = a.qtiles - 1 - rank / nbh;
        bh = rank - (rank / nbh) * nbh;
    } else if (a.causal && a.hgroup > 0) {
        // A grid of several rounds: head by head (heavy tile first) leaves heavy tiles for the very end of the dispatch order
        // and a long tail (measured: a causal launch as slow as the unmasked one).  Take the heads in groups of a.hgroup and
        // hand out the query tiles of a group heaviest first across its heads, so that every group -- the last one included --
        // ends on its light tiles.  When every XCD owns whole heads the groups are formed inside the XCD's own heads.
        const bool whole = rem == 0 && per % a.qtiles == 0;
        const int heads = whole ? per / a.qtiles : nblk / a.qtiles;      // heads the groups are cut from
        const int at = whole ? idx : logical;                            // position among their workgroups
        const int gsz = heads < a.hgroup ? heads : a.hgroup;
        const int per_group = gsz * a.qtiles;
        const int grp = at / per_group, in = at - grp * per_group;
        const int first = grp * gsz;
        const int cur = heads - first < gsz ? heads - first : gsz;       // the last group may be short
        qt = a.qtiles - 1 - in / cur;
        bh = (whole ? xcd * heads : 0) + first + in % cur;
    }
}

// Pool rows of a paged cache for the direct-to-LDS kernels.  A wave loads NK consecutive keys of every key tile (NK = 16 or 8), which
// lie in one block when the block size is a multiple of 16, so one row number serves the wave and its loads keep the form of the
// contiguous case (uniform base, fixed lane offsets).  Lane i of `rows` holds the row of the wave's first key in tile (tile0 + i), 64
// tiles per table read: a tile costs one lane read instead of a table access in front of its loads.
__device__ __forceinline__ int paged_tile_rows(const int* __restrict__ bt, int bsz, FastDiv dbsz, int first_key, int tile_keys, int tile0, int lane,
                                               int last_group)
{
    const int key = min(first_key + (tile0 + lane) * tile_keys, last_group);      // (groups past the end repeat the last one)
    const int blk = (int)fastdiv((uint32_t)key, dbsz);
    return bt[blk] * bsz + (key - blk * bsz);
}
// block sizes the direct-to-LDS kernels take (their rows are at least 128 bytes long: the row numbers of a K and a V pool that fit the
// memory together fit 31 bits)
inline bool paged_block_fits(const int* bt, int bsz) { return !bt || bsz % 16 == 0; }

template <typename T> struct Raw2;
template <> struct Raw2<float> { typedef uint32_t type; };
template <> struct Raw2<f16_t> { typedef uint16_t type; };
template <> struct Raw2<bf16_t> { typedef uint16_t type; };

// 16 bytes = PER16 consecutive elements from p; elements at index >= valid read as zero.
template <typename T>
__device__ __forceinline__ u32x4 ld16(const typename Raw2<T>::type* p, int valid, bool vec)
{
    u32x4 v = {0u, 0u, 0u, 0u};
    if (valid <= 0) return v;
    if (vec && valid >= Elem<T>::PER16) return *(const u32x4*)p;
    if (valid >= Elem<T>::PER16) {
        // rows off the 16-byte grid: a whole chunk is still one load, only element-aligned (the hardware takes such loads)
        typedef u32x4 u32x4_a4 __attribute__((aligned(4)));
        typedef u32x4 u32x4_a2 __attribute__((aligned(2)));
        if constexpr (Elem<T>::BYTES == 4) return *(const u32x4_a4*)p;
        else return *(const u32x4_a2*)p;
    }
    if constexpr (Elem<T>::BYTES == 4) {
#pragma unroll
        for (int e = 0; e < 4; e++) if (e < valid) v[e] = p[e];
    } else {
#pragma unroll
        for (int e = 0; e < 8; e++) if (e < valid) v[e >> 1] |= ((uint32_t)p[e]) << (16 * (e & 1));
    }
    return v;
}

constexpr float LOG2E = 1.4426950408889634f;
constexpr float LN2 = 0.6931471805599453f;

// Direct global -> LDS load of 16 bytes per lane: lane i's data lands at LDS address lds_dst + 16 i (lds_dst wave
// uniform).  Issued from inline asm so the compiler does not order later LDS reads behind it; completion is
// awaited explicitly (s_waitcnt vmcnt(0) + barrier) before the tile is read.
__device__ __forceinline__ void attn_dma16(const void* gptr, uint32_t lds_dst)
{
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, off" ::"s"(lds_dst), "v"(gptr) : "memory");
}
// same, source = wave-uniform base (SGPR pair) + per-lane unsigned 32-bit byte offset
__device__ __forceinline__ void attn_dma16_base(const void* base_uniform, uint32_t lane_off, uint32_t lds_dst)
{
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2" ::"s"(lds_dst), "v"(lane_off), "s"(base_uniform) : "memory");
}

// non-temporal forms for a cache that is read once per launch (decode)
__device__ __forceinline__ void attn_dma16_stream(const void* gptr, uint32_t lds_dst)
{
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, off nt" ::"s"(lds_dst), "v"(gptr) : "memory");
}
__device__ __forceinline__ void attn_dma16_base_stream(const void* base_uniform, uint32_t lane_off, uint32_t lds_dst)
{
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2 nt" ::"s"(lds_dst), "v"(lane_off), "s"(base_uniform) : "memory");
}

typedef short s16x4a __attribute__((ext_vector_type(4)));

// x[i] = cap tanh(x[i] / cap), the soft cap of the logits, N at a time (cap > 0).  The quotient is a product with the reciprocal and what
// that lost.  Up to 0.8 the hyperbolic tangent is an odd polynomial (fitted to the relative error, 3.7e-9; Horner in x^2), beyond it
// 1 - 2 / (1 + e^2|x|) on the vector pipe's exponential and reciprocal; N values that all lie below, which the logits of most models do
// under the caps they use, skip the second part.  An infinity gives +-cap, NaN stays.
// Mean error against float64 (rms relative, caps 2 to 50, this form / an IEEE division and the C library's tanhf in fp32): up to 0.8 4.4e-8 /
// 5.0e-8, to 1.3 4.3e-8 / 4.5e-8, beyond 2.6e-8 / 3.5e-8.
// The device library's function per element was most of the kernels that use it (fp32, with the cap, us of the attention kernel library /
// this: B4 H32 S564 d32 padded 94 / 61, B2 H32 S740 d32 61 / 48; B2 H12 232 x 238 d128 29.4 / 27.1, its probabilities 11.4 / 10.0).
template <int N, typename V>
__device__ __forceinline__ void soft_cap(V& x, float cap)
{
    const float inv = fminf(1.0f / cap, 3.402823466e38f);                         // (a cap below 2^-128 has no finite reciprocal)
    const float lost = inv < 3.4e38f ? fmaf(-cap, inv, 1.0f) * inv : 0.0f;
    float big = 0.0f;
#pragma unroll
    for (int i = 0; i < N; i++) big = fmaxf(big, fabsf(x[i]));
    const bool all_small = __builtin_amdgcn_ballot_w64(big * inv > 0.8f) == 0ull;
    auto quotient = [&](float v) -> float { return fmaf(v, inv, v * lost); };
    auto small = [&](float t) -> float {
        const float z = t * t;
        float p = fmaf(z, 1.584755342e-03f, -7.409555731e-03f);
        p = fmaf(z, p, 2.130298991e-02f);
        p = fmaf(z, p, -5.385233127e-02f);
        p = fmaf(z, p, 1.333222102e-01f);
        p = fmaf(z, p, -3.333329736e-01f);
        return cap * fmaf(t * z, p, t);
    };
    if (all_small) {
#pragma unroll
        for (int i = 0; i < N; i++) {
            x[i] = small(quotient(x[i]));
            if (i % 4 == 3) __builtin_amdgcn_sched_barrier(0);                      // (the kernels that use it are short of registers)
        }
    } else {
#pragma unroll
        for (int i = 0; i < N; i++) {
            const float near = x[i] * inv, t = quotient(x[i]), e = __builtin_amdgcn_exp2f(fabsf(t) * 2.885390082f);       // 2 log2(e)
            const float far = fabsf(near) > 10.0f ? 1.0f : fmaf(-2.0f, __builtin_amdgcn_rcpf(1.0f + e), 1.0f);      // (an infinity has no quotient)
            x[i] = fabsf(near) <= 0.8f ? small(t) : cap * copysignf(far, near);
            if (i % 4 == 3) __builtin_amdgcn_sched_barrier(0);
        }
    }
}

// packed conversions of probabilities and pair sums (shared by both kernels)
template <typename T> __device__ __forceinline__ uint32_t pack2_p(float a, float b);
template <> __device__ __forceinline__ uint32_t pack2_p<f16_t>(float a, float b)
{
    // one packed round-to-nearest-even convert (v_cvt_pk_f16_f32)
    typedef _Float16 h2 __attribute__((ext_vector_type(2)));
    typedef float f2 __attribute__((ext_vector_type(2)));
    f2 x = {a, b};
    h2 v = __builtin_convertvector(x, h2);
    return __builtin_bit_cast(uint32_t, v);
}
// acc + lo + hi of a packed pair (one VALU operation)
template <typename T> __device__ __forceinline__ float add_pair(uint32_t packed, float acc);
template <> __device__ __forceinline__ float add_pair<f16_t>(uint32_t packed, float acc)
{
    typedef _Float16 h2 __attribute__((ext_vector_type(2)));
    const h2 ones = {(_Float16)1.0f, (_Float16)1.0f};
    return __builtin_amdgcn_fdot2(__builtin_bit_cast(h2, packed), ones, acc, false);
}
template <> __device__ __forceinline__ float add_pair<bf16_t>(uint32_t packed, float acc)
{
    typedef __bf16 bf2 __attribute__((ext_vector_type(2)));
    const bf2 ones = {(__bf16)1.0f, (__bf16)1.0f};
    return __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(bf2, packed), ones, acc, false);
}
template <> __device__ __forceinline__ uint32_t pack2_p<bf16_t>(float a, float b)
{
    // probabilities are finite and non-negative: the hardware round-to-nearest-even convert equals the
    // integer rule of float_to_bf16_bits on them
    typedef __bf16 bf2 __attribute__((ext_vector_type(2)));
    bf2 v = {(__bf16)a, (__bf16)b};
    return __builtin_bit_cast(uint32_t, v);
}

// Merge of one query row's partials over key ranges: P = [n][2 + dpad] floats (m, l, unnormalised O), n <= 64, dpad even.  The row
// is merged by WPR waves of the workgroup (1, or all 4), wave `part` of them taking the ranges part, part + WPR, ...; afterwards
// lane i of wave part 0 holds the normalised elements 2 i, 2 i + 1 (and 128 + 2 i, + 1 with NV = 2) and the log-sum-exp.
// Bound by memory latency: eight partial rows per wave are asked for together with the (m, l) pairs, so up to 8 WPR ranges cost one
// round trip; up to eight ranges need no barrier and no LDS.  A range that saw no key weighs zero and adds nothing.
typedef float f32x2p __attribute__((ext_vector_type(2)));
// log(2^m l); rounded once beyond the logarithm and its product (the sum m + log2(l) in units of 2 was a rounding more at nearly twice the size)
__device__ __forceinline__ float log_sum(float m, float l) { return fmaf(m, LN2, __builtin_amdgcn_logf(l) * LN2); }
// KEEP_NAN: a sum that is no number gives NaN instead of zeros, as a single range of the fp32 split kernel does.
template <int NV, int WPR, bool KEEP_NAN = false>
__device__ __forceinline__ float merge_partials(const float* __restrict__ P, int n, int dpad, int D, int part, int lane, f32x2p (&out)[NV])
{
    const long long stride = 2 + dpad;
    const float* ml = P + min(lane, n - 1) * stride;
    const float m = lane < n ? ml[0] : -INFINITY;
    const float l = lane < n ? ml[1] : 0.0f;
    f32x2p v[8][NV];
    auto load8 = [&](int s0) {
#pragma unroll
        for (int u = 0; u < 8; u++)
#pragma unroll
            for (int j = 0; j < NV; j++) {
                v[u][j] = f32x2p{0.0f, 0.0f};
                const int s = s0 + u * WPR;
                if (s < n && 128 * j + 2 * lane < D) v[u][j] = *(const f32x2p*)(P + s * stride + 2 + 128 * j + 2 * lane);
            }
    };
    load8(part);
    float M = m;
#pragma unroll
    for (int off = 8; off >= 1; off >>= 1) M = fmaxf(M, shfl_xor_f(M, off));
    M = max_with_partner32(max_with_partner16(M));
    const float w = __builtin_amdgcn_exp2f(m - (M == -INFINITY ? 0.0f : M));
    float L = l * w;
#pragma unroll
    for (int off = 8; off >= 1; off >>= 1) L += shfl_xor_f(L, off);
    L = sum_with_partner32(sum_with_partner16(L));
#pragma unroll
    for (int j = 0; j < NV; j++) out[j] = f32x2p{0.0f, 0.0f};
    for (int s0 = part; s0 < n; s0 += 8 * WPR) {
        if (s0 != part) load8(s0);
#pragma unroll
        for (int u = 0; u < 8; u++) {
            // (past the last range the row read as zeros; the lane index is only kept inside the wave)
            const float wu = as_f32((uint32_t)__builtin_amdgcn_readlane((int)as_u32(w), (s0 + u * WPR) & 63));
#pragma unroll
            for (int j = 0; j < NV; j++) { out[j][0] = fmaf(v[u][j][0], wu, out[j][0]); out[j][1] = fmaf(v[u][j][1], wu, out[j][1]); }
        }
    }
    if constexpr (WPR > 1) {
        __shared__ f32x2p sums[WPR - 1][NV][64];
        if (part > 0) {
#pragma unroll
            for (int j = 0; j < NV; j++) sums[part - 1][j][lane] = out[j];
        }
        __syncthreads();
        if (part == 0) {
#pragma unroll
            for (int q = 0; q < WPR - 1; q++)
#pragma unroll
                for (int j = 0; j < NV; j++) { out[j][0] += sums[q][j][lane][0]; out[j][1] += sums[q][j][lane][1]; }
        }
    }
    // (divided, as a single range is: a reciprocal would round twice, and a sum that is no number has to give zeros here as there)
#pragma unroll
    for (int j = 0; j < NV; j++)
#pragma unroll
        for (int e = 0; e < 2; e++) out[j][e] = (KEEP_NAN ? L != 0.0f : L > 0.0f) ? out[j][e] / L : 0.0f;
    return L > 0.0f ? log_sum(M, L) : -INFINITY;
}
// waves per row of the merge passes: one (four rows to a workgroup) while a row's ranges fit one round of loads
inline int merge_waves_per_row(int ranges) { return ranges <= 8 ? 1 : 4; }

// fp32 attention on the fp16 matrix pipe (attention_split.hip); options: bias, masks, soft-cap
bool attn_split_applies(const AttnArgs& a);
int attn_split_ranges(const AttnArgs& a);
hipError_t launch_attn_split(const AttnArgs& a, bool options, hipStream_t stream);
hipError_t launch_attn_weights_split(const AttnArgs& a, float* w, hipStream_t stream);
// 16-bit, head dimension 128, plain / causal attention in the software-pipelined form (attention_prefill.hip); kind: 1 fp16, 2 bf16
bool attn_prefill_applies(const AttnArgs& a);
hipError_t launch_attn_prefill(int kind, int out16, AttnArgs a, hipStream_t stream);

}  // namespace aidn
