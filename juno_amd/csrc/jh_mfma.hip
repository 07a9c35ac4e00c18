// jh_mfma.hip -- batched GEMVs (B >= 2) on Q4_K / Q5_K / Q6_K / Q8_0 through
// LDS + fp16 MFMA.
//
// Y[b][r] = sum_c deq(W[r][c]) * X[b][c] is a dense contraction once B >= 16:
// per HBM byte it needs 2B/0.5625 flops (Q4_K), more than the VALU can issue
// without packed fp32, but below the MFMA ridge (~312 flop/B).  The kernels
// keep every weight integer exact and move the arithmetic to
// v_mfma_f32_32x32x16_f16 with x as the A operand and weights as B, so the
// accumulator of a lane holds one weight row (its own) for 16 batch columns:
//
//  * Weights: each format turns its packed integers into exact fp16 integers
//    (or half-integers) and applies its fp32 scales per row in registers: Q4_K,
//    Q5_K and Q2_K fold their small integer scales into the operand (ls * (q - C),
//    one packed FMA per pair, centred where the sub-block has a min) and apply d
//    and dmin per 256 or 128 columns, the min term and the centre as extra MFMAs
//    against sums of x; Q6_K and Q3_K fold per 16-column sub-block with d * sc,
//    Q8_0 per 32-column block with d.
//  * Activations: x is split into fp16 hi + lo limbs (x = hi + lo to ~2^-22,
//    so only the order of summation differs from fp32) after a power-of-two
//    scale per (column, 256-column super-block) that keeps fp16 in range.
//    Each workgroup converts the fp32 x slice of a super-block straight into
//    its LDS image while it stages the weights (no separate prep launch).
//    Up to 16 columns (HL) the two limbs share one MFMA, rows 0..15 and 16..31
//    of its A operand, which takes out half the MFMAs and half the reads of x from
//    LDS (us, 16 columns, before -> after: 2 x 14336 x 4096 Q4_K 36 -> 29, 4096 x 14336
//    Q6_K 30 -> 27, 4096^2 Q4_K 13.5 -> 11.6, 9216 x 3072 Q8_0 18.1 -> 16.0).
//  * What bounds it: no unit alone.  2 x 14336 x 4096 Q4_K at B = 32 (36.7 us) keeps the
//    VALUs busy 46 % of the cycles, LDS 26 %, the matrix cores 22 %, and its waves wait
//    for 27 % of theirs: one workgroup per CU goes through load, conversion, decode,
//    MFMAs and barrier in step.
//  * Work split: a workgroup is kWaves waves x 32 rows, all B columns, and a
//    range of super-blocks.  Per super-block it stages the x slice in LDS
//    (shared by all its rows) and each wave stages its rows' packed blocks in
//    a wave-private LDS window with aligned, coalesced 16-byte loads; the
//    next super-block's loads are in flight during the current one's math.
//    When the row tiles are too few to fill the GPU the K range is split
//    across workgroups; each split writes its partial tile to the workspace
//    and bumps the tile's arrival counter, and the split that arrives last
//    adds all partials in split order into y in the same launch
//    (deterministic; no float atomics; see store_tile).
#include "jh_device.hpp"
#include "jh_kernels.hpp"

#include <limits.h>
#include <mutex>
#include <stdlib.h>
#include <utility>

namespace jh {
namespace {

typedef _Float16 half8 __attribute__((ext_vector_type(8)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
constexpr int kMinWorkgroups = 256;  // split K until the grid has this many

// Timeline builds (-DJH_TIMELINE, juno_amd/timeline.py; never the shipped
// library): per wave of the B <= 32 double-buffered walk, s_memrealtime at entry
// and, per super-block step, after the step's barrier, once its weight chunks
// are parked, once the next x is staged, and after its MFMAs and fold; then in
// the epilogue (store_tile) once its partials are acknowledged, once the
// arrival is counted, and at its end.
#ifdef JH_TIMELINE
constexpr int kMtWg = 512, kMtSteps = 16, kMtEpi = 1 + 4 * kMtSteps, kMtPer = kMtEpi + 3;
__device__ unsigned long long g_mtimeline[kMtWg * 8 * kMtPer];
#define JH_MT(slot)                                                                                         \
    do {                                                                                                    \
        if ((threadIdx.x & 63) == 0 && blockIdx.x < kMtWg && (slot) < kMtPer)                               \
            g_mtimeline[((size_t)blockIdx.x * 8 + (threadIdx.x >> 6)) * kMtPer + (slot)] =                 \
                __builtin_amdgcn_s_memrealtime();                                                           \
    } while (0)
#else
#define JH_MT(slot) do {} while (0)
#endif

constexpr int kRowsPerWave = 32;
constexpr int kWaves = 8;  // waves per workgroup: 256 rows share each staged x slice
constexpr int kThreads = 64 * kWaves;
constexpr int kRowsPerWG = kWaves * kRowsPerWave;
constexpr int kXPad = 8;  // halves of padding per LDS column (spreads banks)

// f(integral_constant i) for i = 0 .. N - 1
template <class F, int... I>
__device__ __forceinline__ void for_seq(F f, std::integer_sequence<int, I...>) {
    (f(std::integral_constant<int, I>{}), ...);
}
template <int N, class F>
__device__ __forceinline__ void for_c(F f) {
    for_seq(f, std::make_integer_sequence<int, N>{});
}

// Maximum and minimum, NaN if an operand is (v_maximum3_f32, v_minimum3_f32).
__device__ __forceinline__ float larger(float a, float b) { return __builtin_elementwise_maximum(a, b); }
__device__ __forceinline__ float smaller(float a, float b) { return __builtin_elementwise_minimum(a, b); }

// Maximum over the 16 lanes of one DPP row (lanes 16 r .. 16 r + 15): xor-1 and
// xor-2 butterflies, then the half-row and row mirrors.
template <int CTRL>
__device__ __forceinline__ float dpp_f(float v) {
    return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), CTRL, 0xF, 0xF, true));
}
__device__ __forceinline__ float row16_max(float v) {
    v = larger(v, dpp_f<0xB1>(v));   // quad_perm 1,0,3,2
    v = larger(v, dpp_f<0x4E>(v));   // quad_perm 2,3,0,1
    v = larger(v, dpp_f<0x141>(v));  // row_half_mirror
    return larger(v, dpp_f<0x140>(v));  // row_mirror
}

// One column and super-block of x as MFMA operands: 16 consecutive lanes hold
// its 256 values, lane q the values 16 q .. +16 (xv).  A power-of-two scale puts
// max |x s| in [2^12, 2^13) (exact, undone on the partial sums by cs = 1 / s),
// then x s is split into fp16 hi + lo limbs by mixed-precision FMAs (x s is
// exact, so hi is x s rounded and lo the rounded rest): two units of 8 values per
// lane and limb, in the order 0 2 1 3 4 6 5 7, in which packed weight bytes
// become fp16 pairs (b0, b2), (b1, b3) by a mask alone.  The 16-value sums times
// 2^-4 and (even q) the 32-value sums times 2^-5 stay in fp16's range for any x.
// All sums run in fixed orders.
//
// EXACT (two vectors and more than 64, which the fp32 kernels took before): what the
// limbs cannot hold.  lo is rounded to 2^-37 of the block's largest |x|, so a block is
// left out -- zeros in place of it, and cs = -1, for which the wave adds its fp32
// products after the walk (add_exact) -- when (unfit)
//  * an element is not finite;
//  * a nonzero one is below 2^-27 of the largest (it would keep fewer than 10 bits);
//  * four neighbours are all below 2^-14 of it, and not all 0 (together they would
//    keep fewer than the 23 bits that the limbs give the others).
// Normal x meets the second about once in 10^7 elements, a product of two about once
// in 10^6, and never the others.  The quick test takes zeros for small elements; the
// right one runs where it fails.  Cost on ordinary x, us, without / with: 2 x 14336 x
// 4096 Q4_K at B = 128 92.5 / 94.7, B = 2 24.3 / 24.6; 9216 x 3072 Q8_0 53.2 / 53.8, 14.6 / 14.75.
constexpr int kXsShift = 5, kX16Shift = 4;
// largest |x|, smallest nonzero one, smallest nonzero maximum of four neighbours
__device__ __forceinline__ bool unfit(float m, float lone, float four) {
    return !(m < INFINITY) || lone < m * 0x1p-27f || four < m * 0x1p-14f;
}
struct XColumn {
    half8 h[2], l[2];
    float s16, s32, cs;
};
template <bool EXACT>
__device__ __forceinline__ XColumn split_x(const float (&x_in)[16]) {
    XColumn r;
    float xv[16], quad[4];
#pragma unroll
    for (int j = 0; j < 16; j++) xv[j] = x_in[j];
#pragma unroll
    for (int j = 0; j < 4; j++)
        quad[j] = larger(larger(fabsf(xv[4 * j]), fabsf(xv[4 * j + 1])), larger(fabsf(xv[4 * j + 2]), fabsf(xv[4 * j + 3])));
    float m = row16_max(larger(larger(quad[0], quad[1]), larger(quad[2], quad[3])));  // the 16 lanes of the column
    bool bad = false;
    if constexpr (EXACT) {
        float lone = fabsf(xv[0]);
#pragma unroll
        for (int j = 1; j < 16; j++) lone = smaller(lone, fabsf(xv[j]));
        const float four = smaller(smaller(quad[0], quad[1]), smaller(quad[2], quad[3]));
        if (__builtin_expect(__builtin_amdgcn_ballot_w64(unfit(m, lone, four)) != 0, 0)) {  // of the wave's four columns
            float lo = INFINITY, lo4 = INFINITY;
#pragma unroll
            for (int j = 0; j < 16; j++) lo = xv[j] != 0.f ? fminf(lo, fabsf(xv[j])) : lo;
#pragma unroll
            for (int j = 0; j < 4; j++) lo4 = quad[j] != 0.f ? fminf(lo4, quad[j]) : lo4;
            bad = ((__builtin_amdgcn_ballot_w64(unfit(m, lo, lo4)) >> (threadIdx.x & 48)) & 0xFFFF) != 0;
            m = bad ? 0.f : m;
#pragma unroll
            for (int j = 0; j < 16; j++) xv[j] = bad ? 0.f : xv[j];
        }
    }
    int k = 0;
    if (m > 0.f) {
        int e;
        (void)frexpf(m, &e);
        k = min(13 - e, 126);  // both 2^k and 2^-k are normal
    }
    const float s = ldexpf(1.f, k);
    r.cs = bad ? -1.f : ldexpf(1.f, -k);
#pragma unroll
    for (int u = 0; u < 2; u++)
#pragma unroll
        for (int i = 0; i < 8; i++) {
            constexpr int ord[8] = {0, 2, 1, 3, 4, 6, 5, 7};
            const float x = xv[8 * u + ord[i]];
            const _Float16 h = (_Float16)(x * s);
            r.h[u][i] = h;
            r.l[u][i] = (_Float16)fmaf(x, s, -(float)h);
        }
    float g[4];  // of x s: sums of x itself pass the largest float from 2^124 on
#pragma unroll
    for (int i = 0; i < 4; i++) g[i] = fmaf(xv[4 * i], s, xv[4 * i + 1] * s) + fmaf(xv[4 * i + 2], s, xv[4 * i + 3] * s);
    const float sub = (g[0] + g[1]) + (g[2] + g[3]);
    r.s16 = ldexpf(sub, -kX16Shift);
    r.s32 = ldexpf(sub + dpp_f<0xB1>(sub), -kXsShift);  // this lane's and its neighbour's
    return r;
}

// ------------------------------------------------------------------ the x operand
// Virtual columns are the 32 rows of the MFMA's A operand for one column group:
//   !HL  32 batch columns, their hi limbs and their lo limbs in two planes (two
//        MFMAs per K-step)
//   HL   16 batch columns, rows 0..15 their hi limbs and rows 16..31 their lo
//        limbs: one MFMA per K-step does both, and half the operand is read from
//        LDS.  (The rows past a batch of 3..16 would be padding otherwise.)
// Contexts give a lane (row lr of A, K half kh) its operands of a super-block:
//   x(n, off) / xlo(n, off)  unit at column offset off, column group n
//   xs(n)                    the 8 32-value sums, limb kh (hi, lo)
//   x16(n, limb)             the 16-value sums 8 kh .. +8
//   cs()                     1 / scale per batch column (-1: the block is left to add_exact)
// The sums' rows 16..31 are zero with HL.
constexpr int COLH = 256 + kXPad;  // halves per LDS column of the staged x slice

// The padded image the fused kernel converts into LDS: column col at col * COLH
// halves, its sums at col * 16 and col * 32.
template <bool HL, int NT>
struct XImage {
    static constexpr int kCols = (HL ? 16 : 32) * NT;
    static constexpr int kLo = (HL ? 16 : 32 * NT) * COLH;     // halves from a column's hi limbs to its lo limbs
    static constexpr int kXs = (HL ? 1 : 2) * 32 * NT * COLH;  // halves: 32 NT x [8 hi, 8 lo]
    static constexpr int kX16 = kXs + 32 * NT * 16;            // halves: 32 NT x [16 hi, 16 lo]
    static constexpr int kCs = 2 * (kX16 + 32 * NT * 32);      // bytes: 32 NT floats
    static constexpr int kBytes = kCs + 32 * NT * 4;
    // one lane's share of column col (lane q of its 16), with the sums that the format reads
    template <int SUMS, bool EXACT>
    static __device__ __forceinline__ void store(uint8_t *buf, const float (&xv)[16], int q, int col) {
        const XColumn x = split_x<EXACT>(xv);
        _Float16 *base = reinterpret_cast<_Float16 *>(buf), *hi = base + col * COLH + 16 * q;
#pragma unroll
        for (int u = 0; u < 2; u++) {
            *reinterpret_cast<half8 *>(hi + 8 * u) = x.h[u];
            *reinterpret_cast<half8 *>(hi + kLo + 8 * u) = x.l[u];
        }
        if (SUMS == 16) {
            const _Float16 h = (_Float16)x.s16;
            base[kX16 + col * 32 + q] = h;
            base[kX16 + col * 32 + 16 + q] = (_Float16)(x.s16 - (float)h);
        }
        if (SUMS == 32 && (q & 1) == 0) {
            const _Float16 h = (_Float16)x.s32;
            base[kXs + col * 16 + (q >> 1)] = h;
            base[kXs + col * 16 + 8 + (q >> 1)] = (_Float16)(x.s32 - (float)h);
        }
        if (q == 0) reinterpret_cast<float *>(buf + kCs)[col] = x.cs;
    }
    // the sums' row of a virtual column that holds lo limbs (HL)
    static __device__ __forceinline__ void zero_sums(uint8_t *buf, int q, int row) {
        _Float16 *base = reinterpret_cast<_Float16 *>(buf);
        base[kXs + row * 16 + q] = (_Float16)0.f;
        base[kX16 + row * 32 + q] = (_Float16)0.f;
        base[kX16 + row * 32 + 16 + q] = (_Float16)0.f;
    }
};
template <bool HL, int NT>
struct Ctx {
    using I = XImage<HL, NT>;
    int lr, kh;
    const uint8_t *buf;
    __device__ __forceinline__ half8 at(int half) const {
        return *reinterpret_cast<const half8 *>(reinterpret_cast<const _Float16 *>(buf) + half);
    }
    __device__ __forceinline__ half8 x(int n, int off) const { return at((32 * n + lr) * COLH + off); }
    __device__ __forceinline__ half8 xlo(int n, int off) const { return at((32 * n + lr) * COLH + off + I::kLo); }
    __device__ __forceinline__ half8 xs(int n) const { return at(I::kXs + (32 * n + lr) * 16 + 8 * kh); }
    __device__ __forceinline__ half8 x16(int n, int limb) const { return at(I::kX16 + (32 * n + lr) * 32 + 16 * limb + 8 * kh); }
    __device__ __forceinline__ const float *cs() const { return reinterpret_cast<const float *>(buf + I::kCs); }
};

// Prepared x (B <= 32): one super-block of the column group, laid out exactly as
// the GEMM's LDS image so that it moves in as a contiguous DMA copy: the plane(s)
// of 32 virtual columns x 32 units, the 32-value sums (32 x 16 halves), cs (32
// floats), padding to whole KB.  Unit u of virtual column v sits at slot v * 32 +
// (u ^ v): the XOR swizzle lets the 32 lanes that read unit u of 32 columns hit
// distinct LDS banks without padding.
template <bool HL>
struct Slab {
    static constexpr int kLo = 16384;  // !HL: the lo limbs' plane
    static constexpr int kXs = HL ? 16384 : 32768, kCs = kXs + 1024;
    static constexpr int kRows = kXs / 1024 + 2;  // 1 KB DMA rows
    static constexpr int kBytes = kRows * 1024;
    static __device__ __forceinline__ int slot(int v, int off) { return 16 * ((v << 5) | ((off >> 3) ^ v)); }
    template <bool EXACT>
    static __device__ __forceinline__ void store(uint8_t *slab, const float (&xv)[16], int q, int col) {
        const XColumn x = split_x<EXACT>(xv);
#pragma unroll
        for (int u = 0; u < 2; u++) {
            *reinterpret_cast<half8 *>(slab + slot(col, 8 * (2 * q + u))) = x.h[u];
            *reinterpret_cast<half8 *>(HL ? slab + slot(16 + col, 8 * (2 * q + u)) : slab + kLo + slot(col, 8 * (2 * q + u))) = x.l[u];
        }
        _Float16 *xs = reinterpret_cast<_Float16 *>(slab + kXs);
        if ((q & 1) == 0) {
            const _Float16 h = (_Float16)x.s32;
            xs[col * 16 + (q >> 1)] = h;
            xs[col * 16 + 8 + (q >> 1)] = (_Float16)(x.s32 - (float)h);
        }
        if (HL) xs[(16 + col) * 16 + q] = (_Float16)0.f;
        if (q == 0) reinterpret_cast<float *>(slab + kCs)[col] = x.cs;
    }
};
template <bool HL>
struct CtxP {
    using I = Slab<HL>;
    int lr, kh;
    const uint8_t *buf;  // the slab in LDS
    __device__ __forceinline__ half8 x(int, int off) const { return *reinterpret_cast<const half8 *>(buf + I::slot(lr, off)); }
    __device__ __forceinline__ half8 xlo(int, int off) const {
        return *reinterpret_cast<const half8 *>(buf + I::kLo + I::slot(lr, off));
    }
    __device__ __forceinline__ half8 xs(int) const { return *reinterpret_cast<const half8 *>(buf + I::kXs + 32 * lr + 16 * kh); }
    __device__ __forceinline__ half8 x16(int, int) const { return half8{}; }  // no format of this path reads them
    __device__ __forceinline__ const float *cs() const { return reinterpret_cast<const float *>(buf + I::kCs); }
};

// Operand roles: x is the A operand and the weights are B, so D[b][r] = sum_k
// x[b][k] w[r][k].  In the 32x32x16 layout lane (lr, kh) supplies weight row lr (K
// elements 8kh .. 8kh+7) and holds D for row lr and A rows 8(i/4) + 4kh + (i%4), i <
// 16: every per-row scale (d, dmin, d*sc) lives in the lane's own registers, and
// consecutive lanes store consecutive rows.  With HL, registers i >= 8 are the lo
// limbs' sums of the columns of registers i - 8.
__device__ __forceinline__ int batch_of(int n, int i, int kh) { return n * 32 + 8 * (i >> 2) + 4 * kh + (i & 3); }
template <bool HL>
constexpr int kOut = HL ? 8 : 16;  // outputs per lane and column group
__device__ __forceinline__ f32x16 mfma(const half8 &x, const half8 &w, const f32x16 &c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_f16(x, w, c, 0, 0, 0);
}
// 1 / scale of the batch columns a lane holds for group n
template <int NI, class C>
__device__ __forceinline__ void col_scales(const C &c, int n, float (&cs)[NI]) {
#pragma unroll
    for (int i = 0; i < NI / 4; i++) {
        const float4 v = *reinterpret_cast<const float4 *>(c.cs() + n * 32 + 8 * i + 4 * c.kh);
        cs[4 * i] = v.x;
        cs[4 * i + 1] = v.y;
        cs[4 * i + 2] = v.z;
        cs[4 * i + 3] = v.w;
    }
}

typedef _Float16 half2v __attribute__((ext_vector_type(2)));
__device__ __forceinline__ half2v dup(float v) { return half2v{(_Float16)v, (_Float16)v}; }
__device__ __forceinline__ half8 join(half2v a, half2v b, half2v c, half2v d) {
    return half8{a[0], a[1], b[0], b[1], c[0], c[1], d[0], d[1]};
}
// a constant held in a register: v_and_or_b32 takes one literal, not two
__device__ __forceinline__ uint32_t in_vgpr(uint32_t v) {
    asm("" : "+v"(v));
    return v;
}
__device__ __forceinline__ half2v as_h2(uint32_t v) { return __builtin_bit_cast(half2v, v); }

// the bytes of two words -> fp16 1024 + u - off in unit order: one byte permute
// per pair takes two bytes and the exponent byte 0x64 from a constant
__device__ __forceinline__ half8 bytes_to_h8(uint32_t w0, uint32_t w1, half2v off) {
    const uint32_t e = 0x64646464u;
    return join(as_h2(__builtin_amdgcn_perm(e, w0, 0x04020400u)) - off, as_h2(__builtin_amdgcn_perm(e, w0, 0x04030401u)) - off,
                as_h2(__builtin_amdgcn_perm(e, w1, 0x04020400u)) - off, as_h2(__builtin_amdgcn_perm(e, w1, 0x04030401u)) - off);
}
// the same in natural order (the operands that meet the sums of x)
__device__ __forceinline__ half8 bytes_to_h8_plain(uint32_t w0, uint32_t w1, half2v off) {
    const uint32_t e = 0x64646464u;
    return join(as_h2(__builtin_amdgcn_perm(e, w0, 0x04010400u)) - off, as_h2(__builtin_amdgcn_perm(e, w0, 0x04030402u)) - off,
                as_h2(__builtin_amdgcn_perm(e, w1, 0x04010400u)) - off, as_h2(__builtin_amdgcn_perm(e, w1, 0x04030402u)) - off);
}

// N dwords at a 2-byte-aligned LDS address, read as aligned dwords and
// realigned in registers with v_alignbyte.  Unaligned 8- and 16-byte LDS reads
// stall the LDS pipeline (and the x-fragment reads queued behind them).  One
// dword past the field is read and ignored when p is dword-aligned, so the
// weight windows end with kWinPad bytes of padding.
constexpr int kWinPad = 16;
template <int N>
__device__ __forceinline__ void lds_read_u(const uint8_t *p, uint32_t (&out)[N]) {
    const uint32_t sh = (uint32_t)(reinterpret_cast<uintptr_t>(p) & 3);
    const uint32_t *b = reinterpret_cast<const uint32_t *>(p - sh);
    uint32_t w[N + 1];
#pragma unroll
    for (int i = 0; i <= N; i++) w[i] = b[i];
#pragma unroll
    for (int i = 0; i < N; i++) out[i] = __builtin_amdgcn_alignbyte(w[i + 1], w[i], sh);
}
__device__ __forceinline__ u32x2 lds_u32x2(const uint8_t *p) {
    uint32_t v[2];
    lds_read_u<2>(p, v);
    return u32x2{v[0], v[1]};
}
__device__ __forceinline__ u32x4 lds_u32x4(const uint8_t *p) {
    uint32_t v[4];
    lds_read_u<4>(p, v);
    return u32x4{v[0], v[1], v[2], v[3]};
}

// 16 bytes at a 2-byte-aligned address in memory (one load on gfx950)
typedef uint32_t u32x4a2 __attribute__((ext_vector_type(4), aligned(2)));
__device__ __forceinline__ u32x4 load16(const uint8_t *p) { return *reinterpret_cast<const u32x4a2 *>(p); }

// Window position (in chunks) of chunk j of a wave's 32 x CH chunk grid when
// rows are RC >= CH chunks apart.
template <int CH, int RC>
__device__ __forceinline__ int win_chunk(int j) { return RC == CH ? j : j + (RC - CH) * (j / CH); }

// ------------------------------------------------------------------ format policies
// Each format supplies, for one 256-column stretch ("super-block") of a row:
//   Regs                  the lane's weight bytes (row lr, K half kh), in VGPRs
//   load(r, p, kh)        p = first byte of the row's stretch, in LDS
//   compute<HL, NT>(...)  the MFMAs and the fold into the fp32 totals
//   run(p, t, ..)         16 columns' quants and scales (p in memory), for add_exact
// K-step t covers 16 columns; lane half kh supplies 8 of them.  Every weight
// enters the MFMA as an exact fp16 integer (or half-integer); scales are applied
// in fp32.  Quants of a sub-block with a nonzero min are centred (Q4_K q - 8, Q5_K
// q - 16, Q2_K q - 1.5): the products then have the size of the weights
// themselves, and what the centre took out comes back with the min term from the
// sums of x.  Uncentred, the accumulators carry that offset through every
// rounding (N(0, 0.02) weights, K = 4096: error against 64 bits 3.95e-7 for Q4_K).
// A sub-block whose min is 0 is not centred: its weights with q = 0 are exactly
// zero, and must stay so under an x of any size.

// acc (+)= x . w over one K-step at column offset off: the hi limbs' MFMA, then the
// lo limbs' into the same sum (HL: one MFMA, the two sums in different registers).
// The hi limbs come first: with the lo limbs' sum as the accumulator input, the
// MFMA drops its low bits always in one direction, a bias that adds up over K
// (Q8_0, K = 14336: 1.73e-7 against 1.24e-7).
template <bool HL, int NT, class C>
__device__ __forceinline__ void mfma_xw(const C &c, const half8 &w, int off, f32x16 (&acc)[NT]) {
#pragma unroll
    for (int n = 0; n < NT; n++) acc[n] = mfma(c.x(n, off), w, acc[n]);
    if constexpr (!HL) {
#pragma unroll
        for (int n = 0; n < NT; n++) acc[n] = mfma(c.xlo(n, off), w, acc[n]);
    }
}
// part += ds * acc
template <int NT>
__device__ __forceinline__ void fold(f32x16 (&part)[NT], float ds, const f32x16 (&acc)[NT]) {
#pragma unroll
    for (int n = 0; n < NT; n++)
#pragma unroll
        for (int i = 0; i < 16; i++) part[n][i] = fmaf(ds, acc[n][i], part[n][i]);
}
// Ends a run of K-steps: the folds are done here, and no operand read of the next
// run has started.  Without it the compiler issues the reads of all K-steps first
// and keeps their sums to the end, which spills.
template <int NT>
__device__ __forceinline__ void step_fence(f32x16 (&part)[NT]) {
#pragma unroll
    for (int n = 0; n < NT; n++) asm volatile("" : "+v"(part[n]));
    __builtin_amdgcn_sched_barrier(0);
}
// How the super-blocks' sums are added up (see kChains): up to 64 columns; chunks of 32; of 64
enum Sums { kPlain, kChained, kWide64 };
// kChained: the folds of a super-block's quarters are summed apart, then in pairs
template <int NT>
__device__ __forceinline__ void next_quarter(int t, f32x16 (&part)[NT], f32x16 (&quarter)[NT], f32x16 (&half)[NT]) {
#pragma unroll
    for (int n = 0; n < NT; n++) {
        if (t == 3 || t == 11) {
            quarter[n] = part[n];
            part[n] = (f32x16){};
        } else if (t == 7) {
#pragma unroll
            for (int i = 0; i < 16; i++) half[n][i] = quarter[n][i] + part[n][i];
            part[n] = (f32x16){};
        } else if (t == 15) {
#pragma unroll
            for (int i = 0; i < 16; i++) part[n][i] = half[n][i] + (quarter[n][i] + part[n][i]);
        }
    }
}
// tot += cs * (the super-block's folded sums)
template <bool HL, int NT, class C>
__device__ __forceinline__ void fold_columns(const C &c, const f32x16 (&part)[NT], float (&tot)[NT][kOut<HL>]) {
#pragma unroll
    for (int n = 0; n < NT; n++) {
        float cs[kOut<HL>];
        col_scales(c, n, cs);
#pragma unroll
        for (int i = 0; i < kOut<HL>; i++)
            tot[n][i] = fmaf(cs[i], HL ? part[n][i] + part[n][(i + 8) & 15] : part[n][i], tot[n][i]);
    }
}

// Q4_K (matVecQ4Kraw, LlamaTransformerHandler.java:1428-1468): w = d*ls*q - dmin*lm.
// B = ls*(q - C), C = 8 where lm is not 0, |.| <= 945: a nibble moved to bits 4..7
// under fp16 64's exponent is 64 + q (one shift, one and-or per pair), and one
// packed FMA gives (64 + q) ls - (64 + C) ls, exact.  Q5_K (Q5 = true,
// matVecQ5Kraw :1525-1576): q has a 5th bit from qh, bits 4..8, C = 16, |.| <= 1953.
template <bool Q5>
struct FmtKQ {
    static constexpr int kBytes = Q5 ? 176 : 144;
    static constexpr int kSums = 32;  // sums of x it reads (0, 16 or 32 values each)
    static constexpr int kChunks = kBytes / 16;  // rows are 16-byte aligned (pitch kBytes * n, aligned base)
    static constexpr int kRowChunks = kChunks;   // LDS window row stride (16-byte chunks)
    static constexpr int kQs = Q5 ? 48 : 16;
    struct Regs {
        u32x4 hd;
        u32x2 qp[4][2];
        u32x2 qh[2];  // Q5_K: qh bytes 16 j + 8 kh .. +8 (bit s for sub-block s)
    };
    static __device__ __forceinline__ void load(Regs &r, const uint8_t *p, int kh) {
        r.hd = *reinterpret_cast<const u32x4 *>(p);
#pragma unroll
        for (int g = 0; g < 4; g++) {
            r.qp[g][0] = *reinterpret_cast<const u32x2 *>(p + kQs + 32 * g + 8 * kh);
            r.qp[g][1] = *reinterpret_cast<const u32x2 *>(p + kQs + 32 * g + 16 + 8 * kh);
        }
        if (Q5) {
            r.qh[0] = *reinterpret_cast<const u32x2 *>(p + 16 + 8 * kh);
            r.qh[1] = *reinterpret_cast<const u32x2 *>(p + 32 + 8 * kh);
        }
    }
    // run t: 16 columns from 16 t on as bytes q + kBias, their scale and min
    static constexpr int kBias = 0;
    static constexpr bool kMin = true;
    static __device__ __forceinline__ u32x4 run(const uint8_t *p, int t, float &sc, float &mn) {
        const int s = t >> 1, hf = t & 1;
        const u32x4 hd = load16(p);
        int ls, lm;
        q4k_scale_min(hd.y, hd.z, hd.w, s, ls, lm);
        sc = half_bits_to_float(hd.x) * (float)ls;
        mn = half_bits_to_float(hd.x >> 16) * (float)lm;
        u32x4 q = (load16(p + kQs + 32 * (s >> 1) + 16 * hf) >> (4 * (s & 1))) & 0x0F0F0F0Fu;
        if (Q5) q |= ((load16(p + 16 + 16 * hf) >> s) & 0x01010101u) << 4;
        return q;
    }
    // the pair of one dword's bytes (odd ? (b1, b3) : (b0, b2)) of sub-block s
    template <int S, int ODD>
    static __device__ __forceinline__ half2v pair(uint32_t w, uint32_t hb, half2v ls, half2v off, uint32_t top) {
        constexpr int sh = (S & 1 ? 4 : 0) + 8 * ODD - 4;  // the nibble's bit within the half word, to bit 4
        if (Q5) {
            constexpr int hs = S + 8 * ODD - 8;  // the 5th bit, to bit 8
            const uint32_t v = hs > 0 ? hb >> (hs > 0 ? hs : 0) : hb << (hs < 0 ? -hs : 0);
            top |= v & 0x01000100u;
        }
        const uint32_t v = sh > 0 ? w >> (sh > 0 ? sh : 0) : w << (sh < 0 ? -sh : 0);
        return __builtin_elementwise_fma(as_h2((v & 0x00F000F0u) | top), ls, off);
    }
    template <bool HL, int NT, Sums SUMS, class C>
    static __device__ __forceinline__ void compute(const Regs &r, const C &c, float (&tot)[NT][kOut<HL>]) {
        // 6-bit scales and mins of the 8 sub-blocks, one per byte (q4kScaleRaw / q4kMinRaw, :1471-1482),
        // and their centres: 8 (Q5_K 16) where the min is not zero
        uint32_t ls4[2], lm4[2], c4[2];
        ls4[0] = r.hd.y & 0x3F3F3F3Fu;
        lm4[0] = r.hd.z & 0x3F3F3F3Fu;
        ls4[1] = (r.hd.w & 0x0F0F0F0Fu) | ((r.hd.y >> 2) & 0x30303030u);
        lm4[1] = ((r.hd.w >> 4) & 0x0F0F0F0Fu) | ((r.hd.z >> 2) & 0x30303030u);
#pragma unroll
        for (int h = 0; h < 2; h++) c4[h] = ((lm4[h] + 0x3F3F3F3Fu) & 0x40404040u) >> (Q5 ? 2 : 3);
        const half2v k1024 = dup(1024.f);
        const uint32_t top = in_vgpr(0x54005400u);
        f32x16 acc[NT];
#pragma unroll
        for (int n = 0; n < NT; n++) acc[n] = (f32x16){};
        for_c<8>([&](auto si) {
            constexpr int S = decltype(si)::value, g = S / 2;
            constexpr uint32_t sel = 0x04000400u + 0x00010001u * (S % 4);  // byte S % 4 under the exponent byte, twice
            const half2v ls = as_h2(__builtin_amdgcn_perm(0x64646464u, ls4[S / 4], sel)) - k1024;
            const half2v off = ls * (dup(960.f) - as_h2(__builtin_amdgcn_perm(0x64646464u, c4[S / 4], sel)));  // -(64 + C) ls
            for_c<2>([&](auto oi) {
                constexpr int o = decltype(oi)::value;
                const u32x2 q = r.qp[g][o], h = Q5 ? r.qh[o] : u32x2{0u, 0u};
                mfma_xw<HL, NT>(c, join(pair<S, 0>(q.x, h.x, ls, off, top), pair<S, 1>(q.x, h.x, ls, off, top),
                                        pair<S, 0>(q.y, h.y, ls, off, top), pair<S, 1>(q.y, h.y, ls, off, top)),
                                16 * (2 * S + o) + 8 * c.kh, acc);
            });
        });
        // the centre's share and the min term, from the sums of x: C ls X and lm X with X = 2^-5 sum(x)
        const half2v mm = dup((float)(1 << kXsShift));
        const half8 wm = bytes_to_h8_plain(lm4[0], lm4[1], k1024) * join(mm, mm, mm, mm);
        const half8 wl = bytes_to_h8_plain(ls4[0], ls4[1], k1024) *
                         (bytes_to_h8_plain(c4[0], c4[1], k1024) * join(mm, mm, mm, mm));
        const float d = half_bits_to_float(r.hd.x), dmin = half_bits_to_float(r.hd.x >> 16);
#pragma unroll
        for (int n = 0; n < NT; n++) {
            if (NT > 1) __builtin_amdgcn_sched_barrier(0);  // one column group's sums at a time
            const half8 xs = c.xs(n);
            const f32x16 a = mfma(xs, wl, acc[n]), mn = mfma(xs, wm, (f32x16){});
            float cs[kOut<HL>];
            col_scales(c, n, cs);
#pragma unroll
            for (int i = 0; i < kOut<HL>; i++)
                tot[n][i] = fmaf(cs[i], fmaf(d, HL ? a[i] + a[(i + 8) & 15] : a[i], -dmin * mn[i]), tot[n][i]);
        }
    }
};

using FmtQ4K = FmtKQ<false>;
using FmtQ5K = FmtKQ<true>;

// Q6_K (matVecQ6Kraw, LlamaTransformerHandler.java:1587-1638): w = (d*sc_j)*(u - 32)
// with u = 4 bits of ql | 2 bits of qh.  A 16-column sub-block is exactly one
// K-step, so B = u - 32 (exact) and each K-step is folded with the fp32
// d*sc_j of the lane's row (the reference's dN).  Step t = 8n + 2qd + j
// covers columns 128n + 32qd + 16j .. +16 and uses scale t.
struct FmtQ6K {
    static constexpr int kSums = 0;
    static constexpr int kBytes = 210;
    static constexpr int kChunks = (kBytes + 14 + 15) / 16;  // a 2-byte-aligned block spans <= 14 chunks
    // window rows 15 chunks (60 dwords) apart: the dword reads of 32 rows hit 16
    // banks (2-way) instead of the 8 of a 56-dword stride
    static constexpr int kRowChunks = kChunks + 1;
    struct Regs {
        u32x2 ql[2][2][2];  // [half n][ql +32 p][j]: bytes 64n + 32p + 16j + 8kh
        u32x2 qh[2][2];     // [n][j]: bytes 128 + 32n + 16j + 8kh
        u32x4 sc;           // bytes 192..207
        uint32_t dw;        // bytes 206..209: d in the high half
    };
    static __device__ __forceinline__ void load(Regs &r, const uint8_t *p, int kh) {
#pragma unroll
        for (int n = 0; n < 2; n++)
#pragma unroll
            for (int j = 0; j < 2; j++) {
                const uint8_t *a = p + 64 * n + 16 * j + 8 * kh;
                r.ql[n][0][j] = lds_u32x2(a);
                r.ql[n][1][j] = lds_u32x2(a + 32);
                r.qh[n][j] = lds_u32x2(p + 128 + 32 * n + 16 * j + 8 * kh);
            }
        r.sc = lds_u32x4(p + 192);
        uint32_t dw[1];
        lds_read_u<1>(p + 206, dw);
        r.dw = dw[0];
    }
    // run t: 16 columns from 16 t on as bytes q + kBias, their scale and min
    static constexpr int kBias = 32;
    static constexpr bool kMin = false;
    static __device__ __forceinline__ u32x4 run(const uint8_t *p, int t, float &sc, float &mn) {
        const int n = t >> 3, qd = (t >> 1) & 3, j = t & 1;
        sc = half_bits_to_float(*reinterpret_cast<const uint16_t *>(p + 208)) * (float)(int8_t)p[192 + t];
        mn = 0.f;
        return ((load16(p + 64 * n + 32 * (qd & 1) + 16 * j) >> (qd >= 2 ? 4 : 0)) & 0x0F0F0F0Fu) |
               (((load16(p + 128 + 32 * n + 16 * j) >> (2 * qd)) & 0x03030303u) << 4);
    }
    template <bool HL, int NT, Sums SUMS, class C>
    static __device__ __forceinline__ void compute(const Regs &r, const C &c, float (&tot)[NT][kOut<HL>]) {
        const half2v off = dup(1056.f);  // 1024 + 32
        const float d = half_bits_to_float(r.dw >> 16);
        f32x16 part[NT], quarter[NT], half[NT];
#pragma unroll
        for (int n = 0; n < NT; n++) part[n] = (f32x16){};
#pragma unroll
        for (int t = 0; t < 16; t++) {
            const int n = t >> 3, qd = (t >> 1) & 3, j = t & 1;
            const u32x2 l = r.ql[n][qd & 1][j], h = r.qh[n][j];
            const uint32_t u0 = ((qd >= 2 ? l.x >> 4 : l.x) & 0x0F0F0F0Fu) | (((h.x >> (2 * qd)) & 0x03030303u) << 4);
            const uint32_t u1 = ((qd >= 2 ? l.y >> 4 : l.y) & 0x0F0F0F0Fu) | (((h.y >> (2 * qd)) & 0x03030303u) << 4);
            f32x16 acc[NT];
#pragma unroll
            for (int m = 0; m < NT; m++) acc[m] = (f32x16){};
            mfma_xw<HL, NT>(c, bytes_to_h8(u0, u1, off), 16 * t + 8 * c.kh, acc);
            fold<NT>(part, d * (float)(int8_t)byte_of(t < 4 ? r.sc.x : t < 8 ? r.sc.y : t < 12 ? r.sc.z : r.sc.w, t & 3), acc);
            if (t % (NT > 1 ? 2 : 4) == (NT > 1 ? 1 : 3)) step_fence(part);
            if (SUMS == kChained) next_quarter<NT>(t, part, quarter, half);
        }
        fold_columns<HL, NT>(c, part, tot);
    }
};

// Q8_0 (matVecQ8_0raw, LlamaTransformerHandler.java:1486-1508): w = d_b * q, 8 blocks
// of 34 B per 256 columns.  Lane half kh holds columns 16kh .. 16kh+15 of
// block b (one 16-byte load), split over the block's two K-steps; B = q exact.
struct FmtQ8_0 {
    static constexpr int kSums = 0;
    static constexpr int kBytes = 8 * 34;
    static constexpr int kChunks = (kBytes + 14 + 15) / 16;
    static constexpr int kRowChunks = kChunks + 1;  // 76-dword window rows (see FmtQ6K)
    struct Regs {
        const uint8_t *p;  // 40 registers of quants and scales would spill: each block is read ahead of its MFMAs
    };
    static __device__ __forceinline__ void load(Regs &r, const uint8_t *p, int) { r.p = p; }
    // run t: 16 columns from 16 t on as bytes q + kBias, their scale and min
    static constexpr int kBias = 128;
    static constexpr bool kMin = false;
    static __device__ __forceinline__ u32x4 run(const uint8_t *p, int t, float &sc, float &mn) {
        sc = half_bits_to_float(*reinterpret_cast<const uint16_t *>(p + 34 * (t >> 1)));
        mn = 0.f;
        return load16(p + 34 * (t >> 1) + 2 + 16 * (t & 1)) ^ 0x80808080u;
    }
    template <bool HL, int NT, Sums SUMS, class C>
    static __device__ __forceinline__ void compute(const Regs &r, const C &c, float (&tot)[NT][kOut<HL>]) {
        const half2v off = dup(1152.f);  // 1024 + 128
        f32x16 part[NT];
#pragma unroll
        for (int n = 0; n < NT; n++) part[n] = (f32x16){};
        u32x4 q = lds_u32x4(r.p + 2 + 16 * c.kh);  // block b: bytes 34b + 2 + 16kh .. +16
        uint32_t d = *reinterpret_cast<const uint16_t *>(r.p);
#pragma unroll
        for (int b = 0; b < 8; b++) {
            const u32x4 qb = q;
            const uint32_t db = d;
            if (b < 7) {
                q = lds_u32x4(r.p + 34 * (b + 1) + 2 + 16 * c.kh);
                d = *reinterpret_cast<const uint16_t *>(r.p + 34 * (b + 1));
            }
            f32x16 acc[NT];
#pragma unroll
            for (int m = 0; m < NT; m++) acc[m] = (f32x16){};
#pragma unroll
            for (int j = 0; j < 2; j++)
                mfma_xw<HL, NT>(c, bytes_to_h8((j ? qb.z : qb.x) ^ 0x80808080u, (j ? qb.w : qb.y) ^ 0x80808080u, off),
                                32 * b + 16 * c.kh + 8 * j, acc);
            fold<NT>(part, half_bits_to_float(db), acc);
            if (HL || NT > 1 || SUMS == kChained) step_fence(part);
        }
        fold_columns<HL, NT>(c, part, tot);
    }
};

// Q2_K (matVecQ2Kraw, LlamaTransformerHandler.java): 84-byte blocks [scales 16]
// [qs 64][d][dmin]; element 128h + 16k + l takes 2 bits at shift 2(k/2) of
// qs[32h + 16(k&1) + l] and sub-block scale byte sc[8h + k] (low nibble scale,
// high nibble min): w = d*(sc&15)*q - dmin*(sc>>4).  A 16-column sub-block is one
// K-step t = 8h + k: B = (sc&15)*(q - C), C = 1.5 where the min is not 0 (|.| <= 45,
// exact: the 2 bits at bits 4..5 under fp16 64's exponent, then one packed FMA);
// the centre's share and the min term are MFMAs per super-block against the
// 16-column sums of x.  The sums are folded with d every 8 K-steps: every 16 is
// 6 % faster at B = 48 but its error against 64 bits (K = 1024: 1.77e-7) is larger
// than the VALU kernel's 1.61e-7; every 8 gives 1.52e-7, every 4 1.40e-7, which
// chunks of 32 columns take; chunks of 64, with one chain of super-blocks, fold every 2
// (folding each K-step with d*(sc&15) is 7 % slower).
// Blocks are 4-byte aligned (84 = 4 * 21).
struct FmtQ2K {
    static constexpr int kSums = 16;
    static constexpr int kBytes = 84;
    static constexpr int kChunks = (kBytes + 12 + 15) / 16;  // a 4-byte-aligned block spans <= 6 chunks
    static constexpr int kRowChunks = kChunks + 1;           // 28-dword window rows (2-way bank conflicts)
    struct Regs {
        u32x2 q[2][2];  // [h][k&1]: qs bytes 32h + 16(k&1) + 8kh .. +8
        u32x4 sc;       // the 16 scale bytes
        uint32_t dm;    // d (low half), dmin (high half)
    };
    static __device__ __forceinline__ void load(Regs &r, const uint8_t *p, int kh) {
#pragma unroll
        for (int h = 0; h < 2; h++)
#pragma unroll
            for (int o = 0; o < 2; o++) r.q[h][o] = lds_u32x2(p + 16 + 32 * h + 16 * o + 8 * kh);
        r.sc = lds_u32x4(p);
        uint32_t dm[1];
        lds_read_u<1>(p + 80, dm);
        r.dm = dm[0];
    }
    // run t: 16 columns from 16 t on as bytes q + kBias, their scale and min
    static constexpr int kBias = 0;
    static constexpr bool kMin = true;
    static __device__ __forceinline__ u32x4 run(const uint8_t *p, int t, float &sc, float &mn) {
        const int k = t & 7;
        const uint32_t dm = *reinterpret_cast<const uint32_t *>(p + 80);
        sc = half_bits_to_float(dm) * (float)(p[t] & 15);
        mn = half_bits_to_float(dm >> 16) * (float)(p[t] >> 4);
        return (load16(p + 16 + 32 * (t >> 3) + 16 * (k & 1)) >> (2 * (k >> 1))) & 0x03030303u;
    }
    template <int J, int ODD>
    static __device__ __forceinline__ half2v pair(uint32_t w, half2v sc, half2v off, uint32_t top) {
        constexpr int sh = 2 * J + 8 * ODD - 4;  // the 2 bits' place within the half word, to bit 4
        const uint32_t v = sh > 0 ? w >> (sh > 0 ? sh : 0) : w << (sh < 0 ? -sh : 0);
        return __builtin_elementwise_fma(as_h2((v & 0x00300030u) | top), sc, off);
    }
    template <bool HL, int NT, Sums SUMS, class C>
    static __device__ __forceinline__ void compute(const Regs &r, const C &c, float (&tot)[NT][kOut<HL>]) {
        constexpr int kFold = SUMS == kPlain ? 8 : SUMS == kChained ? 4 : 2;  // K-steps per fold: see above
        const float d = half_bits_to_float(r.dm), dmin = half_bits_to_float(r.dm >> 16);
        const uint32_t top = in_vgpr(0x54005400u);
        const half2v k = dup(1024.f);
        // the low byte of each sub-block's fp16 64 + C: 0x18 where the min is not 0
        uint32_t c4[4], m4[4], s4[4];
#pragma unroll
        for (int i = 0; i < 4; i++) {
            m4[i] = (r.sc[i] >> 4) & 0x0F0F0F0Fu;
            s4[i] = r.sc[i] & 0x0F0F0F0Fu;
            c4[i] = ((m4[i] + 0x0F0F0F0Fu) & 0x10101010u) * 3u >> 1;
        }
        f32x16 part[NT], acc[NT];
#pragma unroll
        for (int n = 0; n < NT; n++) part[n] = (f32x16){};
        for_c<16>([&](auto ti) {
            constexpr int t = decltype(ti)::value, J = (t & 7) >> 1;
            constexpr uint32_t sel = 0x04000400u + 0x00010001u * (t & 3);
            const u32x2 q = r.q[t >> 3][t & 1];
            const half2v sc = as_h2(__builtin_amdgcn_perm(0x64646464u, s4[t >> 2], sel)) - k;
            const half2v off = -sc * as_h2(__builtin_amdgcn_perm(0x54545454u, c4[t >> 2], sel));  // -(64 + C) sc
            if constexpr (t % kFold == 0) {
#pragma unroll
                for (int m = 0; m < NT; m++) acc[m] = (f32x16){};
            }
            mfma_xw<HL, NT>(c, join(pair<J, 0>(q.x, sc, off, top), pair<J, 1>(q.x, sc, off, top), pair<J, 0>(q.y, sc, off, top),
                                    pair<J, 1>(q.y, sc, off, top)),
                            16 * t + 8 * c.kh, acc);
            if constexpr (t % kFold == kFold - 1) fold<NT>(part, d, acc);
        });
        // centre and min term: sum_t C (sc_t & 15) X16_t and (sc_t >> 4) X16_t with X16 = 2^-4 sum(x), K half kh
        // holding t = 8kh .. 8kh+7
        const half2v mm = dup((float)(1 << kX16Shift)), centre = dup(1.5f);
        // the scales of the centred sub-blocks: bytes with a nonzero min keep theirs
        const uint32_t k0 = (((c.kh ? c4[2] : c4[0]) >> 4) & 0x01010101u) * 15u, k1 = (((c.kh ? c4[3] : c4[1]) >> 4) & 0x01010101u) * 15u;
        const half2v cm = mm * centre;
        const half8 wl = bytes_to_h8_plain((c.kh ? s4[2] : s4[0]) & k0, (c.kh ? s4[3] : s4[1]) & k1, k) * join(cm, cm, cm, cm);
        const half8 wm = bytes_to_h8_plain(c.kh ? m4[2] : m4[0], c.kh ? m4[3] : m4[1], k) * join(mm, mm, mm, mm);
#pragma unroll
        for (int n = 0; n < NT; n++) {
            const half8 xh = c.x16(n, 0), xl = c.x16(n, 1);
            const f32x16 ct = mfma(xl, wl, mfma(xh, wl, (f32x16){})), mn = mfma(xl, wm, mfma(xh, wm, (f32x16){}));
#pragma unroll
            for (int i = 0; i < 16; i++) part[n][i] += fmaf(d, ct[i], -dmin * mn[i]);
        }
        fold_columns<HL, NT>(c, part, tot);
    }
};

// Q3_K (matVecQ3Kraw, LlamaTransformerHandler.java): 110-byte blocks [hmask 32]
// [qs 64][scales 12][d]; sub-block t = 8h + 2j + r covers columns 128h + 32j +
// 16r + l, whose 3-bit quant is 2 bits at shift 2j of qs[32h + 16r + l] and bit
// 4h + j of hmask[16r + l], minus 4, with the 6-bit scale of t minus 32:
// w = d*(sc - 32)*(q - 4).  B = q - 4 (exact), folded per K-step.  Blocks are
// 2-byte aligned: fields are read as aligned dwords and realigned.
struct FmtQ3K {
    static constexpr int kSums = 0;
    static constexpr int kBytes = 110;
    static constexpr int kChunks = (kBytes + 14 + 15) / 16;  // a 2-byte-aligned block spans <= 8 chunks
    static constexpr int kRowChunks = kChunks + 1;           // 36-dword window rows (2-way bank conflicts)
    struct Regs {
        u32x2 q[2][2];  // [h][r]: qs bytes 32 + 32h + 16r + 8kh .. +8
        u32x2 hm[2];    // [r]: hmask bytes 16r + 8kh .. +8
        u32x4 sd;       // scale bytes 96..107 (aux0, aux1, aux2), then d in the low half of .w
    };
    static __device__ __forceinline__ void load(Regs &r, const uint8_t *p, int kh) {
#pragma unroll
        for (int h = 0; h < 2; h++)
#pragma unroll
            for (int o = 0; o < 2; o++) r.q[h][o] = lds_u32x2(p + 32 + 32 * h + 16 * o + 8 * kh);
#pragma unroll
        for (int o = 0; o < 2; o++) r.hm[o] = lds_u32x2(p + 16 * o + 8 * kh);
        r.sd = lds_u32x4(p + 96);
    }
    // run t: 16 columns from 16 t on as bytes q + kBias, their scale and min
    static constexpr int kBias = 4;
    static constexpr bool kMin = false;
    static __device__ __forceinline__ u32x4 run(const uint8_t *p, int t, float &sc, float &mn) {
        const int h = t >> 3, j = (t >> 1) & 3, rr = t & 1;
        const int lo4 = (p[96 + (t & 7)] >> (4 * h)) & 15, hi2 = (p[104 + (t & 3)] >> (2 * (t >> 2))) & 3;
        sc = half_bits_to_float(*reinterpret_cast<const uint16_t *>(p + 108)) * (float)((lo4 | (hi2 << 4)) - 32);
        mn = 0.f;
        return ((load16(p + 32 + 32 * h + 16 * rr) >> (2 * j)) & 0x03030303u) |
               (((load16(p + 16 * rr) >> (4 * h + j)) & 0x01010101u) << 2);
    }
    template <bool HL, int NT, Sums SUMS, class C>
    static __device__ __forceinline__ void compute(const Regs &r, const C &c, float (&tot)[NT][kOut<HL>]) {
        const half2v off = dup(1028.f);  // 1024 + 4
        f32x16 part[NT], quarter[NT], half[NT];
#pragma unroll
        for (int n = 0; n < NT; n++) part[n] = (f32x16){};
        const float d = half_bits_to_float(r.sd.w);
#pragma unroll
        for (int h = 0; h < 2; h++) {
            // the scale words of this half (utmp[2h], utmp[2h+1] of dequantizeQ3K)
            const uint32_t aux2 = r.sd.z;
            const uint32_t ua = ((r.sd.x >> (4 * h)) & 0x0f0f0f0fu) | (((aux2 >> (4 * h)) & 0x03030303u) << 4);
            const uint32_t ub = ((r.sd.y >> (4 * h)) & 0x0f0f0f0fu) | (((aux2 >> (4 * h + 2)) & 0x03030303u) << 4);
#pragma unroll
            for (int j = 0; j < 4; j++)
#pragma unroll
                for (int rr = 0; rr < 2; rr++) {
                    const int t = 8 * h + 2 * j + rr;
                    const u32x2 q = r.q[h][rr], hm = r.hm[rr];
                    const int hb = 4 * h + j;
                    const uint32_t u0 = ((q.x >> (2 * j)) & 0x03030303u) | (((hm.x >> hb) & 0x01010101u) << 2);
                    const uint32_t u1 = ((q.y >> (2 * j)) & 0x03030303u) | (((hm.y >> hb) & 0x01010101u) << 2);
                    f32x16 acc[NT];
#pragma unroll
                    for (int m = 0; m < NT; m++) acc[m] = (f32x16){};
                    mfma_xw<HL, NT>(c, bytes_to_h8(u0, u1, off), 16 * t + 8 * c.kh, acc);
                    const int s6 = (int)byte_of(j < 2 ? ua : ub, 2 * (j & 1) + rr) - 32;
                    fold<NT>(part, d * (float)s6, acc);
                    if (SUMS == kChained && t % 4 == 3) step_fence(part);
                    if (SUMS == kChained) next_quarter<NT>(t, part, quarter, half);
                }
        }
        fold_columns<HL, NT>(c, part, tot);
    }
};

// The columns (bits of a mask) of which a block was left out (see split_x)
template <bool HL, int NT, class C>
__device__ __forceinline__ uint64_t marked_columns(const C &c) {
    const uint64_t b = __builtin_amdgcn_ballot_w64(c.cs()[threadIdx.x & (HL ? 15 : 32 * NT - 1)] < 0.f);
    return HL ? b & 0xFFFF : NT == 1 ? b & 0xFFFFFFFFu : b;
}

// What a walk has met of them: the columns, and the super-blocks modulo 64.  Mostly that
// is a block or two (activations that are products, silu * up, have one in 10^6
// elements), so add_exact looks at the x of those super-blocks only, and one column at a
// time has the loads of four runs in flight.  8B feed-forward at B = 128, us: all
// super-blocks of the walk, four columns at a time 197-206; now 182, as without such
// blocks.  With one outlier, 14336 x 4096 Q4_K 75.9 -> 61.6, 4096 x 14336 Q6_K 100 -> 83.
struct Marks {
    uint64_t cols = 0, blocks = 0;
    __device__ __forceinline__ void add(uint64_t c, int sb) {
        cols |= c;
        blocks |= c ? 1ull << (sb & 63) : 0;
    }
};

// tot += the fp32 products of the blocks that were left out, with x itself and folded
// like those of the fp32 kernels (scale * sum(q x) - min * sum(x)), so that infinities
// and NaN come out as there.  x and p are the columns' and the lane's row's super-block
// 0; half kh of a row's lanes takes 128 columns of a block.  From three columns on four
// at a time share the weights' decode and have their loads in flight
// together: with an outlier in every block of every vector, us, one column at a time /
// four (two vectors: two and four runs) / the fp32 kernels, 14336 x 4096 Q4_K at B = 128
// 2540 / 1345 / 1998, 4096 x 14336 Q6_K 4340 / 1760 / 1440, 9216 x 3072 Q8_0 at B = 2 48 /
// 37 / 25.
template <class F, int K, int kUnroll, int NT, int NI>
__device__ __forceinline__ void add_columns(const Marks &marks, const uint8_t *p, const float *x, size_t ldx, int sb0, int sb1,
                                            int kh, float (&tot)[NT][NI]) {
    for (uint64_t cols = marks.cols; cols;) {
        int b[K];
        uint32_t off[K];
#pragma unroll
        for (int c = 0; c < K; c++) {
            b[c] = cols ? __builtin_ctzll(cols) : -1;
            off[c] = (uint32_t)(b[c] < 0 ? b[0] : b[c]);
            cols &= cols - 1;  // (0 stays 0)
        }
        float acc[K] = {};
#pragma unroll 1
        for (int sb = sb0; sb < sb1; sb++) {
            if (!(marks.blocks >> (sb & 63) & 1)) continue;
            const float *xb[K];
            float4 v[K];
#pragma unroll
            for (int c = 0; c < K; c++) {
                xb[c] = x + off[c] * ldx + 256 * sb;
                v[c] = load_f4(xb[c] + 4 * (threadIdx.x & 63));
            }
            bool bad[K], any = false;
#pragma unroll
            for (int c = 0; c < K; c++) {
                const float e[4] = {fabsf(v[c].x), fabsf(v[c].y), fabsf(v[c].z), fabsf(v[c].w)};
                const float four = larger(larger(e[0], e[1]), larger(e[2], e[3]));
                float lone = INFINITY, m = row16_max(four);
#pragma unroll
                for (int i = 0; i < 4; i++) lone = e[i] != 0.f ? fminf(lone, e[i]) : lone;
                m = larger(m, __shfl_xor(m, 16));
                m = larger(m, __shfl_xor(m, 32));
                bad[c] = __builtin_amdgcn_ballot_w64(unfit(m, lone, four != 0.f ? four : INFINITY)) != 0;
                any |= bad[c];
            }
            if (!any) continue;
            float s[K] = {};
#pragma unroll kUnroll
            for (int t = 8 * kh; t < 8 * kh + 8; t++) {
                float sc, mn;
                const u32x4 q = F::run(p + (size_t)sb * F::kBytes, t, sc, mn);
                float4 u[K][4];
#pragma unroll
                for (int c = 0; c < K; c++)
#pragma unroll
                    for (int i = 0; i < 4; i++) u[c][i] = load_f4(xb[c] + 16 * t + 4 * i);
                float dot[K] = {}, sum[K] = {};
#pragma unroll
                for (int i = 0; i < 4; i++)
#pragma unroll
                    for (int j = 0; j < 4; j++) {
                        const float w = (float)((int)byte_of(q[i], j) - F::kBias);
#pragma unroll
                        for (int c = 0; c < K; c++) {
                            const float e = j == 0 ? u[c][i].x : j == 1 ? u[c][i].y : j == 2 ? u[c][i].z : u[c][i].w;
                            dot[c] = fmaf(w, e, dot[c]);
                            sum[c] += e;
                        }
                    }
#pragma unroll
                for (int c = 0; c < K; c++) {
                    s[c] = fmaf(sc, dot[c], s[c]);
                    if (F::kMin) s[c] = fmaf(-mn, sum[c], s[c]);
                }
            }
#pragma unroll
            for (int c = 0; c < K; c++) acc[c] = bad[c] ? acc[c] + s[c] : acc[c];
        }
#pragma unroll
        for (int c = 0; c < K; c++) {
            acc[c] += __shfl_xor(acc[c], 32);
#pragma unroll
            for (int n = 0; n < NT; n++)
#pragma unroll
                for (int i = 0; i < NI; i++) tot[n][i] = batch_of(n, i, kh) == b[c] ? tot[n][i] + acc[c] : tot[n][i];
        }
    }
}

template <class F, int NT, int NI>
__device__ __forceinline__ void add_exact(const Marks &marks, const uint8_t *p, const float *x, size_t ldx, int sb0, int sb1,
                                          int kh, float (&tot)[NT][NI]) {
    if constexpr (NI == 8) add_columns<F, 2, 4>(marks, p, x, ldx, sb0, sb1, kh, tot);  // (HL: two vectors)
    else if (__builtin_popcountll(marks.cols) <= 2) add_columns<F, 1, 4>(marks, p, x, ldx, sb0, sb1, kh, tot);
    else add_columns<F, 4, 1>(marks, p, x, ldx, sb0, sb1, kh, tot);
}

// A wave's 32 weight rows (past the end: the last row again): a wave-uniform
// 16-byte-aligned base and 32-bit offsets from it, which cost a lane half the
// registers of addresses.  mfma_applies bounds the pitch so that they hold.
struct RowSpan {
    size_t pitch;
    int row0, rbase, nrows;
    __device__ __forceinline__ int row(int rho) const { return min(rbase + rho, nrows - 1); }
    __device__ __forceinline__ size_t first() const { return (size_t)(row0 + row(0)) * pitch; }
    __device__ __forceinline__ size_t base() const { return first() & ~size_t(15); }
    __device__ __forceinline__ uint32_t offset(int rho) const {
        return (uint32_t)(first() & 15) + (uint32_t)(row(rho) - row(0)) * (uint32_t)pitch;
    }
};

// ------------------------------------------------------------------ tile output
// A workgroup's tile goes straight into y when K is not split.  Otherwise
// each split stores its partial tile with coherent (L2-bypassing) stores and
// bumps the tile's counter; the split that arrives last adds all partials in
// split order into y -- a fixed order, whatever the arrival order, so the
// result is deterministic -- and re-arms the counter for the next launch.
// Coherent stores plus a wait for their completion before the counter
// increment avoid a device-scope release, which on a multi-XCD part writes
// back the whole L2 (~100 us per workgroup measured); a separate reduction
// launch costs ~5 us.
constexpr int kMaxTileCounters = kCounterSlots;

template <bool WIDE = false, int NT, int NI>
__device__ __forceinline__ void store_tile(const float (&tot)[NT][NI], int r, int nrows, int kh, int B, float *__restrict__ Y,
                                           float *part, size_t plane, int *counters, int tile, int split, int ksplit) {
    const bool live = r < nrows;
    if (ksplit == 1) {
        if (!live) return;
#pragma unroll
        for (int n = 0; n < NT; n++)
#pragma unroll
            for (int i = 0; i < NI; i++) {
                const int b = batch_of(n, i, kh);
                if (b < B) Y[(size_t)b * nrows + r] = tot[n][i];
            }
        return;
    }
    if (live) {
        float *mine = part + split * plane;
#pragma unroll
        for (int n = 0; n < NT; n++)
#pragma unroll
            for (int i = 0; i < NI; i++) {
                const int b = batch_of(n, i, kh);
                if (b < B) __hip_atomic_store(mine + (size_t)b * nrows + r, tot[n][i], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            }
    }
    // Ordering of the hand-off.  The partials are agent-scope atomic stores, which
    // gfx950 performs at the memory-side coherence point (past the per-XCD L2s);
    // s_waitcnt(0) returns only once each of this wave's stores is acknowledged
    // there, and the barrier makes every wave's acknowledgement precede the
    // counter's fetch_add, itself performed at that point.  The last arriver then
    // reads the partials with agent-scope atomic loads, which are served from the
    // same point.  A release / acquire pair on the counter would order them
    // formally, but an agent-scope release writes back the whole L2 of the XCD
    // (buffer_wbl2), which measured ~100 us per GEMV; there are no non-atomic
    // stores for it to publish.
    __builtin_amdgcn_s_waitcnt(0);  // this wave's partials have reached the coherence point
    JH_MT(kMtEpi);
    __shared__ int s_last;
    __syncthreads();
    if (threadIdx.x == 0) {
        const int old = __hip_atomic_fetch_add(counters + tile * kCounterStride, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        const int last = old == ksplit - 1;
        if (last) __hip_atomic_store(counters + tile * kCounterStride, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        s_last = last;
    }
    __syncthreads();
    JH_MT(kMtEpi + 1);
    if (!s_last || !live) return;
    // KB splits' partials in flight at a time, added in split order
    constexpr int KB = 4 / NT;
    const int ks = ksplit;
    float acc[NT][NI];
#pragma unroll
    for (int n = 0; n < NT; n++)
#pragma unroll
        for (int i = 0; i < NI; i++) acc[n][i] = 0.f;
    for (int k0 = 0; k0 < ks; k0 += KB) {
        float v[KB][NT][NI];
#pragma unroll
        for (int kk = 0; kk < KB; kk++) {
            const int k = k0 + kk;
#pragma unroll
            for (int n = 0; n < NT; n++)
#pragma unroll
                for (int i = 0; i < NI; i++) {
                    // unconditional (clamped) loads, so that they issue back to back;
                    // this split's own partial comes back from memory unchanged
                    const int b = min(batch_of(n, i, kh), B - 1);
                    v[kk][n][i] = __hip_atomic_load(part + min(k, ks - 1) * plane + (size_t)b * nrows + r,
                                                    __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                }
        }
        if constexpr (WIDE) {  // pairs first: see kChains
#pragma unroll
            for (int n = 0; n < NT; n++)
#pragma unroll
                for (int i = 0; i < NI; i++) {
#pragma unroll
                    for (int kk = 1; kk < KB; kk++) v[kk][n][i] = k0 + kk < ks ? v[kk][n][i] : 0.f;
                    const float s = v[0][n][i] + v[1][n][i];
                    acc[n][i] += KB == 4 ? s + (v[KB - 2][n][i] + v[KB - 1][n][i]) : s;
                }
        } else {
#pragma unroll
            for (int kk = 0; kk < KB; kk++)
                if (k0 + kk < ks)
#pragma unroll
                    for (int n = 0; n < NT; n++)
#pragma unroll
                        for (int i = 0; i < NI; i++) acc[n][i] += v[kk][n][i];
        }
    }
#pragma unroll
    for (int n = 0; n < NT; n++)
#pragma unroll
        for (int i = 0; i < NI; i++) {
            const int b = batch_of(n, i, kh);
            if (b < B) Y[(size_t)b * nrows + r] = acc[n][i];
        }
    JH_MT(kMtEpi + 2);
}

// ------------------------------------------------------------------ batched kernel
// One matrix of a grouped launch: the workgroups [wg0, wg0 + tiles * ksplit)
// are its row tiles x column chunks (more than 64 columns) x K splits (split fastest); its partial planes start at
// part0 floats into the group's partial buffer and its tile counters at cnt0.
struct MfmaProblem {
    const uint8_t *w;
    const float *x;
    float *y;
    size_t pitch, part0;
    int type, row0, rows, tiles, wg0, cnt0;
};
struct MfmaGroup {
    MfmaProblem p[kMaxMfmaGroup];
    float *part;
    int *counters;
    int n, nsb, ksb, ksplit, B, chunks;
    // SwiGLU pairs (mfma_group<.., true>): p[0] is gate, w2 the up matrix of the
    // same shape; a workgroup's waves 0-3 take 128 gate rows and waves 4-7 the
    // same up rows, and swiglu[b][r] = silu(gate) * up replaces both outputs
    const uint8_t *w2;
    float *swiglu;
};

// More than 64 columns (WIDE): chunks of 64 columns in one launch, in the kernel of
// 33..64 columns: before, the VALU kernels read the weights again for every 8
// columns (8B feed-forward at B = 128, whole block: 5456 -> 181 us).
// The VALU kernels sum a row in many lanes; one chain of fp32 sums per output over all
// of K is less exact than that.  So chunks of 32, whose accumulators leave the registers
// for it, sum in kChains chains over the super-blocks in turn and Q6_K and Q3_K, whose 16
// folds per super-block are most of their error, in quarters of a super-block as well.
// Groups with one of these two take chunks of 32 only, and those with Q8_0 where a
// workgroup walks more than kLongWalk super-blocks; and the splits' partials are added in
// pairs.  Error against 64 bits at B = 128, one or two chains / now / VALU kernels, 1e-7 of
// the norm: 20480 rows, K = 8192 Q8_0 1.39 / 1.13 / 1.28, Q3_K 1.14 / 1.05 / 1.12, Q6_K 1.14 /
// 1.05 / 1.14; 2048 x 3840 Q3_K 1.014 / 0.959 / 1.000.  us: 4096 x 14336 Q6_K 80.5 / 83, Q3_K
// 70.6 / 72, 16384 x 8192 Q8_0 141 / 150, 20000 x 14336 429 / 487, Q2_K 303 / 378.
template <bool WIDE, int NT>
constexpr Sums kSumsOf = !WIDE ? kPlain : NT == 1 ? kChained : kWide64;
constexpr int kChains = 4, kLongWalk = 16;

// format mask bits: Q4_K, Q5_K, Q6_K, Q8_0, Q2_K, Q3_K
template <int MASK>
__host__ __device__ constexpr int max_chunks() {
    int c = 0;
    if (MASK & 1) c = c > FmtQ4K::kRowChunks ? c : FmtQ4K::kRowChunks;
    if (MASK & 2) c = c > FmtQ5K::kRowChunks ? c : FmtQ5K::kRowChunks;
    if (MASK & 4) c = c > FmtQ6K::kRowChunks ? c : FmtQ6K::kRowChunks;
    if (MASK & 8) c = c > FmtQ8_0::kRowChunks ? c : FmtQ8_0::kRowChunks;
    if (MASK & 16) c = c > FmtQ2K::kRowChunks ? c : FmtQ2K::kRowChunks;
    if (MASK & 32) c = c > FmtQ3K::kRowChunks ? c : FmtQ3K::kRowChunks;
    return c;
}
// LDS: the x image (two of them for NT = 1), then the weight windows
template <bool HL, int NT, int MASK>
__host__ __device__ constexpr int lds_bytes() {
    return (NT == 1 ? 2 : 1) * XImage<HL, NT>::kBytes + kWaves * kRowsPerWave * max_chunks<MASK>() * 16 + kWinPad;
}

// store_tile for a SwiGLU pair workgroup (B <= 32): split partials over virtual
// rows (gate r, up rows + r) in planes of B x 2 rows, the usual hand-off, then
// the up waves pass their totals to the gate waves through LDS and those store
// silu(gate) * up.  r is the lane's row within its matrix, lw its row within
// the workgroup's 128.
template <int NI>
__device__ __forceinline__ void store_pair(const float (&tot)[1][NI], int r, int lw, bool up, int nrows, int kh, int B,
                                           float *__restrict__ out, float *part, int *counters, int tile, int split,
                                           int ksplit, uint8_t *lds) {
    const bool live = r < nrows;
    const int vr = r + (up ? nrows : 0);
    float fin[NI];
#pragma unroll
    for (int i = 0; i < NI; i++) fin[i] = tot[0][i];
    if (ksplit > 1) {
        const size_t plane = (size_t)B * 2 * nrows;
        if (live) {
            float *mine = part + split * plane;
#pragma unroll
            for (int i = 0; i < NI; i++) {
                const int b = batch_of(0, i, kh);
                if (b < B) __hip_atomic_store(mine + (size_t)b * 2 * nrows + vr, tot[0][i], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            }
        }
        __builtin_amdgcn_s_waitcnt(0);  // the same hand-off ordering as store_tile
        __shared__ int s_last;
        __syncthreads();
        if (threadIdx.x == 0) {
            const int old = __hip_atomic_fetch_add(counters + tile * kCounterStride, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            const int last = old == ksplit - 1;
            if (last) __hip_atomic_store(counters + tile * kCounterStride, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            s_last = last;
        }
        __syncthreads();
        if (!s_last) return;  // uniform across the workgroup
        constexpr int KB = 4;
        float acc[NI];
#pragma unroll
        for (int i = 0; i < NI; i++) acc[i] = 0.f;
        const int rr = min(vr, 2 * nrows - 1);
        for (int k0 = 0; k0 < ksplit; k0 += KB) {
            float v[KB][NI];
#pragma unroll
            for (int kk = 0; kk < KB; kk++)
#pragma unroll
                for (int i = 0; i < NI; i++) {
                    const int b = min(batch_of(0, i, kh), B - 1);
                    v[kk][i] = __hip_atomic_load(part + min(k0 + kk, ksplit - 1) * plane + (size_t)b * 2 * nrows + rr,
                                                 __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                }
#pragma unroll
            for (int kk = 0; kk < KB; kk++)
                if (k0 + kk < ksplit)
#pragma unroll
                    for (int i = 0; i < NI; i++) acc[i] += v[kk][i];
        }
#pragma unroll
        for (int i = 0; i < NI; i++) fin[i] = acc[i];
    }
    float *xl = reinterpret_cast<float *>(lds);  // [128 rows][33]: the up totals
    __syncthreads();  // every wave is done with the x buffers
    if (up)
#pragma unroll
        for (int i = 0; i < NI; i++) xl[lw * 33 + batch_of(0, i, kh)] = fin[i];
    __syncthreads();
    if (!up && live)
#pragma unroll
        for (int i = 0; i < NI; i++) {
            const int b = batch_of(0, i, kh);
            if (b < B) out[(size_t)b * nrows + r] = silu_times(fin[i], xl[lw * 33 + b]);
        }
}

// One workgroup's tile (32 rows per wave x all batch columns) over the K
// range of its split, x converted into LDS super-block by super-block.
// WIDE: column chunk `chunk` of g.chunks (32 NT columns each).
// EXACT: see split_x.  NT: column groups of 32 (HL: one of 16)
template <class F, bool HL, int NT, bool PAIR, bool WIDE, bool EXACT>
__device__ __forceinline__ void gemm_body(const MfmaProblem &P, int tile, int chunk, int split, const MfmaGroup &g, uint8_t *lds) {
    constexpr Sums SUMS = kSumsOf<WIDE, NT>;
    const int chunks = WIDE ? g.chunks : 1, col0 = WIDE ? chunk * 32 * NT : 0;
    using I = XImage<HL, NT>;
    constexpr int NI = kOut<HL>;
    constexpr int CH = F::kChunks;          // 16-byte chunks staged per row and super-block
    constexpr int CL = (kRowsPerWave * CH + 63) / 64;  // chunks per lane
    const bool up_half = PAIR && (threadIdx.x >> 6) >= kWaves / 2;  // SwiGLU pairs: waves 4-7 take the up rows
    const uint8_t *W = up_half ? g.w2 : P.w;
    const float *__restrict__ X = P.x + (size_t)col0 * (256 * g.nsb);
    const size_t pitch = P.pitch;
    const int nrows = P.rows, row0 = P.row0, B = WIDE ? min(32 * NT, g.B - col0) : g.B, cols = 256 * g.nsb;

    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int lane = threadIdx.x & 63, lr = lane & 31, kh = lane >> 5;
    const int rbase = PAIR ? tile * (kRowsPerWG / 2) + (wave & (kWaves / 2 - 1)) * kRowsPerWave
                           : tile * kRowsPerWG + wave * kRowsPerWave;
    const int sb0 = split * g.ksb, sb1 = min(g.nsb, sb0 + g.ksb);
    // Weight staging: chunk j = lane + 64 k of the wave's 32 x CH chunk grid is
    // row j / CH, 16-byte piece j % CH of that row's aligned window.  Whole
    // aligned 16-byte lanes, consecutive within a row: few cache accesses per
    // load, instead of 8-byte gathers from 32 rows at 2-byte alignment.
    const RowSpan rows{pitch, row0, rbase, nrows};
    uint32_t coff[CL];
#pragma unroll
    for (int k = 0; k < CL; k++) {
        const int j = min(lane + 64 * k, kRowsPerWave * CH - 1);
        coff[k] = rows.offset(j / CH) + 16 * (j % CH);
    }
    const uint32_t myoff = rows.offset(lr);
    W += rows.base();
    constexpr int RC = NT == 1 ? F::kRowChunks : CH;  // window row stride (chunks): padded for the realigned reads
    uint8_t *wslot = lds + (NT == 1 ? 2 : 1) * I::kBytes + wave * (kRowsPerWave * RC * 16);

    u32x4 ch_n[CL];
    float xv_n[NT][16];  // the next super-block's raw x: column (threadIdx.x >> 4) + 32 i, values 16 q .. +16
    const int xq = threadIdx.x & 15, xcol = threadIdx.x >> 4;
    const bool stager = xcol < I::kCols;  // HL: half of the threads hold the 16 columns
    // (a macro rather than a lambda: the register arrays must stay in VGPRs)
#define JH_LOAD_W(SB)                                                                                      \
    do {                                                                                                   \
        const uint32_t sbo = (uint32_t)(SB) * F::kBytes;                                                       \
        _Pragma("unroll") for (int k = 0; k < CL; k++)                                                     \
            ch_n[k] = *reinterpret_cast<const u32x4 *>(W + ((coff[k] + sbo) & ~15u));               \
    } while (0)
#define JH_LOAD_X(SB)                                                                                      \
    do {                                                                                                   \
        _Pragma("unroll") for (int i = 0; i < NT; i++) {                                                   \
            const int b = xcol + 32 * i;                                                                   \
            const float4 *xp = reinterpret_cast<const float4 *>(X + (size_t)min(b, B - 1) * cols +        \
                                                                (SB) * 256 + 16 * xq);                     \
            _Pragma("unroll") for (int k = 0; k < 4; k++) {                                                \
                const float4 v = b < B ? xp[k] : make_float4(0.f, 0.f, 0.f, 0.f);                         \
                xv_n[i][4 * k] = v.x; xv_n[i][4 * k + 1] = v.y; xv_n[i][4 * k + 2] = v.z; xv_n[i][4 * k + 3] = v.w; \
            }                                                                                              \
        }                                                                                                  \
    } while (0)
#define JH_PARK()                                                                                          \
    do {                                                                                                   \
        _Pragma("unroll") for (int k = 0; k < CL; k++)                                                     \
            if (lane + 64 * k < kRowsPerWave * CH)                                                         \
                *reinterpret_cast<u32x4 *>(wslot + 16 * win_chunk<CH, RC>(lane + 64 * k)) = ch_n[k];       \
    } while (0)

    Marks marked;  // blocks left to add_exact
    float tot[NT][NI], more[kChains - 1][NI];  // (kChained: the other chains)
    if constexpr (SUMS == kChained) {
#pragma unroll
        for (int k = 0; k < kChains - 1; k++)
#pragma unroll
            for (int i = 0; i < NI; i++) more[k][i] = 0.f;
    }
#pragma unroll
    for (int n = 0; n < NT; n++)
#pragma unroll
        for (int i = 0; i < NI; i++) tot[n][i] = 0.f;

    if constexpr (NT == 1) {
        // Two x buffers: super-block sb + 1's x is converted into the free
        // buffer while sb's MFMAs run, with one barrier per super-block.  The
        // buffer a step writes was last read by the previous step's MFMAs,
        // which every wave finished before this step's barrier.
        JH_MT(0);
        if (HL && !stager) {  // the lo limbs' rows carry no sums
            I::zero_sums(lds, xq, xcol);
            I::zero_sums(lds + I::kBytes, xq, xcol);
        }
        if (sb0 < sb1) {
            if (stager) JH_LOAD_X(sb0);
            JH_LOAD_W(sb0);
            if (stager) I::template store<F::kSums, EXACT>(lds, xv_n[0], xq, xcol);
            if (stager && sb0 + 1 < sb1) JH_LOAD_X(sb0 + 1);
        }
        for (int sb = sb0; sb < sb1; sb++) {
            const int buf = (sb - sb0) & 1;
            __syncthreads();  // x of sb is staged; the other buffer is free
            JH_MT(1 + 4 * (sb - sb0));
            JH_PARK();
            JH_MT(2 + 4 * (sb - sb0));
            typename F::Regs w;
            F::load(w, wslot + lr * RC * 16 + ((myoff + (uint32_t)sb * F::kBytes) & 15), kh);
            if (sb + 1 < sb1) {
                if (stager) {
                    I::template store<F::kSums, EXACT>(lds + (buf ^ 1) * I::kBytes, xv_n[0], xq, xcol);
                    if (sb + 2 < sb1) JH_LOAD_X(sb + 2);
                }
                JH_LOAD_W(sb + 1);
            }
            JH_MT(3 + 4 * (sb - sb0));
            const Ctx<HL, NT> c{lr, kh, lds + buf * I::kBytes};
            if constexpr (EXACT) marked.add(marked_columns<HL, NT>(c), sb);
            F::template compute<HL, NT, SUMS>(w, c, tot);
            if constexpr (SUMS == kChained) {
#pragma unroll
                for (int i = 0; i < NI; i++) {
                    const float v = tot[0][i];
                    tot[0][i] = more[0][i];
#pragma unroll
                    for (int k = 0; k + 1 < kChains - 1; k++) more[k][i] = more[k + 1][i];
                    more[kChains - 2][i] = v;
                }
            }
            JH_MT(4 + 4 * (sb - sb0));
        }
    } else {
        if (sb0 < sb1) {
            JH_LOAD_X(sb0);
            JH_LOAD_W(sb0);
        }
        for (int sb = sb0; sb < sb1; sb++) {
            __syncthreads();  // the previous super-block's LDS contents are consumed
#pragma unroll
            for (int i = 0; i < NT; i++) I::template store<F::kSums, EXACT>(lds, xv_n[i], xq, xcol + 32 * i);
            JH_PARK();
            // this lane's row block inside its staged window (same wave: no barrier)
            typename F::Regs w;
            F::load(w, wslot + lr * RC * 16 + ((myoff + (uint32_t)sb * F::kBytes) & 15), kh);
            // The loads below overlap this super-block's math.  They are unconditional (after the last
            // super-block, that one again): a load inside a branch is waited for at the branch's end
            // (2 x 14336 x 4096 Q4_K, B = 64: 65 -> 59 us).
            JH_LOAD_X(min(sb + 1, sb1 - 1));
            JH_LOAD_W(min(sb + 1, sb1 - 1));
            __syncthreads();
            const Ctx<HL, NT> c{lr, kh, lds};
            if constexpr (EXACT) marked.add(marked_columns<HL, NT>(c), sb);
            F::template compute<HL, NT, SUMS>(w, c, tot);
        }
    }
#undef JH_LOAD_X
#undef JH_LOAD_W
#undef JH_PARK

    if constexpr (EXACT) {
        if (__builtin_expect(marked.cols != 0, 0))
            add_exact<F>(marked, W + myoff, X, cols, sb0, sb1, kh, tot);
    }
    if constexpr (PAIR) {
        store_pair(tot, rbase + lr, (wave & (kWaves / 2 - 1)) * kRowsPerWave + lr, up_half, nrows, kh, B,
                   g.swiglu, g.part, g.counters, tile, split, g.ksplit, lds);
        return;
    }
    if constexpr (SUMS == kChained) {
#pragma unroll
        for (int i = 0; i < NI; i++) tot[0][i] = (tot[0][i] + more[0][i]) + (more[1][i] + more[2][i]);
    }
    store_tile<WIDE>(tot, rbase + lr, nrows, kh, B, P.y + (size_t)col0 * nrows, g.part + P.part0 + (size_t)col0 * nrows,
               (size_t)g.B * nrows, g.counters + (size_t)P.cnt0 * kCounterStride, tile * chunks + chunk, split, g.ksplit);
}

// A group of matrices with the same K in one launch (1-D grid): each
// workgroup finds its matrix and runs that matrix's format.
template <bool HL, int NT, int MASK, bool PAIR = false, bool WIDE = false, bool EXACT = WIDE>
__global__ __launch_bounds__(kThreads) void mfma_group(MfmaGroup g) {
    __shared__ __align__(16) uint8_t lds[lds_bytes<HL, NT, MASK>()];
    const int id = blockIdx.x;
    int m = 0;
    for (int i = 1; i < g.n; i++)
        if (id >= g.p[i].wg0) m = i;
    const MfmaProblem &P = g.p[m];
    const int local = id - P.wg0, at = local / g.ksplit, split = local - at * g.ksplit;
    const int tile = WIDE ? at / g.chunks : at, chunk = WIDE ? at - tile * g.chunks : 0;
    switch (P.type) {
        case 12: if constexpr ((MASK & 1) != 0) gemm_body<FmtQ4K, HL, NT, PAIR, WIDE, EXACT>(P, tile, chunk, split, g, lds); break;
        case 13: if constexpr ((MASK & 2) != 0) gemm_body<FmtQ5K, HL, NT, PAIR, WIDE, EXACT>(P, tile, chunk, split, g, lds); break;
        case 14: if constexpr ((MASK & 4) != 0) gemm_body<FmtQ6K, HL, NT, PAIR, WIDE, EXACT>(P, tile, chunk, split, g, lds); break;
        case 10: if constexpr ((MASK & 16) != 0) gemm_body<FmtQ2K, HL, NT, PAIR, WIDE, EXACT>(P, tile, chunk, split, g, lds); break;
        case 11: if constexpr ((MASK & 32) != 0) gemm_body<FmtQ3K, HL, NT, PAIR, WIDE, EXACT>(P, tile, chunk, split, g, lds); break;
        default: if constexpr ((MASK & 8) != 0) gemm_body<FmtQ8_0, HL, NT, PAIR, WIDE, EXACT>(P, tile, chunk, split, g, lds); break;
    }
}

// one workgroup per super-block: 32 (HL: 16) columns x 16 lanes (columns >= B are zero)
template <bool HL, bool EXACT>
__global__ __launch_bounds__(HL ? 256 : 512) void x_prep(const float *__restrict__ X, int B, int cols, uint8_t *__restrict__ slabs) {
    const int sb = blockIdx.x, q = threadIdx.x & 15, col = threadIdx.x >> 4;
    float xv[16];
    const float4 *xp = reinterpret_cast<const float4 *>(X + (size_t)min(col, B - 1) * cols + sb * 256 + 16 * q);
#pragma unroll
    for (int k = 0; k < 4; k++) {
        const float4 v = col < B ? xp[k] : make_float4(0.f, 0.f, 0.f, 0.f);
        xv[4 * k] = v.x;
        xv[4 * k + 1] = v.y;
        xv[4 * k + 2] = v.z;
        xv[4 * k + 3] = v.w;
    }
    Slab<HL>::template store<EXACT>(slabs + (size_t)sb * Slab<HL>::kBytes, xv, q, col);
}

// The B <= 32 kernel on prepared x, for matrices with enough row tiles to
// fill the GPU without splitting K (the output projection).  It reads x once
// per super-block from a slab that x_prep wrote, instead of converting it in
// every workgroup.  Per super-block each wave:
//  1. waits until its share of this super-block's x slab (DMA) and its
//     weight chunks have landed, and meets the others at the one barrier;
//  2. starts the DMA of the next slab into the other LDS buffer (everyone has
//     finished the super-block that used it);
//  3. moves its weight chunks through its LDS window into the format's
//     registers and starts the loads of the super-block after next into the
//     freed register set (two sets alternate: weights stay two super-blocks
//     ahead with no register copies);
//  4. runs the MFMAs.
// Loads are issued unconditionally (addresses clamped to the last super-block
// of the range) so that every wave's count of memory operations in flight is
// the same static number at each wait.
template <class F, bool HL, bool EXACT>
__global__ __launch_bounds__(kThreads) void mfma_px(const uint8_t *W, size_t pitch, int row0, int nrows,
                                                    int nsb, const uint8_t *__restrict__ slabs,
                                                    const float *__restrict__ X, float *__restrict__ Y, int B) {
    constexpr int CH = F::kChunks;
    constexpr int CL = (kRowsPerWave * CH + 63) / 64;
    using I = Slab<HL>;
    constexpr int XI = (I::kRows + kWaves - 1) / kWaves;  // slab rows per wave
    __shared__ __align__(16) uint8_t sh_x[2][I::kBytes];
    constexpr int RC = F::kRowChunks;  // window row stride (chunks)
    __shared__ __align__(16) uint8_t sh_w[kWaves * kRowsPerWave * RC * 16 + kWinPad];

    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int lane = threadIdx.x & 63, lr = lane & 31, kh = lane >> 5;
    const int rbase = blockIdx.x * kRowsPerWG + wave * kRowsPerWave;
    const int sb0 = 0, last = nsb - 1;
    const RowSpan rows{pitch, row0, rbase, nrows};
    uint32_t coff[CL];
#pragma unroll
    for (int k = 0; k < CL; k++) {
        const int j = min(lane + 64 * k, kRowsPerWave * CH - 1);
        coff[k] = rows.offset(j / CH) + 16 * (j % CH);
    }
    const uint32_t myoff = rows.offset(lr);
    W += rows.base();
    uint8_t *wslot = sh_w + wave * (kRowsPerWave * RC * 16);

    // The slab DMA is issued from inline asm, outside the compiler's
    // bookkeeping: its own waits would otherwise drain every load in flight
    // before the first LDS read after a DMA.  Unknown memory operations can
    // only make the compiler's remaining waits stricter, and the order below
    // keeps them exact (each step's weight chunks are waited for before the
    // step issues its DMA).
    auto dma_x = [&](int sb, int buf) {
        const uint8_t *src = slabs + (size_t)min(sb, last) * I::kBytes + 16 * lane;
        const uint32_t dst = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) uint8_t *)sh_x[buf];
#pragma unroll
        for (int k = 0; k < XI; k++) {
            const int r = min(wave + kWaves * k, I::kRows - 1);  // surplus waves repeat the last row (same bytes)
            asm volatile("s_mov_b32 m0, %1\n\tglobal_load_lds_dwordx4 %0, off" ::"v"(src + 1024 * r),
                         "s"(dst + 1024 * r)
                         : "memory", "m0");
        }
    };
    u32x4 wa[CL], wb[CL];
#define JH_LOAD_W(SET, SB)                                                                                 \
    do {                                                                                                   \
        const uint32_t sbo = (uint32_t)min((SB), last) * F::kBytes;                                        \
        _Pragma("unroll") for (int k = 0; k < CL; k++)                                                     \
            SET[k] = *reinterpret_cast<const u32x4 *>(W + ((coff[k] + sbo) & ~15u));                \
    } while (0)

    Marks marked;
    float tot[1][kOut<HL>] = {};
#define JH_STEP(SET, SB, BUF)                                                                              \
    do {                                                                                                   \
        /* this wave's part of slab SB and its chunks of SB have landed (only SB + 1's are in flight) */   \
        asm volatile("s_waitcnt vmcnt(%0)" ::"n"(CL) : "memory");                                        \
        _Pragma("unroll") for (int k = 0; k < CL; k++)                                                     \
            if (lane + 64 * k < kRowsPerWave * CH) *reinterpret_cast<u32x4 *>(wslot + 16 * win_chunk<CH, RC>(lane + 64 * k)) = SET[k]; \
        /* every wave's part of slab SB is in, and every wave is done with slab SB - 1 */                \
        asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");                                   \
        dma_x((SB) + 1, (BUF) ^ 1);                                                                        \
        typename F::Regs w;                                                                                \
        F::load(w, wslot + lr * RC * 16 + ((myoff + (uint32_t)(SB) * F::kBytes) & 15), kh);  \
        JH_LOAD_W(SET, (SB) + 2);                                                                          \
        const CtxP<HL> c{lr, kh, sh_x[BUF]};                                                               \
        if constexpr (EXACT) marked.add(marked_columns<HL, 1>(c), SB);                                     \
        F::template compute<HL, 1, kPlain>(w, c, tot);                                                      \
    } while (0)

    dma_x(sb0, 0);
    JH_LOAD_W(wa, sb0);
    JH_LOAD_W(wb, sb0 + 1);
    int sb = sb0;
    for (; sb < last; sb += 2) {  // pairs of steps: the register sets alternate by name
        JH_STEP(wa, sb, 0);
        JH_STEP(wb, sb + 1, 1);
    }
    if (sb == last) JH_STEP(wa, sb, 0);
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // no DMA into LDS outlives the workgroup
#undef JH_STEP
#undef JH_LOAD_W

    if constexpr (EXACT) {
        if (__builtin_expect(marked.cols != 0, 0)) add_exact<F>(marked, W + myoff, X, (size_t)256 * nsb, 0, nsb, kh, tot);
    }
    store_tile(tot, rbase + lr, nrows, kh, B, Y, nullptr, 0, nullptr, blockIdx.x, 0, 1);
}

}  // namespace

// ------------------------------------------------------------------ host side
// Up to 16 batch columns take the kernels whose MFMAs hold both limbs (HL).
constexpr int kHlMaxBatch = 16;

static bool mfma_applies(const MfmaDesc &d, int B) {
    if ((d.type != 12 && d.type != 13 && d.type != 14 && d.type != 8 && d.type != 10 && d.type != 11) ||
        B < 2 || d.cols % 256 ||
        d.cols <= 0 || d.row_end <= d.row_start)
        return false;
    if (d.pitch > (size_t(1) << 26)) return false;  // 32 rows' offsets in 32 bits
    if ((d.type == 12 || d.type == 13) && ((reinterpret_cast<uintptr_t>(d.w) | d.pitch) & 15))
        return false;  // K-quant rows are staged as whole aligned 16-byte chunks
    return (reinterpret_cast<uintptr_t>(d.x) & 15) == 0;  // x is read as float4
}

namespace {
struct Plan {
    int nsb, ksb, ksplit, grid;
    int chunks, chunk;  // B > 64: column chunks and their width, 64 or 32 columns
    bool prepared;  // one unsplit matrix, B <= 32: x_prep + mfma_px
    size_t slab_bytes, part_floats;
};
}  // namespace

// Two vectors: where this path's fixed 9 to 12 us (15 to 20 from K = 8192 on) are less
// than the fp32 kernels take.  Those read the weights once, bound by their arithmetic,
// in a launch per matrix (and one for silu * up); up to 2048 or 4096 rows all their
// workgroups are resident at once, evenly over the CUs, and their time is that of a
// row.  us, fp32 / here:
//   one matrix, Q4_K   6144 x 4096 10.3 / 10.9, 6656 x 4096 12.7 / 11.0, 9216 x 3072 13.8 / 11.9,
//                      4096 x 8192 12.1 / 14.2, 2048 x 14336 12.3 / 16.3, 2560 x 14336 19.0 / 16.5
//               Q5_K   6144 x 4096 11.7 / 12.7, 6656 x 4096 13.8 / 12.5, 4096 x 8192 14.6 / 16.1,
//                      2560 x 14336 22.4 / 18.9
//               Q8_0   10240 x 2048 12.9 / 13.3, 11008 x 2048 14.9 / 13.4, 5632 x 4096 15.6 / 14.2,
//                      4096 x 8192 20.0 / 17.5, 2048 x 14336 18.0 / 20.5, 2304 x 14336 31.6 / 20.7
//   a group of two     2048 x 2048 Q4_K 7.8 / 9.7, Q8_0 9.3 / 12.1; 2048 x 3072 10.9 / 10.4, 12.1 / 12.9;
//                      1792 x 4096 13.1 / 10.6, 19.3 / 13.1; 4096 x 2048 10.5 / 9.9, 13.5 / 12.7
//   a SwiGLU pair      2048 x 2048 Q4_K 9.9 / 9.8, Q8_0 11.3 / 12.5; 2560 x 2048 12.0 / 10.1, 15.2 / 12.6;
//                      5632 x 2048 14.8 / 10.6, 19.4 / 14.2; it has the limit of the group, whose bits it gives
// Only formats whose error against 64 bits is smaller here (K = 512 .. 28672: Q4_K
// 2.4-2.9e-7 / 1.8-2.0e-7, Q5_K 2.4-2.9e-7 / 1.8-2.0e-7, Q8_0 1.20-1.41e-7 / 0.81-1.25e-7);
// that of Q6_K and Q3_K is not, and Q2_K is not taken either.
static bool two_vectors_pay(int n, bool pair, int type, size_t rows, int cols) {
    const double weights = (double)rows * cols;
    if (pair || n > 1) return weights >= 14e6;
    if (type == 8) return weights >= (rows > 2048 ? 22e6 : 36e6);
    return weights >= (rows > 4096 ? 26e6 : 36e6);
}

// Row tiles of 256 rows; K split the same way for every matrix of the group.  pair:
// d[0] is a SwiGLU pair's virtual matrix, gate's rows and then up's: K is split as for
// the group of the two.
static bool plan_group(int n, const MfmaDesc *d, int B, Plan &p, bool pair = false) {
    if (n < 1 || n > kMaxMfmaGroup) return false;
    int tiles = 0;
    size_t rows = 0;
    bool fine = false, fine_long = false;  // chunks of 32 columns only, always or for long walks (see kChains)
    for (int i = 0; i < n; i++) {
        fine = fine || d[i].type == 14 || d[i].type == 11;
        fine_long = fine_long || d[i].type == 8;
        if (!mfma_applies(d[i], B) || d[i].cols != d[0].cols) return false;
        const int each = (d[i].row_end - d[i].row_start) / (pair ? 2 : 1);
        tiles += (pair ? 2 : 1) * ((each + kRowsPerWG - 1) / kRowsPerWG);
        rows += d[i].row_end - d[i].row_start;
        if (B == 2 && d[i].type != 12 && d[i].type != 13 && d[i].type != 8) return false;
    }
    if (B == 2 && !two_vectors_pay(n, pair, d[0].type, rows, d[0].cols)) return false;
    p.nsb = d[0].cols / 256;
    // One workgroup fits per CU (LDS, VGPRs), so the grid runs in rounds of
    // kMinWorkgroups.  Cost of a split, in super-block steps: rounds x (super-
    // blocks per workgroup + a workgroup's fixed prologue and epilogue, ~5
    // steps), plus one for the hand-off when K is split and a quarter step per
    // split (the partials the last workgroup sums); the smallest split wins
    // ties.  Fitted to the 8B B = 32 shapes ([gate, up]: 2 splits 44 us,
    // 3 splits 57 us, 16 splits 96 us; [o]: 8 splits ahead of 16).
    // More than 64 columns: also over chunks of 32 and of 64 columns, whose steps
    // cost 5 : 8 (2.6 and 4.2 us); a split never needs more scratch than the static
    // one holds.  (9216 x 3072 Q8_0 at B = 128, 36 row tiles: 95 us in chunks of 64, 54 us
    // in chunks of 32; 2 x 14336 x 4096 Q4_K, 112 row tiles: 96 us in chunks of 64.)
    long long best = LLONG_MAX;
    p.ksb = p.nsb;
    p.ksplit = 1;
    const int row_tiles = tiles;
    for (int c = B <= 64 || fine ? 32 : 64; c >= 32; c /= 2) {
        const int chunks = B <= 64 ? 1 : (B + c - 1) / c;
        if ((size_t)row_tiles * chunks > (size_t(1) << 30) / p.nsb) continue;  // the grid is an int
        const int ctiles = row_tiles * chunks;
        for (int ks = 1; ks <= p.nsb; ks++) {
            const int ksb = (p.nsb + ks - 1) / ks, kse = (p.nsb + ksb - 1) / ksb;
            if (c == 64 && fine_long && ksb > kLongWalk) continue;
            if (kse > 1 && ctiles > kMaxTileCounters) break;  // a split needs a counter per tile
            if (kse > 1 && B > 64 && sizeof(float) * (size_t)kse * B * rows > kStaticScratchBytes) break;
            const int rounds = (int)(((long long)ctiles * kse + kMinWorkgroups - 1) / kMinWorkgroups);
            const long long cost = (4ll * ((long long)rounds * (ksb + 5) + (kse > 1 ? 1 : 0)) + (kse > 1 ? kse : 0)) * (c == 64 ? 8 : 5);
            if (cost < best) {
                best = cost;
                p.ksb = ksb;
                p.ksplit = kse;
                p.chunks = chunks;
                p.chunk = c;
            }
        }
    }
    if (best == LLONG_MAX) return false;
    tiles = row_tiles * p.chunks;
    if (const char *f = getenv("JUNO_MFMA_KSPLIT")) {  // tuning runs: a forced split
        const int want = atoi(f);
        if (B <= 64 && want >= 1 && want <= p.nsb && (want == 1 || tiles <= kMaxTileCounters)) {
            p.ksb = (p.nsb + want - 1) / want;
            p.ksplit = (p.nsb + p.ksb - 1) / p.ksb;
        }
    }
    p.grid = tiles * p.ksplit;
    p.prepared = n == 1 && p.ksplit == 1 && B <= 32 && d[0].type != 10 && d[0].type != 11;  // slabs carry no 16-column sums
    p.slab_bytes = p.prepared ? (size_t)p.nsb * (B <= kHlMaxBatch ? Slab<true>::kBytes : Slab<false>::kBytes) : 0;
    p.part_floats = p.ksplit > 1 ? (size_t)p.ksplit * B * rows : 0;
    // two vectors never need more scratch than the static one holds
    return B != 2 || p.slab_bytes + p.part_floats * sizeof(float) <= kStaticScratchBytes;
}

size_t mfma_group_workspace_bytes(int n, const MfmaDesc *d, int B) {
    Plan p;
    if (!plan_group(n, d, B, p)) return 0;
    const size_t bytes = p.slab_bytes + p.part_floats * sizeof(float);
    return bytes > 256 ? bytes : 256;  // nonzero: the MFMA path applies
}

int mfma_group_plan(int n, const MfmaDesc *d, int B, int *ksplit) {
    Plan p;
    if (!plan_group(n, d, B, p)) return 0;
    *ksplit = p.ksplit;
    return p.prepared ? 2 : 1;
}

namespace {
template <bool HL, int NT>
void image_layout(MfmaLayout &l) {
    using I = XImage<HL, NT>;
    l.image_lo = 2 * I::kLo;
    l.image_xs = 2 * I::kXs;
    l.image_x16 = 2 * I::kX16;
    l.image_cs = I::kCs;
    l.image = I::kBytes;
}
template <bool HL>
void slab_layout(MfmaLayout &l) {
    l.image_lo = HL ? 0 : Slab<HL>::kLo;
    l.image_xs = Slab<HL>::kXs;
    l.image_x16 = 0;
    l.image_cs = Slab<HL>::kCs;
    l.image = Slab<HL>::kBytes;
}
template <class F, int MASK>
void format_layout(MfmaLayout &l, bool hl, int nt) {
    l.chunks16 = F::kChunks;
    l.row_chunks16 = nt == 1 ? F::kRowChunks : F::kChunks;
    l.lds = l.kernel == 2 ? 2 * l.image + kWaves * kRowsPerWave * F::kRowChunks * 16 + kWinPad
            : nt == 2     ? lds_bytes<false, 2, MASK>()
            : hl          ? lds_bytes<true, 1, MASK>()
                          : lds_bytes<false, 1, MASK>();
}
}  // namespace

bool mfma_layout(const MfmaDesc &d, int B, MfmaLayout &l) {
    Plan p;
    l = {};
    if (!plan_group(1, &d, B, p)) return false;
    const bool hl = B <= kHlMaxBatch;
    const int nt = B > 64 ? p.chunk / 32 : B > 32 ? 2 : 1;
    l.kernel = p.prepared ? 2 : 1;
    l.ksplit = p.ksplit;
    l.ksb = p.ksb;
    l.columns = B > 64 ? p.chunk : hl ? 16 : 32 * nt;
    l.column_chunks = p.chunks;
    if (p.prepared) hl ? slab_layout<true>(l) : slab_layout<false>(l);
    else if (nt == 2) image_layout<false, 2>(l);
    else hl ? image_layout<true, 1>(l) : image_layout<false, 1>(l);
    switch (d.type) {
        case 12: format_layout<FmtQ4K, 1>(l, hl, nt); break;
        case 13: format_layout<FmtQ5K, 2>(l, hl, nt); break;
        case 14: format_layout<FmtQ6K, 4>(l, hl, nt); break;
        case 10: format_layout<FmtQ2K, 16>(l, hl, nt); break;
        case 11: format_layout<FmtQ3K, 32>(l, hl, nt); break;
        default: format_layout<FmtQ8_0, 8>(l, hl, nt); break;
    }
    return true;
}

// chunks of 64 columns: no Q6_K or Q3_K (plan_group)
static void launch_wide64(const MfmaGroup &g, int mask, int grid, hipStream_t s) {
    switch (mask) {
        case 1: mfma_group<false, 2, 1, false, true><<<grid, kThreads, 0, s>>>(g); break;
        case 2: mfma_group<false, 2, 2, false, true><<<grid, kThreads, 0, s>>>(g); break;
        case 8: mfma_group<false, 2, 8, false, true><<<grid, kThreads, 0, s>>>(g); break;
        case 16: mfma_group<false, 2, 16, false, true><<<grid, kThreads, 0, s>>>(g); break;
        default: mfma_group<false, 2, 27, false, true><<<grid, kThreads, 0, s>>>(g); break;
    }
}

static void launch_wide32(const MfmaGroup &g, int mask, int grid, hipStream_t s) {
    switch (mask) {
        case 1: mfma_group<false, 1, 1, false, true><<<grid, kThreads, 0, s>>>(g); break;
        case 2: mfma_group<false, 1, 2, false, true><<<grid, kThreads, 0, s>>>(g); break;
        case 4: mfma_group<false, 1, 4, false, true><<<grid, kThreads, 0, s>>>(g); break;
        case 8: mfma_group<false, 1, 8, false, true><<<grid, kThreads, 0, s>>>(g); break;
        case 16: mfma_group<false, 1, 16, false, true><<<grid, kThreads, 0, s>>>(g); break;
        case 32: mfma_group<false, 1, 32, false, true><<<grid, kThreads, 0, s>>>(g); break;
        default: mfma_group<false, 1, 63, false, true><<<grid, kThreads, 0, s>>>(g); break;
    }
}

template <bool HL, int NT>
static void launch_group_nt(const MfmaGroup &g, int mask, int grid, hipStream_t s) {
    switch (mask) {
        case 1: mfma_group<HL, NT, 1><<<grid, kThreads, 0, s>>>(g); break;
        case 2: mfma_group<HL, NT, 2><<<grid, kThreads, 0, s>>>(g); break;
        case 4: mfma_group<HL, NT, 4><<<grid, kThreads, 0, s>>>(g); break;
        case 8: mfma_group<HL, NT, 8><<<grid, kThreads, 0, s>>>(g); break;
        case 16: mfma_group<HL, NT, 16><<<grid, kThreads, 0, s>>>(g); break;
        case 32: mfma_group<HL, NT, 32><<<grid, kThreads, 0, s>>>(g); break;
        default: mfma_group<HL, NT, 63><<<grid, kThreads, 0, s>>>(g); break;
    }
}

static void launch_two(const MfmaGroup &g, int mask, int grid, hipStream_t s) {
    switch (mask) {
        case 1: mfma_group<true, 1, 1, false, false, true><<<grid, kThreads, 0, s>>>(g); break;
        case 2: mfma_group<true, 1, 2, false, false, true><<<grid, kThreads, 0, s>>>(g); break;
        case 8: mfma_group<true, 1, 8, false, false, true><<<grid, kThreads, 0, s>>>(g); break;
        default: mfma_group<true, 1, 11, false, false, true><<<grid, kThreads, 0, s>>>(g); break;
    }
}

// JUNO_MFMA_PAIR=0: the batched SwiGLU takes the grouped launch and silu_mul (A/B runs)
static bool mfma_pair_wanted() {
    static const bool on = [] {
        const char *v = getenv("JUNO_MFMA_PAIR");
        return !(v && v[0] == '0');
    }();
    return on;
}

bool mfma_swiglu_applies(const MfmaDesc &gate, const MfmaDesc &up, int B) {
    if (!mfma_pair_wanted()) return false;
    if (B < 2 || B > 32 || gate.type != up.type || gate.cols != up.cols || gate.pitch != up.pitch ||
        gate.x != up.x || gate.row_start != 0 || up.row_start != 0 || gate.row_end != up.row_end)
        return false;
    if (gate.type != 12 && gate.type != 13 && gate.type != 14 && gate.type != 8) return false;
    if (((reinterpret_cast<uintptr_t>(up.w) | up.pitch) & 15) && (up.type == 12 || up.type == 13)) return false;
    MfmaDesc v = gate;
    v.row_end = 2 * gate.row_end;  // the pair's virtual rows
    Plan p;
    return plan_group(1, &v, B, p, true) && (p.ksplit == 1 || (gate.row_end + kRowsPerWG / 2 - 1) / (kRowsPerWG / 2) <= kMaxTileCounters);
}

size_t mfma_swiglu_workspace_bytes(const MfmaDesc &gate, int B) {
    MfmaDesc v = gate;
    v.row_end = 2 * gate.row_end;
    Plan p;
    if (!plan_group(1, &v, B, p, true)) return 0;
    return p.ksplit > 1 ? sizeof(float) * (size_t)p.ksplit * B * v.row_end : 16;
}

hipError_t launch_mfma_swiglu(const MfmaDesc &gate, const MfmaDesc &up, int B, float *out, void *workspace,
                              int *counters, hipStream_t s) {
    if (!mfma_swiglu_applies(gate, up, B)) return hipErrorNotSupported;
    MfmaDesc v = gate;
    v.row_end = 2 * gate.row_end;
    Plan p;
    plan_group(1, &v, B, p, true);
    if (p.ksplit > 1 && !counters) return hipErrorNotSupported;
    MfmaGroup g = {};
    g.part = reinterpret_cast<float *>(workspace);
    g.counters = counters;
    g.n = 1;
    g.nsb = p.nsb;
    g.ksb = p.ksb;
    g.ksplit = p.ksplit;
    g.B = B;
    g.w2 = up.w;
    g.swiglu = out;
    MfmaProblem &q = g.p[0];
    q.w = gate.w;
    q.x = gate.x;
    q.y = nullptr;
    q.pitch = gate.pitch;
    q.type = gate.type;
    q.row0 = 0;
    q.rows = gate.row_end;
    q.tiles = (q.rows + kRowsPerWG / 2 - 1) / (kRowsPerWG / 2);
    q.wg0 = q.cnt0 = 0;
    q.part0 = 0;
    const int grid = q.tiles * p.ksplit;
    auto run = [&](auto *k) { k<<<grid, kThreads, 0, s>>>(g); };
#define JH_PAIR(M)                                                                                    \
    (B == 2 ? run(mfma_group<true, 1, M, true, false, true>)                                          \
            : B <= kHlMaxBatch ? run(mfma_group<true, 1, M, true>) : run(mfma_group<false, 1, M, true>))
    switch (gate.type) {
        case 12: JH_PAIR(1); break;
        case 13: JH_PAIR(2); break;
        case 14: B <= kHlMaxBatch ? run(mfma_group<true, 1, 4, true>) : run(mfma_group<false, 1, 4, true>); break;  // not two
        default: JH_PAIR(8); break;
    }
#undef JH_PAIR
    return hipGetLastError();
}

// ------------------------------------------------------------------ static scratch
// Split-K counters (kCounterSlots lines of kCounterStride ints), then
// kStaticScratchBytes of workspace.  In host code `scratch` names a host-side
// stand-in, not device memory: kernels get the per-device address that
// hipGetSymbolAddress returns.  Every call on a device shares that device's
// copy, so calls that overlap on one device race.
constexpr size_t kStaticCounterBytes = sizeof(int) * (size_t)kCounterSlots * kCounterStride;
static __device__ __align__(256) uint8_t scratch[kStaticCounterBytes + kStaticScratchBytes];

namespace {
__global__ void zero_words(uint32_t *p, int n) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) p[i] = 0u;
}
}  // namespace

hipError_t static_scratch(int device, hipStream_t s, void **workspace, int **counters) {
    static std::mutex mu;
    static uint8_t *ptr[64];
    static bool zeroed[64];
    if (device < 0 || device >= 64) return hipErrorInvalidDevice;
    std::lock_guard<std::mutex> lk(mu);
    if (!ptr[device]) {
        void *p = nullptr;
        const hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));  // the current device's copy
        if (e != hipSuccess) return e;
        ptr[device] = static_cast<uint8_t *>(p);
    }
    if (!zeroed[device]) {
        // a kernel, not a memset: the first call may be under graph capture
        const int n = (int)(kStaticCounterBytes / 4);
        zero_words<<<(n + 255) / 256, 256, 0, s>>>(reinterpret_cast<uint32_t *>(ptr[device]), n);
        const hipError_t e = hipGetLastError();
        if (e != hipSuccess) return e;
        zeroed[device] = true;
    }
    *counters = reinterpret_cast<int *>(ptr[device]);
    *workspace = ptr[device] + kStaticCounterBytes;
    return hipSuccess;
}

hipError_t launch_mfma_group(int n, const MfmaDesc *d, int B, void *workspace, int *counters, hipStream_t s) {
    Plan p;
    if (!plan_group(n, d, B, p)) return hipErrorNotSupported;
    if (!workspace && B <= 64) return hipErrorNotSupported;
    if (!workspace) {  // K whole
        const int tiles = p.grid / (p.ksplit * p.chunks);
        p.ksplit = 1;
        p.ksb = p.nsb;
        for (int i = 0; i < n; i++)
            if (d[i].type == 8 && p.nsb > kLongWalk) p.chunk = 32;
        p.chunks = (B + p.chunk - 1) / p.chunk;
        p.grid = tiles * p.chunks;
    }
    if (p.ksplit > 1 && !counters) return hipErrorNotSupported;
    uint8_t *ws = reinterpret_cast<uint8_t *>(workspace);
    if (p.prepared) {
        const MfmaDesc &m = d[0];
        const int nrows = m.row_end - m.row_start;
        const bool hl = B <= kHlMaxBatch;
        if (B == 2) x_prep<true, true><<<p.nsb, 256, 0, s>>>(m.x, B, m.cols, ws);
        else if (hl) x_prep<true, false><<<p.nsb, 256, 0, s>>>(m.x, B, m.cols, ws);
        else x_prep<false, false><<<p.nsb, 512, 0, s>>>(m.x, B, m.cols, ws);
        auto px = [&](auto *k) { k<<<p.grid, kThreads, 0, s>>>(m.w, m.pitch, m.row_start, nrows, p.nsb, ws, m.x, m.y, B); };
#define JH_PX(F) (B == 2 ? px(mfma_px<F, true, true>) : hl ? px(mfma_px<F, true, false>) : px(mfma_px<F, false, false>))
        if (m.type == 12) JH_PX(FmtQ4K);
        else if (m.type == 13) JH_PX(FmtQ5K);
        else if (m.type == 8) JH_PX(FmtQ8_0);
        else if (hl) px(mfma_px<FmtQ6K, true, false>);  // not with two vectors
        else px(mfma_px<FmtQ6K, false, false>);
#undef JH_PX
        return hipGetLastError();
    }
    MfmaGroup g = {};
    g.part = reinterpret_cast<float *>(ws);
    g.counters = counters;
    g.n = n;
    g.nsb = p.nsb;
    g.ksb = p.ksb;
    g.ksplit = p.ksplit;
    g.B = B;
    int mask = 0, wg = 0, cnt = 0;
    size_t part = 0;
    for (int i = 0; i < n; i++) {
        MfmaProblem &q = g.p[i];
        q.w = d[i].w;
        q.x = d[i].x;
        q.y = d[i].y;
        q.pitch = d[i].pitch;
        q.type = d[i].type;
        q.row0 = d[i].row_start;
        q.rows = d[i].row_end - d[i].row_start;
        q.tiles = (q.rows + kRowsPerWG - 1) / kRowsPerWG;
        q.wg0 = wg;
        q.cnt0 = cnt;
        q.part0 = part;
        wg += q.tiles * p.chunks * p.ksplit;
        cnt += q.tiles * p.chunks;
        part += p.ksplit > 1 ? (size_t)p.ksplit * B * q.rows : 0;
        mask |= q.type == 12 ? 1 : q.type == 13 ? 2 : q.type == 14 ? 4 : q.type == 10 ? 16 : q.type == 11 ? 32 : 8;
    }
    g.chunks = p.chunks;
    if (B > 64 && p.chunk == 64) launch_wide64(g, mask, p.grid, s);
    else if (B > 64) launch_wide32(g, mask, p.grid, s);
    else if (B == 2) launch_two(g, mask, p.grid, s);
    else if (B <= kHlMaxBatch) launch_group_nt<true, 1>(g, mask, p.grid, s);
    else if (B <= 32) launch_group_nt<false, 1>(g, mask, p.grid, s);
    else launch_group_nt<false, 2>(g, mask, p.grid, s);
    return hipGetLastError();
}

hipError_t mfma_timeline_read(unsigned long long *out, size_t n) {
#ifdef JH_TIMELINE
    if (n > (size_t)kMtWg * 8 * kMtPer) n = (size_t)kMtWg * 8 * kMtPer;
    return hipMemcpyFromSymbol(out, HIP_SYMBOL(g_mtimeline), n * sizeof(unsigned long long));
#else
    (void)out;
    (void)n;
    return hipErrorNotSupported;
#endif
}

}  // namespace jh
