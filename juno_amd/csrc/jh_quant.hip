// jh_quant.hip -- dequantization (bit-exact) and quantization kernels.
//
// Dequantization restates LlamaTransformerHandler.dequantize
// (LlamaTransformerHandler.java:873-1135), four elements per lane.
//
// Quantization restates LoraMerge.requantize (LoraMerge.java:226-469) so that
// benchmark and test inputs are the reference quantizer's bytes, produced on
// the device.  A wave per 256 elements; the reference's rounding (Math.round, fp32
// divisions) is reproduced exactly.
#include "jh_dequant.hpp"
#include "jh_device.hpp"
#include "jh_kernels.hpp"

namespace jh {

namespace {

// Words and float quadruples at any alignment: single loads and stores on gfx950.
typedef uint32_t word __attribute__((aligned(1)));
typedef float quadf __attribute__((ext_vector_type(4), aligned(4)));

__device__ __forceinline__ uint32_t load_word(const uint8_t *p) { return *reinterpret_cast<const word *>(p); }
__device__ __forceinline__ void store_word(uint8_t *p, uint32_t v) { *reinterpret_cast<word *>(p) = v; }

// ---------------------------------------------------------------- dequant
// Bound by the writing of the floats (a 4096 x 4096 Q4_K matrix: 9 MB read, 67 MB
// written), so a lane makes four consecutive elements out of one word of quants
// and stores 16 bytes next to its neighbours' 16.  With a lane per sub-block
// (32 elements, 128 bytes apart from the next lane's) every store of a wave
// touched 64 cache lines: 4096 x 4096 Q4_K 25.1 us, now
// 15.3 (5.0 TB/s).
// The arithmetic is deq_unit's (jh_dequant.hpp), element by element.
template <int T>
__device__ __forceinline__ quadf deq_quad(const uint8_t *__restrict__ W, int64_t t) {  // elements 4 t .. 4 t + 3
    quadf v;
    if constexpr (T == 12 || T == 13) {
        const uint8_t *bp = W + (t >> 6) * (T == 12 ? 144 : 176);
        const int j = (int)(t >> 3) & 7, i0 = 4 * ((int)t & 7);
        const uint32_t dm = load_word(bp);
        int ls, lm;
        q4k_scale_min(load_word(bp + 4), load_word(bp + 8), load_word(bp + 12), j, ls, lm);
        const float scale = __fmul_rn(half_bits_to_float(dm & 0xFFFF), (float)ls), mn = __fmul_rn(half_bits_to_float(dm >> 16), (float)lm);
        uint32_t q = (load_word(bp + (T == 12 ? 16 : 48) + 32 * (j >> 1) + i0) >> (4 * (j & 1))) & 0x0F0F0F0Fu;
        if (T == 13) q |= ((load_word(bp + 16 + i0) >> j) & 0x01010101u) << 4;
#pragma unroll
        for (int i = 0; i < 4; i++) v[i] = __fsub_rn(__fmul_rn(scale, (float)byte_of(q, i)), mn);
    } else if constexpr (T == 14) {
        const uint8_t *bp = W + (t >> 6) * 210;
        const int l = (int)t & 63, half = l >> 5, k = (l >> 3) & 3, i0 = 4 * (l & 7);
        const float d = half_bits_to_float(bp[208] | (bp[209] << 8));
        const float dk = __fmul_rn(d, (float)(int8_t)bp[192 + (l >> 2)]);
        const uint32_t q = ((load_word(bp + 64 * half + 32 * (k & 1) + i0) >> (4 * (k >> 1))) & 0x0F0F0F0Fu) |
                           (((load_word(bp + 128 + 32 * half + i0) >> (2 * k)) & 0x03030303u) << 4);
#pragma unroll
        for (int i = 0; i < 4; i++) v[i] = __fmul_rn(dk, (float)((int)byte_of(q, i) - 32));
    } else if constexpr (T == 8) {
        const uint8_t *bp = W + (t >> 3) * 34;
        const float d = half_bits_to_float(bp[0] | (bp[1] << 8));
        const uint32_t q = load_word(bp + 2 + 4 * ((int)t & 7));
#pragma unroll
        for (int i = 0; i < 4; i++) v[i] = __fmul_rn(d, (float)(int8_t)byte_of(q, i));
    } else if constexpr (T == 10) {
        const uint8_t *bp = W + (t >> 6) * 84;
        const int l = (int)t & 63, h = l >> 5, k = (l >> 2) & 7;
        const uint32_t dm = load_word(bp + 80), sc = bp[8 * h + k];
        const float dl = __fmul_rn(half_bits_to_float(dm & 0xFFFF), (float)(sc & 15)), ml = __fmul_rn(half_bits_to_float(dm >> 16), (float)(sc >> 4));
        const uint32_t q = (load_word(bp + 16 + 32 * h + 16 * (k & 1) + 4 * (l & 3)) >> (2 * (k >> 1))) & 0x03030303u;
#pragma unroll
        for (int i = 0; i < 4; i++) v[i] = __fsub_rn(__fmul_rn(dl, (float)byte_of(q, i)), ml);
    } else {
        const uint8_t *bp = W + (t >> 6) * 110;
        const int l = (int)t & 63, is = l >> 2, h = is >> 3, j = (is >> 1) & 3, r = is & 1;
        const float d = half_bits_to_float(bp[108] | (bp[109] << 8));
        const int lo4 = (bp[96 + (is & 7)] >> (is >= 8 ? 4 : 0)) & 15, hi2 = (bp[104 + (is & 3)] >> (2 * (is >> 2))) & 3;
        const float dl = __fmul_rn(d, (float)((lo4 | (hi2 << 4)) - 32));
        const uint32_t q = ((load_word(bp + 32 + 32 * h + 16 * r + 4 * (l & 3)) >> (2 * j)) & 0x03030303u) |
                           (((load_word(bp + 16 * r + 4 * (l & 3)) >> (4 * h + j)) & 0x01010101u) << 2);
#pragma unroll
        for (int i = 0; i < 4; i++) v[i] = __fmul_rn(dl, (float)((int)byte_of(q, i) - 4));
    }
    return v;
}

// unit t of `out`: four elements, F32 one
template <int T> __device__ __forceinline__ void dequant_unit(const uint8_t *W, int64_t t, float *out) {
    if constexpr (T == 0) out[t] = reinterpret_cast<const float *>(W)[t];
    else reinterpret_cast<quadf *>(out)[t] = deq_quad<T>(W, t);
}

template <int T> __global__ void dequant_k(const uint8_t *__restrict__ W, int64_t block0, int64_t units, float *__restrict__ out) {
    const int64_t t = (block0 + blockIdx.x) * blockDim.x + threadIdx.x;
    if (t < units) dequant_unit<T>(W, t, out);
}

// Embedding lookup (getInitialActivation, LlamaTransformerHandler.java:651-660):
// for output row y = blockIdx.y, row clamp(d_tokens[y], 0, rows - 1) of the
// packed matrix, dequantized into out[y].  Tokens are read on the device so
// that a captured step can be replayed.
template <int T>
__global__ void dequant_row_k(const uint8_t *__restrict__ W, const int *__restrict__ d_tokens, int rows, size_t pitch,
                              int64_t units, int64_t row_elems, float *__restrict__ out) {
    const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= units) return;
    const int tok = min(max(d_tokens[blockIdx.y], 0), rows - 1);
    dequant_unit<T>(W + (size_t)tok * pitch, t, out + (int64_t)blockIdx.y * row_elems);
}

// launch(first block, blocks) over `blocks` of 256 threads, 2^31 threads at a time: one
// launch of 2^32 threads or more (from 2^34 elements on, at four a lane) leaves part of
// the array unwritten, without an error
template <class F>
hipError_t in_launches(int64_t blocks, F launch) {
    constexpr int64_t kMax = int64_t(1) << 23;
    for (int64_t b = 0; b < blocks; b += kMax) {
        launch(b, (unsigned)(blocks - b < kMax ? blocks - b : kMax));
        const hipError_t e = hipGetLastError();
        if (e != hipSuccess) return e;
    }
    return hipSuccess;
}

}  // namespace

int64_t dequant_units(int type, int64_t n) {
    switch (type) {
    case 12:
    case 13:
    case 8:
    case 14:
    case 10:
    case 11: return n / 4;
    case 0: return n;
    default: return -1;
    }
}

hipError_t launch_dequant(int type, const uint8_t *w, int rows, int cols, float *out, hipStream_t s) {
    const int64_t units = dequant_units(type, (int64_t)rows * cols);
    if (units < 0) return hipErrorInvalidValue;
    if (units == 0) return hipSuccess;
    return in_launches((units + 255) / 256, [&](int64_t b0, unsigned grid) {
        switch (type) {
        case 12: dequant_k<12><<<grid, 256, 0, s>>>(w, b0, units, out); break;
        case 13: dequant_k<13><<<grid, 256, 0, s>>>(w, b0, units, out); break;
        case 14: dequant_k<14><<<grid, 256, 0, s>>>(w, b0, units, out); break;
        case 8: dequant_k<8><<<grid, 256, 0, s>>>(w, b0, units, out); break;
        case 10: dequant_k<10><<<grid, 256, 0, s>>>(w, b0, units, out); break;
        case 11: dequant_k<11><<<grid, 256, 0, s>>>(w, b0, units, out); break;
        case 0: dequant_k<0><<<grid, 256, 0, s>>>(w, b0, units, out); break;
        }
    });
}

hipError_t launch_dequant_row(int type, const uint8_t *w, int rows, int cols, size_t pitch, const int *d_tokens,
                              int n_out, float *out, hipStream_t s) {
    const int64_t units = dequant_units(type, cols);
    if (units < 0 || rows <= 0 || n_out < 1 || n_out > 65535) return hipErrorInvalidValue;
    dim3 block(64), grid((unsigned)((units + 63) / 64), (unsigned)n_out);
    switch (type) {
    case 12: dequant_row_k<12><<<grid, block, 0, s>>>(w, d_tokens, rows, pitch, units, cols, out); break;
    case 13: dequant_row_k<13><<<grid, block, 0, s>>>(w, d_tokens, rows, pitch, units, cols, out); break;
    case 14: dequant_row_k<14><<<grid, block, 0, s>>>(w, d_tokens, rows, pitch, units, cols, out); break;
    case 8: dequant_row_k<8><<<grid, block, 0, s>>>(w, d_tokens, rows, pitch, units, cols, out); break;
    case 10: dequant_row_k<10><<<grid, block, 0, s>>>(w, d_tokens, rows, pitch, units, cols, out); break;
    case 11: dequant_row_k<11><<<grid, block, 0, s>>>(w, d_tokens, rows, pitch, units, cols, out); break;
    case 0: dequant_row_k<0><<<grid, block, 0, s>>>(w, d_tokens, rows, pitch, units, cols, out); break;
    }
    return hipGetLastError();
}

// ---------------------------------------------------------------- quantize

// clamp(java.lang.Math.round(a), lo, hi) for lo <= 0 <= hi: floor(a + 1/2) without
// the sum's rounding (a - floor(a) is exact where it decides: from 1 on by
// Sterbenz, and a in (-1/2, 0) cannot round below 1/2), NaN -> 0.
__device__ __forceinline__ int round_clamp(float a, float lo, float hi) {
    asm("" : "+v"(a));  // a's own rounding stays: the compiler would contract its product into the difference
    const float f = floorf(a);
    const float r = __fsub_rn(a, f) >= 0.5f ? __fadd_rn(f, 1.f) : f;
    return a != a ? 0 : (int)fminf(fmaxf(r, lo), hi);
}

// LoraMerge.f32ToF16 (LoraMerge.java:589-605): round-to-nearest-even on the
// normal range; NaN becomes infinity; the subnormal branch rounds after a
// truncating shift.  Reproduced as-is so the stored d / dmin bytes match.
__device__ uint32_t f32_to_f16_ref(float value) {
    const int32_t bits = __builtin_bit_cast(int32_t, value);
    const int32_t sign = (int32_t)(((uint32_t)bits >> 31) & 1u);
    int32_t exp = (int32_t)(((uint32_t)bits >> 23) & 0xFFu) - 112;
    int32_t mant = bits & 0x7FFFFF;
    if (exp <= 0) {
        if (exp < -10) return (uint32_t)(sign << 15);
        mant = (mant | 0x800000) >> (1 - exp);
        mant = (mant + 0x0FFF + ((mant >> 13) & 1)) >> 13;
        return (uint32_t)((sign << 15) | mant);
    }
    if (exp >= 31) return (uint32_t)((sign << 15) | 0x7C00);
    const int32_t low = mant & 0x1FFF;
    mant >>= 13;
    if (low > 0x1000 || (low == 0x1000 && (mant & 1))) {
        mant++;
        if (mant == 0x400) {
            mant = 0;
            exp++;
        }
    }
    if (exp >= 31) return (uint32_t)((sign << 15) | 0x7C00);
    return (uint32_t)((sign << 15) | (exp << 10) | mant);
}

namespace {

// A wave quantizes 256 consecutive floats: lane l holds elements 4 l .. 4 l + 3, so
// the source is read 16 bytes a lane side by side and packed bytes are written as
// words.  (One thread per block, as before, put the lanes' reads 1 KB apart and
// its byte stores 144 or more: 4096 x 4096 Q4_K 166 us, now 34,
// Q6_K 437 and 26, Q8_0 261 and 16; what is left at Q4_K is the exact divisions.)  Every
// reduction is a maximum or minimum, so its order does not matter, and the
// arithmetic per element is the reference's.
template <int CTRL>
__device__ __forceinline__ int dpp(int v) {
    return __builtin_amdgcn_update_dpp(0, v, CTRL, 0xF, 0xF, true);
}
constexpr int kXor1 = 0xB1, kXor2 = 0x4E, kHalfMirror = 0x141, kXor8 = 0x128;  // (row_ror:8)
template <int CTRL>
__device__ __forceinline__ float dppf(float v) {
    return __builtin_bit_cast(float, dpp<CTRL>(__builtin_bit_cast(int, v)));
}
__device__ __forceinline__ float larger(float a, float b) { return b > a ? b : a; }
__device__ __forceinline__ float smaller(float a, float b) { return b < a ? b : a; }
__device__ __forceinline__ float max4(float v) {  // over 4 lanes
    v = larger(v, dppf<kXor1>(v));
    return larger(v, dppf<kXor2>(v));
}
__device__ __forceinline__ float max8(float v) {  // over 8 lanes
    v = max4(v);
    return larger(v, dppf<kHalfMirror>(v));
}
__device__ __forceinline__ float min8(float v) {
    v = smaller(v, dppf<kXor1>(v));
    v = smaller(v, dppf<kXor2>(v));
    return smaller(v, dppf<kHalfMirror>(v));
}
__device__ __forceinline__ float max64(float v) {  // over the wave
    v = max8(v);
    v = larger(v, dppf<kXor8>(v));
    v = larger(v, __shfl_xor(v, 16));
    return larger(v, __shfl_xor(v, 32));
}
__device__ __forceinline__ uint32_t pack4(int a, int b, int c, int d) {
    return (uint32_t)(a & 0xFF) | ((uint32_t)(b & 0xFF) << 8) | ((uint32_t)(c & 0xFF) << 16) | ((uint32_t)d << 24);
}

// quantizeQ8_0 (LoraMerge.java:265-277): 8 lanes per block
__global__ __launch_bounds__(256) void quant_q8_0(const float *__restrict__ src, int64_t block0, int64_t quads,
                                                  uint8_t *__restrict__ dst) {
    const int64_t t = (block0 + blockIdx.x) * blockDim.x + threadIdx.x;
    if (t >= quads) return;  // whole groups of 8 lanes
    const quadf v = reinterpret_cast<const quadf *>(src)[t];
    uint8_t *o = dst + (t >> 3) * 34;
    float m = 0.f;
#pragma unroll
    for (int i = 0; i < 4; i++) m = fmaxf(m, fabsf(v[i]));
    const float absMax = max8(m);
    const float d = __fdiv_rn(absMax, 127.f);
    const float invD = d > 0.f ? __fdiv_rn(1.f, d) : 0.f;
    int q[4];
#pragma unroll
    for (int i = 0; i < 4; i++) q[i] = round_clamp(__fmul_rn(v[i], invD), -127.f, 127.f);
    store_word(o + 2 + 4 * ((int)t & 7), pack4(q[0], q[1], q[2], q[3]));
    if ((t & 7) == 0) {
        const uint32_t h = f32_to_f16_ref(d);
        o[0] = (uint8_t)h;
        o[1] = (uint8_t)(h >> 8);
    }
}

// quantizeQ4_K (LoraMerge.java:311-366) and quantizeQ5_K (:376-430): the same
// scale / min search with q in [0, 15] (d = maxRange / 945) or [0, 31]
// (d = maxRange / 1953, 5th bits in qh); the quants use the fp32 d / dmin.
// Sub-block s is lanes 8 s .. 8 s + 7.
template <bool Q5>
__global__ __launch_bounds__(256) void quant_kq(const float *__restrict__ src, int64_t block0, int64_t nblk,
                                                  uint8_t *__restrict__ dst) {
    constexpr int kBytes = Q5 ? 176 : 144, kQs = Q5 ? 48 : 16;
    constexpr float kQmax = Q5 ? 31.f : 15.f, kRange = Q5 ? 1953.f : 945.f;
    const int64_t t = (block0 + blockIdx.x) * 4 + (threadIdx.x >> 6);
    if (t >= nblk) return;  // whole waves
    const int lane = threadIdx.x & 63, s = lane >> 3, i0 = 4 * (lane & 7);
    const quadf v = reinterpret_cast<const quadf *>(src + t * 256)[lane];
    uint8_t *o = dst + t * kBytes;
    float mn = 3.40282347e+38f, mx = -3.40282347e+38f;
#pragma unroll
    for (int i = 0; i < 4; i++) {
        mn = smaller(mn, v[i]);
        mx = larger(mx, v[i]);
    }
    mn = min8(mn);
    mx = max8(mx);
    if (mn > mx) {
        mn = 0.f;
        mx = 0.f;
    }
    const float range = __fsub_rn(mx, mn);
    const float maxRange = max64(larger(0.f, range)), maxAbsMin = max64(larger(0.f, -mn));
    const float d = maxRange > 0.f ? __fdiv_rn(maxRange, kRange) : 0.f;
    const float dmin = maxAbsMin > 0.f ? __fdiv_rn(maxAbsMin, 63.f) : 0.f;
    const int ls = maxRange > 0.f ? round_clamp(__fdiv_rn(__fmul_rn(range, 63.f), maxRange), 0.f, 63.f) : 0;
    const int lm = maxAbsMin > 0.f ? round_clamp(__fdiv_rn(__fmul_rn(-mn, 63.f), maxAbsMin), 0.f, 63.f) : 0;
    uint32_t b1 = 0, b2 = 0, b3 = 0;
#pragma unroll
    for (int j = 0; j < 4; j++) {
        const uint32_t sl = __builtin_amdgcn_readlane(ls, 8 * j), sh = __builtin_amdgcn_readlane(ls, 8 * j + 32);
        const uint32_t ml = __builtin_amdgcn_readlane(lm, 8 * j), mh = __builtin_amdgcn_readlane(lm, 8 * j + 32);
        b1 |= (sl | ((sh & 0x30) << 2)) << (8 * j);
        b2 |= (ml | ((mh & 0x30) << 2)) << (8 * j);
        b3 |= ((sh & 0x0F) | ((mh & 0x0F) << 4)) << (8 * j);
    }
    if (lane < 4) {
        const uint32_t b0 = f32_to_f16_ref(d) | (f32_to_f16_ref(dmin) << 16);
        store_word(o + 4 * lane, lane == 0 ? b0 : lane == 1 ? b1 : lane == 2 ? b2 : b3);
    }
    const float sc = __fmul_rn(d, (float)ls), m = __fmul_rn(dmin, (float)lm);
    int q[4];
#pragma unroll
    for (int i = 0; i < 4; i++) q[i] = sc > 0.f ? round_clamp(__fdiv_rn(__fadd_rn(v[i], m), sc), 0.f, kQmax) : 0;
    const uint32_t w = pack4(q[0], q[1], q[2], q[3]);
    const uint32_t odd = (uint32_t)dpp<kXor8>((int)w);  // even sub-blocks: the odd one's quants of the same bytes
    if ((s & 1) == 0) store_word(o + kQs + 16 * s + i0, (w & 0x0F0F0F0Fu) | ((odd & 0x0F0F0F0Fu) << 4));
    if (Q5) {
        uint32_t h = ((w >> 4) & 0x01010101u) << s;
        h |= (uint32_t)dpp<kXor8>((int)h);
        h |= (uint32_t)__shfl_xor((int)h, 16);
        h |= (uint32_t)__shfl_xor((int)h, 32);
        if (s == 0) store_word(o + 16 + i0, h);
    }
}

// quantizeQ6_K (LoraMerge.java:437-469): sub-block s is lanes 4 s .. 4 s + 3; a
// lane's elements are quarter (lane >> 3) & 3 of half lane >> 5.
__global__ __launch_bounds__(256) void quant_q6k(const float *__restrict__ src, int64_t block0, int64_t nblk,
                                                   uint8_t *__restrict__ dst) {
    const int64_t t = (block0 + blockIdx.x) * 4 + (threadIdx.x >> 6);
    if (t >= nblk) return;  // whole waves
    const int lane = threadIdx.x & 63, half = lane >> 5, quarter = (lane >> 3) & 3, i0 = 4 * (lane & 7);
    const quadf v = reinterpret_cast<const quadf *>(src + t * 256)[lane];
    uint8_t *o = dst + t * 210;
    float m = 0.f;
#pragma unroll
    for (int i = 0; i < 4; i++) m = fmaxf(m, fabsf(v[i]));
    const float subMax = max4(m), globalMax = max64(subMax);
    const float d = globalMax > 0.f ? __fdiv_rn(globalMax, 4064.f) : 0.f;
    const float invD = d > 0.f ? __fdiv_rn(1.f, d) : 0.f;
    const int sc = d > 0.f ? round_clamp(__fdiv_rn(__fmul_rn(subMax, invD), 32.f), -127.f, 127.f) : 0;
    const float eff = __fmul_rn(d, (float)sc);
    int u[4];
#pragma unroll
    for (int i = 0; i < 4; i++) u[i] = (eff != 0.f ? round_clamp(__fdiv_rn(v[i], eff), -32.f, 31.f) : 0) + 32;
    const uint32_t w = pack4(u[0], u[1], u[2], u[3]);
    const uint32_t up = (uint32_t)__shfl_xor((int)w, 16);  // quarters 0, 1: quarters 2, 3
    if (quarter < 2) store_word(o + 64 * half + 32 * quarter + i0, (w & 0x0F0F0F0Fu) | ((up & 0x0F0F0F0Fu) << 4));
    uint32_t h = ((w >> 4) & 0x03030303u) << (2 * quarter);
    h |= (uint32_t)dpp<kXor8>((int)h);
    h |= (uint32_t)__shfl_xor((int)h, 16);
    if (quarter == 0) store_word(o + 128 + 32 * half + i0, h);
    if ((lane & 3) == 0) o[192 + (lane >> 2)] = (uint8_t)(int8_t)sc;
    if (lane < 2) o[208 + lane] = (uint8_t)(f32_to_f16_ref(d) >> (8 * lane));
}

}  // namespace

hipError_t launch_quantize(int type, const float *src, int64_t n, uint8_t *dst, hipStream_t s) {
    int64_t nblk;
    switch (type) {
    case 8: nblk = n / 32; break;
    case 12:
    case 13:
    case 14: nblk = n / 256; break;
    case 0: return hipMemcpyAsync(dst, src, (size_t)n * 4, hipMemcpyDeviceToDevice, s);
    default: return hipErrorInvalidValue;
    }
    if (nblk == 0) return hipSuccess;
    // a wave per 256 elements
    const int64_t waves = type == 8 ? (nblk + 7) / 8 : nblk;
    return in_launches((waves + 3) / 4, [&](int64_t b0, unsigned grid) {
        switch (type) {
        case 8: quant_q8_0<<<grid, 256, 0, s>>>(src, b0, nblk * 8, dst); break;
        case 12: quant_kq<false><<<grid, 256, 0, s>>>(src, b0, nblk, dst); break;
        case 13: quant_kq<true><<<grid, 256, 0, s>>>(src, b0, nblk, dst); break;
        case 14: quant_q6k<<<grid, 256, 0, s>>>(src, b0, nblk, dst); break;
        }
    });
}

}  // namespace jh
