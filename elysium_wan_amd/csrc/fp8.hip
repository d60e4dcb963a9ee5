// fp8.hip -- the fp8 boundary codec of model/fp8.py on gfx950.
//
// quantize (fp8.py:28-49): per row, k = frexp(amax|x|).exponent - ebias and
// q = fp8(x * 2^-k).  Three launch shapes:
//   * rows that fit registers (one vector up to 16 waves x 64 lanes x 4
//     vectors of 16 bytes: 8 to 32,768 bf16 / 4 to 16,384 fp32 columns, any
//     width and any element's alignment): the row is read once into VGPRs, |x|max is a
//     butterfly over the wave, and codes are written from the same
//     registers: one HBM read and one write per element (3 B/elem for bf16
//     -> fp8).  Rows of up to 6 vectors per lane take one wave; longer ones
//     are shared by a block's 4, 8 or 16 waves, whose maxima meet in LDS, so
//     that each wave holds at most 4 vectors and more rows stream at once.  A width
//     that is no whole number of vectors ends in a vector that overlaps the
//     one before it: [16376, 1601] bf16 quantizes in 17 us where element
//     loads with two reads of x took 65 (79 MB: 4.5 against 1.2 TB/s).
//     All of a row's loads are issued before the first is waited for (one
//     vector at a time took C1's round trip from 30.0 to 32.0 us).
//   * longer rows (per-tensor scaling is rows = 1): the row is cut into
//     2048-element segments.  A first launch reduces the row's |x|max into
//     at most 256 partial maxima (each wave strides over its row's segments;
//     integer max, so order-free), a second converts one segment per wave,
//     which folds the partials first.  Two reads of x, no atomics.
//   * rows shorter than a vector: the same launches with element-wise loads.
// Every row whose exponent keeps 2^-k, 2^k and every product exact
// (|k| <= 110, finite |x|max) converts with the instructions: bf16 words go
// straight into v_cvt_scalef32_pk_{fp8,bf8}_bf16 at scale 2^k (the code of
// x * 2^-k in one instruction per two elements), fp32 through a product and
// v_cvt_pk_fp8_f32 / v_cvt_pk_bf8_f32 (proved equal to torch's rounding on
// that domain by ely_selftest_fp8_scaled and ely_selftest_fp8_cvt); the
// other rows follow the bit-level restatement of torch's arithmetic (pow2
// rounded to the dtype, product rounded to the dtype, software conversion),
// uniformly per row.
//
// dequantize (fp8.py:52-53): out = float(q) * 2^k in the output dtype, the
// codes taken as one flat array (a wave's 1,024 codes may span rows), 8 codes
// per lane per step for bf16 output (4 for fp32) so every store instruction
// covers a contiguous 1 KB; bf16 output decodes with
// v_cvt_scalef32_pk_bf16_{fp8,bf8} at scale 2^k unless the vector holds a
// NaN code; a vector that holds the end of one row and the start of the next
// takes each code's own exponent ([16376, 1601] to bf16: 15 us, 41 code by
// code); roundtrip (fp8.py:56-63) fuses both.
#include <algorithm>
#include <map>
#include <mutex>

#include "ely_device.hpp"
#include "ely_host.hpp"

#pragma clang fp contract(off)

#ifndef ELY_DEQ_SEG
#define ELY_DEQ_SEG 1024  // dequantize: codes per wave segment
#endif
#ifndef ELY_DEQ_BATCH
#define ELY_DEQ_BATCH 0  // dequantize: vectors per lane per load batch (0: the whole segment at once)
#endif
#ifndef ELY_SPLIT_WAVES
#define ELY_SPLIT_WAVES 2048  // split path: waves of the partial-max launch (at most)
#endif
#ifndef ELY_SPLIT_CACHED_MB
// split path: MB of x the |x|max launch reads last with plain loads instead
// of nontemporal ones.  C4 per-tensor, when measured: quantize 0.408 -> 0.403 ms, round
// trip 0.509 -> 0.499 ms (0, 192, 256 and 384 MB; a convert launch
// taking the segments last to first, to start on the cached ones, was
// slower)
#define ELY_SPLIT_CACHED_MB 256
#endif
#ifndef ELY_Q_LDS
// wave-per-row quantize: unused dynamic LDS per block, capping it at 16
// blocks (16 waves) per CU.  C1 back to back over 8 inputs, in one process:
// quantize 5.89-5.92 TB/s and round trip 5.92-5.96 against 5.80-5.82 and
// 5.74-5.85 with no cap (256-thread blocks capped at 4 per CU: 5.86-5.88,
// 5.93-5.94)
#define ELY_Q_LDS 10240
#endif
#ifndef ELY_DEQ_LDS
#define ELY_DEQ_LDS 0  // dequantize: unused dynamic LDS per block capping its blocks per CU (caps measured slower)
#endif
#ifndef ELY_RECOVER_KEEP_VPL
#define ELY_RECOVER_KEEP_VPL 16  // longest rows (vectors per lane) whose image reuses the test's codes
#endif
#ifndef ELY_RECOVER_BATCH
#define ELY_RECOVER_BATCH 1  // recover register path: vectors per lane per load batch (0: all)
#endif
#ifndef ELY_RECOVER_WHOLE_VPL
#define ELY_RECOVER_WHOLE_VPL 8  // recover register path: rows of this many vectors per lane or more load at once
#endif

namespace ely {

#ifndef ELY_QBLOCK
// 64: in one process on the same buffers, dequantize 6.55-6.58 TB/s on C4
// and 5.86 on C1 against 6.29-6.46 and 5.68-5.71 on 256-thread blocks;
// the wave-per-row quantize the same (C1 6.0-6.1)
#define ELY_QBLOCK 64
#endif
constexpr int kQBlock = ELY_QBLOCK;            // threads per block; each wave takes its own row or segment
constexpr int kWavesPerBlock = kQBlock / kWave;
constexpr int kRowBlock = 256;                 // the row-max reduce: 4 waves share one row
constexpr int kRowWaves = kRowBlock / kWave;
constexpr int64_t kSegElems = 2048;            // split-path segment, elements
constexpr int64_t kDeqSegCodes = ELY_DEQ_SEG;  // dequantize segment, codes
constexpr int kRecoverKeepVpl = ELY_RECOVER_KEEP_VPL;
constexpr int kFastK = 110;                    // |k| bound of the instruction path

// ----------------------------------------------------------- element helpers

#ifndef ELY_FP8_NT
#define ELY_FP8_NT 3  // bit 0: nontemporal codec loads, bit 1: nontemporal stores
#endif

// Vector accesses carry no alignment beyond the element's: gfx950 loads and
// stores 8- and 16-byte vectors at any address with the same instructions
// (a probe of the quantize's and the dequantize's streams over 200 MB, at
// 2- and 1-byte offsets against aligned: 7.70-7.94 against 8.10 TB/s, 6.22-
// 6.53 against 6.86; nontemporal 5.40-5.83 against 6.75, 5.22-5.53 against
// 6.27), so rows of any width take the vector paths.
// Stores of streamed data; nontemporal when bit 1 of ELY_FP8_NT is set.
typedef uint32_t ev4u __attribute__((ext_vector_type(4), aligned(1)));
typedef uint32_t ev2u __attribute__((ext_vector_type(2), aligned(1)));
typedef uint32_t ev1u __attribute__((aligned(1)));
#define ELY_G1 __attribute__((address_space(1)))
__device__ __forceinline__ void st_vec(void* p, uint4 v) {
#if ELY_FP8_NT & 2
    __builtin_nontemporal_store(ev4u{v.x, v.y, v.z, v.w}, (ELY_G1 ev4u*)p);
#else
    *(ELY_G1 ev4u*)p = ev4u{v.x, v.y, v.z, v.w};
#endif
}
__device__ __forceinline__ void st_vec2(void* p, uint2 v) {
#if ELY_FP8_NT & 2
    __builtin_nontemporal_store(ev2u{v.x, v.y}, (ELY_G1 ev2u*)p);
#else
    *(ELY_G1 ev2u*)p = ev2u{v.x, v.y};
#endif
}
__device__ __forceinline__ void st_u32(void* p, uint32_t v) {
#if ELY_FP8_NT & 2
    __builtin_nontemporal_store(v, (ELY_G1 ev1u*)p);
#else
    *(ELY_G1 ev1u*)p = v;
#endif
}

// 8- and 4-byte loads of streamed data.
__device__ __forceinline__ uint2 ld_vec2(const void* p) {
#if ELY_FP8_NT & 1
    const ev2u v = __builtin_nontemporal_load((const ELY_G1 ev2u*)p);
    return make_uint2(v[0], v[1]);
#else
    const ev2u v = *(const ELY_G1 ev2u*)p;
    return make_uint2(v[0], v[1]);
#endif
}
__device__ __forceinline__ uint32_t ld_u32(const void* p) {
#if ELY_FP8_NT & 1
    return __builtin_nontemporal_load((const ELY_G1 ev1u*)p);
#else
    return *(const ELY_G1 ev1u*)p;
#endif
}

// One 16-byte load of streamed data.
template <bool NT = (ELY_FP8_NT & 1) != 0>
__device__ __forceinline__ uint4 ld_vec(const void* p) {
    ev4u v;
    if (NT) v = __builtin_nontemporal_load((const ELY_G1 ev4u*)p);
    else v = *(const ELY_G1 ev4u*)p;
    return make_uint4(v[0], v[1], v[2], v[3]);
}

template <bool BF16>
__device__ __forceinline__ float load_x(const void* x, int64_t i) {
    if (BF16) return bf16_to_f32(static_cast<const uint16_t*>(x)[i]);
    return static_cast<const float*>(x)[i];
}

__device__ __forceinline__ float round_to(float v, bool bf16) { return bf16 ? bf16_to_f32(f32_to_bf16(v)) : v; }

// Exact-arithmetic (slow-path) quantize of one element: fp8.py:49.
template <int FMT, bool BF16>
__device__ __forceinline__ uint32_t quant_sw(float xv, float s_down) {
    return fp8_from_f32_sw<FMT>(round_to(xv * s_down, BF16));
}

// Exact-arithmetic (slow-path) dequantize of one code: fp8.py:53.
template <int FMT, bool BF16OUT>
__device__ __forceinline__ float dequant_sw(uint32_t c, float s_up) {
    float v = round_to(fp8_to_f32_sw<FMT>(c), BF16OUT);
    return round_to(v * s_up, BF16OUT);
}

// A dequantized value from the instruction path as its output dtype's bits.
// In that path the value is exact in bf16, so truncation is the rounding.
__device__ __forceinline__ uint32_t fast_bf16_bits(float v) { return __float_as_uint(v) >> 16; }

struct RowScale {
    int k;
    bool fast;
    float s_down;   // 2^-k in the input dtype
    float s_up;     // 2^k in the output dtype
};

template <int FMT>
__device__ __forceinline__ RowScale row_scale(uint32_t abits, bool bf16_in, bool bf16_out) {
    RowScale r;
    r.k = scale_exp_from_amax<FMT>(abits);
    r.fast = abits < 0x7F800000u && r.k >= -kFastK && r.k <= kFastK;
    if (r.fast) {
        r.s_down = __uint_as_float((uint32_t)(127 - r.k) << 23);
        r.s_up = __uint_as_float((uint32_t)(127 + r.k) << 23);
    } else {
        r.s_down = pow2_dtype(-r.k, bf16_in);
        r.s_up = pow2_dtype(r.k, bf16_out);
    }
    return r;
}

// |x| bits of 8 bf16 packed in a uint4 / 4 fp32 in a uint4, maxed into m.
template <bool BF16>
__device__ __forceinline__ uint32_t vec_absmax(const uint4& w, uint32_t m) {
    const uint32_t ws[4] = {w.x, w.y, w.z, w.w};
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        if (BF16) {
            const uint32_t lo = ws[j] & 0x7FFFu, hi = (ws[j] >> 16) & 0x7FFFu;
            m = max(m, max(lo, hi));
        } else {
            m = max(m, ws[j] & 0x7FFFFFFFu);
        }
    }
    return m;
}

template <bool BF16>
__device__ __forceinline__ uint32_t to_f32_bits(uint32_t amax) {
    return BF16 ? amax << 16 : amax;
}

// Unpack a uint4 into 8 (bf16) or 4 (fp32) floats.
template <bool BF16>
__device__ __forceinline__ void unpack(const uint4& w, float* f) {
    const uint32_t ws[4] = {w.x, w.y, w.z, w.w};
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        if (BF16) {
            f[2 * j] = bf16_to_f32(ws[j] & 0xFFFFu);
            f[2 * j + 1] = bf16_to_f32(ws[j] >> 16);
        } else {
            f[j] = __uint_as_float(ws[j]);
        }
    }
}

// Quantize one 16-byte input vector (8 bf16 or 4 fp32) of an instruction-path
// row into codes packed in words[0..1] (bf16: 8 codes) or words[0] (fp32: 4
// codes); with `out`, also write the dequantized values in the input dtype at
// out_vec (exact there, so bf16 truncation is the rounding).
template <int FMT, bool BF16>
__device__ __forceinline__ void quant_vec_fast(const uint4& w, const RowScale& rs, uint32_t* words, void* out_vec) {
    if (BF16) {
        // bf16 words straight into the scaled conversions (scale 2^k), no
        // widening or product; no NaN code arises on this path, so the
        // scaled decode gives the output bits too
        words[0] = cvt_scaled_pk_fp8_bf16<FMT, true>(w.y, rs.s_up, cvt_scaled_pk_fp8_bf16<FMT, false>(w.x, rs.s_up, 0u));
        words[1] = cvt_scaled_pk_fp8_bf16<FMT, true>(w.w, rs.s_up, cvt_scaled_pk_fp8_bf16<FMT, false>(w.z, rs.s_up, 0u));
        if (out_vec)
            st_vec(out_vec, make_uint4(cvt_scaled_pk_bf16<FMT, false>(words[0], rs.s_up),
                                       cvt_scaled_pk_bf16<FMT, true>(words[0], rs.s_up),
                                       cvt_scaled_pk_bf16<FMT, false>(words[1], rs.s_up),
                                       cvt_scaled_pk_bf16<FMT, true>(words[1], rs.s_up)));
        return;
    }
    constexpr int EPV = BF16 ? 8 : 4;
    float f[EPV];
    unpack<BF16>(w, f);
#pragma unroll
    for (int j = 0; j < EPV; j += 4) {
        uint32_t pk = cvt_pk_fp8<FMT, false>(f[j] * rs.s_down, f[j + 1] * rs.s_down, 0u);
        pk = cvt_pk_fp8<FMT, true>(f[j + 2] * rs.s_down, f[j + 3] * rs.s_down, pk);
        words[j / 4] = pk;
    }
    if (out_vec) {
        float o[EPV];
#pragma unroll
        for (int j = 0; j < EPV; j += 4) {
            float a, b, c, d;
            cvt_pk_f32<FMT, false>(words[j / 4], a, b);
            cvt_pk_f32<FMT, true>(words[j / 4], c, d);
            o[j] = a * rs.s_up;
            o[j + 1] = b * rs.s_up;
            o[j + 2] = c * rs.s_up;
            o[j + 3] = d * rs.s_up;
        }
        uint4 r;
        if (BF16) {
            uint32_t b[8];
#pragma unroll
            for (int j = 0; j < 8; ++j) b[j] = fast_bf16_bits(o[j]);
            r = make_uint4(b[0] | (b[1] << 16), b[2] | (b[3] << 16), b[4] | (b[5] << 16), b[6] | (b[7] << 16));
        } else {
            r = make_uint4(__float_as_uint(o[0]), __float_as_uint(o[1]), __float_as_uint(o[2]),
                           __float_as_uint(o[3]));
        }
        st_vec(out_vec, r);
    }
}

// Elements [e0, e1) of a row at `base` through the bit-level restatement of
// torch's arithmetic: the rows the instruction path does not cover (|k| >
// 110 or a non-finite |x|max), one element per lane per step.
template <int FMT, bool BF16>
__device__ __forceinline__ void quant_slow(const void* x, int64_t base, int64_t e0, int64_t e1, const RowScale& rs,
                                        uint8_t* q, void* out, int lane) {
    for (int64_t e = e0 + lane; e < e1; e += kWave) {
        const float xv = load_x<BF16>(x, base + e);
        const uint32_t c = quant_sw<FMT, BF16>(xv, rs.s_down);
        if (q) q[base + e] = (uint8_t)c;
        if (out) {
            const float o = dequant_sw<FMT, BF16>(c, rs.s_up);
            if (BF16) static_cast<uint16_t*>(out)[base + e] = (uint16_t)f32_to_bf16(o);
            else static_cast<float*>(out)[base + e] = o;
        }
    }
}

// ------------------------------------------------- wave-per-row (registers)

// A row's vectors: vector i covers elements [i * EPV, i * EPV + EPV), the last
// one of a row that is no whole number of vectors the row's last EPV elements
// (it overlaps the vector before it: both write the same codes there), so a
// row of any width >= EPV is whole vectors with no tail.  row_vec_off gives
// the first element of lane-vector i, clamped to the last vector (lanes past
// the row's end read that again, which no maximum notices).
__device__ __forceinline__ int row_vec_off(int i, int epv, int cols) { return min(i * epv, cols - epv); }

// The codes (and, with orow, the round trip's values) of a row's vectors
// first + lane + kWave * j held in buf.
template <int FMT, bool BF16, int VPL>
__device__ __forceinline__ void store_row_vecs(const uint4 (&buf)[VPL], int first, int cols, const RowScale& rs,
                                               uint8_t* qr, char* orow) {
    constexpr int EPV = BF16 ? 8 : 4;
    constexpr int ESZ = BF16 ? 2 : 4;
#pragma unroll
    for (int j = 0; j < VPL; ++j) {
        const int vi = first + kWave * j;
        if (vi * EPV < cols) {
            const int off = row_vec_off(vi, EPV, cols);
            uint32_t words[2];
            quant_vec_fast<FMT, BF16>(buf[j], rs, words, orow ? orow + off * ESZ : nullptr);
            if (qr) {
                if (BF16) st_vec2(qr + off, make_uint2(words[0], words[1]));
                else st_u32(qr + off, words[0]);
            }
        }
    }
}

template <int FMT, bool BF16, int VPL>
__global__ __launch_bounds__(kQBlock) void quant_rows_kernel(const void* __restrict__ x, int64_t rows, int64_t cols,
                                                             uint8_t* __restrict__ q, int32_t* __restrict__ k,
                                                             void* __restrict__ out) {
    constexpr int EPV = BF16 ? 8 : 4;
    constexpr int ESZ = BF16 ? 2 : 4;
    const int lane = threadIdx.x & (kWave - 1);
    const int64_t row = (int64_t)blockIdx.x * kWavesPerBlock + wave_uniform(threadIdx.x / kWave);
    if (row >= rows) return;  // whole waves leave; the kernel has no block barrier
    const int c = (int)cols;
    const char* xr = static_cast<const char*>(x) + row * cols * ESZ;
    // every load of the row is issued before the first is waited for
    uint4 buf[VPL];
    uint32_t amax = 0;
#pragma unroll
    for (int j = 0; j < VPL; ++j) buf[j] = ld_vec(xr + row_vec_off(lane + kWave * j, EPV, c) * ESZ);
#pragma unroll
    for (int j = 0; j < VPL; ++j) amax = vec_absmax<BF16>(buf[j], amax);
    amax = wave_max_u32(amax);
    const RowScale rs = row_scale<FMT>(to_f32_bits<BF16>(amax), BF16, BF16);
    if (lane == 0 && k) k[row] = rs.k;
    if (!rs.fast) return quant_slow<FMT, BF16>(x, row * cols, 0, cols, rs, q, out, lane);
    store_row_vecs<FMT, BF16, VPL>(buf, lane, c, rs, q ? q + row * cols : nullptr,
                                   out ? static_cast<char*>(out) + row * cols * ESZ : nullptr);
}

// Long rows: the block's W waves share one row, each wave a contiguous run of
// kWave * VPLW vectors; the waves' |x|max meet in LDS across one barrier.
// The host launches exactly one block per row, so every wave of a block
// reaches the barrier.
template <int FMT, bool BF16, int W, int VPLW>
__global__ __launch_bounds__(W * kWave) void quant_block_row_kernel(const void* __restrict__ x, int64_t cols,
                                                                  uint8_t* __restrict__ q, int32_t* __restrict__ k,
                                                                  void* __restrict__ out) {
    constexpr int EPV = BF16 ? 8 : 4;
    constexpr int ESZ = BF16 ? 2 : 4;
    __shared__ uint32_t wmax[W];
    const int lane = threadIdx.x & (kWave - 1);
    const int w = wave_uniform(threadIdx.x / kWave);
    const int64_t row = blockIdx.x;
    const int c = (int)cols;
    const int v0 = w * kWave * VPLW;
    const char* xr = static_cast<const char*>(x) + row * cols * ESZ;
    uint4 buf[VPLW];
    uint32_t amax = 0;
#pragma unroll
    for (int j = 0; j < VPLW; ++j) buf[j] = ld_vec(xr + row_vec_off(v0 + lane + kWave * j, EPV, c) * ESZ);
#pragma unroll
    for (int j = 0; j < VPLW; ++j) amax = vec_absmax<BF16>(buf[j], amax);
    amax = wave_max_u32(amax);
    if (lane == 0) wmax[w] = amax;
    __syncthreads();
    amax = wmax[0];
#pragma unroll
    for (int i = 1; i < W; ++i) amax = max(amax, wmax[i]);
    const RowScale rs = row_scale<FMT>(to_f32_bits<BF16>(amax), BF16, BF16);
    if (threadIdx.x == 0 && k) k[row] = rs.k;
    if (!rs.fast) {
        const int64_t e0 = min((int64_t)v0 * EPV, cols), e1 = min((int64_t)(v0 + kWave * VPLW) * EPV, cols);
        return quant_slow<FMT, BF16>(x, row * cols, e0, e1, rs, q, out, lane);
    }
    store_row_vecs<FMT, BF16, VPLW>(buf, v0 + lane, c, rs, q ? q + row * cols : nullptr,
                                    out ? static_cast<char*>(out) + row * cols * ESZ : nullptr);
}

// ------------------------------------------------------- split long rows

__global__ void fill_u32_kernel(uint32_t* p, int64_t n, uint32_t value) {
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x)
        p[i] = value;
}

// Long rows (and per-tensor scaling, one row) go through segments of
// kSegElems elements.  The row's |x|max is reduced without atomics: block
// (r, j) of the rowmax_partial_kernel folds row r's segments, its waves'
// maxima meeting in LDS, into partial[r * bpr + j], at most 256 a row; every
// wave of the convert launch folds its row's partials itself while its segment
// is on the way.  Per tensor, bf16, back to back, against a launch between
// the two that folded up to 2,048 partials (and blocks of one wave): 0.4 M
// elements 7.1 us against 10.3, 3.1 M 7.6 against 10.6, 16.8 M 12.8 against
// 16.6, 33.6 M 25.4 against 28.5, 537 M 386 against 390; of a length that is
// no whole number of vectors, 3.1 M 7.8 against 29.3.  Values are |x| bit
// patterns (fp32 bits for fp32 input, bf16 bits for bf16), so max is an
// integer max.
constexpr int64_t kSplitWaves = ELY_SPLIT_WAVES;  // waves of the partial-max launch (at most)
constexpr int kSplitBlockWaves = 8;               // ... per block, when a row has that many

// How the partial-max launch shares a row: `waves` per block, `blocks` per row.
struct SplitShape {
    int waves;
    int64_t blocks;
};
static SplitShape split_shape(int64_t rows, int64_t segs) {
    const int64_t wpr = std::max<int64_t>(1, std::min<int64_t>(segs, kSplitWaves / std::max<int64_t>(rows, 1)));
    if (wpr < kSplitBlockWaves) return {1, wpr};
    // a multiple of the 8 XCDs for a single row (see rowmax_partial_kernel)
    const int64_t blocks = (wpr + kSplitBlockWaves - 1) / kSplitBlockWaves;
    return {kSplitBlockWaves, rows == 1 ? (blocks + 7) / 8 * 8 : blocks};
}

// Vectors of one segment a lane holds: 2048 bf16 = 256 x 16 B -> 4 per lane.
template <bool BF16>
struct Seg {
    static constexpr int EPV = BF16 ? 8 : 4;
    static constexpr int VPL = (int)(kSegElems / EPV / kWave);
};

// Segment `seg` of a row of cols elements (at least one vector of them): its
// first element, whether it is a whole one, its vectors, and where vector vi
// lies from e0.  A row that is no whole number of vectors ends in its last
// EPV elements (row_vec_off), which may begin before the segment.
template <bool BF16>
struct SegAt {
    static constexpr int EPV = Seg<BF16>::EPV, ESZ = BF16 ? 2 : 4;
    int64_t e0;
    bool whole;
    int len, nv;
    __device__ __forceinline__ SegAt(int64_t seg, int64_t cols)
        : e0(seg * kSegElems), whole(e0 + kSegElems <= cols), len((int)min(kSegElems, cols - e0)),
          nv((len + EPV - 1) / EPV) {}
    __device__ __forceinline__ int off(int vi) const { return whole ? vi * EPV : min(vi * EPV, len - EPV); }
};

// That segment of the row at xr in registers; lanes past a short segment's
// end load its last vector again.  Whole segments, nearly all of them, load
// without the clamps (with them C4's |x|max pass took 184 us against 153).
template <bool BF16, bool NT = (ELY_FP8_NT & 1) != 0>
__device__ __forceinline__ void load_segment(const char* xr, const SegAt<BF16>& at, int lane,
                                             uint4 (&buf)[Seg<BF16>::VPL]) {
    const char* xs = xr + at.e0 * SegAt<BF16>::ESZ;
    if (at.whole) {
#pragma unroll
        for (int j = 0; j < Seg<BF16>::VPL; ++j) buf[j] = ld_vec<NT>(xs + (lane + kWave * j) * 16);
    } else {
#pragma unroll
        for (int j = 0; j < Seg<BF16>::VPL; ++j) buf[j] = ld_vec<NT>(xs + at.off(lane + kWave * j) * SegAt<BF16>::ESZ);
    }
}

// |x|max bits of segment `seg` of row `row`; vec: the row holds at least one
// vector.
template <bool BF16, bool NT>
__device__ __forceinline__ uint32_t seg_absmax(const void* x, int64_t row, int64_t cols, int64_t seg, int vec, int lane) {
    constexpr int VPL = Seg<BF16>::VPL, ESZ = BF16 ? 2 : 4;
    uint32_t amax = 0;
    if (vec) {
        uint4 buf[VPL];
        load_segment<BF16, NT>(static_cast<const char*>(x) + row * cols * ESZ, SegAt<BF16>(seg, cols), lane, buf);
#pragma unroll
        for (int j = 0; j < VPL; ++j) amax = vec_absmax<BF16>(buf[j], amax);
    } else {
        const int64_t e0 = seg * kSegElems, e1 = min(e0 + kSegElems, cols);
        for (int64_t e = e0 + lane; e < e1; e += kWave) {
            uint32_t b = BF16 ? (uint32_t)static_cast<const uint16_t*>(x)[row * cols + e] & 0x7FFFu
                              : __float_as_uint(static_cast<const float*>(x)[row * cols + e]) & 0x7FFFFFFFu;
            amax = max(amax, b);
        }
    }
    return amax;
}

template <bool BF16, int W>
__global__ __launch_bounds__(W * kWave) void rowmax_partial_kernel(const void* __restrict__ x, int64_t cols,
                                                                   int64_t segs, int64_t bpr, int vec, int64_t cached,
                                                                   uint32_t* __restrict__ partial) {
    __shared__ uint32_t red[W];
    const int lane = threadIdx.x & (kWave - 1), w = wave_uniform(threadIdx.x / kWave);
    const int64_t row = blockIdx.x / bpr, j = blockIdx.x % bpr, step = bpr * W;
    uint32_t amax = 0;
    // a row's last `cached` segments are read last, with plain loads; two
    // loops in sequence keep the two kinds of loads apart
    const int64_t cut = segs - cached;
    // Block j's segments are j, j + bpr, ...: blocks go to the XCDs in turn,
    // so with bpr a multiple of their number a single row's segment is read by
    // the XCD that converts it, whose L2 may still hold it (32 M bf16: the
    // convert launch 15.5 us, against 19 with segments 8 j, 8 j + 1, ...)
    int64_t seg = j + w * bpr;
    for (; seg < cut; seg += step) amax = max(amax, seg_absmax<BF16, (ELY_FP8_NT & 1) != 0>(x, row, cols, seg, vec, lane));
    for (; seg < segs; seg += step) amax = max(amax, seg_absmax<BF16, false>(x, row, cols, seg, vec, lane));
    amax = wave_max_u32(amax);
    if (W == 1) {
        if (lane == 0) partial[blockIdx.x] = amax;
        return;
    }
    if (lane == 0) red[w] = amax;
    __syncthreads();
    if (threadIdx.x == 0) {
#pragma unroll
        for (int i = 1; i < W; ++i) amax = max(amax, red[i]);
        partial[blockIdx.x] = amax;
    }
}

// rowmax[r] = the max of row r's partials, one wave per row (the recovery's
// launches read it).
__global__ __launch_bounds__(kWave) void rowmax_reduce_kernel(const uint32_t* __restrict__ partial, int64_t rows,
                                                              int64_t bpr, uint32_t* __restrict__ rowmax) {
    for (int64_t r = blockIdx.x; r < rows; r += gridDim.x) {
        uint32_t m = 0;
        for (int64_t i = threadIdx.x; i < bpr; i += kWave) m = max(m, partial[r * bpr + i]);
        m = wave_max_u32(m);
        if (threadIdx.x == 0) rowmax[r] = m;
    }
}

// Vector vi of a segment converted at the row's scale rs.
template <int FMT, bool BF16>
__device__ __forceinline__ void convert_seg_vec(const uint4& v, const SegAt<BF16>& at, int vi, int64_t base, const RowScale& rs,
                                                uint8_t* q, void* out) {
    if (vi >= at.nv) return;
    const int64_t e = base + at.e0 + at.off(vi);
    uint32_t words[2];
    quant_vec_fast<FMT, BF16>(v, rs, words, out ? static_cast<char*>(out) + e * SegAt<BF16>::ESZ : nullptr);
    if (q) {
        if (BF16) st_vec2(q + e, make_uint2(words[0], words[1]));
        else st_u32(q + e, words[0]);
    }
}

// A segment converted at the row's scale rs, one vector per lane loaded and
// stored at a time.
template <int FMT, bool BF16>
__device__ __forceinline__ void quant_segment(const void* x, int64_t row, int64_t cols, int64_t seg, int vec,
                                              const RowScale& rs, uint8_t* q, void* out, int lane) {
    const int64_t base = row * cols;
    if (vec && rs.fast) {
        const SegAt<BF16> at(seg, cols);
        const char* xs = static_cast<const char*>(x) + (base + at.e0) * SegAt<BF16>::ESZ;
#pragma unroll
        for (int j = 0; j < Seg<BF16>::VPL; ++j) {
            const int vi = lane + kWave * j;
            const uint4 v = ld_vec(xs + at.off(vi) * SegAt<BF16>::ESZ);
            convert_seg_vec<FMT, BF16>(v, at, vi, base, rs, q, out);
            __builtin_amdgcn_sched_barrier(0);
        }
    } else {
        quant_slow<FMT, BF16>(x, base, seg * kSegElems, min((seg + 1) * kSegElems, cols), rs, q, out, lane);
    }
}

template <int FMT, bool BF16>
__global__ __launch_bounds__(kQBlock) void quant_split_kernel(const void* __restrict__ x, int64_t rows, int64_t cols,
                                                              int64_t segs, int vec,
                                                              const uint32_t* __restrict__ partial, int64_t bpr,
                                                              uint8_t* __restrict__ q, int32_t* __restrict__ k,
                                                              void* __restrict__ out) {
    const int lane = threadIdx.x & (kWave - 1);
    const int64_t gw = (int64_t)blockIdx.x * kWavesPerBlock + wave_uniform(threadIdx.x / kWave);
    const int64_t row = gw / segs, seg = gw % segs;
    if (row >= rows) return;
    // the segment is on its way while the row's partials are folded
    const SegAt<BF16> at(seg, cols);
    uint4 buf[Seg<BF16>::VPL];
    if (vec) load_segment<BF16>(static_cast<const char*>(x) + row * cols * SegAt<BF16>::ESZ, at, lane, buf);
    uint32_t m = 0;
    if (bpr == 1) {
        // short rows: the one word, without the butterfly (8.4 M rows of 4 bf16
        // 4171 -> 3828 us; longer rows the same)
        m = partial[row];
    } else {
#pragma unroll 4
        for (int64_t i = lane; i < bpr; i += kWave) m = max(m, partial[row * bpr + i]);
        m = wave_max_u32(m);
    }
    const RowScale rs = row_scale<FMT>(to_f32_bits<BF16>(m), BF16, BF16);
    if (seg == 0 && lane == 0 && k) k[row] = rs.k;
    if (vec && rs.fast) {
#pragma unroll
        for (int j = 0; j < Seg<BF16>::VPL; ++j)
            convert_seg_vec<FMT, BF16>(buf[j], at, lane + kWave * j, row * cols, rs, q, out);
    } else {
        quant_slow<FMT, BF16>(x, row * cols, at.e0, at.e0 + at.len, rs, q, out, lane);
    }
}

// ------------------------------------------------- per-tensor, with a hint
//
// Per-tensor scaling needs the whole tensor's |x|max before the first code,
// so the split path reads x twice.  Given the exponent a caller expects (the
// previous step's, say), one pass does both: wave w reads segment w once,
// writes its |x|max to partial[w] and its codes at the hinted scale.  A
// small launch folds the partials to kHintBlocks maxima, and a capped fixup
// launch, whose every wave folds those to the tensor's k, writes k (and
// whether it equals the hint) and exits when it does; on a miss its waves
// convert every segment again at the true scale.  The codes depend on k
// alone, so a hit's codes are the split path's, byte for byte.
constexpr int kHintBlocks = 256;         // maxima the reduce launch leaves (4 per lane of a fixup wave)
#ifndef ELY_HINT_FIXUP_WPC
// fixup grid cap, waves per compute unit.  C4 per-tensor (1.07 GB of bf16):
// a hit 6.25-6.32 TB/s with 8 or 32, 6.1 with 128; a miss 2.5 TB/s with 8,
// 3.1 with 32 or 128
#define ELY_HINT_FIXUP_WPC 32
#endif
constexpr int kHintFixupWavesPerCU = ELY_HINT_FIXUP_WPC;
#ifndef ELY_GUESS_MIN_MB
// per-tensor rows of at least this many MiB of x take the sampled guess.
// Back to back on N(0, 1) bf16 (a right guess), per call: 64 MiB 24.0 us
// against 25.3 on the split path, 76 MiB 26.7 against 29.0, 128 MiB 38.8
// against 47.6, 1 GiB 253 against 386 (of fp32, 128 MiB 35 against 44)
#define ELY_GUESS_MIN_MB 64
#endif
#ifndef ELY_GUESS_STRIDE
#define ELY_GUESS_STRIDE 61  // the guess samples every this-many-th segment (a prime)
#endif
constexpr int64_t kGuessStride = ELY_GUESS_STRIDE;

// A segment in registers: its |x|max bits (fp32 bits for fp32 input, bf16 bits
// for bf16), and, where the hint admits the instruction path, its codes at
// the hinted exponent.
template <int FMT, bool BF16>
__device__ __forceinline__ uint32_t hint_segment(const uint4 (&buf)[Seg<BF16>::VPL], const SegAt<BF16>& at, int32_t hint,
                                                 uint8_t* q, void* out, int lane) {
    const bool convert = hint >= -kFastK && hint <= kFastK;
    RowScale hs;
    hs.k = hint;
    hs.fast = true;
    hs.s_down = __uint_as_float((uint32_t)(127 - hint) << 23);
    hs.s_up = __uint_as_float((uint32_t)(127 + hint) << 23);
    uint32_t amax = 0;
#pragma unroll
    for (int j = 0; j < Seg<BF16>::VPL; ++j) {
        amax = vec_absmax<BF16>(buf[j], amax);
        if (convert) convert_seg_vec<FMT, BF16>(buf[j], at, lane + kWave * j, 0, hs, q, out);
    }
    return wave_max_u32(amax);
}

// The hint: k_hint, or *k_hint_dev when that is given (read here, before
// the fixup launch writes k, which may be the same word).  Wave 0 keeps the
// hint it read in hint_copy for the fixup.  A hint outside the instruction
// path's range converts nothing here: the call is then a miss.
template <int FMT, bool BF16>
__global__ __launch_bounds__(kQBlock) void quant_hint_kernel(const void* __restrict__ x, int64_t n, int64_t segs,
                                                             int32_t k_hint, const int32_t* k_hint_dev,
                                                             uint8_t* __restrict__ q, void* __restrict__ out,
                                                             uint32_t* __restrict__ partial,
                                                             int32_t* __restrict__ hint_copy) {
    const int lane = threadIdx.x & (kWave - 1);
    const int64_t seg = (int64_t)blockIdx.x * kWavesPerBlock + wave_uniform(threadIdx.x / kWave);
    if (seg >= segs) return;
    const int32_t hint = k_hint_dev ? __builtin_amdgcn_readfirstlane(*k_hint_dev) : k_hint;
    if (seg == 0 && lane == 0) hint_copy[0] = hint;
    const SegAt<BF16> at(seg, n);
    uint4 buf[Seg<BF16>::VPL];
    load_segment<BF16>(static_cast<const char*>(x), at, lane, buf);
    const uint32_t amax = hint_segment<FMT, BF16>(buf, at, hint, q, out, lane);
    if (lane == 0) partial[seg] = amax;
}

// A per-tensor row's exponent guessed from a sample, in three launches:
//   * guess_amax_kernel: kGuessBlocks blocks fold the |x|max of every
//     kGuessStride-th segment (a prime, so that the sample does not fall in
//     step with a row length or an outlier channel) to one word each, and
//     clear the tops;
//   * quant_guess_kernel: every wave folds those words to the sample's |x|max
//     while its segment is on the way, converts at its exponent, and raises
//     a top where its segment exceeds the sample (none to a few dozen
//     segments of a tensor whose values come in no order; at worst, every
//     segment of a rising one, spread over kTops words, a line each);
//   * the fixup folds the sample and the tops to the row's |x|max: it exits
//     where that has the guessed exponent, and converts again where not.
// All |x|max words here are fp32 bits.  Against five launches (the sample's
// words folded by one, the segments' maxima of the hint path by another),
// bf16, right guesses: 64 MiB 29.4 -> 24.0 us, 128 MiB 45.1 -> 38.8, 1 GiB
// 265 -> 253 (6.37 TB/s).  A miss with every unsampled segment above the
// sample (most atomics): 128 MiB 72.7 -> 66.3 us, 1 GiB 530 -> 515.
constexpr int kGuessBlocks = 256, kGuessBlockWaves = 8;
constexpr int kTops = 64, kTopStride = 32;  // words: a top per lane of a fixup wave, 128 bytes apart
template <bool BF16>
__global__ __launch_bounds__(kGuessBlockWaves * kWave) void guess_amax_kernel(const void* __restrict__ x, int64_t n,
                                                                              int64_t stride, int64_t samples,
                                                                              uint32_t* __restrict__ sampled,
                                                                              uint32_t* __restrict__ tops) {
    __shared__ uint32_t red[kGuessBlockWaves];
    const int lane = threadIdx.x & (kWave - 1), w = wave_uniform(threadIdx.x / kWave);
    uint32_t m = 0;
    for (int64_t i = blockIdx.x + (int64_t)w * kGuessBlocks; i < samples; i += kGuessBlocks * kGuessBlockWaves)
        m = max(m, seg_absmax<BF16, (ELY_FP8_NT & 1) != 0>(x, 0, n, i * stride, 1, lane));
    m = wave_max_u32(m);
    if (lane == 0) red[w] = m;
    __syncthreads();
    if (threadIdx.x == 0) {
#pragma unroll
        for (int i = 1; i < kGuessBlockWaves; ++i) m = max(m, red[i]);
        sampled[blockIdx.x] = to_f32_bits<BF16>(m);
        if (blockIdx.x < kTops) tops[blockIdx.x * kTopStride] = 0;
    }
}

template <int FMT, bool BF16>
__global__ __launch_bounds__(kQBlock) void quant_guess_kernel(const void* __restrict__ x, int64_t n, int64_t segs,
                                                              const uint32_t* __restrict__ sampled,
                                                              uint8_t* __restrict__ q, void* __restrict__ out,
                                                              uint32_t* __restrict__ tops, uint32_t* __restrict__ amax) {
    static_assert(kGuessBlocks == 4 * kWave, "a lane folds four sampled words");
    const int lane = threadIdx.x & (kWave - 1);
    const int64_t seg = (int64_t)blockIdx.x * kWavesPerBlock + wave_uniform(threadIdx.x / kWave);
    if (seg >= segs) return;
    const SegAt<BF16> at(seg, n);
    uint4 buf[Seg<BF16>::VPL];
    load_segment<BF16>(static_cast<const char*>(x), at, lane, buf);
    const uint32_t sample = __builtin_amdgcn_readfirstlane(wave_max_u32(
        max(max(sampled[lane], sampled[lane + kWave]), max(sampled[lane + 2 * kWave], sampled[lane + 3 * kWave]))));
    if (seg == 0 && lane == 0) amax[0] = sample;
    const uint32_t top = to_f32_bits<BF16>(hint_segment<FMT, BF16>(buf, at, scale_exp_from_amax<FMT>(sample), q, out, lane));
    if (lane == 0 && top > sample) atomicMax(tops + (seg % kTops) * kTopStride, top);
}

// partial[0, segs) -> out[b] for b < kHintBlocks (block b folds a contiguous
// share; integer max, so the order does not matter).
__global__ __launch_bounds__(kRowBlock) void hint_reduce_kernel(const uint32_t* __restrict__ partial, int64_t segs,
                                                              uint32_t* __restrict__ out) {
    __shared__ uint32_t red[kRowWaves];
    const int lane = threadIdx.x & (kWave - 1), w = threadIdx.x / kWave;
    const int64_t per = (segs + kHintBlocks - 1) / kHintBlocks;
    const int64_t i0 = (int64_t)blockIdx.x * per, i1 = min(i0 + per, segs);
    uint32_t m = 0;
    for (int64_t i = i0 + threadIdx.x; i < i1; i += kRowBlock) m = max(m, partial[i]);
    m = wave_max_u32(m);
    if (lane == 0) red[w] = m;
    __syncthreads();
    if (threadIdx.x == 0) {
        uint32_t t = red[0];
        for (int j = 1; j < kRowWaves; ++j) t = max(t, red[j]);
        out[blockIdx.x] = t;
    }
}

// The fixup of a hinted or guessed row whose |x|max bits are m: k and the hit
// flag, and, on a miss, every segment again at the true scale.
template <int FMT, bool BF16>
__device__ __forceinline__ void fixup(const void* x, int64_t n, int64_t segs, int32_t hint, uint32_t m, uint8_t* q, int32_t* k,
                                      void* out, int32_t* hit, int lane) {
    const int64_t gw = (int64_t)blockIdx.x * kWavesPerBlock + wave_uniform(threadIdx.x / kWave);
    const int64_t waves = (int64_t)gridDim.x * kWavesPerBlock;
    const RowScale rs = row_scale<FMT>(m, BF16, BF16);
    const bool same = rs.fast && rs.k == hint && hint >= -kFastK && hint <= kFastK;
    if (gw == 0 && lane == 0) {
        k[0] = rs.k;
        if (hit) hit[0] = same ? 1 : 0;
    }
    if (same) return;
    for (int64_t seg = gw; seg < segs; seg += waves) quant_segment<FMT, BF16>(x, 0, n, seg, 1, rs, q, out, lane);
}

template <int FMT, bool BF16>
__global__ __launch_bounds__(kQBlock) void quant_hint_fixup_kernel(const void* __restrict__ x, int64_t n, int64_t segs,
                                                                   const int32_t* __restrict__ hint_copy,
                                                                   const uint32_t* __restrict__ block_max,
                                                                   uint8_t* __restrict__ q, int32_t* __restrict__ k,
                                                                   void* __restrict__ out, int32_t* __restrict__ hit) {
    static_assert(kHintBlocks == 4 * kWave, "a fixup lane folds four block maxima");
    const int lane = threadIdx.x & (kWave - 1);
    const uint32_t m = wave_max_u32(max(max(block_max[lane], block_max[lane + kWave]),
                                        max(block_max[lane + 2 * kWave], block_max[lane + 3 * kWave])));
    fixup<FMT, BF16>(x, n, segs, hint_copy[0], to_f32_bits<BF16>(m), q, k, out, hit, lane);
}

template <int FMT, bool BF16>
__global__ __launch_bounds__(kQBlock) void quant_guess_fixup_kernel(const void* __restrict__ x, int64_t n, int64_t segs,
                                                                    const uint32_t* __restrict__ tops,
                                                                    const uint32_t* __restrict__ amax,
                                                                    uint8_t* __restrict__ q, int32_t* __restrict__ k,
                                                                    void* __restrict__ out) {
    static_assert(kTops == kWave, "a fixup lane reads one top");
    const int lane = threadIdx.x & (kWave - 1);
    const uint32_t sample = amax[0];
    const uint32_t m = wave_max_u32(max(sample, tops[lane * kTopStride]));
    fixup<FMT, BF16>(x, n, segs, scale_exp_from_amax<FMT>(sample), m, q, k, out, nullptr, lane);
}

// -------------------------------------------------------------- dequantize

// The codes are dequantized as one flat array: wave w takes codes
// [S w, S w + S) (S = kDeqSegCodes), which may span rows.  A lane takes CPL
// codes per step (8 for bf16 output, 4 for fp32), so that each store
// instruction of a wave writes one contiguous 1 KB run; every lane issues
// its loads (all of them, or batches of ELY_DEQ_BATCH) before the first is
// used.  When rows are whole vectors (a multiple of 16 codes, 16-byte
// aligned buffers) each CPL-code vector lies in one row; RAGGED takes rows of
// any width >= CPL at any alignment, where a vector may hold the end of one
// row and the start of the next (`cut` codes of it in the first) and the
// array's last vector is its last CPL codes.  Rows at least a segment
// wide give a segment at most two exponents, read once per wave (C1 back to
// back: 5.89-5.94 TB/s against 5.76-5.80 with a division and an exponent
// load per vector); narrower rows look theirs up per vector.  Short
// segments (many short-lived waves) measured fastest.

// CPL codes at e, the first `cut` of them of a row with exponent k1, the rest
// of the next row's k2.
template <int FMT, bool BF16OUT, int CPL>
__device__ __forceinline__ void dequant_two_rows(const uint32_t (&w)[CPL / 4], int k1, int k2, int cut, void* out,
                                                 int64_t e) {
    if (k1 >= -kFastK && k1 <= kFastK && k2 >= -kFastK && k2 <= kFastK) {
        const float s1 = __uint_as_float((uint32_t)(127 + k1) << 23), s2 = __uint_as_float((uint32_t)(127 + k2) << 23);
        float o[CPL];
#pragma unroll
        for (int h = 0; h < CPL / 4; ++h) {
            cvt_pk_f32<FMT, false>(w[h], o[4 * h], o[4 * h + 1]);
            cvt_pk_f32<FMT, true>(w[h], o[4 * h + 2], o[4 * h + 3]);
        }
        uint32_t b[CPL];
#pragma unroll
        for (int t = 0; t < CPL; ++t) {
            const float v = o[t] * (t < cut ? s1 : s2);
            b[t] = BF16OUT ? (v != v ? 0x7FC0u : fast_bf16_bits(v)) : __float_as_uint(v);
        }
        if (BF16OUT)
            st_vec(static_cast<uint16_t*>(out) + e,
                   make_uint4(b[0] | (b[1] << 16), b[2] | (b[3] << 16), b[CPL - 4] | (b[CPL - 3] << 16),
                              b[CPL - 2] | (b[CPL - 1] << 16)));
        else
            st_vec(static_cast<float*>(out) + e, make_uint4(b[0], b[1], b[2], b[3]));
        return;
    }
    const float s1 = pow2_dtype(k1, BF16OUT), s2 = pow2_dtype(k2, BF16OUT);
#pragma unroll 1
    for (int t = 0; t < CPL; ++t) {
        const float o = dequant_sw<FMT, BF16OUT>((w[t / 4] >> (8 * (t % 4))) & 0xFFu, t < cut ? s1 : s2);
        if (BF16OUT) static_cast<uint16_t*>(out)[e + t] = (uint16_t)f32_to_bf16(o);
        else static_cast<float*>(out)[e + t] = o;
    }
}

template <int FMT, bool BF16OUT, bool IDX32, bool RAGGED>
__global__ __launch_bounds__(kQBlock) void dequant_flat_kernel(const uint8_t* __restrict__ q,
                                                               const int32_t* __restrict__ k, int64_t n,
                                                               int64_t cols, void* __restrict__ out) {
    constexpr int CPL = BF16OUT ? 8 : 4;
    constexpr int VPL = (int)(kDeqSegCodes / CPL / kWave);
    const int lane = threadIdx.x & (kWave - 1);
    const int64_t gw = (int64_t)blockIdx.x * kWavesPerBlock + wave_uniform(threadIdx.x / kWave);
    const int64_t e0 = gw * kDeqSegCodes;
    if (e0 >= n) return;
    const int64_t nv = (min(kDeqSegCodes, n - e0) + (RAGGED ? CPL - 1 : 0)) / CPL;
    constexpr int DB = (ELY_DEQ_BATCH <= 0 || ELY_DEQ_BATCH > VPL) ? VPL : ELY_DEQ_BATCH;
    // rows at least a segment wide: the segment meets at most two rows, the
    // one holding code e0 and, from code `split` on, the next; the wave reads
    // their two exponents once (uniform loads) instead of one lookup per vector
    const bool two_rows = cols >= kDeqSegCodes;
    int64_t split = 0;
    int k_lo = 0, k_hi = 0;
    uint32_t buf[VPL][CPL / 4];
#pragma unroll
    for (int j0 = 0; j0 < VPL; j0 += DB) {
#pragma unroll
        for (int j = j0; j < j0 + DB && j < VPL; ++j) {
            const int64_t vi = lane + (int64_t)kWave * j;
            const int64_t ev = e0 + (vi < nv ? vi : nv - 1) * CPL;
            const uint8_t* src = q + (RAGGED ? min(ev, n - CPL) : ev);
            if (CPL == 8) {
                const uint2 w = ld_vec2(src);
                buf[j][0] = w.x;
                buf[j][CPL / 4 - 1] = w.y;
            } else {
                buf[j][0] = ld_u32(src);
            }
        }
        // the exponents are read once the first codes are requested: a wait
        // for these loads ahead of the code loads would hold those back
        if (j0 == 0 && two_rows) {
            // a segment shorter than a vector is the array's last vector, which begins before it
            const int64_t es = RAGGED ? min(e0, n - CPL) : e0;
            const int64_t row0 = IDX32 ? (int64_t)((uint32_t)es / (uint32_t)cols) : es / cols;
            split = (row0 + 1) * cols;
            k_lo = k[row0];
            k_hi = k[split < n ? row0 + 1 : row0];
        }
#pragma unroll
        for (int j = j0; j < j0 + DB && j < VPL; ++j) {
            const int64_t vi = lane + (int64_t)kWave * j;
            if (vi >= nv) continue;
            const int64_t e = RAGGED ? min(e0 + vi * CPL, n - CPL) : e0 + vi * CPL;
            int kk, kk2 = 0, cut = CPL;
            if (two_rows) {
                kk = e < split ? k_lo : k_hi;
                if (RAGGED && e < split && e + CPL > split) {
                    cut = (int)(split - e);
                    kk2 = k_hi;
                }
            } else {
                const int64_t row = IDX32 ? (int64_t)((uint32_t)e / (uint32_t)cols) : e / cols;
                kk = k[row];
                if (RAGGED && e + CPL > (row + 1) * cols) {
                    cut = (int)((row + 1) * cols - e);
                    kk2 = k[row + 1];
                }
            }
            if (RAGGED && cut < CPL && kk2 != kk) {
                dequant_two_rows<FMT, BF16OUT, CPL>(buf[j], kk, kk2, cut, out, e);
                continue;
            }
            if (kk >= -kFastK && kk <= kFastK) {
                const float s_up = __uint_as_float((uint32_t)(127 + kk) << 23);
                if (BF16OUT && !(nan_code_bits<FMT>(buf[j][0]) | nan_code_bits<FMT>(buf[j][CPL / 4 - 1]))) {
                    // no NaN code among the eight: the scaled decode writes the bf16 bits
                    st_vec(static_cast<uint16_t*>(out) + e,
                           make_uint4(cvt_scaled_pk_bf16<FMT, false>(buf[j][0], s_up),
                                      cvt_scaled_pk_bf16<FMT, true>(buf[j][0], s_up),
                                      cvt_scaled_pk_bf16<FMT, false>(buf[j][CPL / 4 - 1], s_up),
                                      cvt_scaled_pk_bf16<FMT, true>(buf[j][CPL / 4 - 1], s_up)));
                    continue;
                }
                float o[CPL];
#pragma unroll
                for (int h = 0; h < CPL / 4; ++h) {
                    float a, b, c, d;
                    cvt_pk_f32<FMT, false>(buf[j][h], a, b);
                    cvt_pk_f32<FMT, true>(buf[j][h], c, d);
                    o[4 * h] = a * s_up;
                    o[4 * h + 1] = b * s_up;
                    o[4 * h + 2] = c * s_up;
                    o[4 * h + 3] = d * s_up;
                }
                if (BF16OUT) {
                    uint32_t b[8];
#pragma unroll
                    for (int t = 0; t < 8; ++t) {
                        // an fp8 NaN is the only non-exact value the instruction path sees
                        const float v = o[t];
                        b[t] = v != v ? 0x7FC0u : fast_bf16_bits(v);
                    }
                    st_vec(static_cast<uint16_t*>(out) + e, make_uint4(b[0] | (b[1] << 16), b[2] | (b[3] << 16),
                                                                       b[4] | (b[5] << 16), b[6] | (b[7] << 16)));
                } else {
                    st_vec(static_cast<float*>(out) + e, make_uint4(__float_as_uint(o[0]), __float_as_uint(o[1]),
                                                                    __float_as_uint(o[2]), __float_as_uint(o[3])));
                }
            } else {
                // the restatement of torch's arithmetic (|k| > 110), code by code
                const float s_up = pow2_dtype(kk, BF16OUT);
#pragma unroll 1
                for (int t = 0; t < CPL; ++t) {
                    const float o = dequant_sw<FMT, BF16OUT>((buf[j][t / 4] >> (8 * (t % 4))) & 0xFFu, s_up);
                    if (BF16OUT) static_cast<uint16_t*>(out)[e + t] = (uint16_t)f32_to_bf16(o);
                    else static_cast<float*>(out)[e + t] = o;
                }
            }
        }
        // the next batch is issued only once this one has been stored
        if (DB < VPL) __builtin_amdgcn_sched_barrier(0);
    }
}

// Any other shape: one wave per (row, kDeqSegCodes-code segment), element by element.
template <int FMT, bool BF16OUT>
__global__ __launch_bounds__(kQBlock) void dequant_any_kernel(const uint8_t* __restrict__ q,
                                                              const int32_t* __restrict__ k, int64_t rows,
                                                              int64_t cols, int64_t segs, void* __restrict__ out) {
    const int lane = threadIdx.x & (kWave - 1);
    const int64_t gw = (int64_t)blockIdx.x * kWavesPerBlock + wave_uniform(threadIdx.x / kWave);
    const int64_t row = gw / segs, seg = gw % segs;
    if (row >= rows) return;
    const int kk = k[row];
    const bool fast = kk >= -kFastK && kk <= kFastK;
    const float s_up = fast ? __uint_as_float((uint32_t)(127 + kk) << 23) : pow2_dtype(kk, BF16OUT);
    const int64_t e0 = seg * kDeqSegCodes, e1 = min(e0 + kDeqSegCodes, cols);
    const int64_t base = row * cols;
    for (int64_t e = e0 + lane; e < e1; e += kWave) {
        const float o = dequant_sw<FMT, BF16OUT>(q[base + e], s_up);
        if (BF16OUT) static_cast<uint16_t*>(out)[base + e] = (uint16_t)f32_to_bf16(o);
        else static_cast<float*>(out)[base + e] = o;
    }
}

// ------------------------------------------------------- recover_exp / wire

// Bit i of the candidate mask stands for offset kDeltas[i] (fp8.py:25).
__constant__ int kDeltas[5] = {0, -1, 1, -2, 2};

// Is v (a value of the tensor's dtype) exactly fp8(v * 2^-c) * 2^c in that
// dtype's arithmetic (fp8.py:85-86)?  `fast` rows use the conversion
// instructions: every candidate's 2^+-c is a normal power of two there and
// every product exact, so the test is just whether v * 2^-c lies on the fp8
// grid; non-finite elements always take the restatement.
template <int FMT, bool BF16>
__device__ __forceinline__ bool exact_at(float v, int c, bool fast) {
    if (fast && __builtin_isfinite(v)) {
        const float y = v * __uint_as_float((uint32_t)(127 - c) << 23);
        const uint32_t code = cvt_pk_fp8<FMT, false>(y, 0.0f, 0u) & 0xFFu;
        float back, unused;
        cvt_pk_f32<FMT, false>(code, back, unused);
        return back * __uint_as_float((uint32_t)(127 + c) << 23) == v;
    }
    const float y = round_to(v * pow2_dtype(-c, BF16), BF16);
    const uint32_t code = fp8_from_f32_sw<FMT>(y);
    const float back = round_to(round_to(fp8_to_f32_sw<FMT>(code), BF16) * pow2_dtype(c, BF16), BF16);
    return back == v;
}

__device__ __forceinline__ uint32_t wave_and_u32(uint32_t v) {
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v &= (uint32_t)__shfl_xor((int)v, o, kWave);
    return v;
}

// The segment's elements, one callback per element (lanes past the end make
// none): vectorized loads, all issued before the first is used, when `vec`
// (16-byte aligned rows whose length is a multiple of the vector), element
// loads otherwise.
template <bool BF16, class F>
__device__ __forceinline__ void for_seg_elems(const void* t, int64_t row, int64_t cols, int64_t e0, int64_t e1,
                                              int vec, int lane, F f) {
    constexpr int EPV = Seg<BF16>::EPV, VPL = Seg<BF16>::VPL, ESZ = BF16 ? 2 : 4;
    if (vec) {
        const uint4* tr = reinterpret_cast<const uint4*>(static_cast<const char*>(t) + (row * cols + e0) * ESZ);
        const int64_t nv = (e1 - e0) / EPV;
        uint4 buf[VPL];
#pragma unroll
        for (int j = 0; j < VPL; ++j) {
            const int64_t vi = lane + (int64_t)kWave * j;
            buf[j] = ld_vec(tr + (vi < nv ? vi : nv - 1));
        }
#pragma unroll
        for (int j = 0; j < VPL; ++j) {
            if (lane + (int64_t)kWave * j >= nv) continue;
            float v[EPV];
            unpack<BF16>(buf[j], v);
#pragma unroll
            for (int e = 0; e < EPV; ++e) f(v[e]);
        }
    } else {
        for (int64_t e = e0 + lane; e < e1; e += kWave) f(load_x<BF16>(t, row * cols + e));
    }
}

// Per (row, segment): the exactness of the candidates over the segment's
// elements, ANDed into rowmask[row] (all candidates set beforehand).  PHASE
// 0 tests the base candidate only; PHASE 1 runs only for rows whose base
// candidate failed somewhere and tests the other four, so a row the base
// exponent recovers (the common case) costs one test per element.
template <int FMT, bool BF16, int PHASE>
__global__ __launch_bounds__(kQBlock) void recover_mask_kernel(const void* __restrict__ t, int64_t rows, int64_t cols,
                                                               int64_t segs, int vec,
                                                               const uint32_t* __restrict__ rowmax,
                                                               uint32_t* __restrict__ rowmask) {
    const int lane = threadIdx.x & (kWave - 1);
    const int64_t gw = (int64_t)blockIdx.x * kWavesPerBlock + wave_uniform(threadIdx.x / kWave);
    const int64_t row = gw / segs, seg = gw % segs;
    if (row >= rows) return;
    if (PHASE == 1 && (rowmask[row] & 1u)) return;  // the base candidate holds for the whole row
    const int base = scale_exp_from_amax<FMT>(to_f32_bits<BF16>(rowmax[row]));
    const bool fast = base - 2 >= -kFastK && base + 2 <= kFastK;
    const int64_t e0 = seg * kSegElems, e1 = min(e0 + kSegElems, cols);
    uint32_t mask = PHASE == 0 ? 0x1u : 0x1Eu;
    for_seg_elems<BF16>(t, row, cols, e0, e1, vec, lane, [&](float v) {
#pragma unroll
        for (int i = (PHASE == 0 ? 0 : 1); i < (PHASE == 0 ? 1 : 5); ++i)
            if ((mask >> i) & 1u)
                if (!exact_at<FMT, BF16>(v, base + kDeltas[i], fast)) mask &= ~(1u << i);
    });
    mask = wave_and_u32(mask);
    const uint32_t keep = PHASE == 0 ? ~0x1u : ~0x1Eu;  // the bits this phase does not test
    if (lane == 0 && (mask | keep) != 0xFFFFFFFFu) atomicAnd(rowmask + row, mask | keep);
}

// k = base + the first exact offset; a row with none counts as bad and keeps
// the last candidate, as the reference's `best` does (fp8.py:82-93).
template <int FMT, bool BF16>
__global__ void recover_final_kernel(int64_t rows, const uint32_t* __restrict__ rowmax,
                                     const uint32_t* __restrict__ rowmask, int32_t* __restrict__ k,
                                     unsigned long long* __restrict__ bad) {
    for (int64_t r = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; r < rows; r += (int64_t)gridDim.x * blockDim.x) {
        const int base = scale_exp_from_amax<FMT>(to_f32_bits<BF16>(rowmax[r]));
        const uint32_t m = rowmask[r];
        int kk = base + 2;
        if (m == 0u) {
            atomicAdd(bad, 1ull);
        } else {
            kk = base + kDeltas[__builtin_ctz(m)];
        }
        k[r] = kk;
    }
}

// q = fp8(x * 2^-k) with the caller's k per row (planes.py:110-111): the
// wire image of a tensor whose exponents recover_exp found.
template <int FMT, bool BF16>
__global__ __launch_bounds__(kQBlock) void quant_k_kernel(const void* __restrict__ x, int64_t rows, int64_t cols,
                                                          int64_t segs, int vec, const int32_t* __restrict__ kin,
                                                          uint8_t* __restrict__ q) {
    constexpr int EPV = Seg<BF16>::EPV, VPL = Seg<BF16>::VPL, ESZ = BF16 ? 2 : 4;
    const int lane = threadIdx.x & (kWave - 1);
    const int64_t gw = (int64_t)blockIdx.x * kWavesPerBlock + wave_uniform(threadIdx.x / kWave);
    const int64_t row = gw / segs, seg = gw % segs;
    if (row >= rows) return;
    const int kk = kin[row];
    const bool fast = kk >= -kFastK && kk <= kFastK;
    const float s_down = fast ? __uint_as_float((uint32_t)(127 - kk) << 23) : pow2_dtype(-kk, BF16);
    const int64_t e0 = seg * kSegElems, e1 = min(e0 + kSegElems, cols);
    const int64_t base = row * cols;
    if (vec && fast) {
        const uint4* xr = reinterpret_cast<const uint4*>(static_cast<const char*>(x) + (base + e0) * ESZ);
        const int64_t nv = (e1 - e0) / EPV;
        uint4 buf[VPL];
#pragma unroll
        for (int j = 0; j < VPL; ++j) {
            const int64_t vi = lane + (int64_t)kWave * j;
            buf[j] = ld_vec(xr + (vi < nv ? vi : nv - 1));
        }
#pragma unroll
        for (int j = 0; j < VPL; ++j) {
            const int64_t vi = lane + (int64_t)kWave * j;
            if (vi >= nv) continue;
            float f[EPV];
            unpack<BF16>(buf[j], f);
            uint32_t words[2];
#pragma unroll
            for (int h = 0; h < EPV; h += 4) {
                uint32_t w = 0;
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    // non-finite values follow the restatement (NaN, Inf codes)
                    const uint32_t c = __builtin_isfinite(f[h + e])
                                           ? cvt_pk_fp8<FMT, false>(f[h + e] * s_down, 0.0f, 0u) & 0xFFu
                                           : quant_sw<FMT, BF16>(f[h + e], s_down);
                    w |= c << (8 * e);
                }
                words[h / 4] = w;
            }
            const int64_t e = e0 + vi * EPV;
            if (BF16) st_vec2(q + base + e, make_uint2(words[0], words[1]));
            else st_u32(q + base + e, words[0]);
        }
    } else {
        for (int64_t e = e0 + lane; e < e1; e += kWave) {
            const float v = load_x<BF16>(x, base + e);
            uint32_t c;
            if (fast && __builtin_isfinite(v)) c = cvt_pk_fp8<FMT, false>(v * s_down, 0.0f, 0u) & 0xFFu;
            else c = quant_sw<FMT, BF16>(v, s_down);
            q[base + e] = (uint8_t)c;
        }
    }
}

// ---------------------------------------------- recover + image, registers

// The first exact candidate of a row outside the register test (a NaN or Inf
// in the row, or candidates outside the instruction path), element by
// element through the restatement, or -1 (the recover_mask_kernel test).
template <int FMT, bool BF16>
__device__ __forceinline__ int recover_slow_row(const void* t, int64_t row, int64_t cols, int base, int lane) {
#pragma unroll 1
    for (int i = 0; i < 5; ++i) {
        bool ok = true;
#pragma unroll 1
        for (int64_t e = lane; e < cols; e += kWave)
            ok = ok && exact_at<FMT, BF16>(load_x<BF16>(t, row * cols + e), base + kDeltas[i], false);
        if (wave_and_u32(ok ? 1u : 0u)) return i;
    }
    return -1;
}

// One candidate exponent c over a row of finite elements held in registers:
// every element's code at 2^-c (packed four to a word, as quant_vec_fast
// packs them) into `codes`, and whether every element of this lane decodes
// back to itself.
template <int FMT, bool BF16, int VPL>
__device__ __forceinline__ bool recover_candidate(const uint4 (&buf)[VPL], int c, uint32_t (&codes)[VPL][BF16 ? 2 : 1]) {
    constexpr int EPV = BF16 ? 8 : 4;
    const float s_down = __uint_as_float((uint32_t)(127 - c) << 23);
    const float s_up = __uint_as_float((uint32_t)(127 + c) << 23);
    bool ok = true;
#pragma unroll
    for (int j = 0; j < VPL; ++j) {
        float v[EPV];
        unpack<BF16>(buf[j], v);  // lanes past the end hold zeros: exact at any c
#pragma unroll
        for (int h = 0; h < EPV; h += 4) {
            uint32_t w = cvt_pk_fp8<FMT, false>(v[h] * s_down, v[h + 1] * s_down, 0u);
            w = cvt_pk_fp8<FMT, true>(v[h + 2] * s_down, v[h + 3] * s_down, w);
            codes[j][h / 4] = w;
            float b[4];
            cvt_pk_f32<FMT, false>(w, b[0], b[1]);
            cvt_pk_f32<FMT, true>(w, b[2], b[3]);
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                ok = ok & (b[e] * s_up == v[h + e]);
            }
        }
    }
    return ok;
}

// One wave per row held in registers (rows of up to kWave * VPL vectors,
// 16-byte aligned): |x|max, the base exponent, the candidates in the
// reference's order, each one wave vote over the registers (the base
// candidate is the only one a recipe round trip usually needs), then, when
// q is given, the row's wire image with the exponent found: one read of t
// and one write of q per element.  A row with no exact candidate counts as
// bad and keeps base + 2 (fp8.py:82-93), the last candidate tested, so in
// either case the codes the last test computed are the image of a row
// without NaN or Inf (the instruction equals the restatement there).
template <int FMT, bool BF16, int VPL>
__global__ __launch_bounds__(kQBlock) void recover_rows_kernel(const void* __restrict__ t, int64_t rows, int64_t cols,
                                                               int32_t* __restrict__ k, uint8_t* __restrict__ q,
                                                               unsigned long long* __restrict__ bad) {
    constexpr int EPV = BF16 ? 8 : 4;
    constexpr int ESZ = BF16 ? 2 : 4;
    // long rows leave few waves per SIMD (registers), so each wave keeps its
    // whole row in flight; short rows batch their loads
    constexpr int QB =
        (VPL >= ELY_RECOVER_WHOLE_VPL || ELY_RECOVER_BATCH <= 0 || ELY_RECOVER_BATCH > VPL) ? VPL : ELY_RECOVER_BATCH;
    const int lane = threadIdx.x & (kWave - 1);
    const int64_t row = (int64_t)blockIdx.x * kWavesPerBlock + wave_uniform(threadIdx.x / kWave);
    if (row >= rows) return;  // whole waves leave; the kernel has no block barrier
    const int64_t nvec = cols / EPV;
    const uint4* tr = reinterpret_cast<const uint4*>(static_cast<const char*>(t) + row * cols * ESZ);
    uint4 buf[VPL];
    uint32_t amax = 0;
#pragma unroll
    for (int j0 = 0; j0 < VPL; j0 += QB) {
#pragma unroll
        for (int j = j0; j < j0 + QB && j < VPL; ++j) {
            const int64_t vi = lane + (int64_t)kWave * j;
            buf[j] = ld_vec(tr + (vi < nvec ? vi : nvec - 1));
        }
#pragma unroll
        for (int j = j0; j < j0 + QB && j < VPL; ++j) {
            const int64_t vi = lane + (int64_t)kWave * j;
            if (vi >= nvec) buf[j] = make_uint4(0u, 0u, 0u, 0u);
            amax = vec_absmax<BF16>(buf[j], amax);
        }
        if (QB < VPL) __builtin_amdgcn_sched_barrier(0);
    }
    amax = wave_max_u32(amax);
    const uint32_t amax_bits = to_f32_bits<BF16>(amax);
    const bool finite_row = amax_bits < 0x7F800000u;  // NaN bits sort above Inf's
    const int base = scale_exp_from_amax<FMT>(amax_bits);
    int chosen = -1;
    bool have_codes = false;
    uint32_t codes[VPL][BF16 ? 2 : 1];
    if (finite_row && base - 2 >= -kFastK && base + 2 <= kFastK) {
#pragma unroll 1
        for (int i = 0; i < 5; ++i) {
            if (wave_and_u32(recover_candidate<FMT, BF16, VPL>(buf, base + kDeltas[i], codes) ? 1u : 0u)) {
                chosen = i;
                break;
            }
        }
        have_codes = VPL <= kRecoverKeepVpl;  // a compile-time false drops the codes
    } else {
        // rows holding NaN or Inf, or outside the instruction's exponent range
        chosen = recover_slow_row<FMT, BF16>(t, row, cols, base, lane);
    }
    const int kk = chosen >= 0 ? base + kDeltas[chosen] : base + 2;
    if (lane == 0) {
        k[row] = kk;
        if (chosen < 0) atomicAdd(bad, 1ull);
    }
    if (!q) return;
    // the image with the exponent found, as quant_k_kernel writes it
    uint8_t* qr = q + row * cols;
    if (have_codes) {
#pragma unroll
        for (int j = 0; j < VPL; ++j) {
            const int64_t vi = lane + (int64_t)kWave * j;
            if (vi >= nvec) continue;
            if (BF16) st_vec2(qr + vi * EPV, make_uint2(codes[j][0], codes[j][BF16 ? 1 : 0]));
            else st_u32(qr + vi * EPV, codes[j][0]);
        }
    } else if (kk >= -kFastK && kk <= kFastK) {
        const float s_down = __uint_as_float((uint32_t)(127 - kk) << 23);
#pragma unroll
        for (int j = 0; j < VPL; ++j) {
            const int64_t vi = lane + (int64_t)kWave * j;
            if (vi >= nvec) continue;
            float f[EPV];
            unpack<BF16>(buf[j], f);
            uint32_t words[2];
#pragma unroll
            for (int h = 0; h < EPV; h += 4) {
                uint32_t w = 0;
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    const uint32_t c = __builtin_isfinite(f[h + e])
                                           ? cvt_pk_fp8<FMT, false>(f[h + e] * s_down, 0.0f, 0u) & 0xFFu
                                           : quant_sw<FMT, BF16>(f[h + e], s_down);
                    w |= c << (8 * e);
                }
                words[h / 4] = w;
            }
            if (BF16) st_vec2(qr + vi * EPV, make_uint2(words[0], words[1]));
            else st_u32(qr + vi * EPV, words[0]);
        }
    } else {
        const float s_down = pow2_dtype(-kk, BF16);
#pragma unroll 1
        for (int64_t e = lane; e < cols; e += kWave) qr[e] = (uint8_t)quant_sw<FMT, BF16>(load_x<BF16>(t, row * cols + e), s_down);
    }
}

// --------------------------------------------------------------- self-test

template <int FMT>
__global__ void selftest_cvt_kernel(uint32_t start, uint64_t count, unsigned long long* mism) {
    using F = Fp8Fmt<FMT>;
    for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < count;
         i += (uint64_t)gridDim.x * blockDim.x) {
        const uint32_t u = (uint32_t)(start + i);
        const float x = __uint_as_float(u);
        const uint32_t sw = fp8_from_f32_sw<FMT>(x);
        const uint32_t lo = cvt_pk_fp8<FMT, false>(x, 0.0f, 0u);
        const uint32_t hi = cvt_pk_fp8<FMT, true>(0.0f, x, 0u);
        const uint32_t hw0 = lo & 0xFFu, hw1 = (hi >> 24) & 0xFFu;
        const bool domain = (u & 0x7FFFFFFFu) <= F::kMaxFiniteBits;
        if (hw0 != sw || hw1 != sw) atomicAdd(mism + (domain ? 0 : 1), 1ull);
        if (u - start < 256u && start == 0u) {
            // decode: every code, instruction vs restatement, both halves of the word
            const uint32_t c = u;
            float a, b, c2, d;
            cvt_pk_f32<FMT, false>(c | (c << 8), a, b);
            cvt_pk_f32<FMT, true>((c << 16) | (c << 24), c2, d);
            const float ref = fp8_to_f32_sw<FMT>(c);
            const float got[4] = {a, b, c2, d};
            bool bad = false;
            for (int j = 0; j < 4; ++j) {
                if (ref != ref) bad |= got[j] == got[j];
                else bad |= __float_as_uint(got[j]) != __float_as_uint(ref);
            }
            if (bad) atomicAdd(mism + 2, 1ull);
        }
    }
}

// One thread per (bf16 pattern u, k), |k| <= kFastK.  Quantize: u and its
// negation in the two halves of a word, converted at scale 2^k into both
// halves of the output, against the restatement quant_sw at 2^-k, over the
// pairs the instruction path meets (finite, |x| 2^-k < 2^ebias) -> mism[0].
// Decode (u < 256, the code): the code in all four bytes, both halves
// decoded at 2^k, against dequant_sw rounded to bf16, NaN codes aside (the
// kernels keep them off the scaled decode) -> mism[1].
template <int FMT>
__global__ void selftest_scaled_kernel(unsigned long long* mism) {
    const uint32_t t = blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= 65536u * (2u * kFastK + 1u)) return;
    const uint32_t u = t & 0xFFFFu;
    const int k = (int)(t >> 16) - kFastK;
    const float s_down = __uint_as_float((uint32_t)(127 - k) << 23);
    const float s_up = __uint_as_float((uint32_t)(127 + k) << 23);
    const float x = bf16_to_f32(u);
    const float lim = __uint_as_float((uint32_t)(127 + Fp8Fmt<FMT>::EBIAS) << 23);
    if ((u & 0x7F80u) != 0x7F80u && __builtin_fabsf(x * s_down) < lim) {
        const uint32_t w = u | ((u ^ 0x8000u) << 16);
        const uint32_t want = quant_sw<FMT, true>(x, s_down), want_neg = quant_sw<FMT, true>(-x, s_down);
        const uint32_t lo = cvt_scaled_pk_fp8_bf16<FMT, false>(w, s_up, 0u);
        const uint32_t hi = cvt_scaled_pk_fp8_bf16<FMT, true>(w, s_up, 0u);
        if ((lo & 0xFFu) != want || ((lo >> 8) & 0xFFu) != want_neg || ((hi >> 16) & 0xFFu) != want ||
            (hi >> 24) != want_neg)
            atomicAdd(mism, 1ull);
    }
    if (u < 256u && (nan_code_bits<FMT>(u) == 0u)) {
        const uint32_t want = f32_to_bf16(dequant_sw<FMT, true>(u, s_up));
        const uint32_t w = u * 0x01010101u;
        const uint32_t lo = cvt_scaled_pk_bf16<FMT, false>(w, s_up), hi = cvt_scaled_pk_bf16<FMT, true>(w, s_up);
        if (lo != (want | (want << 16)) || hi != (want | (want << 16))) atomicAdd(mism + 1, 1ull);
    }
}

__global__ void selftest_sqrt_kernel(uint32_t start, uint64_t count, unsigned long long* mism) {
    for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < count;
         i += (uint64_t)gridDim.x * blockDim.x) {
        const uint32_t u = (uint32_t)(start + i) & 0x7FFFFFFFu;  // non-negative patterns
        const float x = __uint_as_float(u);
        const float a = __builtin_sqrtf(x);
        const float b = (float)__builtin_sqrt((double)x);
        if (__float_as_uint(a) != __float_as_uint(b) && !(a != a && b != b)) atomicAdd(mism, 1ull);
    }
}

// ------------------------------------------------------------------ launch

static void check_fmt(int32_t fmt) {
    if (fmt != ELY_E4M3 && fmt != ELY_E5M2) fail(ELY_EINVAL, "fp8 format must be ELY_E4M3 or ELY_E5M2");
}

static void check_dtype(int32_t dt, const char* what) {
    if (dt != ELY_F32 && dt != ELY_BF16) fail(ELY_EINVAL, std::string(what) + " must be ELY_F32 or ELY_BF16");
}

static void check_shape(int64_t rows, int64_t cols) {
    if (rows < 0 || cols < 0) fail(ELY_EINVAL, "negative rows or cols");
    if (cols > 0 && rows > INT64_MAX / cols) fail(ELY_EINVAL, "rows * cols overflows");
}

static unsigned blocks_for_waves(int64_t waves) {
    const int64_t b = (waves + kWavesPerBlock - 1) / kWavesPerBlock;
    // a dispatch counts its work-items in 32 bits
    if (b > 0xFFFFFFFFLL / kQBlock) fail(ELY_EINVAL, "grid too large: more than 2^32 - 1 threads in one launch");
    return (unsigned)b;
}

// The register paths, by a row's vectors in units of one per lane of a wave
// (rows_units): a wave per row up to kMaxWaveVpl units, a block per row above,
// of as many waves as keep at most 4 vectors per lane in each: 4 waves to 16
// units, 8 to 32, 16 to kMaxRowUnits (32,768 bf16 or 16,384 fp32 columns).
// Against the split path, which reads x twice in two launches (from graphs,
// buffers in turn): [4096, 6144] fp32 quantizes in 21.8 us against 37.6 (5.8
// against 3.3 TB/s), [4096, 20480] bf16 in 41.6 against 66.4, [2048, 16384]
// fp32 in 28.5 against 50.6, [2048, 32768] bf16 in 33.7 against 55.3, 64 rows
// of 32,768 bf16 in 4.4 against 6.9, and one in 3.3 against 4.9.
constexpr int kMaxWaveVpl = 6;
constexpr int kMaxRowUnits = 64;
// Longer rows than this, and rows that are not whole aligned vectors, are
// called with the split path's workspace, whether it is used or not: callers
// size it by ely_fp8_workspace_bytes for every shape, and what was refused
// without it when these rows took the split path still is.
constexpr int kNoWorkspaceUnits = 16;

template <int FMT, bool BF16, int VPL>
static void launch_rows(const void* x, int64_t rows, int64_t cols, uint8_t* q, int32_t* k, void* out, hipStream_t s) {
    hipLaunchKernelGGL((quant_rows_kernel<FMT, BF16, VPL>), dim3(blocks_for_waves(rows)), dim3(kQBlock), ELY_Q_LDS, s, x,
                       rows, cols, q, k, out);
    check_launch("quant_rows_kernel");
}

template <int FMT, bool BF16>
static void dispatch_rows(int vpl, const void* x, int64_t rows, int64_t cols, uint8_t* q, int32_t* k, void* out,
                          hipStream_t s) {
    switch (vpl) {
        case 1: return launch_rows<FMT, BF16, 1>(x, rows, cols, q, k, out, s);
        case 2: return launch_rows<FMT, BF16, 2>(x, rows, cols, q, k, out, s);
        case 3: return launch_rows<FMT, BF16, 3>(x, rows, cols, q, k, out, s);
        case 4: return launch_rows<FMT, BF16, 4>(x, rows, cols, q, k, out, s);
        case 5: return launch_rows<FMT, BF16, 5>(x, rows, cols, q, k, out, s);
        case 6: return launch_rows<FMT, BF16, 6>(x, rows, cols, q, k, out, s);
        default: fail(ELY_EINVAL, "internal: no register path for this row length");
    }
}

// Whether these rows are whole 16-byte vectors at aligned addresses.
static bool whole_vecs(int64_t cols, int32_t dtype, const void* x, const uint8_t* q, const void* out) {
    const int64_t epv = dtype == ELY_BF16 ? 8 : 4;
    return cols % epv == 0 && aligned16(x) && (!out || aligned16(out)) &&
           (!q || reinterpret_cast<uintptr_t>(q) % (uintptr_t)epv == 0);
}

// Whether these rows take the vector paths: at least one vector, at any
// element's alignment.
static bool any_vecs(int64_t cols, int32_t dtype, const void* x, const void* out) {
    const int64_t epv = dtype == ELY_BF16 ? 8 : 4, esz = dtype == ELY_BF16 ? 2 : 4;
    return cols >= epv && reinterpret_cast<uintptr_t>(x) % esz == 0 && reinterpret_cast<uintptr_t>(out) % esz == 0;
}

// A row's vectors in units of one per lane of a wave (kWave vectors), for
// rows that the register paths take; 0 for the others.
static int rows_units(int64_t cols, int32_t dtype, const void* x, const void* out) {
    const int64_t per = (dtype == ELY_BF16 ? 8 : 4) * kWave;
    if (!any_vecs(cols, dtype, x, out)) return 0;
    return cols <= per * kMaxRowUnits ? (int)((cols + per - 1) / per) : 0;
}

// The shapes whose calls carry the split path's workspace.
static bool wants_workspace(int64_t cols, int32_t dtype, const void* x, const uint8_t* q, const void* out) {
    const int units = rows_units(cols, dtype, x, out);
    return !whole_vecs(cols, dtype, x, q, out) || units == 0 || units > kNoWorkspaceUnits;
}

template <int FMT, bool BF16, int W>
static void launch_block_row(int units, const void* x, int64_t rows, int64_t cols, uint8_t* q, int32_t* k, void* out,
                             hipStream_t s) {
    const dim3 g((unsigned)rows), b(W * kWave);
    switch ((units + W - 1) / W) {
        case 2: hipLaunchKernelGGL((quant_block_row_kernel<FMT, BF16, W, 2>), g, b, 0, s, x, cols, q, k, out); break;
        case 3: hipLaunchKernelGGL((quant_block_row_kernel<FMT, BF16, W, 3>), g, b, 0, s, x, cols, q, k, out); break;
        case 4: hipLaunchKernelGGL((quant_block_row_kernel<FMT, BF16, W, 4>), g, b, 0, s, x, cols, q, k, out); break;
        default: fail(ELY_EINVAL, "internal: no block-row path for this row length");
    }
    check_launch("quant_block_row_kernel");
}

// Row maxima, then the partial maxima (at most max(rows, kSplitWaves) of them).
static size_t rowmax_bytes(int64_t rows) { return align_up((size_t)std::max<int64_t>(rows, 1) * 4, 256); }
static size_t split_ws_bytes(int64_t rows) {
    return rowmax_bytes(rows) + align_up((size_t)std::max<int64_t>(rows, kSplitWaves) * 4, 256);
}

// partial[r * shape.blocks + j]: the partial |x|max bits of row r, from the
// split path's first launch.
template <bool BF16>
static SplitShape split_partials(const void* x, int64_t rows, int64_t cols, int vec, uint32_t* partial, hipStream_t s) {
    const int64_t segs = (cols + kSegElems - 1) / kSegElems;
    const SplitShape sh = split_shape(rows, segs);
    if (rows > INT64_MAX / (sh.blocks * sh.waves)) fail(ELY_EINVAL, "too many rows");
    const int64_t blocks = rows * sh.blocks;
    // a dispatch counts its work-items in 32 bits
    if (blocks > 0xFFFFFFFFLL / (sh.waves * kWave)) fail(ELY_EINVAL, "grid too large: more than 2^32 - 1 threads in one launch");
    const int64_t seg_bytes = kSegElems * (BF16 ? 2 : 4);
    const int64_t cached = std::min<int64_t>(segs, ((int64_t)ELY_SPLIT_CACHED_MB << 20) / (seg_bytes * rows));
    if (sh.waves == 1)
        hipLaunchKernelGGL((rowmax_partial_kernel<BF16, 1>), dim3((unsigned)blocks), dim3(kWave), 0, s, x, cols, segs,
                           sh.blocks, vec, cached, partial);
    else
        hipLaunchKernelGGL((rowmax_partial_kernel<BF16, kSplitBlockWaves>), dim3((unsigned)blocks),
                           dim3(kSplitBlockWaves * kWave), 0, s, x, cols, segs, sh.blocks, vec, cached, partial);
    check_launch("rowmax_partial_kernel");
    return sh;
}

// rowmax[r] = |x|max bits of row r, through the split path's first launch and
// a fold of its partials.
template <bool BF16>
static void split_rowmax(const void* x, int64_t rows, int64_t cols, int vec, void* workspace, uint32_t* rowmax,
                         hipStream_t s) {
    const bool one = split_shape(rows, (cols + kSegElems - 1) / kSegElems).blocks == 1;
    uint32_t* partial = one ? rowmax : reinterpret_cast<uint32_t*>(static_cast<char*>(workspace) + rowmax_bytes(rows));
    const SplitShape sh = split_partials<BF16>(x, rows, cols, vec, partial, s);
    if (!one) {
        hipLaunchKernelGGL(rowmax_reduce_kernel, dim3((unsigned)std::min<int64_t>(rows, 65536)), dim3(kWave), 0, s,
                           (const uint32_t*)partial, rows, sh.blocks, rowmax);
        check_launch("rowmax_reduce_kernel");
    }
}

static size_t guess_ws_bytes(int64_t n);
template <int FMT, bool BF16>
static void quantize_guess_impl(const void* x, int64_t n, uint8_t* q, int32_t* k, void* out, void* workspace,
                                int64_t ws_bytes, hipStream_t s);

template <int FMT, bool BF16>
static void quantize_impl(const void* x, int64_t rows, int64_t cols, uint8_t* q, int32_t* k, void* out,
                          void* workspace, int64_t ws_bytes, hipStream_t s, bool allow_guess = true) {
    if (rows == 0) return;
    if (cols == 0) {
        // an empty row has |x|max 0, so k = 0 (fp8.py:38)
        if (k) {
            hipLaunchKernelGGL(fill_u32_kernel, dim3((unsigned)std::min<int64_t>((rows + 255) / 256, 4096)), dim3(256),
                               0, s, reinterpret_cast<uint32_t*>(k), rows, 0u);
            check_launch("fill_u32_kernel");
        }
        return;
    }
    const int32_t dt = BF16 ? ELY_BF16 : ELY_F32;
    const int vec = any_vecs(cols, dt, x, out);
    const bool want_ws = wants_workspace(cols, dt, x, q, out);
    const bool guess = want_ws && allow_guess && rows == 1 && (q || out) && vec &&
                       cols >= ((int64_t)ELY_GUESS_MIN_MB << 20) / (BF16 ? 2 : 4) && workspace &&
                       ws_bytes >= (int64_t)guess_ws_bytes(cols);
    if (want_ws && !guess && (!workspace || ws_bytes < (int64_t)split_ws_bytes(rows)))
        fail(ELY_EWORKSPACE, "fp8 quantize: this shape needs " + std::to_string(split_ws_bytes(rows)) +
                                 " workspace bytes (ely_fp8_workspace_bytes)");
    int units = rows_units(cols, dt, x, out);
    if (units > kMaxWaveVpl) {
        // one block per row; a dispatch counts its threads in 32 bits, and
        // the split path's waves take more rows than that
        const int waves = units <= 16 ? 4 : units <= 32 ? 8 : 16;
        const bool fits = rows <= 0xFFFFFFFFLL / (waves * kWave);
        if (!fits && !want_ws) fail(ELY_EINVAL, "fp8 quantize: too many rows for one launch");
        if (fits)
            return waves == 4 ? launch_block_row<FMT, BF16, 4>(units, x, rows, cols, q, k, out, s)
                   : waves == 8 ? launch_block_row<FMT, BF16, 8>(units, x, rows, cols, q, k, out, s)
                                : launch_block_row<FMT, BF16, 16>(units, x, rows, cols, q, k, out, s);
    } else if (units) {
        return dispatch_rows<FMT, BF16>(units, x, rows, cols, q, k, out, s);
    }
    if (guess) return quantize_guess_impl<FMT, BF16>(x, cols, q, k, out, workspace, ws_bytes, s);
    uint32_t* partial = static_cast<uint32_t*>(workspace);
    const int64_t segs = (cols + kSegElems - 1) / kSegElems;
    if (rows > INT64_MAX / segs) fail(ELY_EINVAL, "too many segments");
    const unsigned blocks = blocks_for_waves(rows * segs);
    const SplitShape sh = split_partials<BF16>(x, rows, cols, vec, partial, s);
    hipLaunchKernelGGL((quant_split_kernel<FMT, BF16>), dim3(blocks), dim3(kQBlock), 0, s, x, rows, cols, segs, vec,
                       (const uint32_t*)partial, sh.blocks, q, k, out);
    check_launch("quant_split_kernel");
}

// Workspace of the hint path over n elements: one maximum per segment, the
// reduce launch's kHintBlocks maxima, the hint as read; at least the split
// path's, which a call falls back to when the one-pass form does not apply.
static size_t hint_ws_bytes(int64_t n) {
    const int64_t segs = std::max<int64_t>((n + kSegElems - 1) / kSegElems, 1);
    return std::max(align_up((size_t)segs * 4, 256) + align_up((size_t)kHintBlocks * 4, 256) + 256, split_ws_bytes(1));
}

template <int FMT, bool BF16>
static void quantize_hint_impl(const void* x, int64_t n, int32_t k_hint, const int32_t* k_hint_dev, uint8_t* q,
                               int32_t* k, void* out, int32_t* hit, void* workspace, int64_t ws_bytes,
                               hipStream_t s) {
    if (!workspace || ws_bytes < (int64_t)hint_ws_bytes(n))
        fail(ELY_EWORKSPACE, "ely_fp8_quantize_hint: workspace of " + std::to_string(ws_bytes) + " bytes, need " +
                                 std::to_string(hint_ws_bytes(n)) + " (ely_fp8_hint_workspace_bytes)");
    // the one-pass form keeps to whole aligned vectors (*hit says so)
    const bool vec = n > 0 && whole_vecs(n, BF16 ? ELY_BF16 : ELY_F32, x, q, out);
    if (!vec || (!k_hint_dev && (k_hint < -kFastK || k_hint > kFastK))) {
        // no one-pass form for this tensor or hint: the split path, a miss
        quantize_impl<FMT, BF16>(x, 1, n, q, k, out, workspace, ws_bytes, s, false);
        if (hit) {
            hipLaunchKernelGGL(fill_u32_kernel, dim3(1), dim3(64), 0, s, reinterpret_cast<uint32_t*>(hit), (int64_t)1, 0u);
            check_launch("fill_u32_kernel");
        }
        return;
    }
    const int64_t segs = (n + kSegElems - 1) / kSegElems;
    uint32_t* partial = static_cast<uint32_t*>(workspace);
    uint32_t* block_max = reinterpret_cast<uint32_t*>(static_cast<char*>(workspace) + align_up((size_t)segs * 4, 256));
    int32_t* hint_copy = reinterpret_cast<int32_t*>(reinterpret_cast<char*>(block_max) + align_up((size_t)kHintBlocks * 4, 256));
    hipLaunchKernelGGL((quant_hint_kernel<FMT, BF16>), dim3(blocks_for_waves(segs)), dim3(kQBlock), 0, s, x, n, segs,
                       k_hint, k_hint_dev, q, out, partial, hint_copy);
    check_launch("quant_hint_kernel");
    hipLaunchKernelGGL(hint_reduce_kernel, dim3(kHintBlocks), dim3(kRowBlock), 0, s, (const uint32_t*)partial, segs,
                       block_max);
    check_launch("hint_reduce_kernel");
    const int64_t waves = std::min<int64_t>(segs, (int64_t)device_info().cus * kHintFixupWavesPerCU);
    hipLaunchKernelGGL((quant_hint_fixup_kernel<FMT, BF16>), dim3(blocks_for_waves(waves)), dim3(kQBlock), 0, s, x, n,
                       segs, (const int32_t*)hint_copy, (const uint32_t*)block_max, q, k, out, hit);
    check_launch("quant_hint_fixup_kernel");
}

// Per-tensor rows of at least ELY_GUESS_MIN_MB MiB (the vector form, a
// workspace of guess_ws_bytes): the exponent is guessed from every
// kGuessStride-th segment's |x|max, and the row is converted at that guess:
// one read of x when the sample holds the row's maximum binade, the fixup (a
// second read and write) when it does not.  Either way the codes and k are
// the split path's, byte for byte.
static size_t guess_ws_bytes(int64_t n) { return hint_ws_bytes(n) + 256; }
static_assert(((int64_t)ELY_GUESS_MIN_MB << 20) / 4 / kSegElems >= kGuessBlocks + kTops * kTopStride,
              "the shortest guessed row's workspace holds the sampled words and the tops");

template <int FMT, bool BF16>
static void quantize_guess_impl(const void* x, int64_t n, uint8_t* q, int32_t* k, void* out, void* workspace,
                                int64_t ws_bytes, hipStream_t s) {
    // after the hint path's layout: the sampled |x|max, and k's word when
    // the caller asked for no k (a round trip); the sampled words and the tops
    // take the first bytes of what the hint path keeps its maxima in
    uint32_t* amax = reinterpret_cast<uint32_t*>(static_cast<char*>(workspace) + hint_ws_bytes(n));
    int32_t* kword = k ? k : reinterpret_cast<int32_t*>(amax + 1);
    uint32_t* sampled = static_cast<uint32_t*>(workspace);
    uint32_t* tops = sampled + kGuessBlocks;
    const int64_t segs = (n + kSegElems - 1) / kSegElems;
    const int64_t samples = (segs + kGuessStride - 1) / kGuessStride;
    hipLaunchKernelGGL((guess_amax_kernel<BF16>), dim3(kGuessBlocks), dim3(kGuessBlockWaves * kWave), 0, s, x, n,
                       (int64_t)kGuessStride, samples, sampled, tops);
    check_launch("guess_amax_kernel");
    hipLaunchKernelGGL((quant_guess_kernel<FMT, BF16>), dim3(blocks_for_waves(segs)), dim3(kQBlock), 0, s, x, n, segs,
                       (const uint32_t*)sampled, q, out, tops, amax);
    check_launch("quant_guess_kernel");
    const int64_t waves = std::min<int64_t>(segs, (int64_t)device_info().cus * kHintFixupWavesPerCU);
    hipLaunchKernelGGL((quant_guess_fixup_kernel<FMT, BF16>), dim3(blocks_for_waves(waves)), dim3(kQBlock), 0, s, x, n,
                       segs, (const uint32_t*)tops, (const uint32_t*)amax, q, kword, out);
    check_launch("quant_guess_fixup_kernel");
}

template <int FMT, bool BF16OUT, bool RAGGED>
static void launch_dequant_flat(const uint8_t* q, const int32_t* k, int64_t n, int64_t cols, void* out, hipStream_t s) {
    const unsigned blocks = blocks_for_waves((n + kDeqSegCodes - 1) / kDeqSegCodes);
    if (n < ((int64_t)1 << 32))
        hipLaunchKernelGGL((dequant_flat_kernel<FMT, BF16OUT, true, RAGGED>), dim3(blocks), dim3(kQBlock), ELY_DEQ_LDS, s, q,
                           k, n, cols, out);
    else
        hipLaunchKernelGGL((dequant_flat_kernel<FMT, BF16OUT, false, RAGGED>), dim3(blocks), dim3(kQBlock), ELY_DEQ_LDS, s, q,
                           k, n, cols, out);
    check_launch("dequant_flat_kernel");
}

template <int FMT, bool BF16OUT>
static void dequantize_impl(const uint8_t* q, const int32_t* k, int64_t rows, int64_t cols, void* out,
                            hipStream_t s) {
    if (rows == 0 || cols == 0) return;
    const int64_t n = rows * cols;
    if ((cols % 16 == 0) && aligned16(q) && aligned16(out))
        return launch_dequant_flat<FMT, BF16OUT, false>(q, k, n, cols, out, s);
    const int64_t segs = (cols + kDeqSegCodes - 1) / kDeqSegCodes;
    if (rows > INT64_MAX / segs) fail(ELY_EINVAL, "too many segments");
    // past the element-wise kernel's grid these rows stay refused, whichever kernel takes them
    const unsigned any_blocks = blocks_for_waves(rows * segs);
    // Few narrow rows to fp32: the element-wise kernel's wave a row is done
    // sooner than the flat one's (124 rows of 33 codes 2.35 us against 2.96, 512
    // of 8 2.34 against 2.98, 64 of 255 2.74 against 2.95); from 4,096 waves, and
    // in less than a wave's codes twice over, the flat kernel is ahead.
    const bool few = !BF16OUT && rows <= 2048 && cols <= 4 * kWave && n > 8 * kWave;
    // rows of at least a vector (a vector then meets at most two rows)
    if (cols >= 8 && !few && reinterpret_cast<uintptr_t>(out) % (BF16OUT ? 2 : 4) == 0)
        return launch_dequant_flat<FMT, BF16OUT, true>(q, k, n, cols, out, s);
    hipLaunchKernelGGL((dequant_any_kernel<FMT, BF16OUT>), dim3(any_blocks), dim3(kQBlock), 0, s, q, k, rows, cols, segs,
                       out);
    check_launch("dequant_any_kernel");
}

// Register path of recover_exp / recover_image: vectors per lane (2, 4, 5,
// 6, 8 or 16) for rows of `cols` elements, or 0 when the row does not fit it.
static int recover_vpl(int64_t cols, bool bf16, const void* t, const uint8_t* q) {
    const int64_t epv = bf16 ? 8 : 4;
    if (cols == 0 || cols % epv != 0 || !aligned16(t)) return 0;
    if (q && reinterpret_cast<uintptr_t>(q) % (uintptr_t)epv != 0) return 0;
    const int64_t nvec = cols / epv;
    for (int v : {2, 4, 5, 6, 8, 16})
        if (nvec <= (int64_t)kWave * v) return v;
    return 0;
}

template <int FMT, bool BF16>
static void launch_recover_rows(int vpl, const void* t, int64_t rows, int64_t cols, int32_t* k, uint8_t* q,
                                unsigned long long* bad, hipStream_t s) {
    const dim3 g(blocks_for_waves(rows)), b(kQBlock);
    switch (vpl) {
        case 2: hipLaunchKernelGGL((recover_rows_kernel<FMT, BF16, 2>), g, b, 0, s, t, rows, cols, k, q, bad); break;
        case 4: hipLaunchKernelGGL((recover_rows_kernel<FMT, BF16, 4>), g, b, 0, s, t, rows, cols, k, q, bad); break;
        case 5: hipLaunchKernelGGL((recover_rows_kernel<FMT, BF16, 5>), g, b, 0, s, t, rows, cols, k, q, bad); break;
        case 6: hipLaunchKernelGGL((recover_rows_kernel<FMT, BF16, 6>), g, b, 0, s, t, rows, cols, k, q, bad); break;
        case 8: hipLaunchKernelGGL((recover_rows_kernel<FMT, BF16, 8>), g, b, 0, s, t, rows, cols, k, q, bad); break;
        case 16: hipLaunchKernelGGL((recover_rows_kernel<FMT, BF16, 16>), g, b, 0, s, t, rows, cols, k, q, bad); break;
        default: fail(ELY_EINVAL, "internal: no register path for this row length");
    }
    check_launch("recover_rows_kernel");
}

static void recover_rows(int vpl, const void* t, bool bf16, int64_t rows, int64_t cols, int32_t fmt, int32_t* k,
                         uint8_t* q, unsigned long long* bad, hipStream_t s) {
    if (fmt == ELY_E4M3) {
        if (bf16) launch_recover_rows<kE4M3, true>(vpl, t, rows, cols, k, q, bad, s);
        else launch_recover_rows<kE4M3, false>(vpl, t, rows, cols, k, q, bad, s);
    } else {
        if (bf16) launch_recover_rows<kE5M2, true>(vpl, t, rows, cols, k, q, bad, s);
        else launch_recover_rows<kE5M2, false>(vpl, t, rows, cols, k, q, bad, s);
    }
}

// The multi-launch recovery for any shape: row maxima, the candidates'
// exactness per segment, then k per row.
static void recover_multi(const void* t, bool bf16, int64_t rows, int64_t cols, int32_t fmt, int32_t* k,
                          unsigned long long* bad_rows_dev, void* workspace, hipStream_t s) {
    uint32_t* rowmax = static_cast<uint32_t*>(workspace);
    uint32_t* rowmask = reinterpret_cast<uint32_t*>(static_cast<char*>(workspace) + split_ws_bytes(rows));
    const unsigned fb = (unsigned)std::min<int64_t>((rows + 255) / 256, 4096);
    hipLaunchKernelGGL(fill_u32_kernel, dim3(fb), dim3(256), 0, s, rowmask, rows, 0x1Fu);
    check_launch("fill_u32_kernel");
    if (cols == 0) {
        hipLaunchKernelGGL(fill_u32_kernel, dim3(fb), dim3(256), 0, s, rowmax, rows, 0u);
        check_launch("fill_u32_kernel");
    } else {
        const int64_t segs = (cols + kSegElems - 1) / kSegElems;
        if (rows > INT64_MAX / segs) fail(ELY_EINVAL, "too many segments");
        const unsigned blocks = blocks_for_waves(rows * segs);
        const int vec = (cols % (bf16 ? 8 : 4) == 0) && aligned16(t);
        if (bf16) split_rowmax<true>(t, rows, cols, vec, workspace, rowmax, s);
        else split_rowmax<false>(t, rows, cols, vec, workspace, rowmax, s);
#define ELY_RECOVER_MASK(F, B)                                                                                    \
    do {                                                                                                          \
        hipLaunchKernelGGL((recover_mask_kernel<F, B, 0>), dim3(blocks), dim3(kQBlock), 0, s, t, rows, cols, segs, \
                           vec, (const uint32_t*)rowmax, rowmask);                                                \
        hipLaunchKernelGGL((recover_mask_kernel<F, B, 1>), dim3(blocks), dim3(kQBlock), 0, s, t, rows, cols, segs, \
                           vec, (const uint32_t*)rowmax, rowmask);                                                \
    } while (0)
        if (fmt == ELY_E4M3) {
            if (bf16) ELY_RECOVER_MASK(kE4M3, true);
            else ELY_RECOVER_MASK(kE4M3, false);
        } else {
            if (bf16) ELY_RECOVER_MASK(kE5M2, true);
            else ELY_RECOVER_MASK(kE5M2, false);
        }
#undef ELY_RECOVER_MASK
        check_launch("recover_mask_kernel");
    }
#define ELY_RECOVER_FINAL(F, B)                                                                                   \
    hipLaunchKernelGGL((recover_final_kernel<F, B>), dim3(fb), dim3(256), 0, s, rows, (const uint32_t*)rowmax,      \
                       (const uint32_t*)rowmask, k, bad_rows_dev)
    if (fmt == ELY_E4M3) {
        if (bf16) ELY_RECOVER_FINAL(kE4M3, true);
        else ELY_RECOVER_FINAL(kE4M3, false);
    } else {
        if (bf16) ELY_RECOVER_FINAL(kE5M2, true);
        else ELY_RECOVER_FINAL(kE5M2, false);
    }
#undef ELY_RECOVER_FINAL
    check_launch("recover_final_kernel");
}

static void quant_k_launch(const void* x, bool bf16, int64_t rows, int64_t cols, int32_t fmt, const int32_t* k,
                           uint8_t* q, hipStream_t s) {
    const int64_t segs = (cols + kSegElems - 1) / kSegElems;
    if (rows > INT64_MAX / segs) fail(ELY_EINVAL, "too many segments");
    const unsigned blocks = blocks_for_waves(rows * segs);
    const int vec = (cols % (bf16 ? 8 : 4) == 0) && aligned16(x) &&
                    (reinterpret_cast<uintptr_t>(q) % (bf16 ? 8 : 4) == 0);
#define ELY_QK(F, B) \
    hipLaunchKernelGGL((quant_k_kernel<F, B>), dim3(blocks), dim3(kQBlock), 0, s, x, rows, cols, segs, vec, k, q)
    if (fmt == ELY_E4M3) {
        if (bf16) ELY_QK(kE4M3, true);
        else ELY_QK(kE4M3, false);
    } else {
        if (bf16) ELY_QK(kE5M2, true);
        else ELY_QK(kE5M2, false);
    }
#undef ELY_QK
    check_launch("quant_k_kernel");
}

// ------------------------------------------------ quantize without allocation

// Scratch of ely_fp8_quantize_noalloc: the split path's row maxima and
// partial maxima live in this file-scope device array instead of a caller
// workspace, so that entry point allocates nothing.  Each GPU holds its own
// copy at its own address until the process ends; host code reaches it only
// through the address hipGetSymbolAddress returns on that device (the
// array's name in host code is a stand-in, not a device address).
constexpr size_t kNoallocScratchBytes = (size_t)1 << 20;
static __device__ __align__(256) unsigned char scratch[kNoallocScratchBytes];

static std::mutex g_scratch_mu;
static std::map<int, void*> g_scratch_ptr;  // device -> address of `scratch` there

// The current device's address of `scratch`, looked up once per device with
// that device current.
static void* noalloc_scratch() {
    int dev = 0;
    check_hip(hipGetDevice(&dev), "hipGetDevice");
    std::lock_guard<std::mutex> lk(g_scratch_mu);
    auto it = g_scratch_ptr.find(dev);
    if (it != g_scratch_ptr.end()) return it->second;
    void* ptr = nullptr;
    check_hip(hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch)), "hipGetSymbolAddress(scratch)");
    if (!ptr) fail(ELY_EHIP, "hipGetSymbolAddress(scratch) returned a null address");
    g_scratch_ptr.emplace(dev, ptr);
    return ptr;
}

}  // namespace ely

using namespace ely;

extern "C" {

int64_t ely_fp8_workspace_bytes(int64_t rows, int64_t cols, int32_t x_dtype) {
    if (rows < 0 || cols < 0) return -1;
    // a long per-tensor row also has room for the sampled-guess path
    if (rows == 1 && cols >= ((int64_t)ELY_GUESS_MIN_MB << 20) / (x_dtype == ELY_F32 ? 4 : 2))
        return (int64_t)std::max(split_ws_bytes(1), guess_ws_bytes(cols));
    return (int64_t)split_ws_bytes(rows);
}

int ely_fp8_quantize(const void* x, int32_t x_dtype, int64_t rows, int64_t cols, int32_t fmt, uint8_t* q, int32_t* k,
                     void* workspace, int64_t ws_bytes, void* stream) {
    return guarded([&] {
        check_fmt(fmt);
        check_dtype(x_dtype, "x_dtype");
        check_shape(rows, cols);
        if (rows * cols > 0 && !x) fail(ELY_EINVAL, "ely_fp8_quantize: null x");
        if (rows > 0 && !k) fail(ELY_EINVAL, "ely_fp8_quantize: null k");
        hipStream_t s = static_cast<hipStream_t>(stream);
        if (fmt == ELY_E4M3) {
            if (x_dtype == ELY_BF16) quantize_impl<kE4M3, true>(x, rows, cols, q, k, nullptr, workspace, ws_bytes, s);
            else quantize_impl<kE4M3, false>(x, rows, cols, q, k, nullptr, workspace, ws_bytes, s);
        } else {
            if (x_dtype == ELY_BF16) quantize_impl<kE5M2, true>(x, rows, cols, q, k, nullptr, workspace, ws_bytes, s);
            else quantize_impl<kE5M2, false>(x, rows, cols, q, k, nullptr, workspace, ws_bytes, s);
        }
    });
}

int ely_fp8_quantize_noalloc(const void* x, int32_t x_dtype, int64_t rows, int64_t cols, int32_t fmt, uint8_t* q,
                             int32_t* k, void* stream) {
    return guarded([&] {
        check_fmt(fmt);
        check_dtype(x_dtype, "x_dtype");
        check_shape(rows, cols);
        if (rows * cols > 0 && !x) fail(ELY_EINVAL, "ely_fp8_quantize_noalloc: null x");
        if (rows > 0 && !k) fail(ELY_EINVAL, "ely_fp8_quantize_noalloc: null k");
        // Only the split path (rows that fit no register path) uses scratch,
        // but every shape that wants_workspace is held to what the static
        // array takes of row maxima and partials.  Every
        // scratch word the split launches read was written by an earlier
        // launch of the same call, so nothing needs clearing between calls.
        const bool split = rows > 0 && cols > 0 && wants_workspace(cols, x_dtype, x, q, nullptr);
        void* ws = nullptr;
        if (split) {
            const size_t need = split_ws_bytes(rows);
            if (need > kNoallocScratchBytes)
                fail(ELY_EINVAL, "ely_fp8_quantize_noalloc: " + std::to_string(rows) + " rows of " + std::to_string(cols) +
                                     " columns need " + std::to_string(need) + " scratch bytes, above the " +
                                     std::to_string(kNoallocScratchBytes) +
                                     "-byte static scratch; use ely_fp8_quantize with a workspace");
            ws = noalloc_scratch();
        }
        hipStream_t s = static_cast<hipStream_t>(stream);
        const int64_t wsb = split ? (int64_t)kNoallocScratchBytes : 0;
        if (fmt == ELY_E4M3) {
            if (x_dtype == ELY_BF16) quantize_impl<kE4M3, true>(x, rows, cols, q, k, nullptr, ws, wsb, s, false);
            else quantize_impl<kE4M3, false>(x, rows, cols, q, k, nullptr, ws, wsb, s, false);
        } else {
            if (x_dtype == ELY_BF16) quantize_impl<kE5M2, true>(x, rows, cols, q, k, nullptr, ws, wsb, s, false);
            else quantize_impl<kE5M2, false>(x, rows, cols, q, k, nullptr, ws, wsb, s, false);
        }
    });
}

int64_t ely_fp8_hint_workspace_bytes(int64_t n) {
    if (n < 0) return -1;
    return (int64_t)hint_ws_bytes(n);
}

int ely_fp8_quantize_hint(const void* x, int32_t x_dtype, int64_t n, int32_t fmt, int32_t k_hint,
                          const int32_t* k_hint_dev, uint8_t* q, int32_t* k, void* out, int32_t* hit_dev,
                          void* workspace, int64_t ws_bytes, void* stream) {
    return guarded([&] {
        check_fmt(fmt);
        check_dtype(x_dtype, "x_dtype");
        check_shape(1, n);
        if (!k) fail(ELY_EINVAL, "ely_fp8_quantize_hint: null k");
        if (n > 0 && (!x || (!q && !out))) fail(ELY_EINVAL, "ely_fp8_quantize_hint: null x, or neither q nor out");
        hipStream_t s = static_cast<hipStream_t>(stream);
        if (fmt == ELY_E4M3) {
            if (x_dtype == ELY_BF16) quantize_hint_impl<kE4M3, true>(x, n, k_hint, k_hint_dev, q, k, out, hit_dev, workspace, ws_bytes, s);
            else quantize_hint_impl<kE4M3, false>(x, n, k_hint, k_hint_dev, q, k, out, hit_dev, workspace, ws_bytes, s);
        } else {
            if (x_dtype == ELY_BF16) quantize_hint_impl<kE5M2, true>(x, n, k_hint, k_hint_dev, q, k, out, hit_dev, workspace, ws_bytes, s);
            else quantize_hint_impl<kE5M2, false>(x, n, k_hint, k_hint_dev, q, k, out, hit_dev, workspace, ws_bytes, s);
        }
    });
}

int ely_fp8_dequantize(const uint8_t* q, const int32_t* k, int64_t rows, int64_t cols, int32_t fmt, void* out,
                       int32_t out_dtype, void* stream) {
    return guarded([&] {
        check_fmt(fmt);
        check_dtype(out_dtype, "out_dtype");
        check_shape(rows, cols);
        if (rows * cols > 0 && (!q || !k || !out)) fail(ELY_EINVAL, "ely_fp8_dequantize: null pointer");
        hipStream_t s = static_cast<hipStream_t>(stream);
        if (fmt == ELY_E4M3) {
            if (out_dtype == ELY_BF16) dequantize_impl<kE4M3, true>(q, k, rows, cols, out, s);
            else dequantize_impl<kE4M3, false>(q, k, rows, cols, out, s);
        } else {
            if (out_dtype == ELY_BF16) dequantize_impl<kE5M2, true>(q, k, rows, cols, out, s);
            else dequantize_impl<kE5M2, false>(q, k, rows, cols, out, s);
        }
    });
}

int ely_fp8_roundtrip(const void* x, int32_t x_dtype, int64_t rows, int64_t cols, int32_t fmt, void* out, uint8_t* q,
                      int32_t* k, void* workspace, int64_t ws_bytes, void* stream) {
    return guarded([&] {
        check_fmt(fmt);
        check_dtype(x_dtype, "x_dtype");
        check_shape(rows, cols);
        if (rows * cols > 0 && (!x || !out)) fail(ELY_EINVAL, "ely_fp8_roundtrip: null x or out");
        hipStream_t s = static_cast<hipStream_t>(stream);
        if (fmt == ELY_E4M3) {
            if (x_dtype == ELY_BF16) quantize_impl<kE4M3, true>(x, rows, cols, q, k, out, workspace, ws_bytes, s);
            else quantize_impl<kE4M3, false>(x, rows, cols, q, k, out, workspace, ws_bytes, s);
        } else {
            if (x_dtype == ELY_BF16) quantize_impl<kE5M2, true>(x, rows, cols, q, k, out, workspace, ws_bytes, s);
            else quantize_impl<kE5M2, false>(x, rows, cols, q, k, out, workspace, ws_bytes, s);
        }
    });
}

int ely_selftest_fp8_cvt(uint32_t start, uint64_t count, int32_t fmt, unsigned long long* mismatches_dev,
                         void* stream) {
    return guarded([&] {
        check_fmt(fmt);
        if (!mismatches_dev) fail(ELY_EINVAL, "null counters");
        if (count > (1ull << 32) || (uint64_t)start + count > (1ull << 32))
            fail(ELY_EINVAL, "range beyond the 2^32 fp32 patterns");
        if (count == 0) return;
        hipStream_t s = static_cast<hipStream_t>(stream);
        const unsigned blocks = (unsigned)std::min<uint64_t>((count + 255) / 256, 65536);
        if (fmt == ELY_E4M3)
            hipLaunchKernelGGL(selftest_cvt_kernel<kE4M3>, dim3(blocks), dim3(256), 0, s, start, count, mismatches_dev);
        else
            hipLaunchKernelGGL(selftest_cvt_kernel<kE5M2>, dim3(blocks), dim3(256), 0, s, start, count, mismatches_dev);
        check_launch("selftest_cvt_kernel");
    });
}

int ely_selftest_fp8_scaled(int32_t fmt, unsigned long long* mismatches_dev, void* stream) {
    return guarded([&] {
        check_fmt(fmt);
        if (!mismatches_dev) fail(ELY_EINVAL, "null counters");
        hipStream_t s = static_cast<hipStream_t>(stream);
        const unsigned blocks = (65536u * (2u * kFastK + 1u) + 255u) / 256u;
        if (fmt == ELY_E4M3)
            hipLaunchKernelGGL(selftest_scaled_kernel<kE4M3>, dim3(blocks), dim3(256), 0, s, mismatches_dev);
        else
            hipLaunchKernelGGL(selftest_scaled_kernel<kE5M2>, dim3(blocks), dim3(256), 0, s, mismatches_dev);
        check_launch("selftest_scaled_kernel");
    });
}

int ely_selftest_sqrt(uint32_t start, uint64_t count, unsigned long long* mismatches_dev, void* stream) {
    return guarded([&] {
        if (!mismatches_dev) fail(ELY_EINVAL, "null counter");
        if (count > (1ull << 32) || (uint64_t)start + count > (1ull << 32))
            fail(ELY_EINVAL, "range beyond the 2^32 fp32 patterns");
        if (count == 0) return;
        hipStream_t s = static_cast<hipStream_t>(stream);
        const unsigned blocks = (unsigned)std::min<uint64_t>((count + 255) / 256, 65536);
        hipLaunchKernelGGL(selftest_sqrt_kernel, dim3(blocks), dim3(256), 0, s, start, count, mismatches_dev);
        check_launch("selftest_sqrt_kernel");
    });
}

int64_t ely_fp8_recover_workspace_bytes(int64_t rows) {
    if (rows < 0) return -1;
    return (int64_t)(split_ws_bytes(rows) + rowmax_bytes(rows));
}

int ely_fp8_recover_exp(const void* t, int32_t t_dtype, int64_t rows, int64_t cols, int32_t fmt, int32_t* k,
                        unsigned long long* bad_rows_dev, void* workspace, int64_t ws_bytes, void* stream) {
    return guarded([&] {
        check_fmt(fmt);
        check_dtype(t_dtype, "t_dtype");
        check_shape(rows, cols);
        if (rows == 0) return;
        if (!k || !bad_rows_dev || (cols > 0 && !t)) fail(ELY_EINVAL, "ely_fp8_recover_exp: null pointer");
        if (!workspace || ws_bytes < ely_fp8_recover_workspace_bytes(rows))
            fail(ELY_EWORKSPACE, "ely_fp8_recover_exp: workspace smaller than ely_fp8_recover_workspace_bytes");
        hipStream_t s = static_cast<hipStream_t>(stream);
        const bool bf16 = t_dtype == ELY_BF16;
        const int vpl = recover_vpl(cols, bf16, t, nullptr);
        if (vpl) return recover_rows(vpl, t, bf16, rows, cols, fmt, k, nullptr, bad_rows_dev, s);
        recover_multi(t, bf16, rows, cols, fmt, k, bad_rows_dev, workspace, s);
    });
}

int ely_fp8_recover_image(const void* t, int32_t t_dtype, int64_t rows, int64_t cols, int32_t fmt, int32_t* k,
                          uint8_t* q, unsigned long long* bad_rows_dev, void* workspace, int64_t ws_bytes,
                          void* stream) {
    return guarded([&] {
        check_fmt(fmt);
        check_dtype(t_dtype, "t_dtype");
        check_shape(rows, cols);
        if (rows == 0) return;
        if (!k || !bad_rows_dev || (cols > 0 && (!t || !q))) fail(ELY_EINVAL, "ely_fp8_recover_image: null pointer");
        if (!workspace || ws_bytes < ely_fp8_recover_workspace_bytes(rows))
            fail(ELY_EWORKSPACE, "ely_fp8_recover_image: workspace smaller than ely_fp8_recover_workspace_bytes");
        hipStream_t s = static_cast<hipStream_t>(stream);
        const bool bf16 = t_dtype == ELY_BF16;
        const int vpl = recover_vpl(cols, bf16, t, q);
        if (vpl) return recover_rows(vpl, t, bf16, rows, cols, fmt, k, q, bad_rows_dev, s);
        recover_multi(t, bf16, rows, cols, fmt, k, bad_rows_dev, workspace, s);
        if (cols > 0) quant_k_launch(t, bf16, rows, cols, fmt, k, q, s);
    });
}

int ely_fp8_quantize_k(const void* x, int32_t x_dtype, int64_t rows, int64_t cols, int32_t fmt, const int32_t* k,
                       uint8_t* q, void* stream) {
    return guarded([&] {
        check_fmt(fmt);
        check_dtype(x_dtype, "x_dtype");
        check_shape(rows, cols);
        if (rows * cols == 0) return;
        if (!x || !k || !q) fail(ELY_EINVAL, "ely_fp8_quantize_k: null pointer");
        quant_k_launch(x, x_dtype == ELY_BF16, rows, cols, fmt, k, q, static_cast<hipStream_t>(stream));
    });
}

}  // extern "C"
