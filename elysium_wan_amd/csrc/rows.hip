// rows.hip -- the row fold of a tied table's step gradient across stages
// (TiedRowFold, runtime/accumulate.py:140-247).  The stock fold is
// acc = g_0, acc += g_i in microbatch order with g_i = h_i + e_i (autograd's
// sum of the table's two uses, e_i = +0 outside the microbatch's rows), one
// rounding per add in the table's dtype.  TiedRowFold reaches the same bits
// without a dense table per microbatch in flight by folding each row as
// soon as its prefix is complete; every fold it makes is one of
//   acc[idx[j]]  = a[rows_a[j]] + 0.0                  (first, free rows)
//   acc[idx[j]] += a[rows_a[j]] + 0.0                  (later, free rows)
//   acc[idx[j]]  = a[j] + e_j       / acc[idx[j]] += a[j] + e_j
//                                                      (held rows resolved)
// over a set of distinct rows, which this kernel runs: a block per row or
// piece of a row, 16-byte vectors across it.  e_j is the embedding row b[b_rows[j]] of a held row the microbatch touched, +0.0 for
// one it did not (b_rows[j] < 0), or b[j] of a compact b.  A second kernel
// takes a whole Head gradient in one pass: its free rows fold, its held
// rows are copied out bit for bit, so that the gradient itself can go.
#include <algorithm>
#include <type_traits>

#include "ely_device.hpp"
#include "ely_host.hpp"

#pragma clang fp contract(off)

namespace ely {
namespace {

// A block of W waves moves V 16-byte vectors per lane of a row and ends, a
// row's pieces across the grid, rows down (a longer list strides).  Launches
// that touch more than the 256 MB MALL holds stream (nontemporal loads, and
// the split's stores of the sum; its held rows stay in the caches, which took
// the split of the table below from 147 to 143 us), one-wave blocks taking the
// pieces; the others keep to plain accesses, for the rows and the sum are read
// again soon, in the shapes of fold_shape and split_shape.  Streaming, against a 256-thread block that
// loops over its row, buffers in turn, a third of the rows held: 32,768 x
// 2,560 fp32 split 166 -> 143 us (5.1 -> 5.9 TB/s) and fold of the held 77 ->
// 58, bf16 84 -> 75 and 40 -> 39; 32,768 x 1,001 bf16, element by element
// before, 90 -> 44 and 40 -> 21.
constexpr int64_t kMallBytes = (int64_t)256 << 20;
constexpr int64_t kRowGrid = 65535;

typedef uint32_t ru4 __attribute__((ext_vector_type(4)));
// ... at any element's address (see the codec's vector types)
typedef uint32_t ru4u __attribute__((ext_vector_type(4), aligned(2)));
#define ROWS_G1 __attribute__((address_space(1)))
template <bool NT>
__device__ __forceinline__ ru4 ld_row(const void* p) {
    if (NT) return __builtin_nontemporal_load((const ROWS_G1 ru4u*)p);
    return *(const ROWS_G1 ru4u*)p;
}
template <bool NT>
__device__ __forceinline__ void st_row(void* p, ru4 v) {
    if (NT) __builtin_nontemporal_store((ru4u)v, (ROWS_G1 ru4u*)p);
    else *(ROWS_G1 ru4u*)p = v;
}

// v = a + b (b = +0.0 when absent) rounded to the dtype, then acc = v or
// acc + v rounded to the dtype: torch's two elementwise adds.
template <bool BF16>
__device__ __forceinline__ float fold1(float acc, float a, float b, bool first) {
    float v = a + b;
    if (BF16) v = bf16_to_f32(f32_to_bf16(v));
    if (first) return v;
    float s = acc + v;
    if (BF16) s = bf16_to_f32(f32_to_bf16(s));
    return s;
}

// One vector of 4 fp32 or 8 bf16 elements: acc (=|+=) x + y, each add rounded
// to the dtype (y = 0 when the row has no b).
template <bool BF16>
__device__ __forceinline__ ru4 fold_vec(ru4 z, ru4 x, ru4 y, int first) {
    ru4 o;
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        if (BF16) {
            const float lo = fold1<true>(bf16_to_f32(z[k] & 0xFFFFu), bf16_to_f32(x[k] & 0xFFFFu), bf16_to_f32(y[k] & 0xFFFFu), first);
            const float hi = fold1<true>(bf16_to_f32(z[k] >> 16), bf16_to_f32(x[k] >> 16), bf16_to_f32(y[k] >> 16), first);
            o[k] = f32_to_bf16(lo) | (f32_to_bf16(hi) << 16);
        } else {
            o[k] = __float_as_uint(fold1<false>(__uint_as_float(z[k]), __uint_as_float(x[k]), __uint_as_float(y[k]), first));
        }
    }
    return o;
}

// Piece `piece` of one row of d elements: ac (=|+=) av + (bv or +0.0), its
// vectors' loads all issued before the first is stored.  The row's last
// elements, short of a vector, go to the last piece's lanes, one each.
template <bool BF16, int V, int W, bool NTL, bool NTS>
__device__ __forceinline__ void fold_piece(char* ac, const char* av, const char* bv, int64_t d, int piece, int first,
                                           int vec) {
    constexpr int EPV = BF16 ? 8 : 4, T = kWave * W;
    const int64_t nvec = vec ? d / EPV : 0;
    const int64_t v0 = (int64_t)piece * (T * V) + threadIdx.x;
    ru4 x[V], y[V], z[V];
#pragma unroll
    for (int u = 0; u < V; ++u) {
        const int64_t v = v0 + u * T;
        const ru4 zero = {0u, 0u, 0u, 0u};
        x[u] = v < nvec ? ld_row<NTL>(av + v * 16) : zero;
        y[u] = (v < nvec && bv) ? ld_row<NTL>(bv + v * 16) : zero;
        z[u] = (v < nvec && !first) ? ld_row<NTL>(ac + v * 16) : zero;
    }
#pragma unroll
    for (int u = 0; u < V; ++u) {
        const int64_t v = v0 + u * T;
        if (v < nvec) st_row<NTS>(ac + v * 16, fold_vec<BF16>(z[u], x[u], y[u], first));
    }
    if (piece != (int)gridDim.x - 1) return;
    for (int64_t c = nvec * EPV + threadIdx.x; c < d; c += T) {
        if (BF16) {
            uint16_t* o = reinterpret_cast<uint16_t*>(ac) + c;
            const float z1 = first ? 0.0f : bf16_to_f32(*o);
            *o = (uint16_t)f32_to_bf16(fold1<true>(z1, bf16_to_f32(reinterpret_cast<const uint16_t*>(av)[c]),
                                                  bv ? bf16_to_f32(reinterpret_cast<const uint16_t*>(bv)[c]) : 0.0f, first));
        } else {
            float* o = reinterpret_cast<float*>(ac) + c;
            *o = fold1<false>(first ? 0.0f : *o, reinterpret_cast<const float*>(av)[c],
                              bv ? reinterpret_cast<const float*>(bv)[c] : 0.0f, first);
        }
    }
}

template <bool BF16, int V, int W, bool NT>
__global__ __launch_bounds__(kWave * W) void rows_fold_kernel(void* __restrict__ acc, const void* __restrict__ a,
                                                              const int64_t* __restrict__ a_rows,
                                                              const void* __restrict__ b,
                                                              const int64_t* __restrict__ b_rows,
                                                              const int64_t* __restrict__ idx, int64_t n_idx,
                                                              int64_t n_rows, int64_t a_total, int64_t b_total,
                                                              int64_t d, int first, int vec) {
    const int64_t esz = BF16 ? 2 : 4;
    for (int64_t j = blockIdx.y; j < n_idx; j += gridDim.y) {
        const int64_t r = idx[j];
        const int64_t ar = a_rows ? a_rows[j] : j;
        const int64_t br = b ? (b_rows ? b_rows[j] : j) : -1;  // < 0: the row adds +0.0
        // the host checks every index; a row outside the tables is skipped, never touched
        if (r < 0 || r >= n_rows || ar < 0 || ar >= a_total || br >= b_total) continue;
        fold_piece<BF16, V, W, NT, false>(static_cast<char*>(acc) + r * d * esz, static_cast<const char*>(a) + ar * d * esz,
                                          br >= 0 ? static_cast<const char*>(b) + br * d * esz : nullptr, d, blockIdx.x,
                                          first, vec);
    }
}

// That piece of a row of d elements copied bit for bit.
template <bool BF16, int V, int W, bool NT>
__device__ __forceinline__ void copy_piece(char* o, const char* x, int64_t d, int piece, int vec) {
    constexpr int EPV = BF16 ? 8 : 4, ESZ = BF16 ? 2 : 4, T = kWave * W;
    const int64_t nvec = vec ? d / EPV : 0;
    const int64_t v0 = (int64_t)piece * (T * V) + threadIdx.x;
    ru4 t[V];
#pragma unroll
    for (int u = 0; u < V; ++u)
        if (v0 + u * T < nvec) t[u] = ld_row<NT>(x + (v0 + u * T) * 16);
#pragma unroll
    for (int u = 0; u < V; ++u)
        if (v0 + u * T < nvec) st_row<false>(o + (v0 + u * T) * 16, t[u]);
    if (piece != (int)gridDim.x - 1) return;
    for (int64_t c = nvec * 16 + threadIdx.x; c < d * ESZ; c += T) o[c] = x[c];
}

// A Head gradient in one pass, a row's pieces across the grid: a row r with
// slot[r] < 0 is free and takes acc[r] = a[r] + 0.0 (first) or
// acc[r] + (a[r] + 0.0), each add rounded to the dtype; a held row
// (slot[r] >= 0) is copied to held_out[slot[r]] bit for bit and acc[r] is
// left for its resolve.
template <bool BF16, int V, int W, bool NTL, bool NTS>
__global__ __launch_bounds__(kWave * W) void rows_split_kernel(void* __restrict__ acc, const void* __restrict__ a,
                                                               const int32_t* __restrict__ slot,
                                                               void* __restrict__ held_out, int64_t n_rows,
                                                               int64_t n_held, int64_t d, int first, int vec) {
    const int64_t row_bytes = d * (BF16 ? 2 : 4);
    for (int64_t r = blockIdx.y; r < n_rows; r += gridDim.y) {
        const int64_t s = slot[r];
        const char* x = static_cast<const char*>(a) + r * row_bytes;
        if (s < 0)
            fold_piece<BF16, V, W, NTL, NTS>(static_cast<char*>(acc) + r * row_bytes, x, nullptr, d, blockIdx.x, first, vec);
        else if (s < n_held)  // the host numbers the held rows 0..n_held-1
            copy_piece<BF16, V, W, NTL>(static_cast<char*>(held_out) + s * row_bytes, x, d, blockIdx.x, vec);
    }
}

// The pieces of a row (`span` vectors a block) across, rows down, for blocks
// of `threads`; a dispatch counts its threads in 32 bits.
dim3 rows_grid(int64_t rows, int64_t nvec, int64_t span, int64_t threads) {
    const int64_t pieces = std::max<int64_t>(1, (nvec + span - 1) / span);
    return dim3((unsigned)pieces, (unsigned)std::min({rows, kRowGrid, (int64_t)0xFFFFFFFFLL / (threads * pieces)}));
}

// The shapes of launches that do not stream, by a row's vectors.  A block that
// holds its whole row is the fastest where the lanes it leaves idle are few: 1,
// 2 and 4 waves of a vector a lane up to 64, 128 and 256 vectors, 4 waves of two
// up to 512.  (A row of two blocks, the second nearly empty, puts the empty
// ones on every second XCD: 320 vectors 12.4 us against 9.8 in one-wave
// pieces.)  Past 512 a row is cut in pieces again (640 vectors in three blocks
// of two waves folded 6.5 us against 8.2 over and over, but 22.2 against 21.3
// within the launches of a whole table).  The fold of few rows, and
// of long bf16 rows, is the faster on one-wave pieces; so is the split of more
// than 32 MB of bf16 (the sum's stores streamed) or of long fp32 rows, two
// vectors a lane.
// The launches of four microbatches (split and fold each), from a graph, in us,
// with a looping 256-thread block per row / one-wave pieces at every size /
// these: fp32 256 x 1,024 17.1 / 18.1 / 16.6, 4,096 x 768 41.8 / 47.0 / 42.5,
// 8,192 x 1,024 82 / 87 / 81, 16,384 x 1,600 230 / 251 / 235; bf16 256 x 768
// 19.6 / 22.5 / 18.9, 8,192 x 2,048 88 / 96 / 90, 32,768 x 768 179 / 142 / 139.
// One by one, a third of 8,192 x 1,024 fp32 rows folded again and again: 5.7 /
// 7.8 / 5.5; 16,384 x 1,600 split 42.5 / 49.0 / 42.0.
struct RowShape {
    int v, w;
};
RowShape fold_shape(int64_t rows, int64_t nvec, bool bf16) {
    if (rows <= 512 || nvec <= kWave || (bf16 && nvec > 4 * kWave)) return {1, 1};
    if (nvec <= 2 * kWave) return {1, 2};
    if (nvec <= 4 * kWave) return {1, 4};
    if (nvec <= 7 * kWave) return {2, 4};
    if (nvec <= 8 * kWave) return {1, 4};
    return {1, 1};
}
RowShape split_shape(int64_t rows, int64_t nvec, bool bf16) {
    if (nvec <= kWave) return {1, 1};
    if (rows * nvec * 16 > kMallBytes / 8 && (bf16 || nvec > 7 * kWave)) return {2, 1};
    if (nvec <= 2 * kWave) return rows <= 512 ? RowShape{1, 1} : RowShape{1, 2};
    if (nvec <= 4 * kWave || rows <= 512 || (rows <= 1024 && nvec > 8 * kWave)) return {1, 4};
    if (nvec <= 8 * kWave) return {2, 4};
    return {2, 1};
}
bool elem_at(const void* p, int64_t esz) { return reinterpret_cast<uintptr_t>(p) % esz == 0; }

// The vectors that a row is moved in; 0 for rows that go element by element
// in a block of 4 waves: those off their elements' addresses, those whose
// pieces no dispatch counts, and few short ones that end in a tail of
// elements, where a vector and then the tail is the longer wait (64 x 257 bf16
// split 3.5 us against 3.0; four microbatches of 256 x 257 24.1 against 21.6).
int64_t row_vecs(int64_t rows, int64_t d, int64_t esz, bool at_elems) {
    const int64_t nvec = d * esz / 16;
    const bool few_tails = rows <= (esz == 2 ? 1024 : 256) && d <= 512 && d * esz % 16 != 0;
    return at_elems && !few_tails && nvec < 0xFFFF0000LL ? nvec : 0;
}

}  // namespace
}  // namespace ely

using namespace ely;

extern "C" int ely_rows_fold(void* acc, const void* a, const int64_t* a_rows, const void* b, const int64_t* b_rows,
                             const int64_t* idx, int64_t n_idx, int64_t n_rows, int64_t a_total, int64_t b_total,
                             int64_t d, int32_t dtype, int32_t first, void* stream) {
    return guarded([&] {
        if (dtype != ELY_F32 && dtype != ELY_BF16) fail(ELY_EINVAL, "ely_rows_fold: dtype must be ELY_F32 or ELY_BF16");
        if (n_idx < 0 || n_rows < 0 || a_total < 0 || b_total < 0 || d < 0) fail(ELY_EINVAL, "ely_rows_fold: negative size");
        if (n_idx == 0 || d == 0) return;
        if (!acc || !a || !idx) fail(ELY_EINVAL, "ely_rows_fold: null pointer");
        if (!a_rows && a_total < n_idx) fail(ELY_EINVAL, "ely_rows_fold: a compact source holds one row per index");
        if (b_rows && !b) fail(ELY_EINVAL, "ely_rows_fold: b_rows without b");
        if (b && !b_rows && b_total < n_idx) fail(ELY_EINVAL, "ely_rows_fold: a compact b holds one row per index");
        const int64_t esz = dtype == ELY_BF16 ? 2 : 4;
        const int64_t nvec = row_vecs(n_idx, d, esz, elem_at(acc, esz) && elem_at(a, esz) && elem_at(b, esz));
        const int vec = nvec > 0;
        const auto launch = [&](auto kern, int v, int w) {
            const dim3 grid = rows_grid(n_idx, nvec, kWave * v * w, kWave * w);
            hipLaunchKernelGGL(kern, grid, dim3(kWave * w), 0, static_cast<hipStream_t>(stream), acc, a, a_rows, b, b_rows,
                               idx, n_idx, n_rows, a_total, b ? b_total : 0, d, first ? 1 : 0, vec);
        };
        const auto shape = [&](auto bf16) {
            constexpr bool B = decltype(bf16)::value;
            if (3 * n_idx * d * esz > kMallBytes) return launch(rows_fold_kernel<B, 1, 1, true>, 1, 1);
            const RowShape sh = vec ? fold_shape(n_idx, nvec, B) : RowShape{1, 4};
            if (sh.v == 2) launch(rows_fold_kernel<B, 2, 4, false>, 2, 4);
            else if (sh.w == 4) launch(rows_fold_kernel<B, 1, 4, false>, 1, 4);
            else if (sh.w == 2) launch(rows_fold_kernel<B, 1, 2, false>, 1, 2);
            else launch(rows_fold_kernel<B, 1, 1, false>, 1, 1);
        };
        dtype == ELY_BF16 ? shape(std::true_type()) : shape(std::false_type());
        check_launch("rows_fold_kernel");
    });
}

extern "C" int ely_rows_split(void* acc, const void* a, const int32_t* slot, void* held_out, int64_t n_rows,
                              int64_t n_held, int64_t d, int32_t dtype, int32_t first, void* stream) {
    return guarded([&] {
        if (dtype != ELY_F32 && dtype != ELY_BF16) fail(ELY_EINVAL, "ely_rows_split: dtype must be ELY_F32 or ELY_BF16");
        if (n_rows < 0 || n_held < 0 || d < 0) fail(ELY_EINVAL, "ely_rows_split: negative size");
        if (n_held > n_rows) fail(ELY_EINVAL, "ely_rows_split: more held rows than rows");
        if (n_rows == 0 || d == 0) return;
        if (!acc || !a || !slot || (n_held && !held_out)) fail(ELY_EINVAL, "ely_rows_split: null pointer");
        const int64_t esz = dtype == ELY_BF16 ? 2 : 4;
        const int64_t nvec = row_vecs(n_rows, d, esz, elem_at(acc, esz) && elem_at(a, esz) && elem_at(held_out, esz));
        const int vec = nvec > 0;
        const auto launch = [&](auto kern, int v, int w) {
            const dim3 grid = rows_grid(n_rows, nvec, kWave * v * w, kWave * w);
            hipLaunchKernelGGL(kern, grid, dim3(kWave * w), 0, static_cast<hipStream_t>(stream), acc, a, slot, held_out,
                               n_rows, n_held, d, first ? 1 : 0, vec);
        };
        const auto shape = [&](auto bf16) {
            constexpr bool B = decltype(bf16)::value;
            if (2 * n_rows * d * esz > kMallBytes) return launch(rows_split_kernel<B, 2, 1, true, true>, 2, 1);
            const RowShape sh = vec ? split_shape(n_rows, nvec, B) : RowShape{1, 4};
            if (sh.v == 2 && sh.w == 4) launch(rows_split_kernel<B, 2, 4, false, false>, 2, 4);
            else if (sh.v == 2 && B && n_rows * d * esz > kMallBytes / 8) launch(rows_split_kernel<B, 2, 1, false, true>, 2, 1);
            else if (sh.v == 2) launch(rows_split_kernel<B, 2, 1, false, false>, 2, 1);
            else if (sh.w == 4) launch(rows_split_kernel<B, 1, 4, false, false>, 1, 4);
            else if (sh.w == 2) launch(rows_split_kernel<B, 1, 2, false, false>, 1, 2);
            else launch(rows_split_kernel<B, 1, 1, false, false>, 1, 1);
        };
        dtype == ELY_BF16 ? shape(std::true_type()) : shape(std::false_type());
        check_launch("rows_split_kernel");
    });
}
