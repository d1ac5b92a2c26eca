// The v2 candidate-scale grid search and the per-channel activation
// importance it weights by, for gfx950.
//
// Search (mround/core/scale_search.py:71-187; oracle
// mround/reference/scale_search.py:130-211): a group in a thread's registers,
// every candidate evaluated against it with the loss summed element by element
// in column order; 2^s neighbouring lanes share a group, each taking every
// 2^s-th candidate, so that small matrices fill the chip and large ones end
// together. The work is VALU-bound: per weight and candidate a product, a
// rounding, a clamp (one v_med3), the residual, its square, the importance and
// the sum, eight instructions; at 2 bits seven, the codes being powers of two
// whose product with the scale is exact, so that one fused multiply-add rounds
// the residual as the two operations do. With importance the lanes of a wave
// take rows of one column group, whose importance then sits in scalar registers
// (64 vector registers fewer: six waves per SIMD instead of three).
// Measured with importance on 11008 x 2048 bf16: groups of 64 at 2 bits (181
// candidates) 725 us with a thread per group, 475 now (2.4 cycles an
// instruction of a SIMD); groups of 128 at 3 bits 1260 -> 590; 192 x 576 at 2
// bits 194 -> 9. Without importance groups of 64 fit six waves per SIMD
// (18944 x 3584 at 3 bits 1832 -> 1561 us; a thread per group 1719, which at
// groups of 128 takes 1836 to the 1867 here and at 192 x 576 190 to 10). (A min
// and max for the v_med3, or the rounding by adding and taking off 1.5 * 2^23,
// measured 7-24 % slower. Ending a candidate when every lane's partial sum
// exceeds its best saves 1-8 % of the elements: not done.)
//
// Importance (the collecting forward of mround/pipeline/runner.py:346-363,
// `sum(square(x), axis=0)` of each linear's input): per-column sums of
// squares in two deterministic passes, row blocks into a workspace, then the
// blocks summed in order and added to the running total.
#include <cmath>
#include <type_traits>

#include "mr_common.h"

namespace mr {
namespace {

constexpr int kBlock = 256;
constexpr int kRowBlocks = 64;

template <typename WT>
__device__ __forceinline__ float ld_as_f32(const WT* p, int64_t i) {
  if constexpr (sizeof(WT) == 4) return reinterpret_cast<const float*>(p)[i];
  else return bf16_to_f32(reinterpret_cast<const uint16_t*>(p)[i]);
}

// The candidates in the order that breaks ties: number 0 is the unclipped
// scale, then the steps -half .. half without 0.
__device__ __forceinline__ int candidate(int o, int half) {
  if (o == 0) return 0;
  const int i = o - 1 - half;
  return i < 0 ? i : i + 1;
}

template <int GS, typename WT, bool IMP>
__global__ __launch_bounds__(kBlock, GS == 32 || (GS == 64 && !IMP) ? 6 : GS == 64 ? 5 : 3) void search_kernel(const WT* __restrict__ w,
                                                        const float* __restrict__ imp,
                                                        int64_t rows, int groups_per_row,
                                                        int bits, double step, int half, int shift,
                                                        float* __restrict__ scale_out) {
  const int lane = threadIdx.x & 63;
  const int64_t wave = static_cast<int64_t>(blockIdx.x) * (kBlock / 64) + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int part = lane & ((1 << shift) - 1);
  const int64_t slot = lane >> shift;
  int64_t g;  // this lane's group
  typedef const __attribute__((address_space(4))) float* uniform_ptr;  // (read into scalar registers)
  uniform_ptr q = nullptr;
  bool active;
  if constexpr (IMP) {
    const int64_t row = wave / groups_per_row * (64 >> shift) + slot;
    const int cg = static_cast<int>(wave % groups_per_row);
    active = row < rows;
    g = (active ? row : rows - 1) * groups_per_row + cg;
    q = (uniform_ptr)(imp + static_cast<int64_t>(cg) * GS);
  } else {
    const int64_t n = rows * groups_per_row;
    g = wave * (64 >> shift) + slot;
    active = g < n;
    if (!active) g = n - 1;
  }
  float x[GS];
#pragma unroll
  for (int j = 0; j < GS; ++j) x[j] = ld_as_f32(w, g * GS + j);
  // anchor: the signed element of largest magnitude, first occurrence
  float gmax = x[0], amax = fabsf(x[0]);
#pragma unroll
  for (int j = 1; j < GS; ++j)
    if (fabsf(x[j]) > amax) {
      amax = fabsf(x[j]);
      gmax = x[j];
    }
  const float recip = gmax == 0.0f ? 0.0f : 1.0f / gmax;
  const double nmax_d = static_cast<double>(1 << (bits - 1));
  const float nmax = static_cast<float>(nmax_d);
  const float lo = -nmax, hi = nmax - 1.0f;
  const int count = 2 * half + 1;

  // Short bfloat16 groups without importance count their loop in scalar
  // registers (18944 x 3584 at 3 bits 1879 -> 1720 us; the other forms 1-4 % slower).
  constexpr bool kCounted = GS == 32 && !IMP && sizeof(WT) == 2;
  const int trips = (count + (1 << shift) - 1) >> shift;

  float best_s = 0.0f, best_l = __builtin_inff();
  int best_o = count;
  auto run = [&](auto fusedc) __attribute__((always_inline)) {
    constexpr bool FUSED = decltype(fusedc)::value;
    for (int n = 0, o = part; kCounted ? n < trips : o < count; ++n, o += 1 << shift) {
      if (kCounted && o >= count) break;
      const float eff = static_cast<float>(nmax_d - step * static_cast<double>(candidate(o, half)));
      const float inverse = (-eff) * recip;
      const float scale = inverse == 0.0f ? 0.0f : 1.0f / inverse;
      // (128 importances outnumber the scalar registers: read again for each candidate)
      if constexpr (IMP && GS > 64) asm volatile("" : "+s"(q));
      float loss = 0.0f;
#pragma unroll
      for (int j = 0; j < GS; ++j) {
        // (a NaN product clamps to lo, as fminf(fmaxf()) does)
        const float c = __builtin_amdgcn_fmed3f(rintf(inverse * x[j]), lo, hi);
        const float r = FUSED ? fmaf(scale, c, -x[j]) : scale * c - x[j];
        float t = r * r;
        if constexpr (IMP) t = t * q[j];
        loss = loss + t;
      }
      // (a NaN loss of candidate 0 is never improved on)
      if (o == 0 && loss != loss) loss = -__builtin_inff();
      if (o == 0 || loss < best_l) {
        best_l = loss;
        best_s = scale;
        best_o = o;
      }
    }
  };
  // The fused residual: |scale| <= amax, so that twice the scale is finite.
  if (bits == 2 && __all(amax < 0x1p126f)) run(std::true_type{});
  else run(std::false_type{});
  for (int off = 1; off < 1 << shift; off <<= 1) {
    const float l = __shfl_xor(best_l, off, 64), sc = __shfl_xor(best_s, off, 64);
    const int o = __shfl_xor(best_o, off, 64);
    if (l < best_l || (l == best_l && o < best_o)) {
      best_l = l;
      best_s = sc;
      best_o = o;
    }
  }
  if (active && part == 0) scale_out[g] = best_s;
}

template <typename XT>
__global__ __launch_bounds__(kBlock) void colsumsq_partial(const XT* __restrict__ x, int64_t rows,
                                                           int64_t cols, int64_t ld,
                                                           float* __restrict__ partial) {
  const int64_t c = static_cast<int64_t>(blockIdx.x) * kBlock + threadIdx.x;
  if (c >= cols) return;
  const int64_t per = (rows + kRowBlocks - 1) / kRowBlocks;
  const int64_t r0 = blockIdx.y * per;
  const int64_t r1 = min(rows, r0 + per);
  float acc = 0.0f;
  for (int64_t r = r0; r < r1; ++r) {
    const float v = ld_as_f32(x, r * ld + c);
    acc = acc + v * v;
  }
  partial[blockIdx.y * cols + c] = acc;
}

__global__ __launch_bounds__(kBlock) void colsumsq_final(const float* __restrict__ partial,
                                                         int64_t cols, float* __restrict__ out) {
  const int64_t c = static_cast<int64_t>(blockIdx.x) * kBlock + threadIdx.x;
  if (c >= cols) return;
  float acc = 0.0f;
  for (int b = 0; b < kRowBlocks; ++b) acc = acc + partial[b * cols + c];
  out[c] = out[c] + acc;
}

template <int GS, typename WT>
int launch_search(const void* w, const float* imp, int64_t rows, int gpr, int bits, double step,
                  int half, float* out, hipStream_t s) {
  // Lanes per group: enough for 8 waves per SIMD (more cost redundant loads of
  // the group), and no more than there are candidates for 4 each.
  auto waves = [&](int shift) {
    const int64_t per = 64 >> shift;
    return imp ? (rows + per - 1) / per * gpr : (rows * gpr + per - 1) / per;
  };
  int shift = 0;
  while (shift < 5 && waves(shift) < 8192 && (2 * half + 1) >> (shift + 1) >= 4) ++shift;
  const int64_t blocks = (waves(shift) + kBlock / 64 - 1) / (kBlock / 64);
  if (blocks > 0x7fffffff) return fail(MR_EINVAL, "mr_search_scales: too large");
  if (imp)
    hipLaunchKernelGGL((search_kernel<GS, WT, true>), dim3(static_cast<unsigned>(blocks)), dim3(kBlock), 0, s,
                       static_cast<const WT*>(w), imp, rows, gpr, bits, step, half, shift, out);
  else
    hipLaunchKernelGGL((search_kernel<GS, WT, false>), dim3(static_cast<unsigned>(blocks)), dim3(kBlock), 0, s,
                       static_cast<const WT*>(w), imp, rows, gpr, bits, step, half, shift, out);
  MR_LAUNCH_CHECK("mr_search_scales");
  return MR_OK;
}

}  // namespace
}  // namespace mr

extern "C" {

int mr_search_scales(const void* w, int w_dtype, const float* importance, int64_t rows,
                     int64_t cols, int group_size, int bits, double step, int half_count,
                     float* scale_out, void* stream) {
  using namespace mr;
  clear_error();
  if (rows <= 0 || cols <= 0) return MR_OK;
  if (!w || !scale_out) return fail(MR_EINVAL, "mr_search_scales: null pointer");
  if (group_size != 32 && group_size != 64 && group_size != 128)
    return fail(MR_EINVAL, "mr_search_scales: group size must be 32, 64 or 128, got %d", group_size);
  if (cols % group_size)
    return fail(MR_EINVAL, "search expects a 2-D weight whose last dimension is a multiple of "
                "group_size=%d, got %lld columns", group_size, (long long)cols);
  if (bits < 2 || bits > 8) return fail(MR_EINVAL, "mr_search_scales: bits must be 2..8");
  if (half_count < 0 || half_count > 100000 || !(step >= 0.0))
    return fail(MR_EINVAL, "mr_search_scales: bad grid");
  if (w_dtype != MR_F32 && w_dtype != MR_BF16)
    return fail(MR_EINVAL, "mr_search_scales: weight must be fp32 or bf16");
  const int gpr = static_cast<int>(cols / group_size);
  hipStream_t s = static_cast<hipStream_t>(stream);
  const bool f32 = w_dtype == MR_F32;
#define MR_SEARCH_CASE(GS)                                                                            \
  return f32 ? launch_search<GS, float>(w, importance, rows, gpr, bits, step, half_count, scale_out, s) \
             : launch_search<GS, uint16_t>(w, importance, rows, gpr, bits, step, half_count, scale_out, s);
  switch (group_size) {
    case 32: { MR_SEARCH_CASE(32) }
    case 64: { MR_SEARCH_CASE(64) }
    default: { MR_SEARCH_CASE(128) }
  }
#undef MR_SEARCH_CASE
}

int64_t mr_colsumsq_workspace_bytes(int64_t cols) {
  return cols > 0 ? static_cast<int64_t>(mr::kRowBlocks) * cols * 4 : 0;
}

int mr_colsumsq(const void* x, int x_dtype, int64_t rows, int64_t cols, int64_t ld, float* out,
                void* workspace, void* stream) {
  using namespace mr;
  clear_error();
  if (rows <= 0 || cols <= 0) return MR_OK;
  if (!x || !out || !workspace) return fail(MR_EINVAL, "mr_colsumsq: null pointer");
  if (ld < cols) return fail(MR_EINVAL, "mr_colsumsq: ld smaller than the row");
  if (x_dtype != MR_F32 && x_dtype != MR_BF16) return fail(MR_EINVAL, "mr_colsumsq: fp32 or bf16 input");
  hipStream_t s = static_cast<hipStream_t>(stream);
  float* partial = static_cast<float*>(workspace);
  const unsigned cb = static_cast<unsigned>((cols + kBlock - 1) / kBlock);
  if (x_dtype == MR_F32)
    hipLaunchKernelGGL(colsumsq_partial<float>, dim3(cb, kRowBlocks), dim3(kBlock), 0, s,
                       static_cast<const float*>(x), rows, cols, ld, partial);
  else
    hipLaunchKernelGGL(colsumsq_partial<uint16_t>, dim3(cb, kRowBlocks), dim3(kBlock), 0, s,
                       static_cast<const uint16_t*>(x), rows, cols, ld, partial);
  hipLaunchKernelGGL(colsumsq_final, dim3(cb), dim3(kBlock), 0, s, partial, cols, out);
  MR_LAUNCH_CHECK("mr_colsumsq");
  return MR_OK;
}

}  // extern "C"
