// Language-model ends of the whole-model scoring pass, for gfx950: the
// embedding lookup that starts the residual stream and the causal-LM
// cross-entropy that ends it.
//
// The reference scores layers with the gradient of the mean shifted
// cross-entropy of the whole model (mround/pipeline/scoring.py:183-192):
// logits = model(tokens[:, :-1]) cast to fp32, loss = mean over positions of
// logsumexp(logits) - logits[label]. Its gradient with respect to the logits
// is (softmax - onehot(label)) / n, which is what the cross-entropy kernel
// writes, as the bf16 operand of the head's input-gradient GEMM.
//
// Logits are bf16 (the model-dtype matmul output the reference casts up); every
// reduction over a row runs in fp32, the loss in fp64 across rows.
#include "mr_common.h"

namespace mr {
namespace {

constexpr int kCeBlock = 512;
constexpr int kCeWaves = kCeBlock / 64;
constexpr float kLog2e = 1.4426950408889634f;
constexpr float kLn2 = 0.6931471805599453f;

// (max, sum of exp(x - max)) pairs, merged; an empty pair has s == 0.
struct MaxSum {
  float m, s;
};

__device__ __forceinline__ MaxSum merge(MaxSum a, MaxSum b) {
  if (a.s == 0.0f) return b;
  if (b.s == 0.0f) return a;
  const float m = fmaxf(a.m, b.m);
  return {m, a.s * exp2f((a.m - m) * kLog2e) + b.s * exp2f((b.m - m) * kLog2e)};
}

// Adds n values held in x[] to the running pair with one rescale. (Values that
// are all -inf sum to zero, an empty pair; taken from themselves they would be
// NaNs, as they are where one of them is a NaN.)
template <int N>
__device__ __forceinline__ MaxSum absorb(MaxSum acc, const float (&x)[N]) {
  float mx = x[0];
#pragma unroll
  for (int k = 1; k < N; ++k) mx = fmaxf(mx, x[k]);
  if (mx == -__builtin_inff()) mx = 0.0f;
  float s = 0.0f;
#pragma unroll
  for (int k = 0; k < N; ++k) s += exp2f((x[k] - mx) * kLog2e);
  return merge(acc, MaxSum{mx, s});
}

__device__ __forceinline__ void unpack8(uint4 r, float (&x)[8]) {
  const uint32_t w[4] = {r.x, r.y, r.z, r.w};
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    x[2 * k] = __uint_as_float(w[k] << 16);
    x[2 * k + 1] = __uint_as_float(w[k] & 0xffff0000u);
  }
}

// One workgroup per row. Pass 1 reads the row once for (max, sum); pass 2
// reads it again and writes the gradient. dlogits may be the logits buffer:
// every element is read and then written by the same thread, after the
// barrier that ends pass 1.
template <bool VEC>
__global__ __launch_bounds__(kCeBlock) void ce_rows(const uint16_t* logits, int64_t ld, int64_t V,
                                                    const int32_t* __restrict__ labels, float scale,
                                                    float* __restrict__ row_loss, uint16_t* dlogits,
                                                    int64_t ldd) {
  __shared__ float sm[kCeWaves], ss[kCeWaves];
  const int64_t row = blockIdx.x;
  const uint16_t* x = logits + row * ld;
  const int label = labels[row];
  MaxSum acc{0.0f, 0.0f};
  if constexpr (VEC) {
    const int64_t n8 = V / 8;
    const uint4* x8 = reinterpret_cast<const uint4*>(x);
    int64_t i = threadIdx.x;
    // Two 16-byte loads in flight per thread per step.
    for (; i + kCeBlock < n8; i += 2 * kCeBlock) {
      const uint4 a = x8[i], b = x8[i + kCeBlock];
      float v[16];
      float lo[8], hi[8];
      unpack8(a, lo);
      unpack8(b, hi);
#pragma unroll
      for (int k = 0; k < 8; ++k) {
        v[k] = lo[k];
        v[8 + k] = hi[k];
      }
      acc = absorb<16>(acc, v);
    }
    if (i < n8) {
      float v[8];
      unpack8(x8[i], v);
      acc = absorb<8>(acc, v);
    }
  } else {
    for (int64_t i = threadIdx.x; i < V; i += kCeBlock) {
      const float v[1] = {bf16_to_f32(x[i])};
      acc = absorb<1>(acc, v);
    }
  }
  // The label's logit is read before the barrier: after it, pass 2 may
  // overwrite the row in place.
  const bool ignored = label < 0;
  const bool bad = label >= V;
  float x_label = 0.0f;
  if (threadIdx.x == 0 && !ignored && !bad) x_label = bf16_to_f32(x[label]);
  // Block merge: waves by shuffles, then the eight wave results.
  for (int off = 32; off > 0; off >>= 1) {
    MaxSum o{__shfl_xor(acc.m, off, 64), __shfl_xor(acc.s, off, 64)};
    acc = merge(acc, o);
  }
  const int wave = threadIdx.x >> 6;
  if ((threadIdx.x & 63) == 0) {
    sm[wave] = acc.m;
    ss[wave] = acc.s;
  }
  __syncthreads();
  MaxSum t{sm[0], ss[0]};
#pragma unroll
  for (int w = 1; w < kCeWaves; ++w) t = merge(t, MaxSum{sm[w], ss[w]});
  const float m = t.m, inv_s = 1.0f / t.s;
  if (threadIdx.x == 0) {
    float l = 0.0f;
    if (bad) {
      l = __builtin_nanf("");
    } else if (!ignored) {
      l = m + log2f(t.s) * kLn2 - x_label;
    }
    row_loss[row] = l;
  }
  if (!dlogits) return;
  uint16_t* d = dlogits + row * ldd;
  const float g = ignored ? 0.0f : scale * inv_s;
  if constexpr (VEC) {
    const int64_t n8 = V / 8;
    const uint4* x8 = reinterpret_cast<const uint4*>(x);
    uint4* d8 = reinterpret_cast<uint4*>(d);
    for (int64_t i = threadIdx.x; i < n8; i += kCeBlock) {
      float v[8];
      unpack8(x8[i], v);
      uint32_t w[4];
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        float p0 = exp2f((v[2 * k] - m) * kLog2e) * g;
        float p1 = exp2f((v[2 * k + 1] - m) * kLog2e) * g;
        const int64_t j = i * 8 + 2 * k;
        if (!ignored && j == label) p0 -= scale;
        if (!ignored && j + 1 == label) p1 -= scale;
        w[k] = pack_bf16x2(p0, p1);
      }
      d8[i] = make_uint4(w[0], w[1], w[2], w[3]);
    }
  } else {
    for (int64_t i = threadIdx.x; i < V; i += kCeBlock) {
      float p = exp2f((bf16_to_f32(x[i]) - m) * kLog2e) * g;
      if (!ignored && i == label) p -= scale;
      d[i] = f32_to_bf16(p);
    }
  }
}

// The same with the row held in registers (rows of up to kHeldMax logits whose
// starts are 16-byte aligned; V itself may be any number: one thread takes a last
// partial piece element by element). What bounds ce_rows is memory, three passes
// over rows that no cache keeps (2048 rows of 151936 logits are 622 MB); here a
// row is read once. THREADS x N pieces of 8 logits cover the row, all of a
// thread's loads in flight together: 1024 threads and 20 pieces fill a CU's
// registers with one row of 163,840.
// The largest logit is known before any exponential, so a logit costs one
// multiply and v_exp_f32 in each of the two uses. That instruction gives zero
// where the result is denormal: the gradient of a row that reaches that far
// below its maximum (or holds an infinity) takes exp2f.
// Measured, 2048 rows: 151936 logits 368 -> 314 us (3.4 -> 4.0 TB/s of one read
// and one write), 65536 143 -> 113, 16384 40 -> 29, 4000 18 -> 13, and 100001,
// which ran the scalar kernel, 551 -> 213. (Whole rows of 1024 threads load, then
// store: with two rows to a CU, up to 65536 logits, the two overlap.) With a -inf in
// every row 151936 logits take 371, 65536 118 and 100001 247 us; second reads of such
// rows an element at a time took 970, 261 and 637.
constexpr int kHeldThreads = 1024, kHeldPieces = 20;
constexpr int64_t kHeldMax = 8ll * kHeldThreads * kHeldPieces;

template <int THREADS, int N>
__global__ __launch_bounds__(THREADS, N <= 8 ? 8 : 4) void ce_rows_held(const uint16_t* logits, int64_t ld, int V,
                                                        const int32_t* __restrict__ labels, float scale,
                                                        float* __restrict__ row_loss, uint16_t* dlogits,
                                                        int64_t ldd) {
  constexpr int W = THREADS / 64;
  constexpr uint32_t kNone = 0xff80ff80u;  // a pair of -inf: no part in the maximum or the sum
  __shared__ float s_max[W], s_min[W], s_sum[W];
  const int64_t row = blockIdx.x;
  const uint16_t* x = logits + row * ld;
  const uint4* x8 = reinterpret_cast<const uint4*>(x);
  const int label = labels[row];
  const int tid = threadIdx.x, n8 = V / 8, rest = V % 8;
  float mx = -__builtin_inff(), mn = __builtin_inff();
  uint4 r[N];
#pragma unroll
  for (int j = 0; j < N; ++j) {
    const int i = j * THREADS + tid;
    r[j] = make_uint4(kNone, kNone, kNone, kNone);
    if (i < n8) r[j] = x8[i];
    else if (i == n8 && rest) {
      uint32_t w[4] = {kNone, kNone, kNone, kNone};
#pragma unroll
      for (int k = 0; k < 7; ++k)
        if (k < rest) {
          const uint32_t v = x[n8 * 8 + k];
          mn = fminf(mn, __uint_as_float(v << 16));
          w[k >> 1] = (k & 1) ? (w[k >> 1] & 0xffffu) | (v << 16) : (w[k >> 1] & 0xffff0000u) | v;
        }
      r[j] = make_uint4(w[0], w[1], w[2], w[3]);
    }
  }
  // the label's logit, before the row may be overwritten in place
  const bool ignored = label < 0;
  const bool bad = label >= V;
  float x_label = 0.0f;
  if (tid == 0 && !ignored && !bad) x_label = bf16_to_f32(x[label]);
  // (the values are unpacked anew in each pass, not kept: fresh hides that they are the same)
  auto fresh = [&]() __attribute__((always_inline)) {
#pragma unroll
    for (int j = 0; j < N; ++j) asm volatile("" : "+v"(r[j].x), "+v"(r[j].y), "+v"(r[j].z), "+v"(r[j].w));
  };
#pragma unroll
  for (int j = 0; j < N; ++j) {
    float v[8];
    unpack8(r[j], v);
    float lo = v[0];
#pragma unroll
    for (int k = 0; k < 8; ++k) {
      mx = fmaxf(mx, v[k]);
      lo = fminf(lo, v[k]);
    }
    if (j * THREADS + tid < n8) mn = fminf(mn, lo);
  }
  for (int off = 32; off > 0; off >>= 1) {
    mx = fmaxf(mx, __shfl_xor(mx, off, 64));
    mn = fminf(mn, __shfl_xor(mn, off, 64));
  }
  const int wave = tid >> 6;
  if ((tid & 63) == 0) {
    s_max[wave] = mx;
    s_min[wave] = mn;
  }
  __syncthreads();
  float m = s_max[0], least = s_min[0];
#pragma unroll
  for (int w = 1; w < W; ++w) {
    m = fmaxf(m, s_max[w]);
    least = fminf(least, s_min[w]);
  }
  // exp2's argument stays above -126 within 87 of the maximum
  const bool normal = __builtin_expect(m - least < 87.0f, 1);
  // A piece for the rows outside: one at a time, its arithmetic apart from what
  // ordinary rows do (shared with theirs, the pieces spilled).
  auto apart = [&](int j, float (&v)[8]) __attribute__((always_inline)) {
    __builtin_amdgcn_sched_barrier(0);
    uint4 p = r[j];
    asm volatile("; below the normal range" : "+v"(p.x), "+v"(p.y), "+v"(p.z), "+v"(p.w));
    unpack8(p, v);
  };
  float s = 0.0f, s1 = 0.0f;
  fresh();
  if (normal) {
#pragma unroll
    for (int j = 0; j < N; ++j) {
      float v[8];
      unpack8(r[j], v);
#pragma unroll
      for (int k = 0; k < 8; k += 2) {
        s += __builtin_amdgcn_exp2f((v[k] - m) * kLog2e);
        s1 += __builtin_amdgcn_exp2f((v[k + 1] - m) * kLog2e);
      }
    }
  } else {  // (terms made zero are under 2^-126 of a sum of at least 1)
#pragma unroll
    for (int j = 0; j < N; ++j) {
      float v[8];
      apart(j, v);
#pragma unroll
      for (int k = 0; k < 8; k += 2) {
        s += __builtin_amdgcn_exp2f((v[k] - m) * kLog2e);
        s1 += __builtin_amdgcn_exp2f((v[k + 1] - m) * kLog2e);
      }
    }
  }
  s += s1;
  for (int off = 32; off > 0; off >>= 1) s += __shfl_xor(s, off, 64);
  if ((tid & 63) == 0) s_sum[wave] = s;
  __syncthreads();  // (and every read of the row is done)
  s = s_sum[0];
#pragma unroll
  for (int w = 1; w < W; ++w) s += s_sum[w];
  if (tid == 0) {
    float l = 0.0f;
    if (bad) {
      l = __builtin_nanf("");
    } else if (!ignored) {
      l = m + log2f(s) * kLn2 - x_label;
    }
    row_loss[row] = l;
  }
  if (!dlogits) return;
  uint16_t* d = dlogits + row * ldd;
  const float g = ignored ? 0.0f : scale * (1.0f / s);
  const int hot = ignored ? -1 : label;
  auto store = [&](int i, float (&v)[8]) __attribute__((always_inline)) {
    if (hot >> 3 == i) {
#pragma unroll
      for (int k = 0; k < 8; ++k)
        if ((hot & 7) == k) v[k] -= scale;
    }
    if (i < n8) {
      reinterpret_cast<uint4*>(d)[i] = make_uint4(pack_bf16x2(v[0], v[1]), pack_bf16x2(v[2], v[3]),
                                                  pack_bf16x2(v[4], v[5]), pack_bf16x2(v[6], v[7]));
    } else {
#pragma unroll
      for (int k = 0; k < 7; ++k)
        if (k < rest) d[i * 8 + k] = f32_to_bf16(v[k]);
    }
  };
  if (!normal) {
#pragma unroll
    for (int j = 0; j < N; ++j) {
      const int i = j * THREADS + tid;
      if (i * 8 >= V) continue;
      float v[8];
      apart(j, v);
#pragma unroll
      for (int k = 0; k < 8; ++k) v[k] = exp2f((v[k] - m) * kLog2e) * g;
      store(i, v);
    }
    return;
  }
  fresh();
#pragma unroll
  for (int j = 0; j < N; ++j) {
    const int i = j * THREADS + tid;
    if (i * 8 >= V) continue;
    float v[8];
    unpack8(r[j], v);
#pragma unroll
    for (int k = 0; k < 8; ++k) v[k] = __builtin_amdgcn_exp2f((v[k] - m) * kLog2e) * g;
    store(i, v);
  }
}

// loss = scale * sum of the row losses, in a fixed order (fp64 partials).
__global__ __launch_bounds__(1024) void ce_finalize(const float* __restrict__ row_loss, int64_t T,
                                                    float scale, float* __restrict__ loss_out) {
  __shared__ double sm[16];
  double acc = 0.0;
  for (int64_t i = threadIdx.x; i < T; i += 1024) acc += static_cast<double>(row_loss[i]);
  for (int off = 32; off > 0; off >>= 1) acc += __shfl_xor(acc, off, 64);
  if ((threadIdx.x & 63) == 0) sm[threadIdx.x >> 6] = acc;
  __syncthreads();
  if (threadIdx.x == 0) {
    double t = 0.0;
    for (int w = 0; w < 16; ++w) t += sm[w];
    loss_out[0] = static_cast<float>(t * static_cast<double>(scale));
  }
}

constexpr int kEmbBlock = 256;

// out[t, :] = table[ids[t], :] widened to fp32; an id outside [0, V) gives a
// row of NaN so that a bad token cannot pass unnoticed.
template <int DT, bool VEC>
__global__ __launch_bounds__(kEmbBlock) void embed_rows(const void* __restrict__ table, int64_t ldt,
                                                        int64_t V, int64_t H,
                                                        const int32_t* __restrict__ ids,
                                                        float* __restrict__ out, int64_t ldo) {
  const int64_t t = blockIdx.x;
  const int id = ids[t];
  float* o = out + t * ldo;
  const bool bad = id < 0 || id >= V;
  if constexpr (VEC) {
    const int64_t n8 = H / 8;
    for (int64_t i = threadIdx.x; i < n8; i += kEmbBlock) {
      float v[8];
      if (bad) {
#pragma unroll
        for (int k = 0; k < 8; ++k) v[k] = __builtin_nanf("");
      } else {
        load8<DT>(table, static_cast<int64_t>(id) * ldt + i * 8, v);
      }
      float4* o4 = reinterpret_cast<float4*>(o + i * 8);
      o4[0] = make_float4(v[0], v[1], v[2], v[3]);
      o4[1] = make_float4(v[4], v[5], v[6], v[7]);
    }
  } else {
    for (int64_t i = threadIdx.x; i < H; i += kEmbBlock)
      o[i] = bad ? __builtin_nanf("") : load_elem<DT>(table, static_cast<int64_t>(id) * ldt + i);
  }
}

}  // namespace
}  // namespace mr

extern "C" {

int mr_cross_entropy(const void* logits, int64_t ld, int64_t T, int64_t V, const int32_t* labels,
                     float scale, float* row_loss, float* loss_out, void* dlogits, int64_t ldd,
                     void* stream) {
  using namespace mr;
  clear_error();
  if (T < 0 || V <= 0) return fail(MR_EINVAL, "mr_cross_entropy: bad sizes T=%lld V=%lld",
                                   static_cast<long long>(T), static_cast<long long>(V));
  if (!logits || !labels || !row_loss) return fail(MR_EINVAL, "mr_cross_entropy: null pointer");
  if (ld < V || (dlogits && ldd < V))
    return fail(MR_EINVAL, "mr_cross_entropy: a leading dimension is smaller than V");
  if (T > 0x7fffffff) return fail(MR_EINVAL, "mr_cross_entropy: too many rows");
  hipStream_t s = static_cast<hipStream_t>(stream);
  if (T > 0) {
    const uint16_t* x = static_cast<const uint16_t*>(logits);
    uint16_t* d = static_cast<uint16_t*>(dlogits);
    const bool rows16 = ld % 8 == 0 && aligned16(x) && (!d || (ldd % 8 == 0 && aligned16(d)));
    const bool vec = V % 8 == 0 && rows16;
    const int64_t pieces = (V + 7) / 8;
#define MR_CE(THREADS, N)                                                                                     \
  hipLaunchKernelGGL((ce_rows_held<THREADS, N>), dim3(static_cast<unsigned>(T)), dim3(THREADS), 0, s, x, ld,  \
                     static_cast<int>(V), labels, scale, row_loss, d, ldd)
    // the fewest threads that hold the row in at most 8 pieces each, then more pieces
    if (rows16 && pieces <= 256 * 4) MR_CE(256, 4);
    else if (rows16 && pieces <= 256 * 8) MR_CE(256, 8);
    else if (rows16 && pieces <= 512 * 8) MR_CE(512, 8);
    else if (rows16 && pieces <= kHeldThreads * 8) MR_CE(kHeldThreads, 8);
    else if (rows16 && pieces <= kHeldThreads * 14) MR_CE(kHeldThreads, 14);
    else if (rows16 && V <= kHeldMax) MR_CE(kHeldThreads, kHeldPieces);
#undef MR_CE
    else if (vec)
      hipLaunchKernelGGL(ce_rows<true>, dim3(static_cast<unsigned>(T)), dim3(kCeBlock), 0, s, x, ld,
                         V, labels, scale, row_loss, d, ldd);
    else
      hipLaunchKernelGGL(ce_rows<false>, dim3(static_cast<unsigned>(T)), dim3(kCeBlock), 0, s, x,
                         ld, V, labels, scale, row_loss, d, ldd);
    MR_LAUNCH_CHECK("mr_cross_entropy");
  }
  if (loss_out) {
    hipLaunchKernelGGL(ce_finalize, dim3(1), dim3(1024), 0, s, row_loss, T, scale, loss_out);
    MR_LAUNCH_CHECK("mr_cross_entropy");
  }
  return MR_OK;
}

int mr_embed_rows(const void* table, int dtype, int64_t V, int64_t H, int64_t ldt,
                  const int32_t* ids, int64_t T, float* out, int64_t ldo, void* stream) {
  using namespace mr;
  clear_error();
  if (T < 0 || V <= 0 || H <= 0) return fail(MR_EINVAL, "mr_embed_rows: bad sizes");
  if (T == 0) return MR_OK;
  if (!table || !ids || !out) return fail(MR_EINVAL, "mr_embed_rows: null pointer");
  if (!valid_dtype(dtype)) return fail(MR_EINVAL, "mr_embed_rows: bad table dtype %d", dtype);
  if (ldt < H || ldo < H) return fail(MR_EINVAL, "mr_embed_rows: a leading dimension is smaller than H");
  if (T > 0x7fffffff) return fail(MR_EINVAL, "mr_embed_rows: too many rows");
  hipStream_t s = static_cast<hipStream_t>(stream);
  const bool vec = H % 8 == 0 && ldt % 8 == 0 && ldo % 4 == 0 && aligned16(table) && aligned16(out);
  const dim3 g(static_cast<unsigned>(T)), b(kEmbBlock);
#define MR_EMB(DT)                                                                          \
  if (vec)                                                                                  \
    hipLaunchKernelGGL((embed_rows<DT, true>), g, b, 0, s, table, ldt, V, H, ids, out, ldo); \
  else                                                                                      \
    hipLaunchKernelGGL((embed_rows<DT, false>), g, b, 0, s, table, ldt, V, H, ids, out, ldo);
  if (dtype == MR_BF16) {
    MR_EMB(MR_BF16)
  } else if (dtype == MR_F16) {
    MR_EMB(MR_F16)
  } else {
    MR_EMB(MR_F32)
  }
#undef MR_EMB
  MR_LAUNCH_CHECK("mr_embed_rows");
  return MR_OK;
}

}  // extern "C"
