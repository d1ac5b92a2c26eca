// fp32 GEMMs of gfx950 for the products that must keep float32 precision: the
// single-layer tuning loop's layer residual x (W' - W)^T and weight gradient
// (dL/dr)^T x, which the reference forms in float32
// (mround/core/tuning.py:140-190).
//
// C[M, N] = sum_k A(m, k) * (B(n, k) - B2(n, k)) (B2 optional), with each
// operand K-major (k contiguous) or MN-major (k the row index), as mr_gemm's
// layouts. Any sizes.
//
// The products run on the bf16 matrix cores, 16 times the rate of the fp32
// MFMA, without giving up float32's bits. Each value is split as it is staged
// into three bfloat16 planes, h = bf16(x), m = bf16(x - h), l = x - h - m: the
// two differences are exact and l has at most 8 significant bits left, so
// h + m + l is x. Of the nine plane products the six down to 2^-16 of the
// largest are formed (each exact in the MFMA): h h into one accumulator and
// h m + m h + h l + m m + l h into a second, added once at the end. The three
// left out are at most 2^-24 of a product together, as much as a float32
// product's own rounding; the sum itself rounds once per 16 k instead of once
// per 2 k. Measured against float64 over K = 64 .. 6000: 0.15-0.4 of the fp32 MFMA
// form's error (normwise 5e-8 .. 4e-7 against 1.4e-7 .. 1.4e-6).
//
// The split is exact while l's last bit stays in bfloat16's range and h does
// not overflow. A block that met a nonzero |x| below 2^-100 (tested on x, not on
// h: below 2^-133 h itself rounds to zero), or whose sums are not all finite (an infinity or a NaN among its operands makes them so, as a
// value that rounds to infinity does), forms its tile again with the fp32
// MFMA, so infinities, NaNs and denormals come out as float32 arithmetic has
// them.
//
// A block of 256 threads (4 waves, 2 x 2) owns a 128 x 128 tile of C, a wave
// 64 x 64 of it, one wave per SIMD. Operand tiles of 32 k move through registers
// (16 values of each operand a thread, B - B2 formed on the way) and are split
// into two LDS stages of 48 KB, rows of 64 bytes whose 16-byte chunk c sits at
// c ^ ((row >> 2) & 3): the 16 rows an LDS cycle serves cover the 64 banks (no
// bank conflicts counted). What bounds it is issue: about 270 VALU
// instructions of splitting a wave and k tile against 48 MFMAs of 32 cycles,
// so the splitting is spread between the MFMAs, six or seven after each, which
// an MFMA hides (as two phases with two blocks to a CU, one splitting while
// the other multiplies, MFMAs were busy 35 % of the time: 3000 x 2048 x 3072
// ran 309 us against 242). Grids that leave CUs idle are cut along K (see
// split_plan), raw partial tiles to the caller's workspace and a fixed-order
// sum after.
// Measured against the fp32 MFMA kernel before it: the 0.5B down projection's
// residual (1000 x 896 x 4864, with B2) 1527 -> 72 us and its gradient
// (896 x 4864 x 1000) 197 -> 83 us; 3000 x 2048 x 3072 718 -> 242 us, 156
// TFLOP/s of float32 product (the fp32 MFMA's peak is 157).
#include <type_traits>

#include "mr_common.h"

namespace mr {
namespace {

typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

constexpr int TM = 128, TN = 128, TK = 32;
constexpr int kThreads = 256;
constexpr int PER = TM * TK / kThreads;  // operand values each thread moves per tile
constexpr int PAD = 4;                   // LDS row padding of the fp32 form (floats)
constexpr int PLANE = TM * TK * 2;       // bytes of one plane of one operand tile
constexpr int kStage = 6 * PLANE;        // both operands
static_assert(TM == TN && 2 * kStage >= 2 * TK * (TM + PAD) * 4, "the fp32 form stages in the same LDS");
// Smallest admissible (bits << 1) - 2 of a nonzero value, 2^-100 (zeros wrap to
// the top).
constexpr uint32_t kKeyLo = ((127u - 100u) << 24) - 2;

struct Operand {
  const float* x;
  const float* minus;  // subtracted element by element, or null (same ld)
  int64_t ld;
  int rows;
};

// Value (r, k) of a K-major (x[r * ld + k]) or MN-major (x[k * ld + r])
// operand, zero outside rows x K.
template <bool KMAJOR>
__device__ __forceinline__ float at(const Operand& o, int r, int k, int K) {
  if (r >= o.rows || k >= K) return 0.0f;
  const int64_t i = KMAJOR ? static_cast<int64_t>(r) * o.ld + k : static_cast<int64_t>(k) * o.ld + r;
  return o.minus ? o.x[i] - o.minus[i] : o.x[i];
}

// A thread's 16 values of an operand tile: two rows (j) of 8 consecutive k.
// K-major: 4 threads read a row's 32 k, 64 rows apart for j. MN-major: a wave
// reads 128 consecutive rows at each of its 8 k.
template <bool KMAJOR>
__device__ __forceinline__ int slot_row(int j) {
  const int t = threadIdx.x;
  return KMAJOR ? (t >> 2) + 64 * j : 2 * (t & 63) + j;
}
template <bool KMAJOR>
__device__ __forceinline__ int slot_chunk() {
  const int t = threadIdx.x;
  return KMAJOR ? t & 3 : t >> 6;
}

// One operand's share of a tile in registers, from row row0 and k0 on, and its
// three planes. PAIRS: an MN-major operand's row pairs lie whole and 8-byte
// aligned (ld and rows even) and are read as such. Rows past the edge repeat
// valid ones (their products are not stored).
struct Planes {
  u32x4 v[2][3];
  template <bool KMAJOR>
  __device__ __forceinline__ void write(uint8_t* lds) const {
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      const int row = slot_row<KMAJOR>(j);
      uint8_t* p = lds + row * (TK * 2) + ((slot_chunk<KMAJOR>() ^ ((row >> 2) & 3)) << 4);
#pragma unroll
      for (int q = 0; q < 3; ++q) *reinterpret_cast<u32x4*>(p + q * PLANE) = v[j][q];
    }
  }
};

template <bool KMAJOR, bool PAIRS, bool MINUS>
struct Share {
  float x[2][8], y[MINUS ? 2 : 1][8];
  // A whole k tile.
  __device__ __forceinline__ void load(const Operand& o, int row0, int k0) {
    const int k = k0 + slot_chunk<KMAJOR>() * 8;
    read(o.x, o, row0, k, x);
    if constexpr (MINUS) read(o.minus, o, row0, k, y);
  }
  // The rest of K past the last whole tile, zeros beyond.
  __device__ __forceinline__ void load_tail(const Operand& o, int row0, int k0, int K) {
    const int k = k0 + slot_chunk<KMAJOR>() * 8;
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        x[j][e] = at<KMAJOR>(o, row0 + slot_row<KMAJOR>(j), k + e, K);
        if constexpr (MINUS) y[j][e] = 0.0f;  // (already subtracted)
      }
  }
  __device__ __forceinline__ static void read(const float* p, const Operand& o, int row0, int k, float (&v)[2][8]) {
    if constexpr (!KMAJOR && PAIRS) {
      const float* q = p + static_cast<int64_t>(k) * o.ld + min(row0 + slot_row<false>(0), o.rows - 2);
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        const float2 a = *reinterpret_cast<const float2*>(q + e * o.ld);
        v[0][e] = a.x;
        v[1][e] = a.y;
      }
    } else {
#pragma unroll
      for (int j = 0; j < 2; ++j) {
        const int r = min(row0 + slot_row<KMAJOR>(j), o.rows - 1);
        const float* q = KMAJOR ? p + static_cast<int64_t>(r) * o.ld + k : p + static_cast<int64_t>(k) * o.ld + r;
#pragma unroll
        for (int e = 0; e < 8; ++e) v[j][e] = q[KMAJOR ? e : e * o.ld];  // (K-major: 16-byte loads)
      }
    }
  }
  // The share's three planes; `key` collects the smallest magnitude key.
  __device__ __forceinline__ void split(Planes& p, uint32_t& key) const {
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        float a = x[j][2 * q], b = x[j][2 * q + 1];
        if constexpr (MINUS) {
          a = a - y[j][2 * q];
          b = b - y[j][2 * q + 1];
        }
        const uint32_t h = pack_bf16x2(a, b);
        key = min(key, min((__float_as_uint(a) << 1) - 2, (__float_as_uint(b) << 1) - 2));
        const float a1 = a - __uint_as_float(h << 16), b1 = b - __uint_as_float(h & 0xffff0000u);
        const uint32_t m = pack_bf16x2(a1, b1);
        p.v[j][0][q] = h;
        p.v[j][1][q] = m;
        p.v[j][2][q] = pack_bf16x2(a1 - __uint_as_float(m << 16), b1 - __uint_as_float(m & 0xffff0000u));
      }
  }
};

// The tile by the fp32 MFMA over k in [k_lo, k_hi), the next k tile's loads in
// flight during this one's MFMAs. (Loaded and multiplied in turn, it took two to
// three times as long: 4096 x 3584 x 3584 with such a value in every block 4400
// us, 1980 here, 1250-1580 on the fp32 MFMA alone; 896 x 4864 x 1000 375, 200 and
// 190-240; 1000 x 896 x 4864 less B2 490, 380 and 1240.)
template <bool A_KMAJOR, bool B_KMAJOR>
__device__ __forceinline__ void tile_fp32(const Operand& A, const Operand& B, int m0, int n0, int k_lo, int k_hi,
                                          uint8_t* lds, f32x16 (&acc)[2][2]) {
  float(*As)[TM + PAD] = reinterpret_cast<float(*)[TM + PAD]>(lds);
  float(*Bs)[TN + PAD] = reinterpret_cast<float(*)[TN + PAD]>(lds + TK * (TM + PAD) * 4);
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int wm = wave >> 1, wn = wave & 1, l32 = lane & 31, kh = lane >> 5;
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j) acc[i][j] = f32x16{};
  float ra[PER], rb[PER];
  auto slot = [](int i, bool kmajor, int& r, int& k) __attribute__((always_inline)) {
    const int idx = i * kThreads + static_cast<int>(threadIdx.x);
    r = kmajor ? idx / TK : idx % TM;
    k = kmajor ? idx % TK : idx / TM;
  };
  auto load = [&](int k0) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < PER; ++i) {
      int r, k;
      slot(i, A_KMAJOR, r, k);
      ra[i] = at<A_KMAJOR>(A, m0 + r, k0 + k, k_hi);
      slot(i, B_KMAJOR, r, k);
      rb[i] = at<B_KMAJOR>(B, n0 + r, k0 + k, k_hi);
    }
  };
  load(k_lo);
  for (int k0 = k_lo; k0 < k_hi; k0 += TK) {
    __syncthreads();  // every read of the previous tile (or of the planes) is done
#pragma unroll
    for (int i = 0; i < PER; ++i) {
      int r, k;
      slot(i, A_KMAJOR, r, k);
      As[k][r] = ra[i];
      slot(i, B_KMAJOR, r, k);
      Bs[k][r] = rb[i];
    }
    __syncthreads();
    if (k0 + TK < k_hi) load(k0 + TK);
#pragma unroll
    for (int kk = 0; kk < TK; kk += 2) {
      float a[2], b[2];
#pragma unroll
      for (int i = 0; i < 2; ++i) a[i] = As[kk + kh][wm * 64 + i * 32 + l32];
#pragma unroll
      for (int j = 0; j < 2; ++j) b[j] = Bs[kk + kh][wn * 64 + j * 32 + l32];
#pragma unroll
      for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j)
          acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x2f32(b[j], a[i], acc[i][j], 0, 0, 0);
    }
  }
}

struct Gemm32 {
  int M, N, K;
  Operand A, B;
  float* C;
  int64_t ldc;
  int grid_m, grid_n;
  // Tiles 0 .. full - 1 take a block each; the `tail` after them ksplit blocks
  // each (of kt_per k tiles), whose TM x TN partials go to ws, tile by tile.
  int full, tail, ksplit, kt_per;
  float* ws;
};

// The MFMA operands of one k16 step: two 32-row blocks of each operand, three planes.
struct Frags {
  bf16x8 a[2][3], b[2][3];
};

template <bool A_KMAJOR, bool B_KMAJOR, bool PAIRS, bool MINUS>
__global__ __launch_bounds__(kThreads, 1) void gemm_f32_kernel(Gemm32 p) {
  __shared__ __attribute__((aligned(1024))) uint8_t lds[2 * kStage];
  // Consecutive tiles (of one split) share operand panels: each XCD (blocks
  // are dealt to the eight round-robin) takes a contiguous run of them.
  const int cut = blockIdx.x >= static_cast<unsigned>(p.full);
  const int blocks = cut ? p.tail * p.ksplit : p.full;
  int bid = static_cast<int>(blockIdx.x) - (cut ? p.full : 0);
  bid = (bid & 7) * (blocks >> 3) + min(bid & 7, blocks & 7) + (bid >> 3);
  const int split = cut ? bid / p.tail : 0, tile = cut ? p.full + bid % p.tail : bid;
  const int m0 = (tile / p.grid_n) * TM, n0 = (tile % p.grid_n) * TN;
  const int k_lo = split * p.kt_per * TK;
  const int k_hi = !cut || split + 1 == p.ksplit ? p.K : k_lo + p.kt_per * TK;
  const int whole = (k_hi - k_lo) / TK;  // k tiles of the pipelined loop
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int wm = wave >> 1, wn = wave & 1;
  const int l32 = lane & 31, kh = lane >> 5;

  f32x16 acc[2][2], low[2][2];
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j) acc[i][j] = low[i][j] = f32x16{};
  uint32_t key = 0xffffffffu;

  Share<A_KMAJOR, PAIRS, false> sa[2];
  Share<B_KMAJOR, PAIRS, MINUS> sb[2];
  Planes pa;
  Frags fr[2];
  auto load = [&](int u, int par) __attribute__((always_inline)) {
    const int k0 = k_lo + min(u, whole - 1) * TK;  // (a repeat of the last tile is never used)
    sa[par].load(p.A, m0, k0);
    sb[par].load(p.B, n0, k0);
  };
  auto frags = [&](const uint8_t* st, int kk, Frags& f) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const int ra = wm * 64 + i * 32 + l32, rb = wn * 64 + i * 32 + l32, c = kk * 2 + kh;
#pragma unroll
      for (int q = 0; q < 3; ++q) {
        f.a[i][q] = *reinterpret_cast<const bf16x8*>(st + q * PLANE + ra * (TK * 2) + ((c ^ ((ra >> 2) & 3)) << 4));
        f.b[i][q] = *reinterpret_cast<const bf16x8*>(st + (3 + q) * PLANE + rb * (TK * 2) + ((c ^ ((rb >> 2) & 3)) << 4));
      }
    }
  };
  // B is the first operand: accumulator register r of lane l holds
  // C[row m = l % 32][column n = (r / 4) * 8 + (l / 32) * 4 + r % 4].
  auto mul = [&](const Frags& f) __attribute__((always_inline)) {
    auto mm = [&](f32x16(&d)[2][2], int qa, int qb) __attribute__((always_inline)) {
#pragma unroll
      for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j)
          d[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(f.b[j][qb], f.a[i][qa], d[i][j], 0, 0, 0);
    };
    mm(acc, 0, 0);
    mm(low, 2, 0);
    mm(low, 0, 2);
    mm(low, 1, 1);
    mm(low, 1, 0);
    mm(low, 0, 1);
  };
  // The order of a half step: each MFMA followed by what it can hide.
  auto order = [](auto first) __attribute__((always_inline)) {
    constexpr bool A = decltype(first)::value;
#pragma unroll
    for (int q = 0; q < 24; ++q) {
      __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);  // MFMA
      if (q & 1) __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);       // LDS read
      else if (A) __builtin_amdgcn_sched_group_barrier(0x200, 1, 0);      // LDS write
      __builtin_amdgcn_sched_group_barrier(0x002, A && MINUS ? 7 : 6, 0);  // VALU
    }
    __builtin_amdgcn_sched_barrier(0);
  };
  // Tile u, in stage u % 2, its first k16 step's operands already read. First
  // half: tile u + 1's B is split and both its operands' planes go to the other
  // stage, and tile u + 3's loads go out. A barrier. Second half: that stage's
  // first operands are read, and tile u + 2's A is split into registers.
  auto step = [&](int u, auto parc) __attribute__((always_inline)) {
    constexpr int par = decltype(parc)::value;
    const uint8_t* cur = lds + par * kStage;
    uint8_t* nxt = lds + (par ^ 1) * kStage;
    frags(cur, 1, fr[1]);
    pa.template write<A_KMAJOR>(nxt);
    Planes pb;
    sb[par ^ 1].split(pb, key);
    pb.template write<B_KMAJOR>(nxt + 3 * PLANE);
    mul(fr[0]);
    order(std::true_type{});
    load(u + 3, par ^ 1);
    // (the loads stay in flight across the barrier)
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_sched_barrier(0);
    frags(nxt, 0, fr[0]);
    sa[par].split(pa, key);
    mul(fr[1]);
    order(std::false_type{});
  };
  if (whole > 0) {
    load(0, 0);
    load(1, 1);
    Planes pb;
    sa[0].split(pa, key);
    sb[0].split(pb, key);
    pa.template write<A_KMAJOR>(lds);
    pb.template write<B_KMAJOR>(lds + 3 * PLANE);
    load(2, 0);
    sa[1].split(pa, key);
    __syncthreads();
    frags(lds, 0, fr[0]);
    for (int u = 0; u < whole; u += 2) {
      step(u, std::integral_constant<int, 0>{});
      if (u + 1 < whole) step(u + 1, std::integral_constant<int, 1>{});
    }
  }
  if (whole * TK < k_hi - k_lo) {
    Planes pb;
    sa[0].load_tail(p.A, m0, k_lo + whole * TK, k_hi);
    sb[0].load_tail(p.B, n0, k_lo + whole * TK, k_hi);
    sa[0].split(pa, key);
    sb[0].split(pb, key);
    __syncthreads();
    pa.template write<A_KMAJOR>(lds);
    pb.template write<B_KMAJOR>(lds + 3 * PLANE);
    __syncthreads();
#pragma unroll
    for (int kk = 0; kk < 2; ++kk) {
      frags(lds, kk, fr[0]);
      mul(fr[0]);
    }
  }
  bool bad = key < kKeyLo;
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const int m = m0 + wm * 64 + i * 32 + l32;
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      acc[i][j] += low[i][j];
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const int n = n0 + wn * 64 + j * 32 + (r >> 2) * 8 + kh * 4 + (r & 3);
        bad |= m < p.M && n < p.N && !(fabsf(acc[i][j][r]) <= 3.402823466e38f);
      }
    }
  }
  if (__syncthreads_or(bad)) tile_fp32<A_KMAJOR, B_KMAJOR>(p.A, p.B, m0, n0, k_lo, k_hi, lds, acc);

  const bool part = cut && p.ksplit > 1;
  float* const out = part ? p.ws + (static_cast<int64_t>(tile - p.full) * p.ksplit + split) * (TM * TN)
                          : p.C + static_cast<int64_t>(m0) * p.ldc + n0;
  const int64_t ld = part ? TN : p.ldc;
  const int rows = part ? TM : p.M - m0, cols = part ? TN : p.N - n0;
  const bool vec = part || ((p.ldc & 3) == 0 && (reinterpret_cast<uintptr_t>(p.C) & 15) == 0);
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const int m = wm * 64 + i * 32 + l32;
    if (m >= rows) continue;
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int g = 0; g < 4; ++g) {
        const int n = wn * 64 + j * 32 + g * 8 + kh * 4;
        float* o = out + m * ld + n;
        if (vec && n + 4 <= cols) {
          *reinterpret_cast<f32x4*>(o) =
              f32x4{acc[i][j][4 * g], acc[i][j][4 * g + 1], acc[i][j][4 * g + 2], acc[i][j][4 * g + 3]};
        } else {
#pragma unroll
          for (int r = 0; r < 4; ++r)
            if (n + r < cols) o[r] = acc[i][j][4 * g + r];
        }
      }
  }
}

// The tail's C from its partial tiles, splits in order; a thread per 4 columns.
__global__ __launch_bounds__(kThreads) void gemm_f32_reduce(Gemm32 p) {
  const int64_t idx = static_cast<int64_t>(blockIdx.x) * kThreads + threadIdx.x;
  const int tile = static_cast<int>(idx / (TM * TN / 4)), rem = static_cast<int>(idx % (TM * TN / 4));
  const int r = rem / (TN / 4), c = rem % (TN / 4) * 4;
  const int m = ((p.full + tile) / p.grid_n) * TM + r, n = ((p.full + tile) % p.grid_n) * TN + c;
  if (m >= p.M || n >= p.N) return;
  const float* part = p.ws + static_cast<int64_t>(tile) * p.ksplit * (TM * TN) + r * TN + c;
  f32x4 s = *reinterpret_cast<const f32x4*>(part);
  for (int sp = 1; sp < p.ksplit; ++sp) s += *reinterpret_cast<const f32x4*>(part + static_cast<int64_t>(sp) * (TM * TN));
  float* o = p.C + static_cast<int64_t>(m) * p.ldc + n;
#pragma unroll
  for (int q = 0; q < 4; ++q)
    if (n + q < p.N) o[q] = s[q];
}

// One block runs on a CU at a time, so tiles go out in whole rounds of 256,
// and what remains (or a grid under one round) is cut along K. The split that
// takes the least time, in k tiles: rounds of the split's k tiles and about 6
// more for a block's start and end, and the partials' round trip, about 8 and
// one for each 128 of them (measured, with B2: 1000 x 896 x 4864, 56 tiles,
// 197 us whole and 70 cut in 4; 896 x 4864 x 1000, 266 tiles, 129 us whole and
// 94 with the last 10 cut in 7). At least 4 k tiles to a split and one round
// of blocks (16 MB of partials).
int split_plan(int64_t tail, int64_t KT) {
  int best = 1;
  double best_t = static_cast<double>(KT + 6);
  for (int sp = 2; sp * 4 <= KT && tail * sp <= 256; ++sp) {
    const double t = static_cast<double>((KT + sp - 1) / sp + 6) + 8.0 + static_cast<double>(tail * sp) / 128.0;
    if (t < best_t) {
      best_t = t;
      best = sp;
    }
  }
  return best;
}

int64_t tiles_of(int64_t M, int64_t N) { return ((M + TM - 1) / TM) * ((N + TN - 1) / TN); }

// Whether an MN-major operand's row pairs lie whole and 8-byte aligned.
bool pairs_ok(const Operand& o) {
  const uintptr_t both = reinterpret_cast<uintptr_t>(o.x) | reinterpret_cast<uintptr_t>(o.minus);
  return (both & 7) == 0 && o.ld % 2 == 0 && o.rows % 2 == 0;
}

}  // namespace
}  // namespace mr

extern "C" {

size_t mr_gemm_f32_workspace_bytes(int64_t M, int64_t N, int64_t K) {
  using namespace mr;
  if (M <= 0 || N <= 0 || K <= 0) return 0;
  const int64_t tail = tiles_of(M, N) % 256;
  const int sp = split_plan(tail, (K + TK - 1) / TK);
  return sp == 1 ? 0 : static_cast<size_t>(tail) * sp * TM * TN * 4;
}

int mr_gemm_f32_ws(int layout, int64_t M, int64_t N, int64_t K, const float* A, int64_t lda, const float* B,
                   const float* B2, int64_t ldb, float* C, int64_t ldc, void* workspace, size_t workspace_bytes,
                   void* stream) {
  using namespace mr;
  clear_error();
  if (M < 0 || N < 0 || K < 0) return fail(MR_EINVAL, "mr_gemm_f32: negative size");
  if (M == 0 || N == 0) return MR_OK;
  if (!A || !B || !C) return fail(MR_EINVAL, "mr_gemm_f32: null operand");
  if (M > 0x7fffffff || N > 0x7fffffff || K > 0x7fffffff) return fail(MR_EINVAL, "mr_gemm_f32: too large");
  if (layout < 0 || layout > 2) return fail(MR_EINVAL, "mr_gemm_f32: unknown layout %d", layout);
  const bool a_kmajor = layout != 2, b_kmajor = layout == 0;
  if (lda < (a_kmajor ? K : M) || ldb < (b_kmajor ? K : N) || ldc < N)
    return fail(MR_EINVAL, "mr_gemm_f32: a leading dimension is smaller than its row");
  if ((M + TM - 1) / TM > 65535) return fail(MR_EINVAL, "mr_gemm_f32: M above %d", 65535 * TM);
  const int64_t tiles = tiles_of(M, N), KT = (K + TK - 1) / TK;
  if (tiles > 0x7fffffff) return fail(MR_EINVAL, "mr_gemm_f32: too large");
  if (workspace && !aligned16(workspace)) return fail(MR_EINVAL, "mr_gemm_f32: workspace must be 16-byte aligned");
  Gemm32 p{};
  p.M = static_cast<int>(M);
  p.N = static_cast<int>(N);
  p.K = static_cast<int>(K);
  p.A = Operand{A, nullptr, lda, p.M};
  p.B = Operand{B, B2, ldb, p.N};
  p.C = C;
  p.ldc = ldc;
  p.grid_m = static_cast<int>((M + TM - 1) / TM);
  p.grid_n = static_cast<int>((N + TN - 1) / TN);
  p.tail = static_cast<int>(tiles % 256);
  p.full = static_cast<int>(tiles - p.tail);
  int sp = workspace ? split_plan(p.tail, KT) : 1;
  if (static_cast<size_t>(p.tail) * sp * TM * TN * 4 > workspace_bytes) sp = 1;
  if (sp > 1) {  // tiles read operand panels while others write their partials
    const int64_t n = static_cast<int64_t>(p.tail) * sp * TM * TN * 4;
    auto span = [](int64_t rows, int64_t ld, int64_t width) { return ((rows - 1) * ld + width) * 4; };
    const int64_t a = a_kmajor ? span(M, lda, K) : span(K, lda, M), b = b_kmajor ? span(N, ldb, K) : span(K, ldb, N);
    if (overlap(workspace, n, A, a) || overlap(workspace, n, B, b) || (B2 && overlap(workspace, n, B2, b)) ||
        overlap(workspace, n, C, span(M, ldc, N)))
      return fail(MR_EINVAL, "mr_gemm_f32: the workspace must not overlap A, B, B2 or C");
  }
  const int64_t per = KT ? (KT + sp - 1) / sp : 0;
  p.kt_per = static_cast<int>(per);
  p.ksplit = per ? static_cast<int>((KT + per - 1) / per) : 1;  // no empty split
  p.ws = static_cast<float*>(workspace);
  const dim3 grid(static_cast<unsigned>(p.full + static_cast<int64_t>(p.tail) * p.ksplit));
  hipStream_t s = static_cast<hipStream_t>(stream);
  const bool pairs = (a_kmajor || pairs_ok(p.A)) && (b_kmajor || pairs_ok(p.B));
#define MR_G32(AK, BK_, P)                                                                             \
  if (B2) hipLaunchKernelGGL((gemm_f32_kernel<AK, BK_, P, true>), grid, dim3(kThreads), 0, s, p);      \
  else hipLaunchKernelGGL((gemm_f32_kernel<AK, BK_, P, false>), grid, dim3(kThreads), 0, s, p)
  if (layout == 0) {
    MR_G32(true, true, false);
  } else if (layout == 1) {
    if (pairs) { MR_G32(true, false, true); }
    else { MR_G32(true, false, false); }
  } else {
    if (pairs) { MR_G32(false, false, true); }
    else { MR_G32(false, false, false); }
  }
#undef MR_G32
  if (p.tail && p.ksplit > 1)
    hipLaunchKernelGGL(gemm_f32_reduce, dim3(static_cast<unsigned>(p.tail * (TM * TN / 4 / kThreads))), dim3(kThreads),
                       0, s, p);
  MR_LAUNCH_CHECK("mr_gemm_f32");
  return MR_OK;
}

int mr_gemm_f32(int layout, int64_t M, int64_t N, int64_t K, const float* A, int64_t lda, const float* B,
                const float* B2, int64_t ldb, float* C, int64_t ldc, void* stream) {
  return mr_gemm_f32_ws(layout, M, N, K, A, lda, B, B2, ldb, C, ldc, nullptr, 0, stream);
}

}  // extern "C"
