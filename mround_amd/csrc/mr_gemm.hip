// bf16 GEMMs on the MFMA cores of gfx950, fp32 accumulation.
//
// C[M, N] = sum_k A(m, k) * B(n, k), with each operand stored either K-major
// (row-major with k contiguous: activations X[t, k], weights W[n, k]) or
// MN-major (k is the row index: dY[t, n] used as A(n, t) for dW = dY^T X, and
// W[k, n] used as B(n, k) for dX = dY W). The three products of a linear
// layer's forward and backward are therefore one kernel:
//   forward  Y  = X  W^T   A = X  (K-major)  B = W  (K-major)
//   input    dX = dY W     A = dY (K-major)  B = W  (MN-major)
//   weight   dW = dY^T X   A = dY (MN-major) B = X  (MN-major)
//
// Tiling: a block of 512 threads (8 waves of 64, 4 x 2) owns a BM x BN tile
// of C; each wave owns (BM/4) x (BN/2) as a grid of 32 x 32 accumulators fed by
// v_mfma_f32_32x32x16_bf16 (lane l: first operand row l%32, second operand
// row l%32, k half l/32; accumulator register r: first-operand index
// (r/4)*8 + (l/32)*4 + r%4, second-operand index l%32; the epilogues that
// stage their tile through LDS pass B first, so a lane holds one row of C and
// runs of 4 consecutive columns). Every
// operand tile moves HBM -> LDS by direct buffer loads (buffer_load ... lds,
// no registers) in the layout it has in memory: a K-major tile as rows of 64
// k, whose MFMA operand is one 16-byte LDS read; an MN-major tile as rows of
// one k, whose operand comes from two transposing LDS reads
// (ds_read_b64_tr_b16). Each lane's load offsets are fixed for the whole k
// loop (one 32-bit register per load); the k advance is in the scalar buffer
// base. The k loop is double-buffered in LDS with the next tile's loads in
// flight during the current tile's MFMAs, and within a tile the operands of
// the next k16 step are read while the current step's MFMAs run.
//
// Blocks are renumbered so that each XCD (blocks are dealt to the 8 XCDs
// round-robin) receives a contiguous run of tiles, grouped along M so that a
// run shares B panels in that XCD's L2.
#include <type_traits>

#include "mr_common.h"

namespace mr {
namespace {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x16 __attribute__((ext_vector_type(16)));

// 8 waves (two per SIMD) in a 4 x 2 grid: a 256 x 256 tile gives each wave
// 64 x 128 (128 accumulator registers), which leaves room for double-buffered
// operands and lets the two waves of a SIMD hide each other's LDS and
// barrier waits. A wave's columns start on a multiple of 64, which the SwiGLU
// epilogue's gate/up pairing needs.
constexpr int kWaves = 8;
constexpr int kThreads = 64 * kWaves;
// Waves 0-3 (one on each SIMD: the waves of a block are dealt to the four
// SIMDs so that waves w and w + 4 share one) issue every operand load of a
// tile, 16 each, right after the barrier; waves 4-7 go straight to their
// fragment reads and MFMAs. A wave stalls while the CU's load path takes its
// burst of direct loads, so this keeps one wave per SIMD issuing MFMAs at
// the start of every tile: measured 3-5 % faster on the 7B block's shapes
// than all eight waves loading (two loaders: 0-30 % slower).
constexpr int kLoaders = 4;
constexpr int kWaveRows = 4;  // waves along M
constexpr int BK = 64;
// LDS tiles are K-major rows of 64 bf16 (128 bytes, 8 chunks of 16 bytes)
// with no padding; chunk c of row r is stored at position c ^ ((r >> 1) & 7)
// (swz below), so the 16 rows one LDS cycle serves cover all 64 banks once.
constexpr int ROW_BYTES = BK * 2;

enum Epi : int {
  EPI_STORE = 0,   // C = acc (+ bias[n])
  EPI_RESID = 1,   // C = resid[m, n] + acc (+ bias[n]), fp32
  EPI_SWIGLU = 2,  // act = silu(g) * u from row-interleaved gate/up weights
  EPI_SWIGLU_BWD = 3,  // dgu (interleaved) from dact = acc and the saved gate/up
  EPI_SWIGLU_SPLIT = 4,  // SWIGLU with act written split, [hi | hi | lo] per row
};
constexpr bool is_swiglu(int epi) { return epi == EPI_SWIGLU || epi == EPI_SWIGLU_SPLIT; }

struct GemmParams {
  int M, N, K;
  const uint16_t* A;
  int64_t lda;
  const uint16_t* B;
  int64_t ldb;
  int n_out;           // SWIGLU: columns of act (B has 2 * n_out interleaved rows)
  void* C;
  int64_t ldc;
  const float* bias;
  const float* resid;
  int64_t ldr;
  uint16_t* gu;        // SWIGLU: gate/up copy, [M, 2 * n_out] bf16, interleaved like B
  int64_t ldgu;        // (SWIGLU_BWD reads the saved gate/up from gu and writes dgu to C)
  uint16_t* act;       // SWIGLU_SPLIT: hi alone, [M, n_out] (with gu), or null; C holds the split rows
  int64_t ldact;
  int grid_m, grid_n;
  // Tiles of this launch: logical tiles tile0 .. tile0 + n_tiles - 1 of the
  // grouped order. ksplit > 1: each tile's k steps are cut into ksplit runs
  // of kt_per steps (one block each), whose raw fp32 accumulators go to
  // ws[(tile - tile0) * ksplit + split] as BM x BN row-major partial tiles.
  int tile0, n_tiles, ksplit, kt_per;
  // sub = 1: this launch's tiles are the four quarters of each of the
  // (2 BM) x (2 BN) tiles tile0 .. of the grid_m x grid_n grid (see launch).
  int sub;
  float* ws;         // k-split partials (caller's workspace), or null: no split
  int64_t ws_bytes;
};

// Logical tile -> (tile row, tile column): groups of 8 tile rows, column by
// column within a group, so that consecutive tiles share B panels.
__device__ __forceinline__ void tile_coords(int lt, int grid_m, int grid_n, int& bm, int& bn) {
  constexpr int GROUP_M = 8;
  const int per_group = GROUP_M * grid_n;
  const int group = lt / per_group;
  const int first_m = group * GROUP_M;
  const int gm = min(grid_m - first_m, GROUP_M);
  bm = first_m + (lt % per_group) % gm;
  bn = (lt % per_group) / gm;
}

// Block i of n, renumbered so that each XCD (blocks are dealt to the eight
// round-robin) works through one contiguous run, whatever n. (Only multiples of
// eight renumbered before: 16384 x 960 x 576 41 us on small tiles, 22 now;
// 1024 x 3584 x 37888 298 -> 245. With up to 8 k-tiles, where the outputs are most
// of the bytes, other numbers stay in the order they are dealt: 532 small tiles
// of 9728 x 896 x 256 13.2 us, renumbered 14.0, 3300 of 6968 x 7680 x 64 with
// the SwiGLU 30.5 and 33.5.)
__device__ __forceinline__ int xcd_order(int i, int n) {
  const int x = i & 7;
  return x * (n >> 3) + min(x, n & 7) + (i >> 3);
}

typedef __attribute__((address_space(3))) void lds_void_t;

// The wave's index in its block as a scalar, so that what derives from it
// (the direct loads' LDS addresses, the wave's tile offsets) stays in scalar
// registers.
__device__ __forceinline__ int wave_id() { return __builtin_amdgcn_readfirstlane(threadIdx.x >> 6); }


// 16 lanes are served per LDS cycle: their 16 rows must cover the 64 banks.
// A row is 128 bytes (half the banks), so even and odd rows take the two
// halves and (row >> 1) & 7 spreads the 8 rows of each half over its 8
// 16-byte positions.
__device__ __forceinline__ int swz_bits(int row) { return (row >> 1) & 7; }

// ---- K-major operand: global -> LDS directly (global_load_lds, 16 B/lane) --
//
// One wave instruction moves 64 chunks = 8 rows; lane l covers row 8q + l/8
// and LDS position l % 8, i.e. global chunk (l % 8) ^ swz_bits(row). Rows past the
// valid range are clamped to the last valid row: they only feed accumulator
// rows or columns that are never stored.
// Buffer resource over `bytes` bytes from `base`. Every offset the loads use
// is already clamped inside the operand (see the loaders), so the resource
// bound is only a second fence (the deep kernel, whose base moves along K,
// sets none).
typedef __amdgpu_buffer_rsrc_t rsrc_t;
constexpr int kRsrcFlags = 0x00020000;  // raw 32-bit dwords, no swizzle
__device__ __forceinline__ rsrc_t make_rsrc(const void* base, int64_t bytes) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(base), 0,
                                           static_cast<int>(bytes < 0x7fffffff ? bytes : 0x7fffffff),
                                           kRsrcFlags);
}

// 16 bytes per lane from the buffer into LDS at lds + 16 * lane. (Kept out of
// the templates: the host pass of hipcc drops the launch stubs of kernels
// whose templates call this builtin directly.)
__device__ __forceinline__ void load_lds16(rsrc_t r, uint8_t* lds, int voff) {
  __builtin_amdgcn_raw_ptr_buffer_load_lds(r, (lds_void_t*)lds, 16, voff, 0, 0, 0);
}

template <int ROWS>
struct KMajorDirect {
  static constexpr int INSTR = ROWS * 8 / 64 / kLoaders;  // instructions per loading wave
  static_assert(INSTR * kLoaders * 64 == ROWS * 8, "the loading waves must cover every chunk of the tile");
  int voff[INSTR];
  __device__ __forceinline__ void init(int64_t ld, int row0, int rows_valid) {
    const int lane = threadIdx.x & 63;
    const int wave = wave_id();
    const int sub = lane >> 3;
#pragma unroll
    for (int i = 0; i < INSTR; ++i) {
      const int q = i * kLoaders + wave % kLoaders;
      const int row = q * 8 + sub;
      const int chunk = (lane & 7) ^ swz_bits(row);
      const int g = min(row0 + row, rows_valid - 1);
      voff[i] = static_cast<int>(((g - row0) * ld + chunk * 8) * 2);
    }
  }
  // The buffer over the operand from row row0, k0 on; then load i of this wave's INSTR into a stage.
  __device__ __forceinline__ static rsrc_t at(const uint16_t* base, int64_t ld, int row0, int rows_valid, int k0) {
    return make_rsrc(base + row0 * ld + k0, (static_cast<int64_t>(rows_valid - row0) * ld - k0) * 2);
  }
  __device__ __forceinline__ void issue_one(rsrc_t r, int i, uint8_t* lds) const {
    load_lds16(r, lds + (i * kLoaders + wave_id() % kLoaders) * 8 * ROW_BYTES, voff[i]);
  }
  __device__ __forceinline__ void issue(const uint16_t* base, int64_t ld, int row0, int rows_valid,
                                        int k0, uint8_t* lds) const {
    const uint16_t* b = base + row0 * ld + k0;
    const rsrc_t r = make_rsrc(b, (static_cast<int64_t>(rows_valid - row0) * ld - k0) * 2);
    const int wave = wave_id();
    if (wave >= kLoaders) return;
#pragma unroll
    for (int i = 0; i < INSTR; ++i) {
      const int q = i * kLoaders + wave % kLoaders;
      load_lds16(r, lds + q * 8 * ROW_BYTES, voff[i]);
    }
  }
};

// ---- MN-major operand: element (row, k) at base[k * ld + row] -------------
//
// Staged as it lies in memory: BK rows (one per k) of ROWS bf16, moved
// HBM -> LDS by direct loads like the K-major tiles, no registers and no
// shuffles. Chunk c of k-row r sits at position c ^ (4 (r & 3)), so the four
// k-rows one transposing read touches land on distinct banks. The MFMA
// operand (8 consecutive k of one m) comes from two ds_read_b64_tr_b16: in
// each 16-lane group, lane i receives element i % 4 of the 8 bytes addressed
// by lane 4 j + i / 4 (j = 0..3); with source lane s addressing k-row
// k0 + s / 4 at column c0 + 4 (s % 4), lane i gets k0..k0+3 of column c0 + i.
typedef short v4i16 __attribute__((ext_vector_type(4)));
typedef short v8i16 __attribute__((ext_vector_type(8)));
typedef __attribute__((address_space(3))) v4i16 lds_v4i16_t;
typedef __attribute__((address_space(3))) bf16x8 lds_bf16x8_t;

template <int ROWS>
struct MNMajorDirect {
  static constexpr int CPR = ROWS / 8;         // 16-byte chunks per k-row
  static constexpr int RPI = 64 / CPR;         // k-rows per wave instruction
  static constexpr int INSTR = BK / RPI / kLoaders;   // instructions per loading wave
  static_assert(INSTR * kLoaders * RPI == BK, "the loading waves must cover every k-row of the tile");
  static constexpr int ROWB = ROWS * 2;        // bytes per k-row
  int voff[INSTR];
  __device__ __forceinline__ void init(int64_t ld, int row0, int rows_valid) {
    const int lane = threadIdx.x & 63;
    const int wave = wave_id();
    const int sub = lane / CPR, pchunk = lane % CPR;
#pragma unroll
    for (int i = 0; i < INSTR; ++i) {
      const int kb = (i * kLoaders + wave % kLoaders) * RPI;
      const int kr = kb + sub;
      const int c = pchunk ^ (4 * (kr & 3));
      const int col = min(row0 + c * 8, rows_valid - 8);
      voff[i] = static_cast<int>((kr * ld + (col - row0)) * 2);
    }
  }
  __device__ __forceinline__ static rsrc_t at(const uint16_t* base, int64_t ld, int row0, int K, int k0) {
    return make_rsrc(base + static_cast<int64_t>(k0) * ld + row0, (static_cast<int64_t>(K - k0) * ld - row0) * 2);
  }
  __device__ __forceinline__ void issue_one(rsrc_t r, int i, uint8_t* lds) const {
    load_lds16(r, lds + (i * kLoaders + wave_id() % kLoaders) * RPI * ROWB, voff[i]);
  }
  __device__ __forceinline__ void issue(const uint16_t* base, int64_t ld, int row0, int K, int k0,
                                        uint8_t* lds) const {
    const uint16_t* b = base + static_cast<int64_t>(k0) * ld + row0;
    const rsrc_t r = make_rsrc(b, (static_cast<int64_t>(K - k0) * ld - row0) * 2);
    const int wave = wave_id();
    if (wave >= kLoaders) return;
#pragma unroll
    for (int i = 0; i < INSTR; ++i) {
      const int kb = (i * kLoaders + wave % kLoaders) * RPI;
      load_lds16(r, lds + kb * ROWB, voff[i]);
    }
  }
  // Lane-dependent byte offset of the k16-step-0 operand for rows rbase.. of
  // a stage (the low 8 bytes; the high 8 are 4 k-rows further, step kk is
  // 16 kk k-rows further).
  __device__ __forceinline__ static uint32_t frag_off(int rbase, int lane) {
    const int h = lane >> 5, q = (lane >> 4) & 1, i = lane & 15;
    const int c = (rbase + q * 16) / 8 + ((i & 3) >> 1);
    return (8 * h + (i >> 2)) * ROWB + ((c ^ (4 * (i >> 2))) << 4) + (i & 1) * 8;
  }
};

// An epilogue's 16-byte global store; NT marks it non-temporal. Measured on
// the 7B block: the plain-store epilogues (the gradients, q/k/v) run 1-2 %
// faster with it, the SwiGLU backward the same, and the SwiGLU forward and
// the in-place residual add 0.7 and 1.5 % slower, so those keep plain stores.
template <bool NT, typename T>
__device__ __forceinline__ void store16(T* p, T v) {
  static_assert(sizeof(T) == 16, "16-byte stores only");
  if constexpr (NT) __builtin_nontemporal_store(v, p);
  else *p = v;
}

// What rounding x to bf16 leaves, exactly.
__device__ __forceinline__ float bf16_rest(float x) { return x - bf16_to_f32(f32_to_bf16(x)); }

// The epilogues of a wave's WM x WN share of a tile from its transposed
// accumulators (see SWAP in the kernels), staged through the wave's REGION
// bytes of LDS at `region` (free once the k loop has ended).
template <int WM, int WN, int REGION, int EPI, bool OUT_BF16, int TM, int TN>
__device__ __forceinline__ void store_tile(const GemmParams& p, f32x16 (&acc)[TM][TN], int m0, int n0, int wm,
                                           int wn, int lane, uint8_t* region) {
  const int lrow = (lane >> 5) * 4;
  const int lcol = lane & 31;
  if constexpr (is_swiglu(EPI)) {
    // B rows interleave 32 gate rows and 32 up rows, and a wave's column
    // range starts on a multiple of 64: block j = 2q holds gate columns and
    // j = 2q + 1 the up columns of the same 32 act columns (accumulators are
    // transposed, see SWAP). Each 32-row slice of the wave's accumulators (JH
    // column blocks at a time, gate and up pairs whole) is staged as fp32 in
    // the wave's LDS share; then a lane takes 8 consecutive act columns of one
    // row, reads their gate and up values, and writes act and the bf16 gate
    // and up copies as one 16-byte store each: whole cache lines instead of
    // 64-byte row pieces. (Computing act while staging made the compiler read
    // the accumulators out of the AGPRs ahead of the silu chains and spill.)
    // SPLIT: act leaves as three pieces, bf16 hi twice and lo, a third of a row
    // apart, and hi and the gate/up copies besides only where a backward will
    // read them. (An fp32 gate/up product and a kernel that read it back moved
    // 28 bytes an act column where this moves 6, a kernel of 157 us for 4096
    // rows of 11008: a split-precision block forward of that size 1895 ->
    // 1756 us, the same bits.)
    typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
    typedef float f32x4 __attribute__((ext_vector_type(4)));
    typedef __attribute__((address_space(3))) uint8_t lds_u8;
    typedef __attribute__((address_space(3))) f32x4 lds_f32x4;
    // Rows are not padded (32 rows of two blocks fill the 8-wave 128 x 128
    // kernel's 8 KB share); instead the 16-byte chunk c of row r sits at
    // chunk c ^ (r % 16), which spreads a write's 32 rows over all banks.
    constexpr int JH = (32 * TN * 32 * 4 <= REGION) ? TN : 2;
    constexpr int PITCH = JH * 32 * 4;
    constexpr int CH = JH * 16 / 8;  // 8-column act pieces per staged row
    constexpr int NIT = 32 * CH / 64;
    static_assert(32 * PITCH <= REGION && TN % JH == 0 && JH % 2 == 0 && NIT * 64 == 32 * CH,
                  "SwiGLU staging does not fit the wave's LDS share");
    auto at = [](int r, int c) __attribute__((always_inline)) { return r * PITCH + ((c ^ (r & 15)) << 4); };
    lds_u8* st = (lds_u8*)region;
    uint16_t* act = static_cast<uint16_t*>(p.C);
    const bool has_gu = p.gu != nullptr;
    constexpr bool SPLIT = EPI == EPI_SWIGLU_SPLIT;
#pragma unroll
    for (int i = 0; i < TM; ++i) {
#pragma unroll
      for (int jb = 0; jb < TN / JH; ++jb) {
#pragma unroll
        for (int jj = 0; jj < JH; ++jj) {
          const int j = jb * JH + jj;
#pragma unroll
          for (int gi = 0; gi < 4; ++gi)
            *(lds_f32x4*)(st + at(lcol, jj * 8 + gi * 2 + lrow / 4)) =
                f32x4{acc[i][j][4 * gi], acc[i][j][4 * gi + 1], acc[i][j][4 * gi + 2], acc[i][j][4 * gi + 3]};
        }
        // The same wave reads back what it wrote (LDS keeps a wave's accesses
        // in order), then the next slice overwrites the region.
        const int row0 = m0 + wm * WM + i * 32;
        const int col0 = n0 + wn * WN + jb * JH * 32;  // gate/up column, a multiple of 64
        // uniform bases of the slice; lane offsets stay 32-bit (ld < 2^22, 32 rows)
        uint16_t* const act_s = act + static_cast<int64_t>(row0) * p.ldc + col0 / 2;
        uint16_t* const gu_s = p.gu + static_cast<int64_t>(row0) * p.ldgu + col0;
        uint16_t* const hi_s = SPLIT ? p.act + static_cast<int64_t>(row0) * p.ldact + col0 / 2 : nullptr;
        // (a slice wholly inside the outputs stores without per-lane guards,
        // as in the plain epilogue; N is a multiple of 32, so an act piece and
        // its gate and up pieces lie inside or past the edge together)
        auto out = [&](auto guardc, auto guc) __attribute__((always_inline)) {
          constexpr bool GUARD = decltype(guardc)::value, GU = decltype(guc)::value;
#pragma unroll
          for (int it = 0; it < NIT; ++it) {
            const int idx = it * 64 + lane, r = idx / CH, ch = idx % CH;
            const int gc = (ch >> 2) * 64 + (ch & 3) * 8;  // staged gate column; up 32 further
            const f32x4 g0 = *(const lds_f32x4*)(st + at(r, gc / 4)), g1 = *(const lds_f32x4*)(st + at(r, gc / 4 + 1));
            const f32x4 u0 = *(const lds_f32x4*)(st + at(r, gc / 4 + 8)), u1 = *(const lds_f32x4*)(st + at(r, gc / 4 + 9));
            if (!GUARD || (row0 + r < p.M && col0 / 2 + ch * 8 < p.n_out)) {
              float a[8];
#pragma unroll
              for (int e = 0; e < 4; ++e) {
                a[e] = silu(g0[e]) * u0[e];
                a[e + 4] = silu(g1[e]) * u1[e];
              }
              const u32x4 hi = {pack_bf16x2(a[0], a[1]), pack_bf16x2(a[2], a[3]), pack_bf16x2(a[4], a[5]),
                                pack_bf16x2(a[6], a[7])};
              uint16_t* const ao = act_s + static_cast<uint32_t>(r * static_cast<int>(p.ldc) + ch * 8);
              store16<false>(reinterpret_cast<u32x4*>(ao), hi);
              if constexpr (SPLIT) {
                store16<false>(reinterpret_cast<u32x4*>(ao + p.n_out), hi);
                store16<false>(reinterpret_cast<u32x4*>(ao + 2 * static_cast<int64_t>(p.n_out)),
                               u32x4{pack_bf16x2(bf16_rest(a[0]), bf16_rest(a[1])), pack_bf16x2(bf16_rest(a[2]), bf16_rest(a[3])),
                                     pack_bf16x2(bf16_rest(a[4]), bf16_rest(a[5])), pack_bf16x2(bf16_rest(a[6]), bf16_rest(a[7]))});
                if constexpr (GU)
                  store16<false>(reinterpret_cast<u32x4*>(hi_s + static_cast<uint32_t>(r * static_cast<int>(p.ldact) + ch * 8)), hi);
              }
              if constexpr (GU) {
                uint16_t* const o = gu_s + static_cast<uint32_t>(r * static_cast<int>(p.ldgu) + gc);
                store16<false>(reinterpret_cast<u32x4*>(o), u32x4{pack_bf16x2(g0[0], g0[1]), pack_bf16x2(g0[2], g0[3]),
                                                           pack_bf16x2(g1[0], g1[1]), pack_bf16x2(g1[2], g1[3])});
                store16<false>(reinterpret_cast<u32x4*>(o + 32), u32x4{pack_bf16x2(u0[0], u0[1]), pack_bf16x2(u0[2], u0[3]),
                                                                pack_bf16x2(u1[0], u1[1]), pack_bf16x2(u1[2], u1[3])});
              }
            }
          }
        };
        const bool full = row0 + 32 <= p.M && col0 / 2 + JH * 16 <= p.n_out;
        if (has_gu) {
          if (full) out(std::false_type{}, std::true_type{});
          else out(std::true_type{}, std::true_type{});
        } else {
          if (full) out(std::false_type{}, std::false_type{});
          else out(std::true_type{}, std::false_type{});
        }
      }
    }
  } else if constexpr (EPI == EPI_SWIGLU_BWD) {
    // acc is dact transposed (SWAP): lane l holds row l % 32 of block (i, j)
    // and, in register group gi, act columns j 32 + 8 gi + 4 (l / 32) .. + 3.
    // Each 32-row slice of the wave's dact (JH column blocks at a time) is
    // staged as fp32 in the wave's LDS share; then a lane takes 8 consecutive
    // act columns of one row: their gate and up values are one 16-byte load
    // each from the saved interleaved gate/up (gate of act column c at
    // (c / 32) 64 + c % 32, up 32 further), all of a slice's loads in flight
    // before any is used, and dgate and dup leave as one 16-byte store each
    // at the same places.
    typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
    typedef float f32x4 __attribute__((ext_vector_type(4)));
    typedef __attribute__((address_space(3))) uint8_t lds_u8;
    constexpr int JH = (32 * (TN * 32 * 4 + 16) <= REGION) ? TN : (32 * (2 * 32 * 4 + 16) <= REGION ? 2 : 1);
    constexpr int PITCH = JH * 32 * 4 + 16;
    constexpr int CH = JH * 32 / 8;  // 8-column pieces per staged row
    constexpr int NIT = 32 * CH / 64;
    static_assert(32 * PITCH <= REGION && TN % JH == 0 && NIT * 64 == 32 * CH, "staging does not fit");
    lds_u8* st = (lds_u8*)region;
    uint16_t* dgu = static_cast<uint16_t*>(p.C);
#pragma unroll
    for (int i = 0; i < TM; ++i) {
#pragma unroll
      for (int jb = 0; jb < TN / JH; ++jb) {
#pragma unroll
        for (int jj = 0; jj < JH; ++jj) {
          const int j = jb * JH + jj;
#pragma unroll
          for (int gi = 0; gi < 4; ++gi)
            *(__attribute__((address_space(3))) f32x4*)(st + lcol * PITCH + (jj * 32 + gi * 8 + lrow) * 4) =
                f32x4{acc[i][j][4 * gi], acc[i][j][4 * gi + 1], acc[i][j][4 * gi + 2], acc[i][j][4 * gi + 3]};
        }
        // The same wave reads back what it wrote (LDS keeps a wave's accesses
        // in order). Loads go to clamped (always valid) places; only the
        // stores are guarded.
        const int row0 = m0 + wm * WM + i * 32;
        const int col0 = n0 + wn * WN + jb * JH * 32;
        const uint16_t* const gu_s = p.gu + static_cast<int64_t>(row0) * p.ldgu;
        uint16_t* const dgu_s = dgu + static_cast<int64_t>(row0) * p.ldc;
        u32x4 gv[NIT], uv[NIT];
#pragma unroll
        for (int it = 0; it < NIT; ++it) {
          const int idx = it * 64 + lane, r = idx / CH, ch = idx % CH;
          const int row = min(row0 + r, p.M - 1), col = min(col0 + ch * 8, p.N - 8);
          // signed: a slice wholly past the edge clamps to row M - 1, below row0
          const int o = (row - row0) * static_cast<int>(p.ldgu) + (col >> 5) * 64 + (col & 31);
          gv[it] = *reinterpret_cast<const u32x4*>(gu_s + o);
          uv[it] = *reinterpret_cast<const u32x4*>(gu_s + o + 32);
        }
        auto out = [&](auto guardc) __attribute__((always_inline)) {  // (guards as in the plain epilogue)
          constexpr bool GUARD = decltype(guardc)::value;
#pragma unroll
        for (int it = 0; it < NIT; ++it) {
          const int idx = it * 64 + lane, r = idx / CH, ch = idx % CH;
          const int row = row0 + r, col = col0 + ch * 8;
          const f32x4 d0 = *(__attribute__((address_space(3))) f32x4*)(st + r * PITCH + ch * 32);
          const f32x4 d1 = *(__attribute__((address_space(3))) f32x4*)(st + r * PITCH + ch * 32 + 16);
          const float da[8] = {d0[0], d0[1], d0[2], d0[3], d1[0], d1[1], d1[2], d1[3]};
          float dg[8], du[8];
#pragma unroll
          for (int e = 0; e < 8; ++e) {
            const uint32_t gw = gv[it][e >> 1], uw = uv[it][e >> 1];
            const float g = __uint_as_float((e & 1) ? (gw & 0xffff0000u) : (gw << 16));
            const float u = __uint_as_float((e & 1) ? (uw & 0xffff0000u) : (uw << 16));
            const float sg = sigmoid(g);
            const float dsilu = sg * (1.0f + g * (1.0f - sg));
            dg[e] = da[e] * u * dsilu;
            du[e] = da[e] * g * sg;
          }
          if (!GUARD || (row < p.M && col < p.N)) {
            const uint32_t od = static_cast<uint32_t>(r * static_cast<int>(p.ldc) + (col >> 5) * 64 + (col & 31));
            store16<true>(reinterpret_cast<u32x4*>(dgu_s + od), u32x4{pack_bf16x2(dg[0], dg[1]), pack_bf16x2(dg[2], dg[3]),
                                                              pack_bf16x2(dg[4], dg[5]), pack_bf16x2(dg[6], dg[7])});
            store16<true>(reinterpret_cast<u32x4*>(dgu_s + od + 32), u32x4{pack_bf16x2(du[0], du[1]), pack_bf16x2(du[2], du[3]),
                                                                   pack_bf16x2(du[4], du[5]), pack_bf16x2(du[6], du[7])});
          }
        }
        };
        if (row0 + 32 <= p.M && col0 + JH * 32 <= p.N) out(std::false_type{});
        else out(std::true_type{});
      }
    }
  } else {  // EPI_STORE, EPI_RESID
    // The transposed accumulators are staged in fp32 per 32-row slice and JH
    // column blocks in the wave's LDS share, then leave as 16-byte row pieces
    // (bias, residual and the bf16 rounding applied on the way): whole cache
    // lines instead of 64-byte (bf16) row pieces, and a quarter of the store
    // instructions. Measured on the 7B block: q/k/v projection 9 %,
    // attention-output input gradient 10 %, fp32 outputs 1-4 % faster. (With
    // the bias added while staging, its branch made the compiler read every
    // accumulator out of the AGPRs ahead of it, 256 values, and spill.)
    typedef float f32x4 __attribute__((ext_vector_type(4)));
    typedef __attribute__((address_space(3))) uint8_t lds_u8;
    typedef __attribute__((address_space(3))) f32x4 lds_f32x4;
    constexpr int JH = (32 * (TN * 32 * 4 + 16) <= REGION) ? TN : (32 * (2 * 32 * 4 + 16) <= REGION ? 2 : 1);
    constexpr int PITCH = JH * 32 * 4 + 16;
    constexpr int OPC = OUT_BF16 ? 8 : 4;   // output columns per 16-byte store
    constexpr int CH = JH * 32 / OPC;       // stores per staged row
    constexpr int NIT = 32 * CH / 64;
    static_assert(32 * PITCH <= REGION && TN % JH == 0 && NIT * 64 == 32 * CH, "staging does not fit");
    static_assert(EPI == EPI_STORE || !OUT_BF16, "the residual epilogue writes fp32");
    lds_u8* st = (lds_u8*)region;
    const bool has_bias = p.bias != nullptr;
#pragma unroll
    for (int i = 0; i < TM; ++i) {
#pragma unroll
      for (int jb = 0; jb < TN / JH; ++jb) {
#pragma unroll
        for (int jj = 0; jj < JH; ++jj) {
          const int j = jb * JH + jj;
#pragma unroll
          for (int gi = 0; gi < 4; ++gi)
            *(lds_f32x4*)(st + lcol * PITCH + (jj * 32 + gi * 8 + lrow) * 4) =
                f32x4{acc[i][j][4 * gi], acc[i][j][4 * gi + 1], acc[i][j][4 * gi + 2], acc[i][j][4 * gi + 3]};
        }
        const int row0 = m0 + wm * WM + i * 32;
        const int col0 = n0 + wn * WN + jb * JH * 32;
        // uniform bases of the slice; lane offsets stay 32-bit (ld < 2^22, 32 rows)
        const int64_t cbase = static_cast<int64_t>(row0) * p.ldc + col0;
        uint16_t* const cb16 = static_cast<uint16_t*>(p.C) + cbase;
        float* const cb32 = static_cast<float*>(p.C) + cbase;
        f32x4 res[EPI == EPI_RESID ? NIT : 1];
        if constexpr (EPI == EPI_RESID) {
          // every residual piece of the slice in flight before any store
          // (the output may be the residual itself, so stores cannot move ahead)
          const float* const rs = p.resid + static_cast<int64_t>(row0) * p.ldr;
#pragma unroll
          for (int it = 0; it < NIT; ++it) {
            const int idx = it * 64 + lane, r = idx / CH, ch = idx % CH;
            const int row = min(row0 + r, p.M - 1), col = min(col0 + ch * 4, p.N - 4);
            // signed: a slice wholly past the edge clamps to row M - 1, below row0
            res[it] = *reinterpret_cast<const f32x4*>(rs + ((row - row0) * static_cast<int>(p.ldr) + col));
          }
        }
        // A slice wholly inside the output stores without per-lane guards:
        // guarded stores each become a branch region of their own, and the
        // LDS reads then wait one by one instead of being in flight together.
        auto out = [&](auto biasc, auto guardc) __attribute__((always_inline)) {
          constexpr bool BIAS = decltype(biasc)::value, GUARD = decltype(guardc)::value;
#pragma unroll
          for (int it = 0; it < NIT; ++it) {
            const int idx = it * 64 + lane, r = idx / CH, ch = idx % CH;
            const int row = row0 + r, col = col0 + ch * OPC;
            const uint32_t oc = static_cast<uint32_t>(r * static_cast<int>(p.ldc) + ch * OPC);
            if (!GUARD || (row < p.M && col < p.N)) {
              // N is a multiple of 8: a store's columns lie wholly inside or past the edge
              const int cb = GUARD ? min(col, p.N - OPC) : col;
              f32x4 w = *(lds_f32x4*)(st + r * PITCH + ch * OPC * 4);
              if constexpr (BIAS) w += f32x4{p.bias[cb], p.bias[cb + 1], p.bias[cb + 2], p.bias[cb + 3]};
              if constexpr (OUT_BF16) {
                typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
                f32x4 w2 = *(lds_f32x4*)(st + r * PITCH + ch * OPC * 4 + 16);
                if constexpr (BIAS)
                  w2 += f32x4{p.bias[cb + 4], p.bias[cb + 5], p.bias[cb + 6], p.bias[cb + 7]};
                store16<true>(reinterpret_cast<u32x4*>(cb16 + oc),
                        u32x4{pack_bf16x2(w[0], w[1]), pack_bf16x2(w[2], w[3]), pack_bf16x2(w2[0], w2[1]),
                              pack_bf16x2(w2[2], w2[3])});
              } else {
                if constexpr (EPI == EPI_RESID) w = res[it] + w;
                store16<EPI == EPI_STORE>(reinterpret_cast<f32x4*>(cb32 + oc), w);
              }
            }
          }
        };
        const bool full = row0 + 32 <= p.M && col0 + JH * 32 <= p.N;
        if (has_bias) {
          if (full) out(std::true_type{}, std::false_type{});
          else out(std::true_type{}, std::true_type{});
        } else {
          if (full) out(std::false_type{}, std::false_type{});
          else out(std::false_type{}, std::true_type{});
        }
      }
    }
  }
}

// A k-split block's raw partial tile, for the reduce kernel: 32 x 32 blocks row
// by row, each as the accumulators hold it (register group gi of the 64 lanes
// contiguous), so that every store is a whole 1 KB. bi, bj: the wave's first
// block.
template <int BM, int BN, int TM, int TN>
__device__ __forceinline__ void store_partial(float* out, const f32x16 (&acc)[TM][TN], int bi, int bj, int lane) {
  typedef float f32x4 __attribute__((ext_vector_type(4)));
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j)
#pragma unroll
      for (int gi = 0; gi < 4; ++gi)
        *reinterpret_cast<f32x4*>(out + (((bi + i) * (BN / 32) + bj + j) * 4 + gi) * 256 + lane * 4) =
            f32x4{acc[i][j][4 * gi], acc[i][j][4 * gi + 1], acc[i][j][4 * gi + 2], acc[i][j][4 * gi + 3]};
}

template <int BM, int BN, bool A_KMAJOR, bool B_KMAJOR, int EPI, bool OUT_BF16>
__global__ __launch_bounds__(kThreads) void gemm_kernel(GemmParams p) {
  constexpr int WM = BM / kWaveRows, WN = BN / (kWaves / kWaveRows);
  constexpr int TM = WM / 32, TN = WN / 32;
  // Every epilogue feeds the MFMA with B as the first operand and A as the
  // second, so that each accumulator holds C transposed: lane l then owns row
  // l % 32 of its 32 x 32 block and, in register group gi, the 4 consecutive
  // columns 8 gi + 4 (l / 32) .. + 3, which the epilogue writes to LDS as one
  // 8- or 16-byte piece. (Every output element is the same k-ordered sum
  // either way.)
  constexpr bool SWAP = true;
  // Two LDS stages as four distinct arrays, indexed only with compile-time
  // stage numbers (the k loop below is unrolled by two), so that the waits
  // for the direct-to-LDS loads into one stage are not placed in front of the
  // operand reads of the other.
  __shared__ __attribute__((aligned(1024))) uint8_t As0[BM * ROW_BYTES];
  __shared__ __attribute__((aligned(1024))) uint8_t As1[BM * ROW_BYTES];
  __shared__ __attribute__((aligned(1024))) uint8_t Bs0[BN * ROW_BYTES];
  __shared__ __attribute__((aligned(1024))) uint8_t Bs1[BN * ROW_BYTES];

  // XCD-aware renumbering, then the grouped order along M. Split launches take
  // the splits of one tile as consecutive blocks.
  int bid = blockIdx.x, split = 0;
  if (p.ksplit > 1) {
    split = bid % p.ksplit;
    bid /= p.ksplit;
  } else if ((p.n_tiles & 7) == 0 || p.K > 8 * BK) {
    bid = xcd_order(bid, p.n_tiles);
  }
  int bm, bn;
  if (p.sub) {
    tile_coords(p.tile0 + (bid >> 2), p.grid_m, p.grid_n, bm, bn);
    bm = 2 * bm + ((bid >> 1) & 1);
    bn = 2 * bn + (bid & 1);
  } else {
    tile_coords(p.tile0 + bid, p.grid_m, p.grid_n, bm, bn);
  }
  const int m0 = bm * BM;
  const int n0 = bn * BN;
  if (m0 >= p.M || n0 >= p.N) return;  // a quarter wholly past the edge (the whole block leaves)

  const int lane = threadIdx.x & 63;
  const int wave = wave_id();
  const int wm = wave / (kWaves / kWaveRows), wn = wave % (kWaves / kWaveRows);

  // Global loads of tile kt, straight into the given LDS stage.
  std::conditional_t<A_KMAJOR, KMajorDirect<BM>, MNMajorDirect<BM>> ld_a;
  std::conditional_t<B_KMAJOR, KMajorDirect<BN>, MNMajorDirect<BN>> ld_b;
  ld_a.init(p.lda, m0, p.M);
  ld_b.init(p.ldb, n0, p.N);
  auto issue_loads = [&](int kt, uint8_t* as_dst, uint8_t* bs_dst) {
    const int k0 = kt * BK;
    if constexpr (A_KMAJOR) ld_a.issue(p.A, p.lda, m0, p.M, k0, as_dst);
    else ld_a.issue(p.A, p.lda, m0, p.K, k0, as_dst);
    if constexpr (B_KMAJOR) ld_b.issue(p.B, p.ldb, n0, p.N, k0, bs_dst);
    else ld_b.issue(p.B, p.ldb, n0, p.K, k0, bs_dst);
  };

  f32x16 acc[TM][TN];
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j) acc[i][j] = f32x16{};

  // MFMAs over one LDS stage, with the operands of the next k16 step read
  // while the current step's MFMAs run.
  // Every k step, fragment slot and accumulator is visited with compile-time
  // indices (StaticFor): left to the loop unroller, a body this large can
  // stay rolled, and a runtime index would move acc and the fragments to
  // scratch memory.
  // LDS operand addresses: the lane-dependent parts are computed once and
  // hidden from the optimizer, so that every operand read is its stage
  // array plus one of these registers plus an immediate (tile, k step). Left
  // alone, the compiler folds the tile and step offsets into a separate
  // register per read and runs out of room for the next step's operands.
  // The reads keep naming their stage array so that the waits for the
  // direct loads into one stage are not put in front of reads of the other.
  constexpr int NA = A_KMAJOR ? BK / 16 : TM, NB = B_KMAJOR ? BK / 16 : TN;
  uint32_t a_reg[NA], b_reg[NB];
  {
    const int h = lane >> 5, l32 = lane & 31;
#pragma unroll
    for (int x = 0; x < NA; ++x) {
      if constexpr (A_KMAJOR)
        a_reg[x] = (wm * WM + l32) * ROW_BYTES + (((2 * x + h) ^ swz_bits(l32)) << 4);
      else
        a_reg[x] = MNMajorDirect<BM>::frag_off(wm * WM + x * 32, lane);
      asm volatile("" : "+v"(a_reg[x]));
    }
#pragma unroll
    for (int x = 0; x < NB; ++x) {
      if constexpr (B_KMAJOR)
        b_reg[x] = (wn * WN + l32) * ROW_BYTES + (((2 * x + h) ^ swz_bits(l32)) << 4);
      else
        b_reg[x] = MNMajorDirect<BN>::frag_off(wn * WN + x * 32, lane);
      asm volatile("" : "+v"(b_reg[x]));
    }
  }
  typedef const __attribute__((address_space(3))) uint8_t* lds_ptr;

  // MFMAs over one LDS stage, with the operands of the next k16 step read
  // while the current step's MFMAs run.
  // Every k step, fragment slot and accumulator is visited with compile-time
  // indices (StaticFor): left to the loop unroller, a body this large can
  // stay rolled, and a runtime index would move acc and the fragments to
  // scratch memory.
  auto compute = [&](auto stagec) {
    constexpr int st = decltype(stagec)::value;
    const lds_ptr la = (lds_ptr)(st ? As1 : As0);
    const lds_ptr lb = (lds_ptr)(st ? Bs1 : Bs0);
    bf16x8 af[2][TM], bfr[2][TN];
    auto read_frags = [&](auto kkc, auto slotc) {
      constexpr int kk = decltype(kkc)::value, slot = decltype(slotc)::value;
      auto ra = [&](auto ic) {
        constexpr int i = decltype(ic)::value;
        if constexpr (A_KMAJOR) {
          af[slot][i] = *(const lds_bf16x8_t*)(la + a_reg[kk] + i * 32 * ROW_BYTES);
        } else {
          constexpr uint32_t R = MNMajorDirect<BM>::ROWB;
          const v4i16 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_v4i16_t*)(la + a_reg[i] + kk * 16 * R));
          const v4i16 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_v4i16_t*)(la + a_reg[i] + kk * 16 * R + 4 * R));
          af[slot][i] = __builtin_bit_cast(bf16x8, __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7));
        }
      };
      auto rb = [&](auto jc) {
        constexpr int j = decltype(jc)::value;
        if constexpr (B_KMAJOR) {
          bfr[slot][j] = *(const lds_bf16x8_t*)(lb + b_reg[kk] + j * 32 * ROW_BYTES);
        } else {
          constexpr uint32_t R = MNMajorDirect<BN>::ROWB;
          const v4i16 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_v4i16_t*)(lb + b_reg[j] + kk * 16 * R));
          const v4i16 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_v4i16_t*)(lb + b_reg[j] + kk * 16 * R + 4 * R));
          bfr[slot][j] = __builtin_bit_cast(bf16x8, __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7));
        }
      };
      StaticFor<0, TM>::run(ra);
      StaticFor<0, TN>::run(rb);
    };
    read_frags(std::integral_constant<int, 0>{}, std::integral_constant<int, 0>{});
    auto kstep = [&](auto kkc) {
      constexpr int kk = decltype(kkc)::value, cur = kk & 1;
      if constexpr (kk + 1 < BK / 16)
        read_frags(std::integral_constant<int, kk + 1>{}, std::integral_constant<int, cur ^ 1>{});
      // The next step's reads stay in front of this step's MFMAs (otherwise
      // the scheduler moves them behind and reuses the same registers).
      __builtin_amdgcn_sched_barrier(0);
      auto mm = [&](auto ijc) {
        constexpr int i = decltype(ijc)::value / TN, j = decltype(ijc)::value % TN;
        if constexpr (SWAP)
          acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(bfr[cur][j], af[cur][i], acc[i][j], 0, 0, 0);
        else
          acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(af[cur][i], bfr[cur][j], acc[i][j], 0, 0, 0);
      };
      StaticFor<0, TM * TN>::run(mm);
    };
    StaticFor<0, BK / 16>::run(kstep);
  };

  // One pipeline step: compute on stage `cur` while tile kt + 1 moves into
  // the other stage, then a barrier.
  auto step = [&](int kt, int KT, auto curc) {
    constexpr int cur = decltype(curc)::value;
    if (kt + 1 < KT) issue_loads(kt + 1, cur ? As0 : As1, cur ? Bs0 : Bs1);
    // Keep the loads of the next tile ahead of this tile's MFMAs: left to
    // itself the scheduler sinks them to the end of the step, right in front
    // of the wait for them, and the whole memory latency is exposed.
    __builtin_amdgcn_sched_barrier(0);
    compute(curc);
    // The direct loads of the next tile and every read of this one are done
    // before any wave moves on.
    __builtin_amdgcn_s_waitcnt(0);
    __syncthreads();
  };

  const int kt_begin = split * p.kt_per;
  const int KT = min(p.K / BK, kt_begin + p.kt_per);
  if (kt_begin < KT) {
    issue_loads(kt_begin, As0, Bs0);
    __builtin_amdgcn_s_waitcnt(0);
    __syncthreads();
    int kt = kt_begin;
    for (; kt + 1 < KT; kt += 2) {
      step(kt, KT, std::integral_constant<int, 0>{});
      step(kt + 1, KT, std::integral_constant<int, 1>{});
    }
    if (kt < KT) step(kt, KT, std::integral_constant<int, 0>{});
  }

  // ---- epilogue ----
  if (p.ksplit > 1) {
    store_partial<BM, BN>(p.ws + (static_cast<int64_t>(bid) * p.ksplit + split) * (BM * BN), acc, wm * TM, wn * TN, lane);
    return;
  }
  {
    // bytes of LDS per wave: two waves per array, or four per A array where A's are the larger
    constexpr int REGION = BM == BN ? (BM + BN) * ROW_BYTES * 2 / kWaves : BM * ROW_BYTES / 4;
    uint8_t* arr = BM == BN ? (wave < 2 ? As0 : wave < 4 ? As1 : wave < 6 ? Bs0 : Bs1) : wave < 4 ? As0 : As1;
    store_tile<WM, WN, REGION, EPI, OUT_BF16>(p, acc, m0, n0, wm, wn, lane, arr + (wave & (BM == BN ? 1 : 3)) * REGION);
  }
}


// ---- 4-wave kernel for 256 x 256 tiles ---------------------------------------
//
// One wave per SIMD, each owning 128 x 128 of the tile (256 accumulator
// registers, held in AGPRs): half the LDS operand reads per MFMA of the 8-wave
// kernel (4 A and 4 B fragments feed 16 MFMAs per k16 step). A has three LDS
// stages and B two (160 KB), so that a k-tile's A loads go out a whole k-tile
// before they are needed; every wave issues 16 loads per k-tile, spread over
// the k16 steps between its MFMAs (4 per step: B of the next k-tile in step 0,
// A of the one after in steps 1 and 2, B of that one in step 3), which keeps
// the CU's load path at about half its rate instead of in bursts. Per k-tile
// there is one barrier, ahead of its last k16 step: every wave has read the
// stage in full, its own loads of the next k-tile have landed (the A loads of
// the k-tile after may still be in flight), and the next k-tile's first
// fragments are read while the last step's MFMAs run. The stage pattern
// repeats every 6 k-tiles (A stage u % 3, B stage u % 2, all compile-time);
// a K of KT k-tiles enters the first group of 6 at position (6 - KT % 6) % 6.
// Loads past the last k-tile repeat it into a stage nobody reads again.
// Measured on the 7B block's plain products: 3-11 % faster than the 8-wave
// kernel (gate/up 16384 x 37888 x 3584: 1340 against 1220 TFLOP/s).
constexpr int kWaves4 = 4;
template <bool A_KMAJOR, bool B_KMAJOR, int EPI, bool OUT_BF16>
__global__ __launch_bounds__(64 * kWaves4) __attribute__((amdgpu_waves_per_eu(1, 1))) void gemm4_kernel(GemmParams p) {
  constexpr int BM = 256, BN = 256, WM = 128, WN = 128, TM = WM / 32, TN = WN / 32;
  constexpr int STAGE = 256 * ROW_BYTES;  // bytes of one operand stage (either layout)
  static_assert(STAGE == MNMajorDirect<256>::ROWB * BK, "both layouts stage 32 KB");
  __shared__ __attribute__((aligned(1024))) uint8_t As0[STAGE];
  __shared__ __attribute__((aligned(1024))) uint8_t As1[STAGE];
  __shared__ __attribute__((aligned(1024))) uint8_t As2[STAGE];
  __shared__ __attribute__((aligned(1024))) uint8_t Bs0[STAGE];
  __shared__ __attribute__((aligned(1024))) uint8_t Bs1[STAGE];

  // A k-split launch takes the splits of one tile as consecutive blocks, each
  // over kt_per k-tiles (the last over what remains).
  int bid = blockIdx.x, split = 0;
  if (p.ksplit > 1) {
    split = bid % p.ksplit;
    bid /= p.ksplit;
  } else {
    bid = xcd_order(bid, p.n_tiles);
  }
  int bm, bn;
  tile_coords(p.tile0 + bid, p.grid_m, p.grid_n, bm, bn);
  const int m0 = bm * BM, n0 = bn * BN;
  const int lane = threadIdx.x & 63;
  const int wave = wave_id();
  const int wm = wave >> 1, wn = wave & 1;

  std::conditional_t<A_KMAJOR, KMajorDirect<BM>, MNMajorDirect<BM>> ld_a;
  std::conditional_t<B_KMAJOR, KMajorDirect<BN>, MNMajorDirect<BN>> ld_b;
  ld_a.init(p.lda, m0, p.M);
  ld_b.init(p.ldb, n0, p.N);
  const int kt0 = split * p.kt_per;
  const int KT = min(p.K / BK - kt0, p.kt_per);  // this block's k-tiles: kt0 .. kt0 + KT - 1
  auto tk = [&](int u) { return kt0 + min(u, KT - 1); };
  auto ra_at = [&](int kt) { return ld_a.at(p.A, p.lda, m0, A_KMAJOR ? p.M : p.K, kt * BK); };
  auto rb_at = [&](int kt) { return ld_b.at(p.B, p.ldb, n0, B_KMAJOR ? p.N : p.K, kt * BK); };

  f32x16 acc[TM][TN];
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j) acc[i][j] = f32x16{};

  // fragment addresses, as in the 8-wave kernel
  constexpr int NA = A_KMAJOR ? BK / 16 : TM, NB = B_KMAJOR ? BK / 16 : TN;
  uint32_t a_reg[NA], b_reg[NB];
  {
    const int h = lane >> 5, l32 = lane & 31;
#pragma unroll
    for (int x = 0; x < NA; ++x) {
      if constexpr (A_KMAJOR)
        a_reg[x] = (wm * WM + l32) * ROW_BYTES + (((2 * x + h) ^ swz_bits(l32)) << 4);
      else
        a_reg[x] = MNMajorDirect<BM>::frag_off(wm * WM + x * 32, lane);
      asm volatile("" : "+v"(a_reg[x]));
    }
#pragma unroll
    for (int x = 0; x < NB; ++x) {
      if constexpr (B_KMAJOR)
        b_reg[x] = (wn * WN + l32) * ROW_BYTES + (((2 * x + h) ^ swz_bits(l32)) << 4);
      else
        b_reg[x] = MNMajorDirect<BN>::frag_off(wn * WN + x * 32, lane);
      asm volatile("" : "+v"(b_reg[x]));
    }
  }
  typedef const __attribute__((address_space(3))) uint8_t* lds_ptr;
  bf16x8 af[2][TM], bfr[2][TN];
  auto rd = [&](lds_ptr la, lds_ptr lb, int kk, int slot) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < TM; ++i) {
      if constexpr (A_KMAJOR) {
        af[slot][i] = *(const lds_bf16x8_t*)(la + a_reg[kk] + i * 32 * ROW_BYTES);
      } else {
        constexpr uint32_t R = MNMajorDirect<BM>::ROWB;
        const v4i16 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_v4i16_t*)(la + a_reg[i] + kk * 16 * R));
        const v4i16 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_v4i16_t*)(la + a_reg[i] + kk * 16 * R + 4 * R));
        af[slot][i] = __builtin_bit_cast(bf16x8, __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7));
      }
    }
#pragma unroll
    for (int j = 0; j < TN; ++j) {
      if constexpr (B_KMAJOR) {
        bfr[slot][j] = *(const lds_bf16x8_t*)(lb + b_reg[kk] + j * 32 * ROW_BYTES);
      } else {
        constexpr uint32_t R = MNMajorDirect<BN>::ROWB;
        const v4i16 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_v4i16_t*)(lb + b_reg[j] + kk * 16 * R));
        const v4i16 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_v4i16_t*)(lb + b_reg[j] + kk * 16 * R + 4 * R));
        bfr[slot][j] = __builtin_bit_cast(bf16x8, __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7));
      }
    }
  };
  auto mm = [&](int slot) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
      for (int j = 0; j < TN; ++j)
        acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(bfr[slot][j], af[slot][i], acc[i][j], 0, 0, 0);
  };
  // The order of a k16 step: its next-step fragment reads (8, 12 or 16 LDS
  // instructions) and the loads spread between its 16 MFMAs.
  constexpr int NR = (A_KMAJOR ? TM : 2 * TM) + (B_KMAJOR ? TN : 2 * TN);
  auto order = [](bool loads) __attribute__((always_inline)) {
#pragma unroll
    for (int q = 0; q < 8; ++q) {
      if constexpr (NR == 12) {
        if (q & 1) __builtin_amdgcn_sched_group_barrier(0x100, 2, 0);
        else __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
      } else {
        __builtin_amdgcn_sched_group_barrier(0x100, NR / 8, 0);
      }
      __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
      if (loads && (q & 1)) __builtin_amdgcn_sched_group_barrier(0x010, 1, 0);
      __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
    }
  };

  const int phase = (6 - KT % 6) % 6;
  {
    // k-tile 0 whole, then k-tile 1's A and the first half of its B, into the
    // stages of positions phase and phase + 1
    auto pro = [&](uint8_t* a0, uint8_t* b0, uint8_t* a1, uint8_t* b1) __attribute__((always_inline)) {
      const rsrc_t r_a0 = ra_at(tk(0)), r_b0 = rb_at(tk(0));
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        ld_a.issue_one(r_a0, i, a0);
        ld_b.issue_one(r_b0, i, b0);
      }
      __builtin_amdgcn_s_waitcnt(0);
      __syncthreads();
      const rsrc_t r_a1 = ra_at(tk(1)), r_b1 = rb_at(tk(1));
#pragma unroll
      for (int i = 0; i < 8; ++i) ld_a.issue_one(r_a1, i, a1);
#pragma unroll
      for (int i = 0; i < 4; ++i) ld_b.issue_one(r_b1, i, b1);
      rd((lds_ptr)a0, (lds_ptr)b0, 0, 0);
    };
    switch (phase) {
      case 0: pro(As0, Bs0, As1, Bs1); break;
      case 1: pro(As1, Bs1, As2, Bs0); break;
      case 2: pro(As2, Bs0, As0, Bs1); break;
      case 3: pro(As0, Bs1, As1, Bs0); break;
      case 4: pro(As1, Bs0, As2, Bs1); break;
      default: pro(As2, Bs1, As0, Bs0); break;
    }
    __builtin_amdgcn_sched_barrier(0);
  }
  // k-tile u on A stage SA and B stage SB
  auto tile = [&](int u, auto sac, auto sbc) __attribute__((always_inline)) {
    constexpr int SA = decltype(sac)::value, SB = decltype(sbc)::value;
    uint8_t* la_ = SA == 0 ? As0 : SA == 1 ? As1 : As2;
    uint8_t* na_ = SA == 0 ? As1 : SA == 1 ? As2 : As0;
    uint8_t* fa_ = SA == 0 ? As2 : SA == 1 ? As0 : As1;  // A of k-tile u + 2
    uint8_t* lb_ = SB == 0 ? Bs0 : Bs1;                  // after the barrier: B of k-tile u + 2
    uint8_t* nb_ = SB == 0 ? Bs1 : Bs0;                  // B of k-tile u + 1
    const lds_ptr la = (lds_ptr)la_, lb = (lds_ptr)lb_;
    const rsrc_t r_b1 = rb_at(tk(u + 1)), r_a2 = ra_at(tk(u + 2)), r_b2 = rb_at(tk(u + 2));
    rd(la, lb, 1, 1);
#pragma unroll
    for (int i = 4; i < 8; ++i) ld_b.issue_one(r_b1, i, nb_);
    mm(0);
    order(true);
    __builtin_amdgcn_sched_barrier(0);
    rd(la, lb, 2, 0);
#pragma unroll
    for (int i = 0; i < 4; ++i) ld_a.issue_one(r_a2, i, fa_);
    mm(1);
    order(true);
    __builtin_amdgcn_sched_barrier(0);
    rd(la, lb, 3, 1);
#pragma unroll
    for (int i = 4; i < 8; ++i) ld_a.issue_one(r_a2, i, fa_);
    mm(0);
    order(true);
    __builtin_amdgcn_sched_barrier(0);
    // Every read of this stage done, k-tile u + 1 landed (the 8 A loads of
    // k-tile u + 2 may be in flight): a plain barrier, no memory fence.
    asm volatile("s_waitcnt vmcnt(8) lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_sched_barrier(0);
    rd((lds_ptr)na_, (lds_ptr)nb_, 0, 0);
#pragma unroll
    for (int i = 0; i < 4; ++i) ld_b.issue_one(r_b2, i, lb_);
    mm(1);
    order(true);
    __builtin_amdgcn_sched_barrier(0);
  };
  {
    int u = 0;
    if (phase <= 0) tile(u++, std::integral_constant<int, 0>{}, std::integral_constant<int, 0>{});
    if (phase <= 1) tile(u++, std::integral_constant<int, 1>{}, std::integral_constant<int, 1>{});
    if (phase <= 2) tile(u++, std::integral_constant<int, 2>{}, std::integral_constant<int, 0>{});
    if (phase <= 3) tile(u++, std::integral_constant<int, 0>{}, std::integral_constant<int, 1>{});
    if (phase <= 4) tile(u++, std::integral_constant<int, 1>{}, std::integral_constant<int, 0>{});
    tile(u++, std::integral_constant<int, 2>{}, std::integral_constant<int, 1>{});
    for (; u < KT; u += 6) {
      tile(u, std::integral_constant<int, 0>{}, std::integral_constant<int, 0>{});
      tile(u + 1, std::integral_constant<int, 1>{}, std::integral_constant<int, 1>{});
      tile(u + 2, std::integral_constant<int, 2>{}, std::integral_constant<int, 0>{});
      tile(u + 3, std::integral_constant<int, 0>{}, std::integral_constant<int, 1>{});
      tile(u + 4, std::integral_constant<int, 1>{}, std::integral_constant<int, 0>{});
      tile(u + 5, std::integral_constant<int, 2>{}, std::integral_constant<int, 1>{});
    }
  }
  // the repeated last loads land, every wave is past its reads: LDS is free
  __builtin_amdgcn_s_waitcnt(0);
  __syncthreads();
  if (p.ksplit > 1) {
    store_partial<BM, BN>(p.ws + (static_cast<int64_t>(bid) * p.ksplit + split) * (BM * BN), acc, wm * TM, wn * TN, lane);
    return;
  }
  uint8_t* region = wave == 0 ? As0 : wave == 1 ? As1 : wave == 2 ? As2 : Bs0;
  store_tile<WM, WN, STAGE, EPI, OUT_BF16>(p, acc, m0, n0, wm, wn, lane, region);
}

// ---- deep-pipelined 4-wave kernel, 128 x 128 or 256 x 128 tiles, one block per CU --
//
// Where a launch has no more tiles than CUs (the small models' products, cut
// along K or not), nothing but a block's own loads can hide the memory latency:
// the double-buffered kernel spends about 0.7 us on each 64-k tile of 0.2 us
// of MFMAs. Here a block has the CU's LDS to itself: four stages of 32 KB, so
// that three k-tiles are in flight while one is multiplied. One wave per SIMD
// owns 64 x 64. As in the 256 x 256 kernel, the k-tile's barrier stands ahead
// of its last k16 step: every wave has then read the stage in full, so the
// loads of k-tile u + 4 go into it at once, half behind that step's MFMAs and
// half behind the next k-tile's first, and the next k-tile's first operands
// are read while the last step multiplies. What bounds it then is LDS: 64 KB
// of operand reads and 32 KB of loads a k-tile, 0.33 us with few CUs at work
// (0.2 us of MFMAs) and 0.42 with all 256 (measured, K = 4096).
// Measured against the two-per-CU form: 576 x 576 x 4096 (25 tiles) 45 us, 26
// here whole and 16 cut in 5; 4096 x 576 x 3072 34 -> 22; the residual products
// 4096 x 576 x 1536 22 -> 16 and, on large tiles, 36; 2048 x 2048 x 2048 28 -> 20.
//
// With BM = 256 (wide) a wave owns 128 x 64 and three stages of 48 KB take the
// LDS: per product 3/4 of the operand reads and loads of the 128 x 128 form, for
// grids that have too few 256 x 256 tiles and enough of these (operands in cache
// and from memory, against the best other plan: 4096 x 1536 x 2048 30 -> 28 and
// 40 -> 33 us; 1536 x 5120 x 4096 63 -> 55 and 69 -> 66; 9728 x 896 x 4096 75 ->
// 70 and 84 -> 83; 8192 x 896 x 9728 131 -> 116 in cache).
template <int BM, bool A_KMAJOR, bool B_KMAJOR, int EPI, bool OUT_BF16>
__global__ __launch_bounds__(64 * kWaves4) __attribute__((amdgpu_waves_per_eu(1, 1))) void gemm_deep_kernel(GemmParams p) {
  constexpr int BN = 128, WM = BM / 2, WN = 64, TM = WM / 32, TN = 2;
  constexpr int STAGE_A = BM * ROW_BYTES, STAGE_B = BN * ROW_BYTES;
  constexpr int NS = BM == 256 ? 3 : 4;      // stages
  constexpr int LA = BM / 32, LB = BN / 32;  // a wave's loads of a k-tile
  __shared__ __attribute__((aligned(1024))) uint8_t As0[STAGE_A];
  __shared__ __attribute__((aligned(1024))) uint8_t As1[STAGE_A];
  __shared__ __attribute__((aligned(1024))) uint8_t As2[STAGE_A];
  __shared__ __attribute__((aligned(1024))) uint8_t As3[NS > 3 ? STAGE_A : 16];
  __shared__ __attribute__((aligned(1024))) uint8_t Bs0[STAGE_B];
  __shared__ __attribute__((aligned(1024))) uint8_t Bs1[STAGE_B];
  __shared__ __attribute__((aligned(1024))) uint8_t Bs2[STAGE_B];
  __shared__ __attribute__((aligned(1024))) uint8_t Bs3[NS > 3 ? STAGE_B : 16];

  // The first p.tile0 blocks take a whole tile each, the rest the (split, tile)
  // pairs of the tail, tiles fastest: each XCD a contiguous run of either, so
  // that its blocks share operand panels.
  const bool cut = static_cast<int>(blockIdx.x) >= p.tile0;
  const int blocks = cut ? p.n_tiles * p.ksplit : p.tile0;
  int bid = static_cast<int>(blockIdx.x) - (cut ? p.tile0 : 0);
  bid = xcd_order(bid, blocks);
  const int split = cut ? bid / p.n_tiles : 0;
  bid -= split * p.n_tiles;
  int bm, bn;
  tile_coords((cut ? p.tile0 : 0) + bid, p.grid_m, p.grid_n, bm, bn);
  const int m0 = bm * BM, n0 = bn * BN;
  const int lane = threadIdx.x & 63;
  const int wave = wave_id();
  const int wm = wave >> 1, wn = wave & 1;

  std::conditional_t<A_KMAJOR, KMajorDirect<BM>, MNMajorDirect<BM>> ld_a;
  std::conditional_t<B_KMAJOR, KMajorDirect<BN>, MNMajorDirect<BN>> ld_b;
  ld_a.init(p.lda, m0, p.M);
  ld_b.init(p.ldb, n0, p.N);
  const int kt0 = split * p.kt_per;
  const int KT = cut ? min(p.K / BK - kt0, p.kt_per) : p.K / BK;  // this block's k-tiles: kt0 .. kt0 + KT - 1
  // The k-tile being loaded: its operands' first elements. Offsets from them
  // are clamped inside the operands by the loaders, and the k-tiles stop at the
  // last (loads past it repeat it into a stage nobody reads again).
  const int64_t step_a = A_KMAJOR ? BK : BK * p.lda, step_b = B_KMAJOR ? BK : BK * p.ldb;
  const uint16_t* at_a = p.A + (A_KMAJOR ? m0 * p.lda : m0) + kt0 * step_a;
  const uint16_t* at_b = p.B + (B_KMAJOR ? n0 * p.ldb : n0) + kt0 * step_b;
  auto advance = [&](int u) __attribute__((always_inline)) {  // to k-tile u
    at_a += u < KT ? step_a : 0;
    at_b += u < KT ? step_b : 0;
  };

  f32x16 acc[TM][TN];
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j) acc[i][j] = f32x16{};

  // fragment addresses, as in the 8-wave kernel
  constexpr int NA = A_KMAJOR ? BK / 16 : TM, NB = B_KMAJOR ? BK / 16 : TN;
  uint32_t a_reg[NA], b_reg[NB];
  {
    const int h = lane >> 5, l32 = lane & 31;
#pragma unroll
    for (int x = 0; x < NA; ++x) {
      if constexpr (A_KMAJOR)
        a_reg[x] = (wm * WM + l32) * ROW_BYTES + (((2 * x + h) ^ swz_bits(l32)) << 4);
      else
        a_reg[x] = MNMajorDirect<BM>::frag_off(wm * WM + x * 32, lane);
      asm volatile("" : "+v"(a_reg[x]));
    }
#pragma unroll
    for (int x = 0; x < NB; ++x) {
      if constexpr (B_KMAJOR)
        b_reg[x] = (wn * WN + l32) * ROW_BYTES + (((2 * x + h) ^ swz_bits(l32)) << 4);
      else
        b_reg[x] = MNMajorDirect<BN>::frag_off(wn * WN + x * 32, lane);
      asm volatile("" : "+v"(b_reg[x]));
    }
  }
  typedef const __attribute__((address_space(3))) uint8_t* lds_ptr;
  bf16x8 af[2][TM], bfr[2][TN];
  auto rd_tr = [](lds_ptr l, uint32_t reg, int kk, uint32_t R) __attribute__((always_inline)) {  // R: bytes of a k-row
    const v4i16 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_v4i16_t*)(l + reg + kk * 16 * R));
    const v4i16 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_v4i16_t*)(l + reg + kk * 16 * R + 4 * R));
    return __builtin_bit_cast(bf16x8, __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7));
  };
  auto rd = [&](lds_ptr la, lds_ptr lb, int kk, int slot) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < TM; ++i) {
      if constexpr (A_KMAJOR) af[slot][i] = *(const lds_bf16x8_t*)(la + a_reg[kk] + i * 32 * ROW_BYTES);
      else af[slot][i] = rd_tr(la, a_reg[i], kk, MNMajorDirect<BM>::ROWB);
    }
#pragma unroll
    for (int j = 0; j < TN; ++j) {
      if constexpr (B_KMAJOR) bfr[slot][j] = *(const lds_bf16x8_t*)(lb + b_reg[kk] + j * 32 * ROW_BYTES);
      else bfr[slot][j] = rd_tr(lb, b_reg[j], kk, MNMajorDirect<BN>::ROWB);
    }
  };
  auto mm = [&](int slot) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
      for (int j = 0; j < TN; ++j)
        acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(bfr[slot][j], af[slot][i], acc[i][j], 0, 0, 0);
  };
  // The order of a k16 step: the next step's fragment reads and the loads
  // between its MFMAs.
  constexpr int NR = (A_KMAJOR ? TM : 2 * TM) + (B_KMAJOR ? TN : 2 * TN);
  auto order = [](bool loads) __attribute__((always_inline)) {
#pragma unroll
    for (int q = 0; q < TM * TN; ++q) {
      if (q < TM * TN / 2) __builtin_amdgcn_sched_group_barrier(0x100, NR / (TM * TN / 2), 0);
      __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
      if (loads && q < (LA + LB) / 2) __builtin_amdgcn_sched_group_barrier(0x010, 1, 0);
    }
    __builtin_amdgcn_sched_barrier(0);
  };
  auto issue = [&](uint8_t* a, uint8_t* b, int h0, int h1) __attribute__((always_inline)) {  // halves h0 .. h1 - 1 of a k-tile
    const rsrc_t r_a = make_rsrc(at_a, 0x7fffffff), r_b = make_rsrc(at_b, 0x7fffffff);
#pragma unroll
    for (int i = h0 * (LA / 2); i < h1 * (LA / 2); ++i) ld_a.issue_one(r_a, i, a);
#pragma unroll
    for (int i = h0 * (LB / 2); i < h1 * (LB / 2); ++i) ld_b.issue_one(r_b, i, b);
  };
  const int phase = (NS - KT % NS) % NS;  // the stage k-tile 0 takes
  {
    // The asm at the end differs between the phases, so that their first reads
    // stay in place: merged behind the branches, their waits could not tell the
    // stages apart (every load in flight was waited for), and with three phases
    // the merged read lost its address in one of them.
    auto pro = [&](uint8_t* a0, uint8_t* b0, uint8_t* a1, uint8_t* b1, uint8_t* a2, uint8_t* b2, uint8_t* a3,
                   uint8_t* b3, auto sc) __attribute__((always_inline)) {
      issue(a0, b0, 0, 2);
      advance(1);
      issue(a1, b1, 0, 2);
      advance(2);
      if constexpr (NS == 4) {
        issue(a2, b2, 0, 2);
        advance(3);
        issue(a3, b3, 0, 1);
        asm volatile("s_waitcnt vmcnt(20)" ::: "memory");
      } else {
        issue(a2, b2, 0, 1);
        asm volatile("s_waitcnt vmcnt(18)" ::: "memory");
      }
      __builtin_amdgcn_s_barrier();
      __builtin_amdgcn_sched_barrier(0);
      rd((lds_ptr)a0, (lds_ptr)b0, 0, 0);
      asm volatile("; k-tile 0 in stage %0" ::"i"(decltype(sc)::value) : "memory");
    };
    if constexpr (NS == 4) {
      switch (phase) {
        case 0: pro(As0, Bs0, As1, Bs1, As2, Bs2, As3, Bs3, std::integral_constant<int, 0>{}); break;
        case 1: pro(As1, Bs1, As2, Bs2, As3, Bs3, As0, Bs0, std::integral_constant<int, 1>{}); break;
        case 2: pro(As2, Bs2, As3, Bs3, As0, Bs0, As1, Bs1, std::integral_constant<int, 2>{}); break;
        default: pro(As3, Bs3, As0, Bs0, As1, Bs1, As2, Bs2, std::integral_constant<int, 3>{}); break;
      }
    } else {
      switch (phase) {
        case 0: pro(As0, Bs0, As1, Bs1, As2, Bs2, As3, Bs3, std::integral_constant<int, 0>{}); break;
        case 1: pro(As1, Bs1, As2, Bs2, As0, Bs0, As3, Bs3, std::integral_constant<int, 1>{}); break;
        default: pro(As2, Bs2, As0, Bs0, As1, Bs1, As3, Bs3, std::integral_constant<int, 2>{}); break;
      }
    }
    __builtin_amdgcn_sched_barrier(0);
  }
  // k-tile u, in stage S
  auto tile = [&](int u, auto sc) __attribute__((always_inline)) {
    constexpr int S = decltype(sc)::value;
    uint8_t* la_ = S == 0 ? As0 : S == 1 ? As1 : S == 2 ? As2 : As3;
    uint8_t* lb_ = S == 0 ? Bs0 : S == 1 ? Bs1 : S == 2 ? Bs2 : Bs3;
    constexpr int N1 = (S + 1) % NS, P = (S + NS - 1) % NS;  // the stages of k-tiles u + 1 and u + NS - 1
    uint8_t* na_ = N1 == 0 ? As0 : N1 == 1 ? As1 : N1 == 2 ? As2 : As3;
    uint8_t* nb_ = N1 == 0 ? Bs0 : N1 == 1 ? Bs1 : N1 == 2 ? Bs2 : Bs3;
    uint8_t* pa_ = P == 0 ? As0 : P == 1 ? As1 : P == 2 ? As2 : As3;
    uint8_t* pb_ = P == 0 ? Bs0 : P == 1 ? Bs1 : P == 2 ? Bs2 : Bs3;
    const lds_ptr la = (lds_ptr)la_, lb = (lds_ptr)lb_;
    rd(la, lb, 1, 1);
    issue(pa_, pb_, 1, 2);
    mm(0);
    order(true);
    rd(la, lb, 2, 0);
    mm(1);
    order(false);
    rd(la, lb, 3, 1);
    advance(u + NS);
    mm(0);
    order(false);
    // Every read of this stage done, k-tile u + 1 landed (the loads of the
    // k-tiles after it may be in flight): a plain barrier, no fence.
    if constexpr (NS == 4) asm volatile("s_waitcnt vmcnt(16) lgkmcnt(0)" ::: "memory");
    else asm volatile("s_waitcnt vmcnt(12) lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_sched_barrier(0);
    rd((lds_ptr)na_, (lds_ptr)nb_, 0, 0);
    issue(la_, lb_, 0, 1);
    mm(1);
    order(true);
  };
  int u = 0;
  if (phase <= 0) tile(u++, std::integral_constant<int, 0>{});
  if (phase <= 1) tile(u++, std::integral_constant<int, 1>{});
  if constexpr (NS == 4)
    if (phase <= 2) tile(u++, std::integral_constant<int, 2>{});
  tile(u++, std::integral_constant<int, NS - 1>{});
  for (; u < KT; u += NS) {
    tile(u, std::integral_constant<int, 0>{});
    tile(u + 1, std::integral_constant<int, 1>{});
    tile(u + 2, std::integral_constant<int, 2>{});
    if constexpr (NS == 4) tile(u + 3, std::integral_constant<int, 3>{});
  }
  // the repeated last loads land, every wave is past its reads: LDS is free
  __builtin_amdgcn_s_waitcnt(0);
  __syncthreads();
  if (cut && p.ksplit > 1) {
    store_partial<BM, BN>(p.ws + (static_cast<int64_t>(bid) * p.ksplit + split) * (BM * BN), acc, wm * TM, wn * TN, lane);
    return;
  }
  constexpr int REGION = 128 * ROW_BYTES;
  uint8_t* region = wave == 0 ? As0 : wave == 1 ? As1 : wave == 2 ? As2 : NS == 4 ? As3 : Bs0;
  store_tile<WM, WN, REGION, EPI, OUT_BF16>(p, acc, m0, n0, wm, wn, lane, region);
}

// Sums the k-split partial tiles of a launch in split order and applies the
// epilogue the whole-K kernel would have. A block of 256 threads takes a
// 32 x 32 block of a tile (for SwiGLU a pair: gate and up sit 32 columns
// apart), a thread 4 columns of a row: the partials and the outputs both move
// in whole 128-byte lines. (Against row-major partials and element-wise output:
// the 3B split-precision products' reduces 33 -> 24 and 31 -> 25 us.)
template <int BM, int BN, int EPI, bool OUT_BF16>
__global__ __launch_bounds__(256) void gemm_reduce(GemmParams p) {
  typedef float f32x4 __attribute__((ext_vector_type(4)));
  constexpr int NB = is_swiglu(EPI) ? BN / 64 : BN / 32;  // blocks (or pairs) across a tile
  constexpr int PER_TILE = (BM / 32) * NB;
  const int t = static_cast<int>(blockIdx.x) / PER_TILE, rem = static_cast<int>(blockIdx.x) % PER_TILE;
  const int bi = rem / NB, bj = rem % NB;
  int bm, bn;
  tile_coords(p.tile0 + t, p.grid_m, p.grid_n, bm, bn);
  const int r = threadIdx.x >> 3, c = threadIdx.x & 7;  // row and 4-column piece of the block
  const int row = bm * BM + bi * 32 + r;
  if (row >= p.M) return;
  auto sum4 = [&](int b) __attribute__((always_inline)) {  // piece of block column b, splits in order
    const float* part = p.ws + static_cast<int64_t>(t) * p.ksplit * (BM * BN) +
                        ((bi * (BN / 32) + b) * 4 + (c >> 1)) * 256 + ((c & 1) * 32 + r) * 4;
    f32x4 a = *reinterpret_cast<const f32x4*>(part);
#pragma unroll 4
    for (int sp = 1; sp < p.ksplit; ++sp) a += *reinterpret_cast<const f32x4*>(part + static_cast<int64_t>(sp) * (BM * BN));
    return a;
  };
  auto pack4 = [](f32x4 v) { return make_uint2(pack_bf16x2(v[0], v[1]), pack_bf16x2(v[2], v[3])); };
  if constexpr (is_swiglu(EPI)) {
    const int col = (bn * BN) / 2 + bj * 32 + c * 4;  // act column; N and n_out are multiples of 32
    if (col >= p.n_out) return;
    const f32x4 g = sum4(2 * bj), u = sum4(2 * bj + 1);
    f32x4 a;
#pragma unroll
    for (int k = 0; k < 4; ++k) a[k] = silu(g[k]) * u[k];
    uint16_t* const ao = static_cast<uint16_t*>(p.C) + static_cast<int64_t>(row) * p.ldc + col;
    *reinterpret_cast<uint2*>(ao) = pack4(a);
    if constexpr (EPI == EPI_SWIGLU_SPLIT) {
      *reinterpret_cast<uint2*>(ao + p.n_out) = pack4(a);
      *reinterpret_cast<uint2*>(ao + 2 * static_cast<int64_t>(p.n_out)) =
          pack4(f32x4{bf16_rest(a[0]), bf16_rest(a[1]), bf16_rest(a[2]), bf16_rest(a[3])});
      if (p.gu) *reinterpret_cast<uint2*>(p.act + static_cast<int64_t>(row) * p.ldact + col) = pack4(a);
    }
    if (p.gu) {
      uint16_t* o = p.gu + static_cast<int64_t>(row) * p.ldgu + bn * BN + bj * 64 + c * 4;
      *reinterpret_cast<uint2*>(o) = pack4(g);
      *reinterpret_cast<uint2*>(o + 32) = pack4(u);
    }
  } else {
    const int col = bn * BN + bj * 32 + c * 4;
    if (col >= p.N) return;  // N is a multiple of 8: the piece lies wholly inside or past the edge
    f32x4 x = sum4(bj);
    if constexpr (EPI == EPI_SWIGLU_BWD) {
      const int gcol = (col >> 5) * 64 + (col & 31);
      const uint16_t* gu = p.gu + static_cast<int64_t>(row) * p.ldgu + gcol;
      const uint2 gv = *reinterpret_cast<const uint2*>(gu), uv = *reinterpret_cast<const uint2*>(gu + 32);
      f32x4 dg, du;
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        const uint32_t gw = k < 2 ? gv.x : gv.y, uw = k < 2 ? uv.x : uv.y;
        const float g = __uint_as_float((k & 1) ? (gw & 0xffff0000u) : (gw << 16));
        const float u = __uint_as_float((k & 1) ? (uw & 0xffff0000u) : (uw << 16));
        const float sg = sigmoid(g);
        const float dsilu = sg * (1.0f + g * (1.0f - sg));
        dg[k] = x[k] * u * dsilu;
        du[k] = x[k] * g * sg;
      }
      uint16_t* o = static_cast<uint16_t*>(p.C) + static_cast<int64_t>(row) * p.ldc + gcol;
      *reinterpret_cast<uint2*>(o) = pack4(dg);
      *reinterpret_cast<uint2*>(o + 32) = pack4(du);
    } else {
      if (p.bias) {
#pragma unroll
        for (int k = 0; k < 4; ++k) x[k] += p.bias[col + k];
      }
      const int64_t o = static_cast<int64_t>(row) * p.ldc + col;
      if constexpr (EPI == EPI_RESID)
        x = *reinterpret_cast<const f32x4*>(p.resid + static_cast<int64_t>(row) * p.ldr + col) + x;
      if constexpr (OUT_BF16) *reinterpret_cast<uint2*>(static_cast<uint16_t*>(p.C) + o) = pack4(x);
      else *reinterpret_cast<f32x4*>(static_cast<float*>(p.C) + o) = x;
    }
  }
}

template <int BM, int BN, int EPI, bool OUT_BF16>
void launch_reduce(const GemmParams& p, hipStream_t s) {
  constexpr int PER_TILE = (BM / 32) * (is_swiglu(EPI) ? BN / 64 : BN / 32);
  hipLaunchKernelGGL((gemm_reduce<BM, BN, EPI, OUT_BF16>), dim3(static_cast<unsigned>(p.n_tiles) * PER_TILE), dim3(256),
                     0, s, p);
}

// The k-split tails' partial tiles live in a workspace the caller passes in
// (mr_gemm_workspace_bytes gives the size the plan below wants; a smaller or
// absent one narrows or drops the split). kSplitCapBytes bounds the plan.
constexpr int64_t kSplitCapBytes = 128ll << 20;
constexpr int kSplitMinKt = 96;

// Blocks per tile for the remainder past the last whole wave of large tiles
// (1 = no split), with its partials within ws_bytes.
int split_plan(int64_t tiles, int KT, int64_t ws_bytes) {
  constexpr int64_t wave = 256, tile_bytes = 256ll * 256 * 4;
  const int64_t tail = tiles % wave;
  int split = 1;
  if (!tail || KT < kSplitMinKt) return 1;
  const int64_t cap = ws_bytes < kSplitCapBytes ? ws_bytes : kSplitCapBytes;
  double best = 1.0;
  for (int sp = 2; sp <= 16 && sp <= KT; ++sp) {
    if (tail * sp * tile_bytes > cap) break;
    const double t = static_cast<double>((tail * sp + wave - 1) / wave) / sp;
    if (t < best - 1e-9) {
      best = t;
      split = sp;
    }
  }
  return split;
}

// How a product runs is whichever of four plans the times below expect to take
// least, with the margins of plan_for. The constants are microseconds, fitted to
// 304 products (the twelve of a block over geometries of hidden 576 .. 3584 and
// 256 .. 8192 tokens, and the vocabulary heads), each run by every plan, with its
// operands in cache and, for half of them, from memory, and the deep kernel's
// slope over long runs to 667 from memory (those over 128 .. 8192 tokens, the
// split-precision products and 120 of random sizes). Over these 667 the plan
// chosen is on average 1.5 % slower than the best of the plans, and 10 % of them
// and more slower than the large and small tiles alone for one (2560 x 2048 x
// 4096 of MR_TN on 160 wide tiles, 59 -> 67; on average they gain 29 %). The start
// and epilogue of a round of tiles depend on the kind of output.
enum Output { OUT_B16, OUT_F32, OUT_RESID, OUT_SWIGLU, OUT_SWIGLU_BWD, OUTPUTS };

// 128 x 128 or (wide) 256 x 128 tiles on the deep kernel, one block per CU:
// rounds of 256, the tail past them cut along K into `split` blocks a tile, whose
// partials take a round trip and a second kernel. A k-tile takes longer the more
// CUs work, and, with operands from memory, `more` longer from the 25th of a run
// on (128 x 128 tiles 0.6 us and more a k-tile: 1024 x 2560 x 6144 in one run 62
// us, 49 on large tiles; of 46 such products with runs of 72 k-tiles and more 45
// were slower than another plan, of 44 on wide tiles with runs of 120 and more 38).
struct DeepTimes {
  double launch, start[OUTPUTS], round, tail, busy, reduce, partial, more;
};
constexpr DeepTimes kDeepTimes = {0.9, {3.0, 4.0, 5.4, 4.9, 6.7}, 0.453, 0.305, 0.149, 1.2, 0.035, 0.15};
constexpr DeepTimes kWideTimes = {0.6, {4.3, 5.4, 7.5, 6.9, 11.0}, 0.838, 0.526, 0.266, 1.1, 0.051, 0.06};
double deep_time(const DeepTimes& c, int64_t tiles, int KT, int split, Output o) {
  auto late = [&](int kt) { return kt > 24 ? c.more * (kt - 24) : 0.0; };
  const int64_t tail = tiles % 256, blocks = tail * split;
  const int run = (KT + split - 1) / split;
  double t = c.launch + static_cast<double>(tiles / 256) * (c.start[o] + c.round * KT + late(KT));
  if (tail) t += c.start[o] + run * (c.tail + c.busy * static_cast<double>(blocks) / 256.0) + late(run);
  if (split > 1) t += c.reduce + c.partial * static_cast<double>(blocks);
  return t;
}

// The double-buffered 128 x 128 tiles, two blocks per CU: rounds of 512.
double small_time(int64_t tiles, int KT, Output o) {
  constexpr double start[OUTPUTS] = {2.0, 3.6, 4.8, 4.2, 7.7};
  const int64_t r = tiles % 512;
  double t = static_cast<double>(tiles / 512) * (start[o] + 1.011 * KT);
  if (r) t += start[o] + KT * (r <= 256 ? 0.642 : 0.832 + 0.195 * static_cast<double>(r - 256) / 256.0);
  return t;
}

// 256 x 256 tiles, one per CU: rounds of 256, the tail in `split` blocks a tile
// or, up to half a round of plain stores, as quarter tiles (see launch).
double big_time(int64_t tiles, int KT, int split, Output o) {
  constexpr double start[OUTPUTS] = {7.5, 9.2, 12.1, 10.4, 18.9};
  const int64_t tail = tiles % 256, blocks = tail * split;
  double t = static_cast<double>(tiles / 256) * (start[o] + 1.481 * KT);
  if (tail && split == 1 && o <= OUT_F32 && tiles >= 256 && tail <= 128) {
    t += start[o] + 0.809 * KT;
  } else if (tail) {
    const double busy = blocks < 256 ? static_cast<double>(blocks) / 256.0 : 1.0;
    t += static_cast<double>((blocks + 255) / 256) * (start[o] + (KT + split - 1) / split * (0.87 + 0.578 * busy));
  }
  if (split > 1) t += 0.9 + 0.065 * static_cast<double>(blocks);
  return t;
}

enum Kind { BIG, SMALL, DEEP, WIDE };
struct Plan {
  Kind kind;
  int split;  // DEEP, WIDE: blocks per tail tile
};

// The plan of an M x N x (64 KT) product with ws_bytes for partials. rows: M
// counts activation rows (NT, NN), not weight rows (TN). There a product of
// under kSplitMinKt k-tiles is never cut along K, so that a row's sums are the
// same bits whatever other rows come with it: a step in pieces has the
// activations of the whole batch's step. (Cutting them too gained 9 us of a
// 0.5B scoring batch's 2,397.) The deep kernel is taken for 1.5 % or more, and of up
// to kShortKt k-tiles large tiles over small ones for 12 % or more: within these
// the times do not tell them apart, and the wrong one cost more than the right one
// gave (weight gradients of 512 tokens and fewer, whose outputs are most of
// their bytes: 3584 x 18944 x 512 100 us on small tiles, 108 on large).
constexpr int kShortKt = 8;
Plan plan_for(int64_t M, int64_t N, int KT, bool rows, Output o, int64_t ws_bytes) {
  const int64_t big = ((M + 255) / 256) * ((N + 255) / 256);
  const int64_t small = ((M + 127) / 128) * ((N + 127) / 128);
  const int64_t wide = ((M + 255) / 256) * ((N + 127) / 128);
  Plan p{BIG, 1};
  double best = big_time(big, KT, split_plan(big, KT, ws_bytes), o);
  const double t_small = small_time(small, KT, o);
  if (t_small * (KT <= kShortKt ? 0.88 : 1.0) < best) {
    best = t_small;
    p.kind = SMALL;
  }
  best *= 0.985;
  auto deep = [&](Kind kind, const DeepTimes& times, int64_t tiles, int64_t tile_bytes) {
    const int64_t tail = tiles % 256;
    for (int sp = 1; sp <= 16; ++sp) {
      if (sp > 1 && (!tail || (rows && KT < kSplitMinKt) || tail * sp > 256 || sp * 2 > KT || tail * sp * tile_bytes > ws_bytes)) break;
      const double t = deep_time(times, tiles, KT, sp, o);
      if (t < best) {
        best = t;
        p = Plan{kind, sp};
      }
    }
  };
  deep(DEEP, kDeepTimes, small, 128ll * 128 * 4);
  deep(WIDE, kWideTimes, wide, 256ll * 128 * 4);
  return p;
}

// Bytes of partials the plan uses for an M x N x K product (0: no split),
// whatever its layout and output.
int64_t split_bytes(int64_t M, int64_t N, int64_t K) {
  const int KT = static_cast<int>(K / BK);
  int64_t bytes = 0;
  for (int v = 0; v < 2 * OUTPUTS; ++v) {
    const int o = v >> 1;
    const bool rows = v & 1;
    const Plan p = plan_for(M, N, KT, rows, static_cast<Output>(o), kSplitCapBytes);
    int64_t b = 0;
    if ((p.kind == DEEP || p.kind == WIDE) && p.split > 1) {
      const int64_t bm = p.kind == WIDE ? 256 : 128;
      b = (((M + bm - 1) / bm) * ((N + 127) / 128) % 256) * p.split * bm * 128 * 4;
    } else if (p.kind == BIG) {
      const int64_t tiles = ((M + 255) / 256) * ((N + 255) / 256);
      const int split = split_plan(tiles, KT, kSplitCapBytes);
      if (split > 1) {
        const int kt_per = (KT + split - 1) / split;
        b = (tiles % 256) * ((KT + kt_per - 1) / kt_per) * 256ll * 256 * 4;
      }
    }
    bytes = b > bytes ? b : bytes;
  }
  return bytes;
}

// Whether the last wave of a large-tile launch runs as quarter tiles (see launch).
bool quarter_tail(int64_t tiles, int split) { return split == 1 && tiles >= 256 && tiles % 256 && tiles % 256 <= 128; }

// Large tiles go out in whole waves of 256 (one per CU). When K is long (at
// least kSplitMinKt steps, so a tile takes far longer than the partial-tile
// round trip), a remainder that would leave CUs idle in a last, partial wave
// (or a whole grid under one wave) is cut along K instead: ksplit blocks per
// tile, chosen (up to 16) to minimise the remainder's time in tile units,
// ceil(tail * ksplit / 256) / ksplit, within the workspace.
// Whole 256 x 256 tiles tile0 .. tile0 + n - 1 of p, without a k split: the
// 4-wave kernel (K of at least two k-tiles), else the 8-wave one.
// MR_GEMM_8WAVE=1 in the environment keeps every launch on the 8-wave kernel
// (read at every launch; the two kernels give bit-identical results, which
// the tests check).
bool use_4wave(int KT) {
  const char* e = getenv("MR_GEMM_8WAVE");
  return !(e && e[0] == '1') && KT >= 2;
}

template <bool AK, bool BKM, int EPI, bool OB>
void launch_whole(GemmParams q, int tile0, int64_t n, hipStream_t s) {
  q.tile0 = tile0;
  q.n_tiles = static_cast<int>(n);
  q.ksplit = 1;
  q.kt_per = q.K / BK;
  q.sub = 0;
  if (use_4wave(q.K / BK))
    hipLaunchKernelGGL((gemm4_kernel<AK, BKM, EPI, OB>), dim3(static_cast<unsigned>(n)), dim3(64 * kWaves4), 0, s, q);
  else
    hipLaunchKernelGGL((gemm_kernel<256, 256, AK, BKM, EPI, OB>), dim3(static_cast<unsigned>(n)), dim3(kThreads), 0,
                       s, q);
}

template <int BM, int BN, bool AK, bool BKM, int EPI, bool OB>
int launch(GemmParams p, hipStream_t s) {
  p.grid_m = (p.M + BM - 1) / BM;
  p.grid_n = (p.N + BN - 1) / BN;
  const int64_t tiles = static_cast<int64_t>(p.grid_m) * p.grid_n;
  if (tiles > 0x7fffffff) return fail(MR_EINVAL, "mr_gemm: problem too large");
  const int KT = p.K / BK;
  constexpr int64_t wave = 256;
  const int64_t tail = tiles % wave, full = tiles - tail;
  const int split = BM == 256 && p.ws ? split_plan(tiles, KT, p.ws_bytes) : 1;
  if constexpr (BM == 256 && (EPI == EPI_STORE || EPI == EPI_SWIGLU_SPLIT)) {
    // A last wave at most half full runs as quarter tiles (two per CU)
    // instead of leaving half the CUs or more idle: measured 5-6 % faster on
    // the 7B block's q/k/v projection (4.5 waves) and its attention-output and
    // q/k/v input gradients (3.5 waves). (The residual and SwiGLU-backward
    // epilogues ran no faster or slower on quarter tiles.)
    if (quarter_tail(tiles, split)) {
      launch_whole<AK, BKM, EPI, OB>(p, 0, full, s);
      GemmParams q = p;
      q.ksplit = 1;
      q.kt_per = KT;
      q.tile0 = static_cast<int>(full);
      q.n_tiles = static_cast<int>(4 * tail);
      q.sub = 1;
      hipLaunchKernelGGL((gemm_kernel<BM / 2, BN / 2, AK, BKM, EPI, OB>),
                         dim3(static_cast<unsigned>(4 * tail)), dim3(kThreads), 0, s, q);
      MR_LAUNCH_CHECK("mr_gemm");
      return MR_OK;
    }
  }
  if (split == 1) {
    if constexpr (BM == 256) {
      launch_whole<AK, BKM, EPI, OB>(p, 0, tiles, s);
    } else {
      p.tile0 = 0;
      p.n_tiles = static_cast<int>(tiles);
      p.ksplit = 1;
      p.kt_per = KT;
      hipLaunchKernelGGL((gemm_kernel<BM, BN, AK, BKM, EPI, OB>), dim3(static_cast<unsigned>(tiles)),
                         dim3(kThreads), 0, s, p);
    }
    MR_LAUNCH_CHECK("mr_gemm");
    return MR_OK;
  }
  if (full) launch_whole<AK, BKM, EPI, OB>(p, 0, full, s);
  p.tile0 = static_cast<int>(full);
  p.n_tiles = static_cast<int>(tail);
  p.kt_per = (KT + split - 1) / split;
  p.ksplit = (KT + p.kt_per - 1) / p.kt_per;  // no empty split
  if (BM == 256 && use_4wave(p.kt_per))
    hipLaunchKernelGGL((gemm4_kernel<AK, BKM, EPI, OB>), dim3(static_cast<unsigned>(tail * p.ksplit)),
                       dim3(64 * kWaves4), 0, s, p);
  else
    hipLaunchKernelGGL((gemm_kernel<BM, BN, AK, BKM, EPI, OB>),
                       dim3(static_cast<unsigned>(tail * p.ksplit)), dim3(kThreads), 0, s, p);
  launch_reduce<BM, BN, EPI, OB>(p, s);
  MR_LAUNCH_CHECK("mr_gemm");
  return MR_OK;
}

// BM x 128 tiles on the deep kernel: whole rounds of 256, then the tail cut along K.
template <int BM, bool AK, bool BKM, int EPI, bool OB>
int launch_deep(GemmParams p, int split, hipStream_t s) {
  p.grid_m = (p.M + BM - 1) / BM;
  p.grid_n = (p.N + 127) / 128;
  const int64_t tiles = static_cast<int64_t>(p.grid_m) * p.grid_n;
  const int KT = p.K / BK;
  p.n_tiles = static_cast<int>(tiles % 256);
  p.tile0 = static_cast<int>(tiles) - p.n_tiles;
  p.kt_per = (KT + split - 1) / split;
  p.ksplit = (KT + p.kt_per - 1) / p.kt_per;  // no empty split
  if (use_4wave(KT)) {
    hipLaunchKernelGGL((gemm_deep_kernel<BM, AK, BKM, EPI, OB>), dim3(static_cast<unsigned>(p.tile0 + p.n_tiles * p.ksplit)),
                       dim3(64 * kWaves4), 0, s, p);
  } else {  // the same tiles and splits on the 8-wave kernel
    GemmParams q = p;
    q.n_tiles = p.tile0;
    q.tile0 = 0;
    q.ksplit = 1;
    q.kt_per = KT;
    if (q.n_tiles)
      hipLaunchKernelGGL((gemm_kernel<BM, 128, AK, BKM, EPI, OB>), dim3(static_cast<unsigned>(q.n_tiles)), dim3(kThreads),
                         0, s, q);
    if (p.n_tiles)
      hipLaunchKernelGGL((gemm_kernel<BM, 128, AK, BKM, EPI, OB>), dim3(static_cast<unsigned>(p.n_tiles * p.ksplit)),
                         dim3(kThreads), 0, s, p);
  }
  if (p.n_tiles && p.ksplit > 1) launch_reduce<BM, 128, EPI, OB>(p, s);
  MR_LAUNCH_CHECK("mr_gemm");
  return MR_OK;
}

template <bool AK, bool BKM, int EPI, bool OB>
int dispatch(GemmParams p, hipStream_t s) {
  constexpr Output o = EPI == EPI_RESID        ? OUT_RESID
                       : EPI == EPI_SWIGLU     ? OUT_SWIGLU
                       : EPI == EPI_SWIGLU_BWD ? OUT_SWIGLU_BWD
                       : EPI == EPI_SWIGLU_SPLIT ? OUT_F32  // the fp32 product's plan, so its bits
                       : OB                    ? OUT_B16
                                               : OUT_F32;
  const Plan plan = plan_for(p.M, p.N, p.K / BK, AK, o, p.ws ? p.ws_bytes : 0);
  if (plan.kind == WIDE) return launch_deep<256, AK, BKM, EPI, OB>(p, plan.split, s);
  if (plan.kind == DEEP) return launch_deep<128, AK, BKM, EPI, OB>(p, plan.split, s);
  if (plan.kind == SMALL) return launch<128, 128, AK, BKM, EPI, OB>(p, s);
  return launch<256, 256, AK, BKM, EPI, OB>(p, s);
}

// Load offsets are 32-bit: 256 rows of a K-major tile span 256 * ld * 2 bytes;
// the epilogues' lane offsets within a 32-row slice of an output are 32-bit too.
constexpr int kMaxLd = 1 << 22;

bool ok16(const void* p, int64_t ld) {
  return aligned16(p) && (ld % 8) == 0;
}

// The caller's k-split workspace: null or zero bytes disable the split.
bool set_workspace(GemmParams& p, void* ws, size_t bytes) {
  if (!ws || !bytes) {
    p.ws = nullptr;
    p.ws_bytes = 0;
    return true;
  }
  if (!aligned16(ws)) return false;
  p.ws = static_cast<float*>(ws);
  p.ws_bytes = static_cast<int64_t>(bytes);
  return true;
}

}  // namespace
}  // namespace mr

namespace mr {
namespace {

// Bytes from the first element of a rows x width matrix (leading dimension
// ld, esize-byte elements) to one past its last.
int64_t span_bytes(int64_t rows, int64_t ld, int64_t width, int64_t esize) {
  return ((rows - 1) * ld + width) * esize;
}

// A region the launch writes (outputs, k-split partials) against the regions
// it reads: tiles read operand panels while other tiles write, so any shared
// byte changes results. Each pair is (pointer, bytes); null pointers are
// skipped. Returns whether any written region overlaps any other region.
struct Region {
  const void* p;
  int64_t n;
};
template <int NW, int NR>
bool writes_overlap(const Region (&w)[NW], const Region (&r)[NR]) {
  for (int a = 0; a < NW; ++a) {
    if (!w[a].p) continue;
    for (int b = 0; b < NR; ++b)
      if (r[b].p && overlap(w[a].p, w[a].n, r[b].p, r[b].n)) return true;
    for (int b = a + 1; b < NW; ++b)
      if (w[b].p && overlap(w[a].p, w[a].n, w[b].p, w[b].n)) return true;
  }
  return false;
}

// mr_gemm_swiglu, or with `split` (rows of 3N) mr_gemm_swiglu_split, where
// act is optional.
int swiglu_product(const char* fn, int64_t M, int64_t N, int64_t K, const void* X, int64_t ldx, const void* Wgu,
                   int64_t ldw, void* split, int64_t ldsplit, void* act, int64_t ldact, void* gu, int64_t ldgu,
                   void* workspace, size_t workspace_bytes, void* stream) {
  if (M <= 0 || N <= 0) return MR_OK;
  if (!X || !Wgu || (!act && !split)) return fail(MR_EINVAL, "%s: null operand", fn);
  if (M % 8 || N % 32 || K % BK || K <= 0)
    return fail(MR_EINVAL, "%s: M %% 8, N %% 32 and K %% %d must be 0", fn, BK);
  if (!ok16(X, ldx) || !ok16(Wgu, ldw) || (act && !ok16(act, ldact)) || (gu && !ok16(gu, ldgu)) ||
      (split && !ok16(split, ldsplit)))
    return fail(MR_EINVAL, "%s: operands and outputs must be 16-byte aligned with leading "
                "dimensions multiples of 8", fn);
  if (ldx < K || ldw < K || (act && ldact < N) || (gu && ldgu < 2 * N) || (split && ldsplit < 3 * N) || ldx > kMaxLd ||
      ldw > kMaxLd || (act && ldact > kMaxLd) || (gu && ldgu > kMaxLd) || (split && ldsplit > kMaxLd))
    return fail(MR_EINVAL, "%s: bad leading dimension", fn);
  {
    const Region w[4] = {{act, act ? span_bytes(M, ldact, N, 2) : 0}, {gu, gu ? span_bytes(M, ldgu, 2 * N, 2) : 0},
                         {split, split ? span_bytes(M, ldsplit, 3 * N, 2) : 0},
                         {workspace, static_cast<int64_t>(workspace_bytes)}};
    const Region r[2] = {{X, span_bytes(M, ldx, K, 2)}, {Wgu, span_bytes(2 * N, ldw, K, 2)}};
    if (writes_overlap(w, r))
      return fail(MR_EINVAL, "%s: act, gu and the workspace must not overlap X, Wgu or each other", fn);
  }
  GemmParams p{};
  p.M = static_cast<int>(M);
  p.N = static_cast<int>(2 * N);
  p.n_out = static_cast<int>(N);
  p.K = static_cast<int>(K);
  p.A = static_cast<const uint16_t*>(X);
  p.lda = ldx;
  p.B = static_cast<const uint16_t*>(Wgu);
  p.ldb = ldw;
  p.C = split ? split : act;
  p.ldc = split ? ldsplit : ldact;
  p.gu = static_cast<uint16_t*>(gu);
  p.ldgu = ldgu;
  if (!set_workspace(p, workspace, workspace_bytes))
    return fail(MR_EINVAL, "%s: workspace must be 16-byte aligned", fn);
  const hipStream_t s = static_cast<hipStream_t>(stream);
  if (!split) return dispatch<true, true, EPI_SWIGLU, true>(p, s);
  p.act = static_cast<uint16_t*>(act);
  p.ldact = ldact;
  return dispatch<true, true, EPI_SWIGLU_SPLIT, true>(p, s);
}

}  // namespace
}  // namespace mr

extern "C" {

size_t mr_gemm_workspace_bytes(int64_t M, int64_t N, int64_t K) {
  if (M <= 0 || N <= 0 || K <= 0) return 0;
  return static_cast<size_t>(mr::split_bytes(M, N, K));
}

int mr_gemm_plan(int layout, int output, int64_t M, int64_t N, int64_t K, size_t workspace_bytes, int* tiles_out,
                 int* split_out, int64_t* tail_out) {
  using namespace mr;
  clear_error();
  if (layout < 0 || layout > 2 || output < MR_OUT_F32 || output > MR_OUT_SWIGLU_BWD)
    return fail(MR_EINVAL, "mr_gemm_plan: unknown layout %d or output %d", layout, output);
  if (M <= 0 || N <= 0 || K <= 0 || K % BK || M > 0x7fffffff || N > 0x7fffffff || K > 0x7fffffff)
    return fail(MR_EINVAL, "mr_gemm_plan: M and N positive, K a positive multiple of %d", BK);
  if (!tiles_out || !split_out || !tail_out) return fail(MR_EINVAL, "mr_gemm_plan: null output");
  constexpr Output kinds[] = {OUT_F32, OUT_B16, OUT_RESID, OUT_SWIGLU, OUT_F32, OUT_SWIGLU_BWD};
  const int KT = static_cast<int>(K / BK);
  const int64_t ws = static_cast<int64_t>(workspace_bytes < kSplitCapBytes ? workspace_bytes : kSplitCapBytes);
  const Plan p = plan_for(M, N, KT, layout != MR_TN, kinds[output], ws);
  const int64_t bm = p.kind == BIG || p.kind == WIDE ? 256 : 128, bn = p.kind == BIG ? 256 : 128;
  const int64_t tiles = ((M + bm - 1) / bm) * ((N + bn - 1) / bn);
  int split = p.kind == BIG ? split_plan(tiles, KT, ws) : p.split;
  if (p.kind != SMALL && split > 1) split = (KT + (KT + split - 1) / split - 1) / ((KT + split - 1) / split);  // no empty split
  const bool quarters = p.kind == BIG && (output <= MR_OUT_BF16 || output == MR_OUT_SWIGLU_SPLIT) && quarter_tail(tiles, split);
  *tiles_out = p.kind == BIG ? (quarters ? MR_TILES_LARGE_QUARTERS : MR_TILES_LARGE)
                             : p.kind == SMALL ? MR_TILES_SMALL : p.kind == DEEP ? MR_TILES_DEEP : MR_TILES_WIDE;
  *split_out = split;
  *tail_out = p.kind == SMALL ? tiles : tiles % 256;
  return MR_OK;
}

int mr_gemm(int layout, int64_t M, int64_t N, int64_t K, const void* A, int64_t lda,
            const void* B, int64_t ldb, void* C, int c_dtype, int64_t ldc, const float* bias,
            const float* resid, int64_t ldr, void* workspace, size_t workspace_bytes, void* stream) {
  using namespace mr;
  clear_error();
  if (M < 0 || N < 0 || K < 0) return fail(MR_EINVAL, "mr_gemm: negative size");
  if (M == 0 || N == 0) return MR_OK;
  if (!A || !B || !C) return fail(MR_EINVAL, "mr_gemm: null operand");
  if (M % 8 || N % 8 || K % BK || K == 0)
    return fail(MR_EINVAL, "mr_gemm: M and N must be multiples of 8 and K a positive multiple of %d "
                "(M=%lld N=%lld K=%lld)", BK, (long long)M, (long long)N, (long long)K);
  if (M > 0x7fffffff || N > 0x7fffffff || K > 0x7fffffff) return fail(MR_EINVAL, "mr_gemm: too large");
  if (lda > kMaxLd || ldb > kMaxLd || ldc > kMaxLd || (resid && ldr > kMaxLd))
    return fail(MR_EINVAL, "mr_gemm: leading dimensions above %d are not supported", kMaxLd);
  if (!ok16(A, lda) || !ok16(B, ldb))
    return fail(MR_EINVAL, "mr_gemm: operands must be 16-byte aligned with ld a multiple of 8");
  if (c_dtype != MR_F32 && c_dtype != MR_BF16) return fail(MR_EINVAL, "mr_gemm: C must be fp32 or bf16");
  if (!aligned16(C) || ldc % (c_dtype == MR_BF16 ? 8 : 4) || (resid && (!aligned16(resid) || ldr % 4)))
    return fail(MR_EINVAL, "mr_gemm: C and resid must be 16-byte aligned with 16-byte rows");
  if (resid && c_dtype != MR_F32) return fail(MR_EINVAL, "mr_gemm: the residual form writes fp32");
  if (layout < 0 || layout > 2) return fail(MR_EINVAL, "mr_gemm: unknown layout %d", layout);
  {
    const bool a_kmajor = layout != 2, b_kmajor = layout == 0;
    if (lda < (a_kmajor ? K : M) || ldb < (b_kmajor ? K : N) || ldc < N || (resid && ldr < N))
      return fail(MR_EINVAL, "mr_gemm: a leading dimension is smaller than its row");
    // C may be the residual itself (same place, same rows), nothing else it reads
    const int64_t nc = span_bytes(M, ldc, N, c_dtype == MR_BF16 ? 2 : 4);
    const bool in_place = resid == C && ldr == ldc;
    const Region w[2] = {{C, nc}, {workspace, static_cast<int64_t>(workspace_bytes)}};
    const Region r[3] = {{A, a_kmajor ? span_bytes(M, lda, K, 2) : span_bytes(K, lda, M, 2)},
                         {B, b_kmajor ? span_bytes(N, ldb, K, 2) : span_bytes(K, ldb, N, 2)},
                         {in_place ? nullptr : resid, resid ? span_bytes(M, ldr, N, 4) : 0}};
    if (writes_overlap(w, r) || (in_place && workspace && overlap(workspace, workspace_bytes, C, nc)))
      return fail(MR_EINVAL, "mr_gemm: C and the workspace must not overlap A, B, the residual (unless C is "
                  "the residual itself) or each other");
  }
  GemmParams p{};
  p.M = static_cast<int>(M);
  p.N = static_cast<int>(N);
  p.K = static_cast<int>(K);
  p.A = static_cast<const uint16_t*>(A);
  p.lda = lda;
  p.B = static_cast<const uint16_t*>(B);
  p.ldb = ldb;
  p.C = C;
  p.ldc = ldc;
  p.bias = bias;
  p.resid = resid;
  p.ldr = ldr;
  if (!set_workspace(p, workspace, workspace_bytes))
    return fail(MR_EINVAL, "mr_gemm: workspace must be 16-byte aligned");
  hipStream_t s = static_cast<hipStream_t>(stream);
  const bool ob = c_dtype == MR_BF16;
#define MR_GEMM_CASE(AK, BKM)                                                             \
  if (resid) return dispatch<AK, BKM, EPI_RESID, false>(p, s);                            \
  return ob ? dispatch<AK, BKM, EPI_STORE, true>(p, s)                                    \
            : dispatch<AK, BKM, EPI_STORE, false>(p, s);
  switch (layout) {
    case 0: { MR_GEMM_CASE(true, true) }    // NT: Y = X W^T
    case 1: { MR_GEMM_CASE(true, false) }   // NN: dX = dY W
    case 2: { MR_GEMM_CASE(false, false) }  // TN: dW = dY^T X
    default: return fail(MR_EINVAL, "mr_gemm: unknown layout %d", layout);
  }
#undef MR_GEMM_CASE
}

int mr_gemm_swiglu(int64_t M, int64_t N, int64_t K, const void* X, int64_t ldx, const void* Wgu,
                   int64_t ldw, void* act, int64_t ldact, void* gu, int64_t ldgu, void* workspace,
                   size_t workspace_bytes, void* stream) {
  mr::clear_error();
  return mr::swiglu_product("mr_gemm_swiglu", M, N, K, X, ldx, Wgu, ldw, nullptr, 0, act, ldact, gu, ldgu, workspace,
                            workspace_bytes, stream);
}

int mr_gemm_swiglu_split(int64_t M, int64_t N, int64_t K, const void* X, int64_t ldx, const void* Wgu,
                         int64_t ldw, void* act_split, int64_t ldsplit, void* act, int64_t ldact, void* gu,
                         int64_t ldgu, void* workspace, size_t workspace_bytes, void* stream) {
  mr::clear_error();
  if (M <= 0 || N <= 0) return MR_OK;
  if (!act_split) return mr::fail(MR_EINVAL, "mr_gemm_swiglu_split: null operand");
  if (!act != !gu) return mr::fail(MR_EINVAL, "mr_gemm_swiglu_split: act and gu come together");
  return mr::swiglu_product("mr_gemm_swiglu_split", M, N, K, X, ldx, Wgu, ldw, act_split, ldsplit, act, ldact, gu,
                            ldgu, workspace, workspace_bytes, stream);
}

int mr_gemm_swiglu_bwd(int64_t M, int64_t N, int64_t K, const void* dd, int64_t ldd,
                       const void* Wd, int64_t ldw, const void* gu, int64_t ldgu, void* dgu,
                       int64_t lddgu, void* workspace, size_t workspace_bytes, void* stream) {
  using namespace mr;
  clear_error();
  if (M <= 0 || N <= 0) return MR_OK;
  if (!dd || !Wd || !gu || !dgu) return fail(MR_EINVAL, "mr_gemm_swiglu_bwd: null operand");
  if (M % 8 || N % 32 || K % BK || K == 0)
    return fail(MR_EINVAL, "mr_gemm_swiglu_bwd: M %% 8, N %% 32 and K %% %d must be 0", BK);
  if (!ok16(dd, ldd) || !ok16(Wd, ldw) || !ok16(gu, ldgu) || !ok16(dgu, lddgu))
    return fail(MR_EINVAL, "mr_gemm_swiglu_bwd: operands and gu/dgu must be 16-byte aligned with leading "
                "dimensions multiples of 8");
  if (ldd < K || ldw < N || lddgu < 2 * N || ldd > kMaxLd || ldw > kMaxLd || lddgu > kMaxLd)
    return fail(MR_EINVAL, "mr_gemm_swiglu_bwd: bad leading dimension");
  if (ldgu != lddgu) return fail(MR_EINVAL, "mr_gemm_swiglu_bwd: gu and dgu must share a layout");
  {
    // dgu may be written over gu itself: each piece of gu is read before the
    // same piece of dgu is written, by the same lane
    const int64_t ng = span_bytes(M, ldgu, 2 * N, 2);
    const Region w[2] = {{dgu, ng}, {workspace, static_cast<int64_t>(workspace_bytes)}};
    const Region r[3] = {{dd, span_bytes(M, ldd, K, 2)}, {Wd, span_bytes(K, ldw, N, 2)},
                         {dgu == gu ? nullptr : gu, ng}};
    if (writes_overlap(w, r) || (dgu == gu && workspace && overlap(workspace, workspace_bytes, gu, ng)))
      return fail(MR_EINVAL, "mr_gemm_swiglu_bwd: dgu and the workspace must not overlap dd, Wd, gu (unless dgu "
                  "is gu itself) or each other");
  }
  GemmParams p{};
  p.M = static_cast<int>(M);
  p.N = static_cast<int>(N);
  p.K = static_cast<int>(K);
  p.A = static_cast<const uint16_t*>(dd);
  p.lda = ldd;
  p.B = static_cast<const uint16_t*>(Wd);
  p.ldb = ldw;
  p.C = dgu;
  p.ldc = lddgu;
  p.gu = const_cast<uint16_t*>(static_cast<const uint16_t*>(gu));
  p.ldgu = ldgu;
  if (!set_workspace(p, workspace, workspace_bytes))
    return fail(MR_EINVAL, "mr_gemm_swiglu_bwd: workspace must be 16-byte aligned");
  return dispatch<true, false, EPI_SWIGLU_BWD, true>(p, static_cast<hipStream_t>(stream));
}

}  // extern "C"
