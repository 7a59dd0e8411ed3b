// Prefill projections: Y = X W^T for many rows on the MFMA units.
//
// Four waves in a 2x2 arrangement, MFMA 16x16x32, B fragments from the tiled
// weight layout shared with the decode GEMV (one 16-byte piece per lane per
// 16x32 fragment):
// - small grids (gemm_small_kernel): tiles of 32 to 128 rows x 32 to 128
//   columns, dense or Q8_0, chosen so that the grid covers the CUs (try_small);
// - dense 16-bit weights (gemm_dma_kernel, 128 or 256 rows x 128 columns):
//   both operands go global -> LDS by direct-to-LDS loads through a ring of
//   32-k stages; waves hold 64 x 64 or 128 x 64;
// - Q8_0 (gemm_q8_kernel, 64 rows x 128 columns): K step 64, X staged global ->
//   registers -> LDS, double-buffered with one barrier per K step (row pitch
//   padded to 72 elements so the MFMA-order 16-byte reads are bank-conflict
//   free), fragments read straight from global memory one K step ahead.
// Every global load is unconditional (out-of-range rows and tiles read
// clamped addresses), so no wait depends on a branch.  Work-groups are
// mapped to tiles over an XCD grid chosen per shape (see tile_of).  Q8_0
// weights are converted to f16 exactly and each 32-wide block's partial
// product is scaled by its f16 scale in f32.
//
// Reference: Linear::forward / FusedLinear::forward (linear.rs:29-100) over
// (b*t, in) rows; call sites qwen3.rs:213, 258, 288-291.
#include <type_traits>

#include "fmd_common.h"
#include "fmd_kernels.h"

namespace {

constexpr int BM = 128, BK = 64, LDA = BK + 8;

template <int A>
__device__ __forceinline__ f32x4 mfma16(u32x4 a, u32x4 b, f32x4 c) {
  if constexpr (A == ACT_F16)
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8, a),
                                                  __builtin_bit_cast(f16x8, b), c, 0, 0, 0);
  else
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a),
                                                   __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
}

__device__ __forceinline__ u32x4 q8_to_f16x8(uint32_t w0, uint32_t w1) {
  uint32_t a, b, c, d;
  i8x4_to_f16x4(w0, a, b);
  i8x4_to_f16x4(w1, c, d);
  return u32x4{a, b, c, d};
}

// 16-byte load at a byte offset (< 4 GiB) from a work-group-uniform base: one
// 32-bit offset register per load instead of 64-bit address arithmetic.
__device__ __forceinline__ u32x4 ld16(const void* ubase, uint32_t byte_off) {
  return *(const u32x4*)((const char*)ubase + byte_off);
}
__device__ __forceinline__ uint32_t ld4(const void* ubase, uint32_t byte_off) {
  return *(const uint32_t*)((const char*)ubase + byte_off);
}

// Weight n-tile handled by a wave's ni-th fragment column in column group cg.
template <int EPI>
__device__ __forceinline__ int wave_tile(int cg, int ntiles, int wn, int ni) {
  if constexpr (EPI == EPI_SWIGLU) {
    const int base = cg * 4 + wn * 2 + (ni & 1);
    return ni < 2 ? base : base + ntiles / 2;
  } else {
    return cg * 8 + wn * 4 + ni;
  }
}

// Row tile mt and column group cg of work-group id.  Work-groups are dealt
// to the 8 XCDs round-robin (id % 8), each XCD with its own L2.  The XCDs
// form an a x (8/a) grid over (row tiles x column groups): XCD x takes the
// row-tile block x / (8/a) and the column-group block x % (8/a), so the X
// rows are fetched by 8/a XCDs and each weight tile by a of them (a is
// chosen per shape by the host to minimise that traffic).  The grid holds
// 8 * Ma * Cb work-groups (Ma = ceil(mtiles / a), Cb = cols / (8/a));
// those past the last row tile return at once (mt >= mtiles).
__device__ __forceinline__ void tile_of(int id, int mtiles, int cols, int a, int& mt, int& cg) {
  const int b = 8 / a, x = id & 7, j = id >> 3;
  const int Ma = (mtiles + a - 1) / a, Cb = cols / b;
  if (Cb < 16) {
    mt = (x / b) * Ma + j / Cb;
    cg = (x % b) * Cb + j % Cb;
    return;
  }
  // A wide block (16 or more column groups): groups of GM row tiles with the
  // row tile fastest, so that an XCD's concurrent work-groups (about 64)
  // span GM row tiles x 64/GM column groups, whose X and weight tiles fit
  // its L2 better than 64/Cb row tiles x all Cb column groups (audio path
  // q|k|v and fc1 at 24,016 rows: 439.5 -> 449.8 windows/s with GM = 8;
  // GM = 16 another +0.6-0.8%, q|k|v 178 -> 171 us; 4 and 32 no better,
  // grouping blocks of 8 column groups too slower; prefill unchanged).
  constexpr int GM = 16;
  const int g = j / (GM * Cb), r = j - g * (GM * Cb);
  const int gm = min(GM, Ma - g * GM);
  mt = (x / b) * Ma + g * GM + r % gm;
  cg = (x % b) * Cb + r / gm;
}

// Four values rounded to the 16-bit activation dtype (round to nearest even).
template <int A>
__device__ __forceinline__ uint2 pack4(f32x4 v) {
  if constexpr (A == ACT_BF16) {
    typedef __bf16 b2 __attribute__((ext_vector_type(2)));
    typedef float f2 __attribute__((ext_vector_type(2)));
    return uint2{__builtin_bit_cast(uint32_t, __builtin_convertvector((f2){v[0], v[1]}, b2)),
                 __builtin_bit_cast(uint32_t, __builtin_convertvector((f2){v[2], v[3]}, b2))};
  } else {
    return uint2{(uint32_t)st_act<A>(v[0]) | ((uint32_t)st_act<A>(v[1]) << 16),
                 (uint32_t)st_act<A>(v[2]) | ((uint32_t)st_act<A>(v[3]) << 16)};
  }
}

// EPI_ROPE: the work-group's 128 columns are head slot cg of q|k|v, and the
// tile (64 or 128 rows) goes on through Attention::forward's q/k RMSNorm,
// RoPE and KvCache::append (qwen3.rs:214-227, 139-144, 86-101) instead of
// being stored.  Its rounded products (rd(x W^T), qwen3.rs:213) are staged
// in LDS, chunk c of row r at chunk position c ^ rope_sw(r), so that the
// 2-byte stores of a wave's four 16-lane groups (rows 4 apart) fall in
// distinct banks; then each 16-lane group finishes
// rows gi, gi + 16, ... (8 dims per lane): q and k heads through norm_rope8,
// the decode attention's routine for the new token (so prefill and decode
// store the same bits for a token), into q_out or the K cache, v heads as
// projected into the V cache.
__device__ __forceinline__ int rope_sw(int r) { return ((r >> 2) & 3) << 1; }

// Position and batch index (pos * 16 + b: b < 16, the prefill batch bound)
// of the rows gi + 16 j (j < BMT / 16) of the tile that this thread's 16-lane
// group finishes, loaded before the K loop; rows past M read row M - 1's
// (they are not stored).
template <int BMT>
struct RopeRows {
  int pb[BMT / 16];
};

template <int BMT>
__device__ __forceinline__ RopeRows<BMT> rope_rows(const GemmArgs& p, int m0) {
  RopeRows<BMT> rr;
  const int gi = threadIdx.x >> 4;
#pragma unroll
  for (int j = 0; j < BMT / 16; ++j) {
    const int gr = min(m0 + gi + 16 * j, p.M - 1);
    rr.pb[j] = p.rope.row_pos[gr] * 16 + p.rope.row_b[gr];
  }
  return rr;
}

// acc: the wave's BMT/2 x 64 accumulators (2 x 2 waves, as the epilogues
// below); stg: BMT x 128 activations of LDS, free once the caller's K loop
// has ended.
// CROSS: the accumulators' layout (dense tiles: see cross below); their 8-byte
// writes (16 rows x 32 bytes) then take the swizzle R & 15.
template <int A, int BMT, int MI, bool CROSS>
__device__ __forceinline__ void rope_epilogue(const GemmArgs& p, const f32x4 (&acc)[MI][4],
                                              typename ActT<A>::T* stg, int m0, int cg,
                                              const RopeRows<BMT>& rr) {
  static_assert(BMT == 32 || BMT == 64 || BMT == 128, "rope tiles");
  typedef typename ActT<A>::T T;
  constexpr int NJ = BMT / 16;   // rows per 16-lane group
  const RopeArgs& q = p.rope;
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6, wm = w >> 1, wn = w & 1;
  const int row = lane & 15, kg = lane >> 4;
  const int dc = threadIdx.x & 15, gi = threadIdx.x >> 4;
  const int slot = cg;
  const bool is_q = slot < q.nh, is_v = slot >= q.nh + q.nkv;
  float g[8];
  u32x4 cr[NJ], sr[NJ];
  if (!is_v) {
    // gain and cos / sin rows, in flight while the tile is staged
    unpack8<A>(*(const u32x4*)((const T*)(is_q ? q.qn_w : q.kn_w) + dc * 8), g);
#pragma unroll
    for (int j = 0; j < NJ; ++j) {
      const size_t o = (size_t)(rr.pb[j] >> 4) * 64 + (dc & 7) * 8;
      cr[j] = *(const u32x4*)((const T*)q.cos + o);
      sr[j] = *(const u32x4*)((const T*)q.sin + o);
    }
  }
  barrier_lds();   // every wave is done with the K loop's LDS
  const int gsw = CROSS ? gi : rope_sw(gi);   // of rows gi + 16 j
  if constexpr (CROSS) {
    T* const wb = stg + (wm * (BMT / 2) + row) * 128 + 4 * (kg & 1);
#pragma unroll
    for (int mi = 0; mi < MI; ++mi)
#pragma unroll
      for (int ni = 0; ni < 4; ++ni)
        *(uint2*)(wb + mi * 16 * 128 + (((wn * 8 + ni * 2 + (kg >> 1)) ^ row) << 3)) =
            pack4<A>(acc[mi][ni]);
  } else {
    // The rows this lane writes are 4 kg + (a multiple of 4) + r, r < 4, so
    // their rope_sw is 2 kg and column wn*64 + ni*16 + row lands at wn*64 +
    // (ni ^ kg)*16 + row.
    T* const wb = stg + (wm * (BMT / 2) + 4 * kg) * 128 + wn * 64 + row;
#pragma unroll
    for (int mi = 0; mi < MI; ++mi)
#pragma unroll
      for (int r = 0; r < 4; ++r)
#pragma unroll
        for (int ni = 0; ni < 4; ++ni) wb[(mi * 16 + r) * 128 + (ni ^ kg) * 16] = st_act<A>(acc[mi][ni][r]);
  }
  barrier_lds();
  const T* const rb = stg + gi * 128 + ((dc ^ gsw) << 3);
#pragma unroll
  for (int j = 0; j < NJ; ++j) {
    const int gr = m0 + gi + 16 * j;
    // a whole 16-lane group leaves together (norm_rope8 reads its lanes)
    if (gr >= p.M) break;
    const u32x4 raw = *(const u32x4*)(rb + j * 16 * 128);
    const int b = rr.pb[j] & 15, pos = rr.pb[j] >> 4;
    if (is_v) {
      T* dst = (T*)q.vc + (((size_t)b * q.nkv + (slot - q.nh - q.nkv)) * q.cap + pos) * 128;
      *(u32x4*)(dst + dc * 8) = raw;
      continue;
    }
    float x[8], c[8], sn[8];
    unpack8<A>(raw, x);
    unpack8<A>(cr[j], c);
    unpack8<A>(sr[j], sn);
    norm_rope8<A>(x, g, c, sn, dc, q.eps);
    uint32_t o[4];
#pragma unroll
    for (int t = 0; t < 4; ++t)
      o[t] = (uint32_t)st_act<A>(x[2 * t]) | ((uint32_t)st_act<A>(x[2 * t + 1]) << 16);
    T* dst = is_q ? (T*)q.q_out + ((size_t)gr * q.nh + slot) * 128
                  : (T*)q.kc + (((size_t)b * q.nkv + (slot - q.nh)) * q.cap + pos) * 128;
    *(u32x4*)(dst + dc * 8) = u32x4{o[0], o[1], o[2], o[3]};
  }
}

// GELU-erf, 0.5 v (1 + erf(v / sqrt 2)), branch-free, from Abramowitz &
// Stegun 7.1.26: erfc(x) ~ t (a1 + t (a2 + t (a3 + t (a4 + t a5)))) exp(-x^2)
// with t = 1 / (1 + p x), |error| <= 1.5e-7 for x >= 0.  With
// h = erfc(|v| / sqrt 2) / 2, the GELU is max(v, 0) - |v| h for either sign
// of v (v - v h for v > 0, v h for v < 0: no cancellation for negative v),
// one fma.  1/sqrt 2 is folded into p, 1/2 into the a_k (exact), and
// exp(-v^2 / 2) is exp2(v (v (-log2(e) / 2))).  The device erff branches on
// the size of its argument, which diverges within a wave.
__device__ __forceinline__ float gelu_erf(float v) {
  constexpr float kP = 0.3275911f;
  constexpr float kA1 = 0.254829592f, kA2 = -0.284496736f, kA3 = 1.421413741f,
                  kA4 = -1.453152027f, kA5 = 1.061405429f;
  constexpr float kRsqrt2 = 0.70710678118654752f, kE = -0.72134752044448170f;
  const float av = fabsf(v);
  const float t = __builtin_amdgcn_rcpf(fmaf(kP * kRsqrt2, av, 1.0f));
  const float poly =
      t * fmaf(t, fmaf(t, fmaf(t, fmaf(t, 0.5f * kA5, 0.5f * kA4), 0.5f * kA3), 0.5f * kA2), 0.5f * kA1);
  const float h = poly * __builtin_amdgcn_exp2f(v * (v * kE));
  // max(v, 0) as one v_max_f32 (fmaxf adds a canonicalising max(v, v) per
  // element; a NaN v makes h NaN, so the result is NaN either way)
  float pos;
  asm("v_max_f32 %0, 0, %1" : "=v"(pos) : "v"(v));
  return fmaf(-av, h, pos);
}

// EPI_AFFINE for an output element from its f32 accumulator (the steps and
// their rounding as AffineArgs states), given the element's bias, residual
// and table values (each used only when its pointer is set).
template <int A>
__device__ __forceinline__ float affine_steps(const GemmArgs& p, float acc, int col, float bias,
                                              float resid, float table) {
  const AffineArgs& f = p.aff;
  float v = rd<A>(acc);
  if (f.bias) v = rd<A>(v + bias);
  if (col < f.scale_cols) v = rd<A>(v * f.scale);
  if (f.act == 1) v = rd<A>(gelu_erf(v));
  else if (f.act == 2) v = rd<A>(v / (1.0f + __expf(-v)));
  if (p.resid) v = rd<A>(resid + v);
  if (f.table) v = rd<A>(v + table);
  return v;
}
// affine_steps over N elements at once, step by step: the same operations
// in the same order for each element, but every step's uniform branch is
// taken once for the block, so the elements' chains are independent
// instructions the compiler can interleave (element by element, each step
// sat in its own basic block and only one chain was in flight).
// Inputs already rounded to the dtype (ROUNDED) skip the first rounding.
// The scale step multiplies each element by its scl (f.scale for the
// scaled columns, 1 for the others: rd(v * 1) = v for a rounded v), so it
// needs no per-element select.  The residual and table values arrive as
// stored (rv, tv) and are widened inside their steps, so the wait for their
// loads falls after the steps that do not need them.
template <int A, int N, bool ROUNDED>
__device__ __forceinline__ void affine_block(const GemmArgs& p, float (&v)[N], const float (&scl)[N],
                                             const float (&bias)[N],
                                             const typename ActT<A>::T (&rv)[N],
                                             const typename ActT<A>::T (&tv)[N]) {
  const AffineArgs& f = p.aff;
  if constexpr (!ROUNDED) {
#pragma unroll
    for (int e = 0; e < N; ++e) v[e] = rd<A>(v[e]);
  }
  if (f.bias) {
#pragma unroll
    for (int e = 0; e < N; ++e) v[e] = rd<A>(v[e] + bias[e]);
  }
  if (f.scale_cols > 0) {
#pragma unroll
    for (int e = 0; e < N; ++e) v[e] = rd<A>(v[e] * scl[e]);
  }
  if (f.act == 1) {
#pragma unroll
    for (int e = 0; e < N; ++e) v[e] = rd<A>(gelu_erf(v[e]));
  } else if (f.act == 2) {
#pragma unroll
    for (int e = 0; e < N; ++e) v[e] = rd<A>(v[e] / (1.0f + __expf(-v[e])));
  }
  if (p.resid) {
#pragma unroll
    for (int e = 0; e < N; ++e) v[e] = rd<A>(ld_act<A>(rv[e]) + v[e]);
  }
  if (f.table) {
#pragma unroll
    for (int e = 0; e < N; ++e) v[e] = rd<A>(v[e] + ld_act<A>(tv[e]));
  }
}

// The same for output element (gr, col), loading its values.
template <int A>
__device__ __forceinline__ float affine_value(const GemmArgs& p, float acc, int gr, int col) {
  typedef typename ActT<A>::T T;
  const AffineArgs& f = p.aff;
  const float bias = f.bias ? ld_act<A>(((const T*)f.bias)[col]) : 0.f;
  const float resid = p.resid ? ld_act<A>(((const T*)p.resid)[(size_t)gr * p.ldy + col]) : 0.f;
  const float table = f.table ? ld_act<A>(((const T*)f.table)[(size_t)(gr % f.period) * p.W.out + col]) : 0.f;
  return affine_steps<A>(p, acc, col, bias, resid, table);
}
// Whether output row gr is stored (EPI_AFFINE skips the rows between windows).
__device__ __forceinline__ bool affine_row(const GemmArgs& p, int gr) {
  return p.aff.period <= 0 || gr % p.aff.period < p.aff.valid;
}

// EPI_RESID: the residual of every output element a lane stores (rows
// 4 kg + r of each 16-row fragment, column `row` of tile[ni]), loaded before
// the K loop so that these scattered 2-byte loads are in flight behind it
// instead of exposed in the epilogue.  Rows past M and tiles past the end
// read clamped addresses (they are not stored).  MI is 2 or 4: the 64- and
// 128-row tiles.
template <int A, int MI>
struct ResidRows {
  typename ActT<A>::T v[MI][4][4];
};

template <int A, int BMT, int MI>
__device__ __forceinline__ ResidRows<A, MI> load_resid(const GemmArgs& p, int m0, const int (&tile)[4],
                                                       const bool (&tv)[4]) {
  typedef typename ActT<A>::T T;
  ResidRows<A, MI> rr;
  const int lane = threadIdx.x & 63, wm = (threadIdx.x >> 6) >> 1;
  const int row = lane & 15, kg = lane >> 4;
#pragma unroll
  for (int mi = 0; mi < MI; ++mi)
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int gr = min(m0 + wm * (BMT / 2) + mi * 16 + 4 * kg + r, p.M - 1);
#pragma unroll
      for (int ni = 0; ni < 4; ++ni)
        rr.v[mi][r][ni] = ((const T*)p.resid)[(size_t)gr * p.ldy + (tv[ni] ? tile[ni] : 0) * 16 + row];
    }
  return rr;
}

// EPI_RESID of the 64-row Q8_0 tiles and the 128-row dense ones: y = rd(resid +
// rd(acc)), 2 bytes at a time, 16 lanes to 32 consecutive bytes of a row.  8-byte
// pieces of the dense tiles' other layout, 16 rows to an instruction, are slower
// (medians of five alternating runs, 2-byte | 8-byte, us, bf16): O at 12,288 rows
// 66.7 | 68.9, 8000 42.0 | 43.2, 4800 33.0 | 35.3; down 87.3 | 90.7, 56.7 | 57.9,
// 45.0 | 47.5; f16 at 6400 rows 36.6 | 39.1 and 52.0 | 54.4.
template <int A, int BMT, int MI>
__device__ __forceinline__ void resid_epilogue(const GemmArgs& p, const f32x4 (&acc)[MI][4], int m0,
                                               const int (&tile)[4], const bool (&tv)[4],
                                               const ResidRows<A, MI>& rr) {
  typedef typename ActT<A>::T T;
  const int lane = threadIdx.x & 63, wm = (threadIdx.x >> 6) >> 1;
  const int row = lane & 15, kg = lane >> 4;
#pragma unroll
  for (int mi = 0; mi < MI; ++mi)
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int gr = m0 + wm * (BMT / 2) + mi * 16 + 4 * kg + r;
      if (gr >= p.M) continue;
#pragma unroll
      for (int ni = 0; ni < 4; ++ni)
        if (tv[ni])
          ((T*)p.y)[(size_t)gr * p.ldy + tile[ni] * 16 + row] =
              st_act<A>(ld_act<A>(rr.v[mi][r][ni]) + rd<A>(acc[mi][ni][r]));
    }
}

// EPI_STORE of the 64-row Q8_0 tiles and the 128- and 256-row dense ones, in the
// same layout, to any alignment.  Against 8-byte pieces of the other layout (us,
// medians of four alternating runs, bf16): K = 1024, N = 6144 at 3200 rows 51.5 |
// 54.8, 6000 90.8 | 96.5, 12,288 174.3 | 185.8, 24,016 331.9 | 351.7; N = 4096
// 36.8 | 38.2, 58.8 | 60.5, 115.0 | 122.0, 257.4 | 262.1.
template <int A, int BMT, int MI>
__device__ __forceinline__ void store_epilogue(const GemmArgs& p, const f32x4 (&acc)[MI][4], int m0,
                                               const int (&tile)[4], const bool (&tv)[4]) {
  typedef typename ActT<A>::T T;
  const int lane = threadIdx.x & 63, wm = (threadIdx.x >> 6) >> 1;
  const int row = lane & 15, kg = lane >> 4;
#pragma unroll
  for (int mi = 0; mi < MI; ++mi)
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int gr = m0 + wm * (BMT / 2) + mi * 16 + 4 * kg + r;
      if (gr >= p.M) continue;
#pragma unroll
      for (int ni = 0; ni < 4; ++ni)
        if (tv[ni]) ((T*)p.y)[(size_t)gr * p.ldy + tile[ni] * 16 + row] = st_act<A>(acc[mi][ni][r]);
    }
}

// EPI_SWIGLU epilogue (Mlp::forward's silu(gate) * up, qwen3.rs:288-291):
// tiles 0, 1 of the wave hold gate columns, tiles 2, 3 the matching up
// columns.  Each 16-row fragment's eight products are computed before any
// of them is stored -- rd(gate), rd(up), rd(silu(gate)), rd(s * u) in that
// order per element -- with no branch between them, so their chains (an
// exponential and a division each) interleave; the row and tile checks
// only guard the stores.
template <int A, int BMT, int MI>
__device__ __forceinline__ void swiglu_epilogue(const GemmArgs& p, const f32x4 (&acc)[MI][4], int m0,
                                                const int (&tile)[4], const bool (&tv)[4]) {
  typedef typename ActT<A>::T T;
  const int lane = threadIdx.x & 63, wm = (threadIdx.x >> 6) >> 1;
  const int row = lane & 15, kg = lane >> 4;
#pragma unroll
  for (int mi = 0; mi < MI; ++mi) {
    float o[4][2];
#pragma unroll
    for (int r = 0; r < 4; ++r)
#pragma unroll
      for (int ni = 0; ni < 2; ++ni) {
        const float gg = rd<A>(acc[mi][ni][r]), u = rd<A>(acc[mi][ni + 2][r]);
        o[r][ni] = rd<A>(gg / (1.0f + __expf(-gg))) * u;
      }
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int gr = m0 + wm * (BMT / 2) + mi * 16 + 4 * kg + r;
#pragma unroll
      for (int ni = 0; ni < 2; ++ni)
        if (gr < p.M && tv[ni]) ((T*)p.y)[(size_t)gr * p.ldy + tile[ni] * 16 + row] = st_act<A>(o[r][ni]);
    }
  }
}

// Q8_0 weights (f16 activations) past the small grids: 64 x 128 tiles, K step
// 64, X staged global -> registers -> LDS, weight fragments and scales read
// straight from global memory one K step ahead.  The tiles scale each block's
// product in f32 on the VALU, so their accumulators live in VGPRs.
template <int EPI>
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2)))
gemm_q8_kernel(GemmArgs p) {
  constexpr int A = ACT_F16, BMT = 64;
  typedef typename ActT<A>::T T;
  constexpr int MI = BMT / 32;   // 16-row fragments per wave (waves are 2 x 2)
  constexpr int NA = BMT / 32;   // 16-byte pieces of the X tile per thread
  __shared__ uint16_t sA[2 * BMT * LDA];
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const int wm = w >> 1, wn = w & 1;
  const int K = p.W.in, ntiles = p.W.out / 16;
  const int cols = EPI == EPI_SWIGLU ? (ntiles / 2 + 3) / 4 : (ntiles + 7) / 8;
  int mt, cg;
  tile_of(blockIdx.x, (p.M + BMT - 1) / BMT, cols, p.map, mt, cg);
  if (mt * BMT >= p.M) return;   // padding of the last row-tile block
  const int m0 = mt * BMT;
  const int row = lane & 15, kg = lane >> 4;
  [[maybe_unused]] RopeRows<EPI == EPI_ROPE ? BMT : 16> rrows;
  if constexpr (EPI == EPI_ROPE) rrows = rope_rows<BMT>(p, m0);

  // Every global load below is unconditional (a branch around a load makes
  // the compiler wait for all outstanding loads at the next join, which
  // serialises the prefetch): rows past M read row M - 1 and weight tiles
  // past the end read the last tile.  Each output depends only on its own X
  // row and weight tile, and those outputs are never stored.
  int tile[4], ltile[4];
  bool tv[4];
#pragma unroll
  for (int ni = 0; ni < 4; ++ni) {
    tile[ni] = wave_tile<EPI>(cg, ntiles, wn, ni);
    tv[ni] = (EPI == EPI_SWIGLU) ? (cg * 4 + wn * 2 + (ni & 1)) < ntiles / 2
                                 : tile[ni] < ntiles;
    ltile[ni] = tv[ni] ? tile[ni] : ntiles - 1;
  }
  [[maybe_unused]] ResidRows<A, EPI == EPI_RESID ? MI : 1> rres;
  if constexpr (EPI == EPI_RESID) rres = load_resid<A, BMT, MI>(p, m0, tile, tv);

  // Global -> register staging of the X tile (BMT rows x 64 k), two register
  // sets: X of step j lives in set j & 1 from its load, two steps ahead,
  // until it is written to LDS.
  // byte offsets of this thread's X pieces from the work-group's first row
  const uint16_t* xbase = (const uint16_t*)p.x + (size_t)m0 * p.ldx;
  uint32_t xoff[NA];
#pragma unroll
  for (int i = 0; i < NA; ++i) {
    const int idx = threadIdx.x + 256 * i;
    const int r = idx >> 3, c = idx & 7;
    xoff[i] = (uint32_t)((min(m0 + r, p.M - 1) - m0) * p.ldx + c * 8) * 2u;
  }
  u32x4 ra[2][NA];
  auto load_a = [&](int kt, int set) {
#pragma unroll
    for (int i = 0; i < NA; ++i) ra[set][i] = ld16(xbase, xoff[i] + (uint32_t)(kt * BK * 2));
  };
  auto store_a = [&](int buf, int set) {
#pragma unroll
    for (int i = 0; i < NA; ++i) {
      const int idx = threadIdx.x + 256 * i;
      const int r = idx >> 3, c = idx & 7;
      *(u32x4*)&sA[buf * BMT * LDA + r * LDA + c * 8] = ra[set][i];
    }
  };
  // B fragments, double-buffered by step parity: step kt reads set kt & 1,
  // which was loaded during step kt - 1, and loads set (kt + 1) & 1.
  u32x4 rb[2][4];
  uint32_t rs[2][4];
  auto load_b = [&](int kt, int set) {
#pragma unroll
    for (int ni = 0; ni < 4; ++ni) {
      const uint32_t ch = (uint32_t)ltile[ni] * (K / 64) + kt;
      rb[set][ni] = ld16(p.W.w, (ch * 64 + lane) * 16u);
      rs[set][ni] = ld4(p.W.sc, (ch * 16 + row) * 4u);
    }
  };

  f32x4 acc[MI][4];
#pragma unroll
  for (int mi = 0; mi < MI; ++mi)
#pragma unroll
    for (int ni = 0; ni < 4; ++ni) acc[mi][ni] = f32x4{0.f, 0.f, 0.f, 0.f};

  // Pipeline: step kt computes from LDS buffer kt & 1 and the B fragments
  // loaded during the previous step; at its end X of step kt + 1 goes from
  // registers into the other buffer and X of step kt + 3 is loaded.  One
  // barrier per step: it orders this step's writes of buffer (kt+1) & 1
  // before the next step's reads, and this step's reads of buffer kt & 1
  // before the next step's writes to it.  The loop is unrolled by two so that
  // every register set index is a compile-time constant.  Loads past the last
  // step re-read it; their data is never used.
  const int KT = K / BK;
  load_a(0, 0);
  load_b(0, 0);
  load_a(min(1, KT - 1), 1);
  store_a(0, 0);
  load_a(min(2, KT - 1), 0);
  __syncthreads();
  auto step = [&](auto par, int kt) {
    constexpr int P = decltype(par)::value;
    u32x4 cb[4];
    uint32_t cs[4];
#pragma unroll
    for (int ni = 0; ni < 4; ++ni) {
      cb[ni] = rb[P][ni];
      cs[ni] = rs[P][ni];
    }
    load_b(min(kt + 1, KT - 1), P ^ 1);
    const uint16_t* a = sA + P * BMT * LDA;
    u32x4 fa[MI][2];
#pragma unroll
    for (int mi = 0; mi < MI; ++mi)
#pragma unroll
      for (int ks = 0; ks < 2; ++ks)
        fa[mi][ks] = *(const u32x4*)&a[(wm * (BMT / 2) + mi * 16 + row) * LDA + ks * 32 + kg * 8];
#pragma unroll
    for (int ni = 0; ni < 4; ++ni) {
      const u32x4 b0 = q8_to_f16x8(cb[ni][0], cb[ni][1]);
      const u32x4 b1 = q8_to_f16x8(cb[ni][2], cb[ni][3]);
      const float d0 = f16_to_f32((uint16_t)(cs[ni] & 0xffffu));
      const float d1 = f16_to_f32((uint16_t)(cs[ni] >> 16));
      const f32x4 z = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int mi = 0; mi < MI; ++mi) {
        const f32x4 t0 = mfma16<ACT_F16>(fa[mi][0], b0, z);
        const f32x4 t1 = mfma16<ACT_F16>(fa[mi][1], b1, z);
        acc[mi][ni] += d0 * t0;
        acc[mi][ni] += d1 * t1;
      }
    }
    store_a(P ^ 1, P ^ 1);
    load_a(min(kt + 3, KT - 1), P ^ 1);
    __syncthreads();
  };
  for (int kt = 0; kt < KT; kt += 2) {
    step(std::integral_constant<int, 0>{}, kt);
    if (kt + 1 < KT) step(std::integral_constant<int, 1>{}, kt + 1);
  }

  if constexpr (EPI == EPI_ROPE) {
    rope_epilogue<A, BMT, MI, false>(p, acc, sA, m0, cg, rrows);
    return;
  }
  if constexpr (EPI == EPI_SWIGLU) {
    swiglu_epilogue<A, BMT, MI>(p, acc, m0, tile, tv);
    return;
  }
  if constexpr (EPI == EPI_RESID) {
    resid_epilogue<A, BMT, MI>(p, acc, m0, tile, tv, rres);
    return;
  }
  store_epilogue<A, BMT, MI>(p, acc, m0, tile, tv);
}

// 16-bit activations with dense 16-bit weights, both operands copied global
// -> LDS by the direct-to-LDS loads (no register staging): a ring of NS
// stages of BK2 = 32 k, NS - 1 steps in flight, one barrier per step.  Tile
// BMT x 128 (BMT 128 or 256), four waves of BMT/2 x 64 (same fragments and
// XCD work order as gemm_q8_kernel).  X stage: BMT rows x 4
// chunks of 8 elements, chunk c of row r at slot r * 4 + (c ^ swz(r)), so
// that the fragment reads of any 8 consecutive lanes fall in distinct
// 16-byte bank groups of 128 bytes and those of any 16 in distinct groups of
// 256 bytes; W stage: the work-group's 8 weight tiles, each one 1 KiB
// fragment of the tiled layout.  LDS: NS * (BMT * 64 + 8192) bytes, so two
// work-groups per CU at (128, 4) and (256, 3).
constexpr int BK2 = 32;

__device__ __forceinline__ int swz(int r) { return ((r >> 1) ^ (r >> 3)) & 3; }

// Two values already rounded to the 16-bit activation dtype, packed (lo in
// the low half).  bf16: the high halves of the two f32 (their low halves are
// zero), one v_perm_b32.
template <int A>
__device__ __forceinline__ uint32_t pack2_rounded(float lo, float hi) {
  if constexpr (A == ACT_BF16)
    return __builtin_amdgcn_perm(__builtin_bit_cast(uint32_t, hi), __builtin_bit_cast(uint32_t, lo), 0x07060302u);
  else
    return (uint32_t)st_act<A>(lo) | ((uint32_t)st_act<A>(hi) << 16);
}

// Dense tiles run their MFMAs with the weights as the A operand (both operands'
// fragments have the same layout), Y^T = W X^T per 16 x 16 piece: a lane then
// holds four consecutive output columns 4 kg .. 4 kg + 3 of tile[ni] for X row
// 16 mi + lane % 16, so residuals, tables and outputs move 8 bytes at a time
// straight from the registers, and what is staged through LDS is written 8
// bytes at a time.  Against 2-byte accesses in the other layout (the same
// bits): encoder layer at 16 windows 936 -> 927 us, 5 x 1137 306.5 -> 304.4 us.
// gate|up's stores from this layout, against 16-byte stores of products staged
// through LDS (medians of five alternating runs, bf16): 12,288 rows 151.1 |
// 148.2 us, 8000 100.3 | 99.9, 4800 64.2 | 65.8, 3200 50.2 | 50.1; f16 12,288
// 155.6 | 154.5, 6400 95.4 | 96.2 -- within 2.5% either way, so not staged.
// Residuals and plain stores of the 128- and 256-row tiles keep the other layout
// (resid_epilogue, store_epilogue).

// Four consecutive 16-bit values at q (VEC: 8-byte aligned).
template <bool VEC>
__device__ __forceinline__ uint2 load4(const uint16_t* q) {
  if constexpr (VEC) return *(const uint2*)q;
  else return uint2{q[0] | ((uint32_t)q[1] << 16), q[2] | ((uint32_t)q[3] << 16)};
}
template <bool VEC>
__device__ __forceinline__ void store4(uint16_t* q, uint2 v) {
  if constexpr (VEC) {
    *(uint2*)q = v;
  } else {
    q[0] = (uint16_t)v.x;
    q[1] = (uint16_t)(v.x >> 16);
    q[2] = (uint16_t)v.y;
    q[3] = (uint16_t)(v.y >> 16);
  }
}
__device__ __forceinline__ uint16_t elem4(uint2 v, int r) {
  return (uint16_t)((r < 2 ? v.x : v.y) >> (16 * (r & 1)));
}

// The residual, or the table value, of every output a lane stores (a product
// has at most one of the two; with neither, unused values of y); rows past M
// and tiles past the end read clamped addresses (they are not stored).  mb: the
// wave's first row.
template <bool VEC, int MI, int NI>
__device__ __forceinline__ void cross_resid(const GemmArgs& p, int mb, const int (&tile)[NI], const bool (&tv)[NI],
                                            uint2 (&rr)[MI][NI]) {
  const int lane = threadIdx.x & 63, row = lane & 15, kg = lane >> 4;
  const bool tab = !p.resid && p.aff.table;
  const uint16_t* rp = (const uint16_t*)(p.resid ? p.resid : tab ? p.aff.table : p.y) + 4 * kg;
  const int ld = tab ? p.W.out : p.ldy;
#pragma unroll
  for (int mi = 0; mi < MI; ++mi) {
    int r = min(mb + mi * 16 + row, p.M - 1);
    if (tab) r = min(r % p.aff.period, p.aff.valid - 1);
#pragma unroll
    for (int ni = 0; ni < NI; ++ni) rr[mi][ni] = load4<VEC>(rp + (size_t)r * ld + (tv[ni] ? tile[ni] : 0) * 16);
  }
}

// Epilogue of a wave's MI x NI pieces (EPI_STORE, RESID, SWIGLU, AFFINE).
// SWIGLU: tiles [0, NI / 2) hold gate columns, the others the matching up
// columns.  rr: cross_resid's values (EPI_RESID, and EPI_AFFINE with a
// residual or a table; every load comes before the first store, since a vector-memory wait
// also counts the stores issued before it).
template <int A, int EPI, bool VEC, int MI, int NI>
__device__ __forceinline__ void cross_epilogue(const GemmArgs& p, const f32x4 (&acc)[MI][NI], int mb,
                                               const int (&tile)[NI], const bool (&tv)[NI],
                                               const uint2 (&rr)[MI][NI]) {
  const int lane = threadIdx.x & 63, row = lane & 15, kg = lane >> 4;
  uint16_t* const y = (uint16_t*)p.y + 4 * kg;
  if constexpr (EPI == EPI_SWIGLU) {
    constexpr int G = NI / 2;
#pragma unroll
    for (int mi = 0; mi < MI; ++mi) {
      f32x4 o[G];
#pragma unroll
      for (int ni = 0; ni < G; ++ni)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const float gg = rd<A>(acc[mi][ni][r]), u = rd<A>(acc[mi][ni + G][r]);
          o[ni][r] = rd<A>(gg / (1.0f + __expf(-gg))) * u;
        }
      const int gr = mb + mi * 16 + row;
#pragma unroll
      for (int ni = 0; ni < G; ++ni)
        if (gr < p.M && tv[ni]) store4<VEC>(y + (size_t)gr * p.ldy + tile[ni] * 16, pack4<A>(o[ni]));
    }
  } else if constexpr (EPI == EPI_AFFINE) {
    const AffineArgs& f = p.aff;
    constexpr int N = NI * 4;
    float bs[N], sc[NI];
#pragma unroll
    for (int ni = 0; ni < NI; ++ni) {
      const int col = (tv[ni] ? tile[ni] : 0) * 16 + 4 * kg;
      const uint2 b = f.bias ? load4<VEC>((const uint16_t*)f.bias + col) : uint2{0, 0};
#pragma unroll
      for (int r = 0; r < 4; ++r) bs[ni * 4 + r] = ld_act<A>(elem4(b, r));
      sc[ni] = col < f.scale_cols ? f.scale : 1.0f;   // scale_cols is a multiple of 4
    }
#pragma unroll
    for (int mi = 0; mi < MI; ++mi) {
      float v[N], sv[N];
      uint16_t xv[N];
#pragma unroll
      for (int e = 0; e < N; ++e) {
        v[e] = acc[mi][e >> 2][e & 3];
        sv[e] = sc[e >> 2];
        xv[e] = elem4(rr[mi][e >> 2], e & 3);
      }
      affine_block<A, N, false>(p, v, sv, bs, xv, xv);
      const int gr = mb + mi * 16 + row;
      if (gr >= p.M || !affine_row(p, gr)) continue;
      uint16_t* const yr = y + (size_t)gr * p.ldy;
#pragma unroll
      for (int ni = 0; ni < NI; ++ni)
        if (tv[ni])
          store4<VEC>(yr + tile[ni] * 16, uint2{pack2_rounded<A>(v[4 * ni], v[4 * ni + 1]),
                                                pack2_rounded<A>(v[4 * ni + 2], v[4 * ni + 3])});
    }
  } else {
#pragma unroll
    for (int mi = 0; mi < MI; ++mi) {
      const int gr = mb + mi * 16 + row;
      if (gr >= p.M) continue;
#pragma unroll
      for (int ni = 0; ni < NI; ++ni) {
        if (!tv[ni]) continue;
        f32x4 v = acc[mi][ni];
        if constexpr (EPI == EPI_RESID) {
#pragma unroll
          for (int r = 0; r < 4; ++r) v[r] = ld_act<A>(elem4(rr[mi][ni], r)) + rd<A>(v[r]);
        }
        store4<VEC>(y + (size_t)gr * p.ldy + tile[ni] * 16, pack4<A>(v));
      }
    }
  }
}

// EPI_AFFINE on the direct-to-LDS BMT x 128 tiles, through LDS: the
// accumulators, rounded to the activation dtype (the first affine step), are
// staged row-major in the freed ring, 8 bytes (four columns) at a time -- the
// 16-byte chunk c of tile row R at chunk position c ^ (R & 15) -- then 16 lanes
// per row finish 8 columns each, two rows per pass (16 independent chains through
// affine_block), with 16-byte residual and table loads and 16-byte stores: 8-byte
// stores straight from the accumulators cost the 128- and 256-row tiles 17-20%
// (fc1 at 16 windows 243 -> 283 us, q|k|v 167 -> 200).
template <int A, int BMT, int MI>
__device__ __forceinline__ void staged_affine_epilogue(const GemmArgs& p, const f32x4 (&acc)[MI][4], int m0,
                                                       int cg, uint16_t* stg) {
  typedef typename ActT<A>::T T;
  const AffineArgs& f = p.aff;
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const int wm = w >> 1, wn = w & 1, row = lane & 15, kg = lane >> 4;
  const int ch = threadIdx.x & 15, r0 = threadIdx.x >> 4;   // chunk, first row
  const int gc = cg * 128 + ch * 8;                          // its first output column
  const bool col_ok = gc < p.W.out;
  const int rows = min(BMT, p.M - m0);
  // The bias and the residual or table values (a product has at most one
  // of the two) of the lane's rows r0, r0 + 16, ... are loaded
  // first, so the loads run under the staging below and none follows a
  // store: a vector-memory wait also counts the stores issued before it, so
  // a load placed after a store would hold the lane until that store
  // completed.  A lane loads the residual of exactly the outputs it stores
  // (the output may be the residual itself).  The loads are unconditional
  // (a load inside a branch is waited for where the branches join): without
  // a residual or table every row reads the tile's first output row, and
  // without a bias the bias load reads that row too (values affine_block
  // does not use); rows past the tile read its last row and lanes past the
  // last column read column 0 (neither is stored).
  constexpr int NR = BMT / 16;
  const int gl = col_ok ? gc : 0;
  const T* xb = (const T*)p.y + (size_t)m0 * p.ldy + gl;
  int xs = 0;
  if (p.resid) {
    xb = (const T*)p.resid + (size_t)m0 * p.ldy + gl;
    xs = p.ldy;
  } else if (f.table) {
    xb = (const T*)f.table + gl;
    xs = p.W.out;
  }
  const bool by_period = f.table && !p.resid;
  const u32x4 bias4 = *(const u32x4*)(f.bias ? (const T*)f.bias + gl : xb);
  u32x4 xv4[NR];
#pragma unroll
  for (int i = 0; i < NR; ++i) {
    const int R = min(r0 + 16 * i, rows - 1);
    const int xr = by_period ? max(min((m0 + R) % f.period, f.valid - 1), 0) : R;
    xv4[i] = *(const u32x4*)(xb + (size_t)xr * xs);
  }
  barrier_lds();   // every wave's last fragment reads are done
  {
    uint16_t* const wb = stg + (wm * (BMT / 2) + row) * 128 + 4 * (kg & 1);
#pragma unroll
    for (int mi = 0; mi < MI; ++mi)
#pragma unroll
      for (int ni = 0; ni < 4; ++ni)
        *(uint2*)(wb + mi * 16 * 128 + (((wn * 8 + ni * 2 + (kg >> 1)) ^ row) << 3)) =
            pack4<A>(acc[mi][ni]);
  }
  barrier_lds();
  if (!col_ok) return;                                       // (no barrier follows)
  T* const y = (T*)p.y + (size_t)m0 * p.ldy + gc;
  float bias[8], scl[8];
  unpack8<A>(bias4, bias);
#pragma unroll
  for (int e = 0; e < 8; ++e) scl[e] = gc + e < f.scale_cols ? f.scale : 1.0f;
  // two rows (16 independent chains) per pass
#pragma unroll
  for (int i = 0; i < NR; i += 2) {
    if (r0 + 16 * i >= rows) break;
    float v[16], bs[16], sc[16];
    T xv[16];
#pragma unroll
    for (int q = 0; q < 2; ++q) {
      const int R = min(r0 + 16 * (i + q), rows - 1);
      unpack8<A>(*(const u32x4*)&stg[R * 128 + ((ch ^ (R & 15)) << 3)], &v[8 * q]);
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        xv[8 * q + e] = (T)(xv4[i + q][e / 2] >> (16 * (e & 1)));
        bs[8 * q + e] = bias[e];
        sc[8 * q + e] = scl[e];
      }
    }
    affine_block<A, 16, true>(p, v, sc, bs, xv, xv);
#pragma unroll
    for (int q = 0; q < 2; ++q) {
      const int R = r0 + 16 * (i + q);
      if (R >= rows || !affine_row(p, m0 + R)) continue;
      uint32_t o[4];
#pragma unroll
      for (int e = 0; e < 8; e += 2) o[e / 2] = pack2_rounded<A>(v[8 * q + e], v[8 * q + e + 1]);
      *(u32x4*)(y + (size_t)R * p.ldy) = u32x4{o[0], o[1], o[2], o[3]};
    }
  }
}

template <int A, int EPI, int BMT, int NS>
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2)))
gemm_dma_kernel(GemmArgs p) {
  typedef typename ActT<A>::T T;
  static_assert((BMT == 128 && NS == 4) || (BMT == 256 && NS == 3), "tile / ring");
  constexpr int MI = BMT / 32;           // 16-row fragments per wave
  constexpr bool CROSS = EPI != EPI_RESID && EPI != EPI_STORE;   // weights as the A operand
  constexpr int NX = BMT / 64;           // X copies per thread per stage
  constexpr int PER = NX + 2;            // copies per thread per stage
  constexpr int SA = BMT * BK2;          // X elements per stage
  constexpr int SB = 8 * 512;            // weight elements per stage (8 KB)
  static_assert(NS * (SA + SB) >= BMT * 128, "the staged epilogues reuse the ring");
  __shared__ __attribute__((aligned(1024))) uint16_t smem[NS * (SA + SB)];
  uint16_t* const sA = smem;
  uint16_t* const sB = smem + NS * SA;
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const int wm = w >> 1, wn = w & 1;
  const int K = p.W.in, ntiles = p.W.out / 16;
  const int cols = EPI == EPI_SWIGLU ? (ntiles / 2 + 3) / 4 : (ntiles + 7) / 8;
  int mt, cg;
  tile_of(blockIdx.x, (p.M + BMT - 1) / BMT, cols, p.map, mt, cg);
  if (mt * BMT >= p.M) return;
  const int m0 = mt * BMT;
  const int row = lane & 15, kg = lane >> 4;
  [[maybe_unused]] RopeRows<EPI == EPI_ROPE ? BMT : 16> rrows;
  if constexpr (EPI == EPI_ROPE) rrows = rope_rows<BMT>(p, m0);
  int tile[4];
  bool tv[4];
#pragma unroll
  for (int ni = 0; ni < 4; ++ni) {
    tile[ni] = wave_tile<EPI>(cg, ntiles, wn, ni);
    tv[ni] = (EPI == EPI_SWIGLU) ? (cg * 4 + wn * 2 + (ni & 1)) < ntiles / 2 : tile[ni] < ntiles;
  }
  const int mb = m0 + wm * (BMT / 2);
  static_assert(EPI != EPI_RESID || BMT <= 128, "residual prefetch: 128-row tiles");
  [[maybe_unused]] ResidRows<A, EPI == EPI_RESID ? MI : 1> rres;   // in flight behind the K loop
  if constexpr (EPI == EPI_RESID) rres = load_resid<A, BMT, MI>(p, m0, tile, tv);
  // This thread's copies per stage: X slots j * 64 + lane of instructions
  // j = NX w .. NX w + NX - 1 (rows 16 j + lane / 4; rows past M read row
  // M - 1), weight tiles t = 2w, 2w + 1 (past the end: the last tile).
  const uint16_t* xbase = (const uint16_t*)p.x + (size_t)m0 * p.ldx;
  uint32_t xoff[NX], woff[2];
#pragma unroll
  for (int i = 0; i < NX; ++i) {
    const int j = NX * w + i;
    const int slot = j * 64 + lane, r = slot >> 2, cs = slot & 3;
    const int c = cs ^ swz(r);
    xoff[i] = (uint32_t)((min(m0 + r, p.M - 1) - m0) * p.ldx + c * 8) * 2u;
  }
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const int t = 2 * w + i;
    int tl = wave_tile<EPI>(cg, ntiles, t >> 2, t & 3);
    const bool ok = (EPI == EPI_SWIGLU) ? (cg * 4 + (t >> 2) * 2 + (t & 1)) < ntiles / 2 : tl < ntiles;
    tl = ok ? tl : ntiles - 1;
    woff[i] = ((uint32_t)tl * (K / 32) * 64 + lane) * 16u;
  }
  const int wu = __builtin_amdgcn_readfirstlane(w);
  const uint32_t la = lds_addr(sA) + (uint32_t)wu * (NX * 1024u);
  const uint32_t lb = lds_addr(sB) + (uint32_t)wu * 2048u;
  auto issue = [&](int kt, int buf) {
#pragma unroll
    for (int i = 0; i < NX; ++i)
      lds_copy16(xbase, xoff[i] + (uint32_t)(kt * BK2 * 2), la + (uint32_t)(buf * SA * 2 + i * 1024));
#pragma unroll
    for (int i = 0; i < 2; ++i)
      lds_copy16(p.W.w, woff[i] + (uint32_t)(kt * 1024), lb + (uint32_t)(buf * SB * 2 + i * 1024));
  };

  f32x4 acc[MI][4];
#pragma unroll
  for (int mi = 0; mi < MI; ++mi)
#pragma unroll
    for (int ni = 0; ni < 4; ++ni) acc[mi][ni] = f32x4{0.f, 0.f, 0.f, 0.f};

  // Stages past the last step re-read it (their copies only make the waits
  // below conservative).
  const int KT = K / BK2;
#pragma unroll
  for (int s0 = 0; s0 < NS - 1; ++s0) issue(min(s0, KT - 1), s0);
  for (int kt = 0; kt < KT; ++kt) {
    // this step's copies have landed (those of the `after` later stages may
    // still be in flight, PER copies each), then every thread's are visible
    const int after = min(NS - 2, KT - 1 - kt);
    if (after == 2) wait_vm<2 * PER>();
    else if (after == 1) wait_vm<PER>();
    else wait_vm<0>();
    barrier_lds();
    // refill the stage computed in the previous step
    if (kt + NS - 1 < KT) issue(kt + NS - 1, (kt + NS - 1) % NS);
    const uint16_t* a = sA + (kt % NS) * SA;
    const uint16_t* bb = sB + (kt % NS) * SB;
    u32x4 fb[4];
#pragma unroll
    for (int ni = 0; ni < 4; ++ni) fb[ni] = *(const u32x4*)&bb[(wn * 4 + ni) * 512 + lane * 8];
#pragma unroll
    for (int mi = 0; mi < MI; ++mi) {
      const int r = wm * (BMT / 2) + mi * 16 + row;
      const u32x4 fa = *(const u32x4*)&a[(r * 4 + (kg ^ swz(r))) * 8];
#pragma unroll
      for (int ni = 0; ni < 4; ++ni)
        acc[mi][ni] = CROSS ? mfma16<A>(fb[ni], fa, acc[mi][ni]) : mfma16<A>(fa, fb[ni], acc[mi][ni]);
    }
  }

  if constexpr (EPI == EPI_ROPE) {
    rope_epilogue<A, BMT, MI, true>(p, acc, smem, m0, cg, rrows);
  } else if constexpr (EPI == EPI_AFFINE) {
    staged_affine_epilogue<A, BMT, MI>(p, acc, m0, cg, smem);
  } else if constexpr (EPI == EPI_RESID) {
    resid_epilogue<A, BMT, MI>(p, acc, m0, tile, tv, rres);
  } else if constexpr (EPI == EPI_STORE) {
    store_epilogue<A, BMT, MI>(p, acc, m0, tile, tv);
  } else {   // EPI_SWIGLU
    const uint2 none[MI][4] = {};   // (read for a residual or a table only)
    cross_epilogue<A, EPI, true, MI, 4>(p, acc, mb, tile, tv, none);
  }
}

// ---------------------------------------------------------------------------
// Small grids: BM x BN tiles (32, 64 or 128 rows x 32, 64 or 128 columns), four
// waves in 2 x 2 (BM/2 x BN/2 each), for products whose 64 x 128 tiles would
// leave most CUs without a work-group.
//
// What bounds them is the serial K loop of one work-group, not bytes: 64 x 128
// register-staged tiles, which ran them before, took 23 us for K = 3072 at any M
// up to 2048 (32 work-groups on 256 CUs at M = 256), Q8_0 ones 33 us.  A
// smaller tile has less to copy, read and multiply per k and the ring keeps
// 30-70 KB of it in flight per work-group: 7.6 us (dense, 32 x 32) and 11.8 us
// (Q8_0) at M = 256, N = 1024, K = 3072 (try_small has the rule and figures).
//
// Both operands (for Q8_0 the quants and the scales too) go global -> LDS by
// direct-to-LDS loads through a ring of NS stages of KS k, NS - 1 in flight,
// one barrier per stage.  KS is 64 or 128 for dense weights and 128 or 256 for
// Q8_0 (a stage is then a whole number of copies per wave).  X stage: row r is KS / 8
// chunks of 16 bytes, chunk c at position c ^ swx(r), so that the fragment
// reads (16 rows, one chunk) fall in distinct banks.  Weight stage: the tiles'
// fragments as stored; Q8_0 scales: 16 x 2 u32 per tile.  Each output is
// summed over k in the order of the other tiles by the same MFMAs, so tile
// kinds give the same bits.
template <int KS>
__device__ __forceinline__ int swx(int r) {
  return KS == 64 ? (r >> 1) & 7 : r & 15;
}

// Column tile lt (0 .. BN/16 - 1; wave column lt / NI, its fragment lt % NI)
// of column group cg: EPI_SWIGLU pairs gate tiles (the first half of a wave's
// fragments) with the matching up tiles.  ok: whether it lies in the product.
template <int EPI, int BN>
__device__ __forceinline__ int small_tile(int cg, int ntiles, int lt, bool& ok) {
  constexpr int NI = BN / 32;
  if constexpr (EPI == EPI_SWIGLU) {
    constexpr int G = NI / 2;
    const int wn = lt / NI, ni = lt % NI;
    const int base = cg * (BN / 32) + wn * G + ni % G;
    ok = base < ntiles / 2;
    return ni < G ? base : base + ntiles / 2;
  } else {
    const int t = cg * (BN / 16) + lt;
    ok = t < ntiles;
    return t;
  }
}

template <int A, int WK, int EPI, int BM, int BN, int KS, int NS, bool VEC>
__global__ void __launch_bounds__(256) gemm_small_kernel(GemmArgs p) {
  typedef typename ActT<A>::T T;
  constexpr bool Q8 = WK == WK_Q8;
  constexpr int MI = BM / 32, NI = BN / 32, NT = BN / 16;
  static_assert(EPI != EPI_SWIGLU || NI >= 2, "gate and up tiles in one wave");
  static_assert(EPI != EPI_ROPE || BN == 128, "one head slot per work-group");
  constexpr int XB = BM * KS * 2;                 // stage bytes: X rows,
  constexpr int WB = Q8 ? BN * KS : BN * KS * 2;  // weights,
  constexpr int SCB = Q8 ? NT * KS : 0;           // scales
  constexpr int TK = Q8 ? KS / 64 : KS / 32;      // KiB of weights per tile
  constexpr int SCL = SCB / 64;                   // 16-byte pieces of scales per wave
  constexpr int SB = XB + WB + SCB;
  constexpr int NXC = XB / 4096, NWC = WB / 4096; // 1 KiB copies per wave
  static_assert(XB % 4096 == 0 && WB % 4096 == 0, "whole copies per wave");
  constexpr int PER = NXC + NWC + (Q8 ? 1 : 0);
  static_assert((NS - 2) * PER < 64, "vmcnt");
  constexpr int EPIB = EPI == EPI_ROPE ? BM * 256 : 0;
  __shared__ __attribute__((aligned(1024))) uint8_t smem[NS * SB > EPIB ? NS * SB : EPIB];
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const int wm = w >> 1, wn = w & 1, row = lane & 15, kg = lane >> 4;
  const int K = p.W.in, ntiles = p.W.out / 16;
  constexpr int CW = EPI == EPI_SWIGLU ? BN / 32 : NT;   // (gate) tiles per column group
  const int cols = ((EPI == EPI_SWIGLU ? ntiles / 2 : ntiles) + CW - 1) / CW;
  int mt, cg;
  tile_of(blockIdx.x, (p.M + BM - 1) / BM, cols, p.map, mt, cg);
  if (mt * BM >= p.M) return;
  const int m0 = mt * BM;
  [[maybe_unused]] RopeRows<EPI == EPI_ROPE ? BM : 16> rrows;
  if constexpr (EPI == EPI_ROPE) rrows = rope_rows<BM>(p, m0);
  int tile[NI];
  bool tv[NI];
#pragma unroll
  for (int ni = 0; ni < NI; ++ni) tile[ni] = small_tile<EPI, BN>(cg, ntiles, wn * NI + ni, tv[ni]);

  // The residuals of the elements this lane stores, loaded before the K loop
  // (rows past M and tiles past the end read clamped addresses).
  const int mb = m0 + wm * (BM / 2);
  [[maybe_unused]] uint2 rres[Q8 ? 1 : MI][NI];          // dense
  [[maybe_unused]] T qres[Q8 ? MI : 1][4][Q8 ? NI : 1];  // Q8_0: rows 4 kg + r, column `row`
  if constexpr (!Q8 && (EPI == EPI_RESID || EPI == EPI_AFFINE)) cross_resid<VEC, MI, NI>(p, mb, tile, tv, rres);
  if constexpr (Q8 && EPI == EPI_RESID) {
#pragma unroll
    for (int mi = 0; mi < MI; ++mi)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int gr = min(mb + mi * 16 + 4 * kg + r, p.M - 1);
#pragma unroll
        for (int ni = 0; ni < NI; ++ni)
          qres[mi][r][ni] = ((const T*)p.resid)[(size_t)gr * p.ldy + (tv[ni] ? tile[ni] : 0) * 16 + row];
      }
  }

  // This wave's copies per stage.
  const int wu = __builtin_amdgcn_readfirstlane(w);
  const uint16_t* xbase = (const uint16_t*)p.x + (size_t)m0 * p.ldx;
  uint32_t xoff[NXC], woff[NWC], soff = 0;
#pragma unroll
  for (int i = 0; i < NXC; ++i) {
    constexpr int CH = KS / 8;
    const int piece = (wu * NXC + i) * 64 + lane, r = piece / CH, pos = piece % CH;
    xoff[i] = (uint32_t)(min(m0 + r, p.M - 1) - m0) * (uint32_t)p.ldx * 2u + (uint32_t)((pos ^ swx<KS>(r)) * 16);
  }
#pragma unroll
  for (int i = 0; i < NWC; ++i) {
    // copy j is KiB j % TK of column tile j / TK's stage (a KiB is 32 k of
    // dense weights, 64 k of Q8_0)
    const int j = wu * NWC + i;
    bool ok;
    int tl = small_tile<EPI, BN>(cg, ntiles, j / TK, ok);
    tl = ok ? tl : ntiles - 1;
    woff[i] = ((uint32_t)tl * (K / (KS / TK)) + (j % TK)) * 1024u + lane * 16u;
  }
  if constexpr (Q8) {
    const int q = wu * SCL + min(lane, SCL - 1);
    bool ok;
    int tl = small_tile<EPI, BN>(cg, ntiles, q / (KS / 16), ok);
    tl = ok ? tl : ntiles - 1;
    soff = (uint32_t)tl * K + (q % (KS / 16)) * 16u;
  }
  const uint32_t ls = lds_addr(smem);
  auto issue = [&](int kt, int buf) {
    const uint32_t b = ls + (uint32_t)(buf * SB);
#pragma unroll
    for (int i = 0; i < NXC; ++i)
      lds_copy16(xbase, xoff[i] + (uint32_t)(kt * KS * 2), b + (uint32_t)((wu * NXC + i) * 1024));
#pragma unroll
    for (int i = 0; i < NWC; ++i)
      lds_copy16(p.W.w, woff[i] + (uint32_t)(kt * TK * 1024), b + (uint32_t)(XB + (wu * NWC + i) * 1024));
    if constexpr (Q8) {
      // a quarter of the scales per wave: lanes past its pieces copy nothing
      if (lane < SCL) lds_copy16(p.W.sc, soff + (uint32_t)(kt * KS), b + (uint32_t)(XB + WB + wu * (SCL * 16)));
    }
  };

  f32x4 acc[MI][NI];
#pragma unroll
  for (int mi = 0; mi < MI; ++mi)
#pragma unroll
    for (int ni = 0; ni < NI; ++ni) acc[mi][ni] = f32x4{0.f, 0.f, 0.f, 0.f};
  const int KT = K / KS;
#pragma unroll
  for (int s0 = 0; s0 < NS - 1; ++s0) issue(min(s0, KT - 1), s0);
  int slot = 0;   // kt % NS
  for (int kt = 0; kt < KT; ++kt) {
    // this stage's copies have landed; the last NS - 2 stages wait for all
    if (KT - 1 - kt >= NS - 2) wait_vm<(NS - 2) * PER>();
    else wait_vm<0>();
    barrier_lds();
    // refill the slot computed in the previous step
    if (kt + NS - 1 < KT) issue(kt + NS - 1, slot == 0 ? NS - 1 : slot - 1);
    const uint16_t* a = (const uint16_t*)(smem + slot * SB);
    const uint8_t* bb = smem + slot * SB + XB;
    if constexpr (Q8) {
      const uint32_t* sc = (const uint32_t*)(bb + WB);
#pragma unroll
      for (int c = 0; c < TK; ++c) {
        u32x4 fa[MI][2];
#pragma unroll
        for (int mi = 0; mi < MI; ++mi)
#pragma unroll
          for (int ks = 0; ks < 2; ++ks) {
            const int r = wm * (BM / 2) + mi * 16 + row;
            fa[mi][ks] = *(const u32x4*)&a[r * KS + (((8 * c + 4 * ks + kg) ^ swx<KS>(r)) << 3)];
          }
#pragma unroll
        for (int ni = 0; ni < NI; ++ni) {
          const int lt = wn * NI + ni;
          const u32x4 cb = *(const u32x4*)(bb + (lt * TK + c) * 1024 + lane * 16);
          const uint32_t cs = sc[(lt * TK + c) * 16 + row];
          const u32x4 b0 = q8_to_f16x8(cb[0], cb[1]);
          const u32x4 b1 = q8_to_f16x8(cb[2], cb[3]);
          const float d0 = f16_to_f32((uint16_t)(cs & 0xffffu));
          const float d1 = f16_to_f32((uint16_t)(cs >> 16));
          const f32x4 z = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
          for (int mi = 0; mi < MI; ++mi) {
            const f32x4 t0 = mfma16<ACT_F16>(fa[mi][0], b0, z);
            const f32x4 t1 = mfma16<ACT_F16>(fa[mi][1], b1, z);
            acc[mi][ni] += d0 * t0;
            acc[mi][ni] += d1 * t1;
          }
        }
      }
    } else {
#pragma unroll
      for (int ks = 0; ks < TK; ++ks) {
        u32x4 fb[NI];
#pragma unroll
        for (int ni = 0; ni < NI; ++ni)
          fb[ni] = *(const u32x4*)(bb + ((wn * NI + ni) * TK + ks) * 1024 + lane * 16);
#pragma unroll
        for (int mi = 0; mi < MI; ++mi) {
          const int r = wm * (BM / 2) + mi * 16 + row;
          const u32x4 fa = *(const u32x4*)&a[r * KS + (((4 * ks + kg) ^ swx<KS>(r)) << 3)];
#pragma unroll
          for (int ni = 0; ni < NI; ++ni) acc[mi][ni] = mfma16<A>(fb[ni], fa, acc[mi][ni]);
        }
      }
    }
    slot = slot + 1 == NS ? 0 : slot + 1;
  }

  if constexpr (EPI == EPI_ROPE) {
    rope_epilogue<A, BM, MI, !Q8>(p, acc, (T*)smem, m0, cg, rrows);
  } else if constexpr (!Q8) {
    cross_epilogue<A, EPI, VEC, MI, NI>(p, acc, mb, tile, tv, rres);
  } else {
    // Q8_0 (each column's block scale sits in the lane of that column): a lane
    // holds rows 4 kg + r of each fragment, column `row`
    constexpr int NO = EPI == EPI_SWIGLU ? NI / 2 : NI;
#pragma unroll
    for (int mi = 0; mi < MI; ++mi)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int gr = mb + mi * 16 + 4 * kg + r;
#pragma unroll
        for (int ni = 0; ni < NO; ++ni) {
          float v = acc[mi][ni][r];
          if constexpr (EPI == EPI_SWIGLU) {
            const float gg = rd<A>(v), u = rd<A>(acc[mi][ni + NO][r]);
            v = rd<A>(gg / (1.0f + __expf(-gg))) * u;
          }
          if constexpr (EPI == EPI_RESID) v = ld_act<A>(qres[mi][r][ni]) + rd<A>(v);
          if (gr < p.M && tv[ni]) ((T*)p.y)[(size_t)gr * p.ldy + tile[ni] * 16 + row] = st_act<A>(v);
        }
      }
  }
}

// f32 activations / weights on v_mfma_f32_16x16x4f32; same tiling, K chunks of 16.
template <int EPI>
__global__ void __launch_bounds__(256) gemm32_kernel(GemmArgs p) {
  constexpr int LDF = BK + 4;
  __shared__ float sA[BM * LDF];
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const int wm = w >> 1, wn = w & 1;
  const int K = p.W.in, ntiles = p.W.out / 16;
  const int m0 = blockIdx.x * BM;
  const int row = lane & 15, kg = lane >> 4;
  int tile[4];
  bool tv[4];
#pragma unroll
  for (int ni = 0; ni < 4; ++ni) {
    tile[ni] = wave_tile<EPI>(blockIdx.y, ntiles, wn, ni);
    tv[ni] = (EPI == EPI_SWIGLU) ? (blockIdx.y * 4 + wn * 2 + (ni & 1)) < ntiles / 2
                                 : tile[ni] < ntiles;
  }
  f32x4 acc[4][4];
#pragma unroll
  for (int mi = 0; mi < 4; ++mi)
#pragma unroll
    for (int ni = 0; ni < 4; ++ni) acc[mi][ni] = f32x4{0.f, 0.f, 0.f, 0.f};
  const int KT = K / BK;
  for (int kt = 0; kt < KT; ++kt) {
    __syncthreads();
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const int idx = threadIdx.x + 256 * i;  // 2048 float4 pieces
      const int r = idx >> 4, c = idx & 15;
      const int gr = m0 + r;
      *(f32x4*)&sA[r * LDF + c * 4] =
          gr < p.M ? *(const f32x4*)((const float*)p.x + (size_t)gr * p.ldx + kt * BK + c * 4)
                   : f32x4{0.f, 0.f, 0.f, 0.f};
    }
    __syncthreads();
#pragma unroll
    for (int c = 0; c < 4; ++c) {
      f32x4 fb[4];
#pragma unroll
      for (int ni = 0; ni < 4; ++ni) {
        const size_t ch = (size_t)tile[ni] * (K / 16) + kt * 4 + c;
        fb[ni] = tv[ni] ? ((const f32x4*)p.W.w)[ch * 64 + lane] : f32x4{0.f, 0.f, 0.f, 0.f};
      }
#pragma unroll
      for (int mi = 0; mi < 4; ++mi) {
        const f32x4 fa = *(const f32x4*)&sA[(wm * 64 + mi * 16 + row) * LDF + c * 16 + kg * 4];
#pragma unroll
        for (int ni = 0; ni < 4; ++ni)
#pragma unroll
          for (int j = 0; j < 4; ++j)
            acc[mi][ni] = __builtin_amdgcn_mfma_f32_16x16x4f32(fa[j], fb[ni][j], acc[mi][ni], 0, 0, 0);
      }
    }
  }
#pragma unroll
  for (int mi = 0; mi < 4; ++mi) {
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int gr = m0 + wm * 64 + mi * 16 + 4 * kg + r;
      if (gr >= p.M) continue;
      if constexpr (EPI == EPI_SWIGLU) {
#pragma unroll
        for (int ni = 0; ni < 2; ++ni) {
          if (!tv[ni]) continue;
          const float gg = acc[mi][ni][r], u = acc[mi][ni + 2][r];
          ((float*)p.y)[(size_t)gr * p.ldy + tile[ni] * 16 + row] = (gg / (1.0f + __expf(-gg))) * u;
        }
      } else {
        if constexpr (EPI == EPI_AFFINE)
          if (!affine_row(p, gr)) continue;
#pragma unroll
        for (int ni = 0; ni < 4; ++ni) {
          if (!tv[ni]) continue;
          const size_t o = (size_t)gr * p.ldy + tile[ni] * 16 + row;
          if constexpr (EPI == EPI_RESID)
            ((float*)p.y)[o] = ((const float*)p.resid)[o] + acc[mi][ni][r];
          else if constexpr (EPI == EPI_AFFINE)
            ((float*)p.y)[o] = affine_value<ACT_F32>(p, acc[mi][ni][r], gr, tile[ni] * 16 + row);
          else
            ((float*)p.y)[o] = acc[mi][ni][r];
        }
      }
    }
  }
}

// Rows of the 16-bit dense tiles past the small grids (512 work-groups = two
// per CU): 256 where those tiles fill about 4/5 of the slots and do not end in a
// last round of fewer than 128 work-groups, else 128.  It decides for gate|up,
// the encoder's products and plain stores; q|k|v with its RoPE epilogue and the
// residual products of the decoder take 128 rows wherever it says 256 (dispatch).
// us, 256 | 128 rows, bf16, by tiles of 256 rows:
//   gate|up at 2240 rows (432 tiles) 36.4 | 37.4, 2560 (480) 36.6 | 40.0, but
//   3072 (576) 52.5 | 48.9; 4096 (768) 56.3 | 59.5, 12,288 (2304) 158.1 | 178.3;
//   the encoder's fc1 at 3300 (416) 43.7 | 44.9, 4500 (576) 64.0 | 60.9, 12,000
//   (1504) 128.9 | 147.4; its q|k|v at 3300 (312) 37.6 | 35.2, 4500 (432) 39.8 |
//   41.9, 24,000 (2256) 165.6 | 198.0; its fc2 at 12,000 (376) 119.5 | 118.3,
//   14,000 (440) 125.5 | 141.2, 18,000 (568) 187.5 | 176.7.
// (64-row tiles were slower than 128-row ones past the small grids: O at 4503
// rows 33.8 against 31.3, 7505 44.8 against 37.0; down 47.7 against 43.3 and 66.2
// against 53.3.)
int gemm_tile_rows(int M, int col_groups) {
  const int tiles256 = (M + 255) / 256 * col_groups;
  return tiles256 >= 400 && (tiles256 % 512 == 0 || tiles256 % 512 >= 128) ? 256 : 128;
}

// Whether the dense tiles may move 16 bytes of output, bias, residual and table
// rows at a time.
bool vec_ok(const GemmArgs& a) {
  auto al = [](const void* q) { return ((uintptr_t)q & 15) == 0; };
  return a.ldy % 8 == 0 && al(a.y) && al(a.aff.bias) && al(a.aff.table) && al(a.resid);
}

template <int A, int BMT, int NS>
hipError_t launch_dma(int epi, dim3 grid, const GemmArgs& a, hipStream_t s) {
  switch (epi) {
    case EPI_STORE: hipLaunchKernelGGL((gemm_dma_kernel<A, EPI_STORE, BMT, NS>), grid, dim3(256), 0, s, a); break;
    case EPI_RESID:
      if constexpr (BMT > 128) return hipErrorInvalidValue;
      else hipLaunchKernelGGL((gemm_dma_kernel<A, EPI_RESID, BMT, NS>), grid, dim3(256), 0, s, a);
      break;
    case EPI_SWIGLU: hipLaunchKernelGGL((gemm_dma_kernel<A, EPI_SWIGLU, BMT, NS>), grid, dim3(256), 0, s, a); break;
    case EPI_ROPE:
      if constexpr (BMT > 128) return hipErrorInvalidValue;
      else hipLaunchKernelGGL((gemm_dma_kernel<A, EPI_ROPE, BMT, NS>), grid, dim3(256), 0, s, a);
      break;
    case EPI_AFFINE: hipLaunchKernelGGL((gemm_dma_kernel<A, EPI_AFFINE, BMT, NS>), grid, dim3(256), 0, s, a); break;
    default: return hipErrorInvalidValue;
  }
  return hipGetLastError();
}

hipError_t launch_q8(int epi, dim3 grid, const GemmArgs& a, hipStream_t s) {
  switch (epi) {
    case EPI_STORE: hipLaunchKernelGGL((gemm_q8_kernel<EPI_STORE>), grid, dim3(256), 0, s, a); break;
    case EPI_RESID: hipLaunchKernelGGL((gemm_q8_kernel<EPI_RESID>), grid, dim3(256), 0, s, a); break;
    case EPI_SWIGLU: hipLaunchKernelGGL((gemm_q8_kernel<EPI_SWIGLU>), grid, dim3(256), 0, s, a); break;
    case EPI_ROPE: hipLaunchKernelGGL((gemm_q8_kernel<EPI_ROPE>), grid, dim3(256), 0, s, a); break;
    default: return hipErrorInvalidValue;  // the audio path is dense
  }
  return hipGetLastError();
}

// XCD rows a (1, 2, 4 or 8; the XCD grid is a x 8/a) for an M x N x K
// product: the X bytes are fetched 8/a times and the weight bytes a times;
// the column groups must split evenly over 8/a.
int xcd_rows(const GemmArgs& p, int cols) {
  const double xb = (double)p.M * p.W.in * 2;
  const double wb = (double)p.W.out * p.W.in * (p.W.kind == WK_Q8 ? 34.0 / 32 : 2.0);
  int best = 1;
  double cost = 1e300;
  for (int a = 1; a <= 8; a *= 2) {
    if (cols % (8 / a)) continue;
    const double c = (8 / a) * xb + a * wb;
    if (c < cost) cost = c, best = a;
  }
  return best;
}

template <int A, int WK, int BM, int BN, int KS, int NS, bool VEC = true>
hipError_t launch_small(int epi, const GemmArgs& a, hipStream_t s) {
  const int ntiles = a.W.out / 16;
  const int cw = epi == EPI_SWIGLU ? BN / 32 : BN / 16;
  const int cols = ((epi == EPI_SWIGLU ? ntiles / 2 : ntiles) + cw - 1) / cw;
  GemmArgs g = a;
  g.map = xcd_rows(a, cols);
  const int mtiles = (a.M + BM - 1) / BM, Ma = (mtiles + g.map - 1) / g.map;
  const dim3 grid(8 * Ma * (cols / (8 / g.map)));
#define SMALL(E) hipLaunchKernelGGL((gemm_small_kernel<A, WK, E, BM, BN, KS, NS, VEC>), grid, dim3(256), 0, s, g)
  switch (epi) {
    case EPI_STORE:
      if constexpr (BN < 128) { SMALL(EPI_STORE); break; }
      return hipErrorInvalidValue;
    case EPI_ROPE:
      if constexpr (BN == 128) { SMALL(EPI_ROPE); break; }
      return hipErrorInvalidValue;
    case EPI_SWIGLU:
      if constexpr (BN == 64 && VEC) { SMALL(EPI_SWIGLU); break; }
      return hipErrorInvalidValue;
    case EPI_AFFINE:   // the audio path is dense
      if constexpr (BN < 128 && WK != WK_Q8 && VEC) { SMALL(EPI_AFFINE); break; }
      return hipErrorInvalidValue;
    case EPI_RESID:
      if constexpr (BN < 128 && VEC) { SMALL(EPI_RESID); break; }
      return hipErrorInvalidValue;
    default: return hipErrorInvalidValue;
  }
#undef SMALL
  return hipGetLastError();
}

// Tiles of the small grids: the smallest tile whose grid does not exceed
// `most` work-groups (one or two per CU), so that every CU has one while each
// work-group's serial K loop stays short; past all of them the tiles above.
// us per product (this rule's tile | the 64- and 128-row tiles above):
//   dense N = 1024, K = 3072: M = 100 7.2 | 22.4, 256 7.6 | 22.8, 450 10.6 |
//   22.7, 1024 14.6 | 23.0, 2048 20.7 | 24.0, 4096 31.1 | 34.6;
//   dense N = 4096, K = 1024: M = 24 4.5 | 12.3, 100 5.1 | 12.7, 256 6.9 |
//   12.9, 450 9.4 | 13.3, 1024 13.7 | 14.7, but 1501 (768 work-groups) 21.4 |
//   19.1;
//   Q8_0 N = 1024, K = 3072: M = 100 11.4 | 33.1, 256 11.8 | 33.2, 1024 20.7 |
//   34.4, 2048 33.8 | 35.1, but 3002 52.0 | 48.0;
//   Q8_0 N = 4096, K = 1024: M = 24 5.0 | 13.7, 256 8.9 | 13.7, 450 13.8 |
//   14.4, but 700 21.5 | 19.4.
// EPI_ROPE needs 128 columns (a head slot) and EPI_SWIGLU 64 (a gate and an up
// tile in each wave).  false: no tile applies.
template <int A, int WK>
bool try_small(int epi, const GemmArgs& a, hipStream_t s, hipError_t* e) {
  const int ntiles = epi == EPI_SWIGLU ? a.W.out / 32 : a.W.out / 16, K = a.W.in;
  const bool n32 = epi != EPI_ROPE && epi != EPI_SWIGLU, n64 = epi != EPI_ROPE;
  // grid of BM x BN tiles (a gate and an up tile count as one)
  auto fits = [&](int bm, int bn, int ks, int most) {
    const int cw = epi == EPI_SWIGLU ? bn / 32 : bn / 16;
    return K % ks == 0 && (int64_t)((a.M + bm - 1) / bm) * ((ntiles + cw - 1) / cw) <= most;
  };
  if constexpr (WK == WK_Q8) {
    if (n32 && fits(32, 32, 256, 256)) *e = launch_small<A, WK, 32, 32, 256, 3>(epi, a, s);
    else if (n32 && fits(64, 32, 128, 512)) *e = launch_small<A, WK, 64, 32, 128, 3>(epi, a, s);
    else if (n64 && fits(64, 64, 128, 512)) *e = launch_small<A, WK, 64, 64, 128, 3>(epi, a, s);
    else if (!n64 && fits(32, 128, 128, 256)) *e = launch_small<A, WK, 32, 128, 128, 3>(epi, a, s);
    else return false;
  } else {
    // a caller's unaligned output (EPI_STORE only: every other product works on
    // the library's buffers) is stored element by element, by one kind of small
    // tile, and past it by the larger tiles, which always store so
    if (epi == EPI_STORE && !vec_ok(a)) {
      if (!fits(128, 64, 64, 512)) return false;
      *e = launch_small<A, WK, 128, 64, 64, 3, false>(epi, a, s);
    } else if (epi != EPI_ROPE && !vec_ok(a)) *e = hipErrorInvalidValue;
    else if (n32 && fits(32, 32, 128, 256)) *e = launch_small<A, WK, 32, 32, 128, 4>(epi, a, s);
    else if (n64 && fits(32, 64, 128, 256)) *e = launch_small<A, WK, 32, 64, 128, 3>(epi, a, s);
    else if (n64 && fits(64, 64, 128, 256)) *e = launch_small<A, WK, 64, 64, 128, 3>(epi, a, s);
    else if (n64 && fits(64, 64, 64, 512)) *e = launch_small<A, WK, 64, 64, 64, 4>(epi, a, s);
    else if (n64 && fits(128, 64, 64, 512)) *e = launch_small<A, WK, 128, 64, 64, 3>(epi, a, s);
    else if (!n64 && fits(32, 128, 64, 256)) *e = launch_small<A, WK, 32, 128, 64, 4>(epi, a, s);
    else if (!n64 && fits(64, 128, 64, 512)) *e = launch_small<A, WK, 64, 128, 64, 3>(epi, a, s);
    else return false;
  }
  return true;
}

template <int A, int WK>
hipError_t dispatch(int epi, const GemmArgs& a, hipStream_t s) {
  const int ntiles = a.W.out / 16;
  const int cols = epi == EPI_SWIGLU ? (ntiles / 2 + 3) / 4 : (ntiles + 7) / 8;
  if constexpr (A == ACT_F32) {
    const dim3 grid((a.M + BM - 1) / BM, cols);
    switch (epi) {
      case EPI_STORE: hipLaunchKernelGGL(gemm32_kernel<EPI_STORE>, grid, dim3(256), 0, s, a); break;
      case EPI_RESID: hipLaunchKernelGGL(gemm32_kernel<EPI_RESID>, grid, dim3(256), 0, s, a); break;
      case EPI_SWIGLU: hipLaunchKernelGGL(gemm32_kernel<EPI_SWIGLU>, grid, dim3(256), 0, s, a); break;
      case EPI_AFFINE: hipLaunchKernelGGL(gemm32_kernel<EPI_AFFINE>, grid, dim3(256), 0, s, a); break;
      default: return hipErrorInvalidValue;
    }
    return hipGetLastError();
  } else {
    {
      hipError_t e = hipSuccess;
      if (try_small<A, WK>(epi, a, s, &e)) return e;
    }
    int bm = WK == WK_Q8 ? 64 : gemm_tile_rows(a.M, cols);
    // the fused q/k norm + RoPE epilogue stages at most 128 rows (a 256-row
    // tile would spill), and the residuals a 256-row tile would prefetch do
    // not fit its registers: 128-row tiles instead
    if ((epi == EPI_ROPE || epi == EPI_RESID) && bm == 256) bm = 128;
    GemmArgs g = a;
    g.map = xcd_rows(a, cols);
    const int mtiles = (a.M + bm - 1) / bm, Ma = (mtiles + g.map - 1) / g.map;
    const dim3 grid(8 * Ma * (cols / (8 / g.map)));
    if constexpr (WK == WK_Q8) return launch_q8(epi, grid, g, s);
    else if (bm == 256) return launch_dma<A, 256, 3>(epi, grid, g, s);
    else return launch_dma<A, 128, 4>(epi, grid, g, s);
  }
}

}  // namespace

hipError_t launch_gemm(int act, int epi, const GemmArgs& a, hipStream_t s) {
  if (a.M <= 0) return hipSuccess;
  if (a.W.in % BK || a.W.out % 16 || (epi == EPI_SWIGLU && a.W.out % 32))
    return hipErrorInvalidValue;
  // 16-bit rows go global -> LDS by copies that read 16 aligned bytes
  if (act != ACT_F32 && ((uintptr_t)a.x % 16 || a.ldx % 8)) return hipErrorInvalidValue;
  // EPI_ROPE: 16-bit activations, one 128-wide head slot per column group,
  // at most 16 sequences (a row's position and sequence travel as pos * 16 + b)
  if (epi == EPI_ROPE && (act == ACT_F32 || a.W.out != (a.rope.nh + 2 * a.rope.nkv) * 128 ||
                          !a.rope.row_b || !a.rope.row_pos || a.rope.batch < 1 ||
                          a.rope.batch > 16))
    return hipErrorInvalidValue;
  if (epi == EPI_AFFINE && ((a.aff.table && (a.aff.period <= 0 || a.aff.valid < 1)) ||
                            (a.aff.period > 0 && (a.aff.valid < 0 || a.aff.valid > a.aff.period)) ||
                            a.aff.act < 0 || a.aff.act > 2 || a.aff.scale_cols < 0 ||
                            a.aff.scale_cols % 4 || (a.resid && a.aff.table)))
    return hipErrorInvalidValue;
  if (a.W.kind == WK_Q8) {
    if (act != ACT_F16) return hipErrorInvalidValue;
    return dispatch<ACT_F16, WK_Q8>(epi, a, s);
  }
  switch (act) {
    case ACT_F32: return dispatch<ACT_F32, WK_DENSE>(epi, a, s);
    case ACT_F16: return dispatch<ACT_F16, WK_DENSE>(epi, a, s);
    case ACT_BF16: return dispatch<ACT_BF16, WK_DENSE>(epi, a, s);
  }
  return hipErrorInvalidValue;
}
