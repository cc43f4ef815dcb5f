// Learned relaxation kernels (BF16 MFMA, FP32 accumulation) for gfx950.
//
// v_mfma_f32_32x32x16_bf16 operand layouts (lane l, g = l / 32, c = l % 32):
//   A (32 x 16): lane holds A[c][8g + t], t = 0..7
//   B (16 x 32): lane holds B[8g + t][c]
//   C (32 x 32): register r holds C[8(r/4) + 4g + (r%4)][c]
// (v_mfma_f32_32x32x8_bf16, the layout self-test's other form: A[c][4g + t],
// B[4g + t][c], t = 0..3, the same C.)  The MFMA self-tests check both
// layouts against host matrix products.
//
// Pair layer: one wave serves 64 particles, one per lane.  Each lane walks its
// own particle's candidates (the three row ranges of its 3x3 cells) and stops
// at its next in-range pair; the wave's 64 current pairs are two 32-row MFMA
// tiles (rows = lanes 0..31 and lanes 32..63), one K = 16 MFMA per tile and
// hidden half gives the pre-activations z.  A lane without a pair left
// contributes a zero feature row, whose messages are relu(0) = 0 because the
// bias is a feature.  relu(z) is taken on BF16: two values are converted with
// one v_cvt_pk_bf16_f32 and clamped at 0 with one v_pk_max_i16 (a negative
// BF16 is a negative 16-bit integer).  The per-particle sum H_i += relu(z_ij)
// runs on the matrix core: in the C layout, registers 8s .. 8s + 7 of a lane
// hold exactly the B operand (K = 16 rows of z, the lane's hidden column) of
// a K = 16 MFMA, and a 0/1 selection matrix as A sends row k of z to its
// particle's row of H; with one nonzero product per output, the MFMA adds
// each BF16 value to the FP32 accumulator exactly as an FP32 add would.
#include "nbs_device.hpp"
#include "nbs_surrogate.hpp"

#include <algorithm>
#include <cmath>

namespace nbs {

typedef short bf16x4 __attribute__((__vector_size__(4 * sizeof(short))));
typedef float floatx16 __attribute__((__vector_size__(16 * sizeof(float))));

typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef float f32x2 __attribute__((ext_vector_type(2)));

// FP32 -> BF16, round to nearest even: one v_cvt_pk_bf16_f32 for both values
// (converting the elements one at a time costs two conversions and a permute
// when the inputs are MFMA results).
__device__ __forceinline__ uint32_t pack2(float lo, float hi) {
  const f32x2 f = {lo, hi};
  return __builtin_bit_cast(uint32_t, __builtin_convertvector(f, bf16x2));
}
__device__ __forceinline__ uint16_t f2bf(float x) { return __builtin_bit_cast(uint16_t, (__bf16)x); }

__device__ __forceinline__ floatx16 mfma(bf16x4 a, bf16x4 b, floatx16 c) {
  return __builtin_amdgcn_mfma_f32_32x32x8bf16_1k(a, b, c, 0, 0, 0);
}

__device__ __forceinline__ floatx16 zero16() {
  floatx16 z;
#pragma unroll
  for (int k = 0; k < 16; ++k) z[k] = 0.0f;
  return z;
}

// relu(z) as an integer maximum of the bit pattern with 0: negative values
// (and -0) become +0, others are unchanged.  One instruction; fmaxf costs two
// here (the IEEE-mode canonicalisation of its operand).
__device__ __forceinline__ float relu(float z) { return __int_as_float(max(__float_as_int(z), 0)); }

// K = 16 operands: eight BF16 values in four words.
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef short s16x2 __attribute__((ext_vector_type(2)));

__device__ __forceinline__ bf16x8 bf8(uint32_t w0, uint32_t w1, uint32_t w2, uint32_t w3) {
  const u32x4 u = {w0, w1, w2, w3};
  return __builtin_bit_cast(bf16x8, u);
}

__device__ __forceinline__ floatx16 mfma16(bf16x8 a, bf16x8 b, floatx16 c) {
  return __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, c, 0, 0, 0);
}

// relu of two values rounded to BF16 (round to nearest even), packed: one
// v_cvt_pk_bf16_f32, then one v_pk_max_i16 with 0 (negative values and -0 are
// negative 16-bit integers and become +0).
__device__ __forceinline__ uint32_t relu2_bf16(float lo, float hi) {
  const s16x2 v = __builtin_bit_cast(s16x2, pack2(lo, hi));
  const s16x2 z = {0, 0};
  return __builtin_bit_cast(uint32_t, __builtin_elementwise_max(v, z));
}

// K = 16 B operand of a row-major BF16 matrix W (rows = outputs, K inputs):
// B[k][n] = W[n0 + n][k0 + k].  K and k0 are multiples of 8 (16-byte loads).
__device__ __forceinline__ bf16x8 load_wb16(const uint16_t *W, int K, int n0, int k0) {
  const int c = threadIdx.x & 31, g = (threadIdx.x >> 5) & 1;
  const uint4 w = *reinterpret_cast<const uint4 *>(W + (size_t)(n0 + c) * K + k0 + 8 * g);
  return bf8(w.x, w.y, w.z, w.w);
}

// Eight BF16 values at p (a row of an LDS buffer, 4-byte aligned).
__device__ __forceinline__ bf16x8 lds_bf8(const uint16_t *p) {
  const uint32_t *w = reinterpret_cast<const uint32_t *>(p);
  return bf8(w[0], w[1], w[2], w[3]);
}

__device__ __forceinline__ void lds_put8(uint16_t *p, bf16x8 v) {
  const u32x4 u = __builtin_bit_cast(u32x4, v);
  uint32_t *w = reinterpret_cast<uint32_t *>(p);
#pragma unroll
  for (int k = 0; k < 4; ++k) w[k] = u[k];
}

// B operand of step s (K = 16 rows of a 32-row C-layout tile z): this lane's
// registers 8s .. 8s + 7, relu'd in BF16.
__device__ __forceinline__ bf16x8 relu_rows(const floatx16 &z, int s) {
  return bf8(relu2_bf16(z[8 * s + 0], z[8 * s + 1]), relu2_bf16(z[8 * s + 2], z[8 * s + 3]),
             relu2_bf16(z[8 * s + 4], z[8 * s + 5]), relu2_bf16(z[8 * s + 6], z[8 * s + 7]));
}

// C-layout row of register r for lane group g.
__device__ __forceinline__ int c_row(int r, int g) { return 8 * (r >> 2) + 4 * g + (r & 3); }

// A operand of step s of the pair sum: 32 x 16, A[p][k] = 1 when the K index k
// (K = 16 rows of z as relu_rows supplies them: lane group g', register
// 8s + t for k = 8g' + t) is row p of the tile.  Lane (c, g) holds row c.
__device__ __forceinline__ bf16x8 selection(int s) {
  const int c = threadIdx.x & 31, g = (threadIdx.x >> 5) & 1;
  uint32_t w[4];
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    const uint32_t lo = c_row(8 * s + 2 * q, g) == c ? 0x3F80u : 0u;  // BF16 1.0
    const uint32_t hi = c_row(8 * s + 2 * q + 1, g) == c ? 0x3F80u : 0u;
    w[q] = lo | (hi << 16);
  }
  return bf8(w[0], w[1], w[2], w[3]);
}

// B operand (K = 16) of the 16 x 32 matrix with ones where k + first == n.
__device__ __forceinline__ bf16x8 identity16(int first) {
  const int c = threadIdx.x & 31, g = (threadIdx.x >> 5) & 1;
  uint32_t w[4];
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    const int k = first + 8 * g + 2 * q;
    w[q] = k == c ? 0x3F80u : (k + 1 == c ? 0x3F800000u : 0u);  // BF16 1.0
  }
  return bf8(w[0], w[1], w[2], w[3]);
}

constexpr int kWaveRows = 64;    // particles per wave in the pair kernels
constexpr int kHbStride = 68;    // BF16 per row of the head operand buffer (padded)
constexpr int kTileCap = 512;    // staged candidates (positions, previous positions, densities)
constexpr int kStageBytes = 3 * kTileCap * 8;
static_assert(kSurRows * kHbStride * 2 <= kStageBytes, "a row tile's BF16 activations fit the staging pool");

// Per-particle inputs of the pair layer.
struct PartInfo {
  float2 xi;
  float vix, viy;
  float fr, fn;  // normalised density, near density
};

// A particle's own loads for part_info, requested before the tile is staged
// (the staging's waits then cover them) and turned into PartInfo after.
struct PartRaw {
  uint32_t key;
  float2 x, pv, d;
};
__device__ __forceinline__ PartRaw part_raw(const Buffers &b, int i) { return {b.keys[i], b.x1[i], b.prev[i], b.dens[i]}; }

__device__ __forceinline__ float2 velocity(float2 x, float2 prev, const DevParams &p) {
  return make_float2((x.x - prev.x) * p.invDt, (x.y - prev.y) * p.invDt);
}
__device__ __forceinline__ float2 normalised(float2 d, const float *norm) {
  return make_float2((d.x - norm[1]) * norm[2], (d.y - norm[3]) * norm[4]);
}
__device__ __forceinline__ PartInfo part_info(const DevParams &p, const float *norm, const PartRaw &r) {
  const float2 v = velocity(r.x, r.pv, p), f = normalised(r.d, norm);
  return {r.x, v.x, v.y, f.x, f.y};
}

// A lane's walk over its particle's candidates: the rows dy = -1..1 of the
// 3x3 cells, each a contiguous slot range (demo4.cpp:188-203 order).  tb maps
// a slot of the current row to its index in the neighbour source.
struct Cursor {
  uint32_t j, jend, tb;
  int d;
  bool done;
  // In-range candidates of the chunk being taken (bit b is entry mbase + b of
  // the source) and of the next two, in order.
  uint32_t mask, mbase, m1, b1, m2, b2;
  RowRange r0, r1, r2;  // the rows not walked yet
};

// Neighbour data of a wave's candidates: an LDS copy of the three candidate
// slot ranges of the wave's 64 particles (the layout of TilePlan) when they
// fit, else the slot arrays.  The tile holds velocities and normalised
// densities, computed once per candidate instead of once per pair, in place of
// the slot arrays' previous positions and densities (with the square root for
// waves without tiny operands, 262,144 particles 46.5 -> 44.6 us).

struct PairSrc {
  const float2 *x, *pv, *d;
  uint32_t rowStart0, rowStart1, rowStart2, off0, off1, off2;
  bool tiled;
  // slot j of candidate row r sits at j + base(r)
  __device__ __forceinline__ uint32_t base(int r) const {
    if (!tiled) return 0u;
    return r == 0 ? off0 - rowStart0 : (r == 1 ? off1 - rowStart1 : off2 - rowStart2);
  }
};

__device__ __forceinline__ bool cursor_next_row(Cursor &cu, const PairSrc &src) {
  while (cu.d < 3) {
    const int r = cu.d++;
    cu.j = cu.r0.j0;
    cu.jend = cu.r0.j1;
    cu.r0 = cu.r1;
    cu.r1 = cu.r2;
    if (cu.j < cu.jend) {
      cu.tb = src.base(r);
      return true;
    }
  }
  return false;
}

// Stages the planned tile when it fits (every lane must call it).
__device__ __forceinline__ PairSrc stage_pairs(const Buffers &b, const DevParams &p, const float *norm,
                                               const TilePlan &plan, unsigned char *pool) {
  PairSrc src;
  src.tiled = plan.use != 0;
  src.rowStart0 = plan.rowStart[0], src.rowStart1 = plan.rowStart[1], src.rowStart2 = plan.rowStart[2];
  src.off0 = plan.off[0], src.off1 = plan.off[1], src.off2 = plan.off[2];
  if (src.tiled) {
    float2 *tx = reinterpret_cast<float2 *>(pool);
    float2 *tp = tx + kTileCap, *td = tp + kTileCap;
    const float2 *const from[3] = {b.x1, b.prev, b.dens};
    float2 *const to[3] = {tx, tp, td};
    // the three arrays' loads in flight together
    stage_arrays<3>(plan, from, to, [&](float2 (&w)[3]) {
      w[1] = velocity(w[0], w[1], p);
      w[2] = normalised(w[2], norm);
    });
    src.x = tx;
    src.pv = tp;
    src.d = td;
  } else {
    src.x = b.x1;
    src.pv = b.prev;
    src.d = b.dens;
  }
  __syncthreads();
  return src;
}

// The source with its pointers re-derived from the LDS pool (tiled) or the
// slot arrays, for code that handles one kind only.
__device__ __forceinline__ PairSrc tile_src(PairSrc s, unsigned char *pool) {
  s.tiled = true;
  s.x = reinterpret_cast<const float2 *>(pool);
  s.pv = s.x + kTileCap;
  s.d = s.pv + kTileCap;
  return s;
}
__device__ __forceinline__ PairSrc slot_src(PairSrc s, const Buffers &b) {
  s.tiled = false;
  s.x = b.x1;
  s.pv = b.prev;
  s.d = b.dens;
  return s;
}

// Cut-off mask of the cnt <= 32 candidates at xs[0 .. cnt): bit k is set when
// candidate k lies within h of xi.
__device__ __forceinline__ uint32_t chunk_bits(const float2 *xs, uint32_t cnt, float2 xi, float h2) {
  // m = 2 * m + (d2 < h2), last candidate first, so candidate k ends at bit
  // k: the compare's lane mask is the add's carry-in
  uint32_t m = 0;
  auto push = [&](float d2) {
    asm("v_cmp_gt_f32_e32 vcc, %1, %2\n\tv_addc_co_u32_e32 %0, vcc, %0, %0, vcc" : "+v"(m) : "s"(h2), "v"(d2) : "vcc");
  };
  auto dist2 = [&](uint32_t k) {
    const float2 x = xs[k];
    const float dx = x.x - xi.x, dy = x.y - xi.y;
    return dx * dx + dy * dy;
  };
  uint32_t u = cnt;
  for (; u >= 8u; u -= 8u) {  // eight position loads in flight
    float d2[8];
#pragma unroll
    for (int k = 0; k < 8; ++k) d2[k] = dist2(u - 1 - k);
#pragma unroll
    for (int k = 0; k < 8; ++k) push(d2[k]);
  }
  for (; u >= 4u; u -= 4u) {
    const float a0 = dist2(u - 1), a1 = dist2(u - 2), a2 = dist2(u - 3), a3 = dist2(u - 4);
    push(a0);
    push(a1);
    push(a2);
    push(a3);
  }
  for (; u > 0u; --u) push(dist2(u - 1));
  return m;
}

// Rows of at most kWalkRowMax candidates can be tested up front: when every
// lane's three rows fit (rows_fit, wave-uniform), cursor_rows tests all of
// them with the wave's lanes together and next_pair then only moves from one
// row's mask to the next.  Otherwise, when a lane runs out of marked candidates,
// every lane with room tests its next chunk of kWalkChunk (cursor_chunk).
constexpr uint32_t kWalkChunk = 32;
constexpr uint32_t kWalkRowMax = 32;

// rows: the lane's three candidate rows (row_ranges; ignored for a lane past
// n).
__device__ __forceinline__ bool rows_fit(const RowRange (&rows)[3], bool live) {
  bool fit = true;
  if (live)
#pragma unroll
    for (int d = 0; d < 3; ++d) fit = fit && rows[d].j1 - rows[d].j0 <= kWalkRowMax;
  return __ballot(!fit) == 0ull;
}

// Tests the lane's three rows (every row at most kWalkRowMax candidates) and
// loads their masks into the cursor; the particle itself is no pair.
__device__ __forceinline__ void cursor_rows(Cursor &cu, const RowRange (&rows)[3], const DevParams &p,
                                            const PairSrc &src, const PartInfo &q, int i) {
  uint32_t m[3], base[3];
#pragma unroll
  for (int r = 0; r < 3; ++r) {
    const RowRange rr = rows[r];
    const uint32_t cnt = rr.j1 - rr.j0;
    // the row's first index in the source: j0 + base(r) wraps modulo 2^32
    // (off - rowStart on the LDS tile), so it is formed in 32 bits first
    base[r] = (uint32_t)(rr.j0 + src.base(r));
    m[r] = chunk_bits(src.x + base[r], cnt, q.xi, p.h2);
    const uint32_t self = (uint32_t)i - rr.j0;
    if (self < cnt) m[r] &= ~(1u << self);
  }
  cu.mask = m[0], cu.mbase = base[0];
  cu.m1 = m[1], cu.b1 = base[1], cu.m2 = m[2], cu.b2 = base[2];
}

// Tests the lane's next chunk and appends its mask, if any candidate is in
// range, to the cursor's (which has room); done when there is none left.
__device__ __forceinline__ void cursor_chunk(Cursor &cu, const DevParams &p, const PairSrc &src, const PartInfo &q,
                                             int i) {
  if (cu.j >= cu.jend && !cursor_next_row(cu, src)) {
    cu.done = true;
    return;
  }
  const uint32_t cnt = min(kWalkChunk, cu.jend - cu.j);
  // the chunk's first index in the source: j + tb wraps modulo 2^32 (tb is
  // off - rowStart on the LDS tile), so it is formed in 32 bits first
  const uint32_t base = (uint32_t)(cu.j + cu.tb);
  uint32_t m = chunk_bits(src.x + base, cnt, q.xi, p.h2);
  const uint32_t self = (uint32_t)i - cu.j;  // the particle itself is no pair
  if (self < cnt) m &= ~(1u << self);
  cu.j += cnt;
  if (m == 0u) return;
  if (cu.mask == 0u)
    cu.mask = m, cu.mbase = base;
  else if (cu.m1 == 0u)
    cu.m1 = m, cu.b1 = base;
  else
    cu.m2 = m, cu.b2 = base;
}

// Advances to the lane's next pair (j != i, r^2 < h^2); false when exhausted.
// t is the pair's index in src.  The masks' bits are taken lowest first
// (candidate order); with rows (the cursor loaded by cursor_rows) the masks of
// all three rows are there already, else every lane keeps up to three chunks'
// masks and the wave refills them together, once some lane has none: in crowded
// states refilled a lane at a time, the rest of the wave waiting for each of its
// chunks, the 4,096-particle dam break at step 400 (up to 370 candidates) took
// 369 us per network step and 632 per training step, now 215 and 387.  All lanes
// of the wave must call it.
__device__ __forceinline__ bool next_pair(Cursor &cu, const DevParams &p, const PairSrc &src, const PartInfo &q, int i,
                                          bool rows, uint32_t &t, float2 &xj, float &Rx, float &Ry, float &r2) {
  if (cu.mask == 0u) {
    const bool next = cu.m1 != 0u;
    cu.mask = next ? cu.m1 : cu.m2;
    cu.mbase = next ? cu.b1 : cu.b2;
    cu.m1 = next ? cu.m2 : 0u;
    cu.b1 = cu.b2;
    cu.m2 = 0u;
  }
  if (!rows)
    while (__ballot(cu.mask == 0u && !cu.done))  // wave-uniform
      if (cu.m2 == 0u && !cu.done) cursor_chunk(cu, p, src, q, i);
  if (cu.mask == 0u) return false;
  t = cu.mbase + (uint32_t)__builtin_ctz(cu.mask);
  cu.mask &= cu.mask - 1u;
  xj = src.x[t];
  Rx = xj.x - q.xi.x;
  Ry = xj.y - q.xi.y;
  r2 = Rx * Rx + Ry * Ry;
  return true;
}

// Runs walk(source, whether the rows were tested up front).  One copy of the
// walk per source, so that the tile's loads are LDS loads (a pointer that may be
// either is a flat address), and per kind of walk: their cursors hold different
// registers.
template <typename Walk>
__device__ __forceinline__ void pair_pass(const PairSrc &src, unsigned char *pool, const Buffers &b, const DevParams &p,
                                          const PartInfo &q, const RowRange (&rr)[3], int i, int n, Cursor &cu,
                                          Walk &&walk) {
  auto pass = [&](const PairSrc &sp) {
    if (rows_fit(rr, i < n)) {
      if (i < n) cursor_rows(cu, rr, p, sp, q, i);
      walk(sp, std::true_type());
    } else {
      walk(sp, std::false_type());
    }
  };
  if (src.tiled)
    pass(tile_src(src, pool));
  else
    pass(slot_src(src, b));
}

// The pair's 16 BF16 features as 8 words (features 2k, 2k+1 in word k).
__device__ __forceinline__ void pair_words(uint32_t w[8], const PairSrc &src, const DevParams &p, const float *norm,
                                           const PartInfo &q, uint32_t t, float2 xj, float Rx, float Ry, float r2,
                                           bool near) {
  const float2 pj = src.pv[t], dj = src.d[t];
  const float2 vj = src.tiled ? pj : velocity(xj, pj, p), fj = src.tiled ? dj : normalised(dj, norm);
  const float r = root_of(near, r2);
  const float qq = 1.0f - r * p.invH;
  w[0] = pack2(Rx * p.invH, Ry * p.invH);
  w[1] = pack2((vj.x - q.vix) * norm[0], (vj.y - q.viy) * norm[0]);
  w[2] = pack2(q.fr, q.fn);
  w[3] = pack2(fj.x, fj.y);
  w[4] = pack2(1.0f, qq);
  w[5] = pack2(qq * qq, 0.0f);
  w[6] = 0u;
  w[7] = 0u;
}

struct W1Operands {
  bf16x8 lo, hi;  // hidden 0..31 / 32..63
};

__device__ __forceinline__ W1Operands load_w1(const uint16_t *w1b) {
  return {load_wb16(w1b, kFeat, 0, 0), load_wb16(w1b, kFeat, 32, 0)};
}

// A operands (K = 16) of the two row tiles from each lane's own feature words:
// tile 0 rows are lanes 0..31, tile 1 rows lanes 32..63; lane (c, g) supplies
// features 8g .. 8g + 7 of its row, so one half of each tile's words crosses
// the lane halves (words 6, 7 are zero): one exchange per word (with shuffles
// through the LDS unit the 262,144-particle forward took 62 us instead of 60).
struct PairA {
  bf16x8 t0, t1;
};

__device__ __forceinline__ PairA pair_operands(const uint32_t w[8]) {
  // swap(x, y): y's lower half moves to x's upper half and back
  const auto r0 = __builtin_amdgcn_permlane32_swap(w[0], w[4], false, false);
  const auto r1 = __builtin_amdgcn_permlane32_swap(w[1], w[5], false, false);
  const auto r2 = __builtin_amdgcn_permlane32_swap(w[2], 0u, false, false);
  const auto r3 = __builtin_amdgcn_permlane32_swap(w[3], 0u, false, false);
  return {bf8(r0[0], r1[0], r2[0], r3[0]), bf8(r0[1], r1[1], r2[1], r3[1])};
}

// Pre-activations z = F W1^T of one row tile (C layout, lane = hidden unit).
__device__ __forceinline__ void pair_layer(bf16x8 a, const W1Operands &w, floatx16 &zlo, floatx16 &zhi) {
  zlo = mfma16(a, w.lo, zero16());
  zhi = mfma16(a, w.hi, zero16());
}

// ---------------------------------------------------------------------------
// Forward
// ---------------------------------------------------------------------------
// C layout to K order: registers 8s .. 8s + 7 of a lane hold rows 16s + 4g + {0
// .. 3, 8 .. 11}; swapping four of them between the wave's halves leaves rows
// 16s + 8g + {0 .. 7} in both, the K index order of a 32x32x16 operand.
__device__ __forceinline__ floatx16 k_order(floatx16 z) {
#pragma unroll
  for (int s = 0; s < 2; ++s)
#pragma unroll
    for (int t = 0; t < 4; ++t) {
      const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(z[8 * s + t]), __float_as_uint(z[8 * s + 4 + t]),
                                                      false, false);
      z[8 * s + t] = __uint_as_float(r[0]);
      z[8 * s + 4 + t] = __uint_as_float(r[1]);
    }
  return z;
}

// The training activations of a row tile leave the forward as operands of the
// backward pass's weight gradients (K = 16 particles): a lane's eight rows of
// one hidden column are 16 bytes of BF16, and every store is 1 KiB of
// consecutive words for the wave.
__device__ __forceinline__ uint4 pack8(const floatx16 &z, int s) {
  return make_uint4(pack2(z[8 * s], z[8 * s + 1]), pack2(z[8 * s + 2], z[8 * s + 3]),
                    pack2(z[8 * s + 4], z[8 * s + 5]), pack2(z[8 * s + 6], z[8 * s + 7]));
}
__device__ __forceinline__ void store_tile_bf16(uint4 *dst, floatx16 lo, floatx16 hi) {
  lo = k_order(lo), hi = k_order(hi);
  dst[0 * 64 + threadIdx.x] = pack8(lo, 0);
  dst[1 * 64 + threadIdx.x] = pack8(lo, 1);
  dst[2 * 64 + threadIdx.x] = pack8(hi, 0);
  dst[3 * 64 + threadIdx.x] = pack8(hi, 1);
}
// One word of it from LDS: particles 16 s + 8 g + {0 .. 7} of hidden column h.
__device__ __forceinline__ uint4 lds_column(const uint16_t (*rows)[kHbStride], int h, int s) {
  const uint16_t(*r)[kHbStride] = rows + 16 * s + 8 * (int)((threadIdx.x >> 5) & 1);
  auto two = [&](int k) { return (uint32_t)r[k][h] | ((uint32_t)r[k + 1][h] << 16); };
  return make_uint4(two(0), two(2), two(4), two(6));
}
// Word q of an FP32 tile: rows 2q and 2q + 1 of the lane's two columns.
__device__ __forceinline__ void store_tile_f32(float4 *dst, int lane, const floatx16 &lo, const floatx16 &hi) {
#pragma unroll
  for (int q = 0; q < 8; ++q) dst[q * 64 + lane] = make_float4(lo[2 * q], hi[2 * q], lo[2 * q + 1], hi[2 * q + 1]);
}

// Operands (K = hidden) of a half of a tile whose C layout has the particle as
// its lane: k_order on packed BF16 words.
__device__ __forceinline__ void k_operands(const floatx16 &z, bf16x8 &op0, bf16x8 &op1) {
#pragma unroll
  for (int s = 0; s < 2; ++s) {
    const int r = 8 * s;
    const auto a = __builtin_amdgcn_permlane32_swap(pack2(z[r], z[r + 1]), pack2(z[r + 4], z[r + 5]), false, false);
    const auto b = __builtin_amdgcn_permlane32_swap(pack2(z[r + 2], z[r + 3]), pack2(z[r + 6], z[r + 7]), false, false);
    (s ? op1 : op0) = bf8(a[0], b[0], a[1], b[1]);
  }
}

// Registers of a C-layout tile from a vector indexed by its row: v[c_row(r, g)].
__device__ __forceinline__ floatx16 by_row(const float *v) {
  floatx16 z;
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    const float4 f = *reinterpret_cast<const float4 *>(v + 8 * q + 4 * ((threadIdx.x >> 5) & 1));
    z[4 * q] = f.x, z[4 * q + 1] = f.y, z[4 * q + 2] = f.z, z[4 * q + 3] = f.w;
  }
  return z;
}

// The head, without LDS.  The pair sums h[tile][hidden half] have the particle
// as their lane (column) and the hidden units in their registers, so that a
// layer's packed outputs are, after one exchange between the wave's halves, the
// next layer's operands, both row tiles share the weights' operands, and lane l
// ends with all 64 values of G of particle l for the output layer's FP32 sum (k
// ascending).  262,144 particles: one tile after the other through LDS 20 of
// the forward's 60 us, all of it 46 us after.
// TRAIN also writes the activations, whose layout has the hidden unit as the
// lane: H and M, whose BF16 operands are the values kept, times the identity,
// and G as a second product with the operands' roles exchanged.  An infinite or
// NaN value times the identity's zeros would make its particle's others NaN, so
// a wave that holds one stores them again, transposed through LDS (pool); it
// shows in any one of the next layer's pre-activations, which add infinity or
// NaN times a weight.
template <bool TRAIN>
__device__ __forceinline__ float2 head_output(const floatx16 (&h)[2][2], uint32_t np, const SurrogateBufs &m,
                                              int base, int n, unsigned char *pool) {
  const float *prm = m.params;
  const int c = threadIdx.x & 31;
  const auto cnt = __builtin_amdgcn_permlane32_swap(__float_as_uint((float)np), __float_as_uint((float)np), false, false);
  uint4 *act[2];
  if (TRAIN)
#pragma unroll
    for (int t = 0; t < 2; ++t) act[t] = m.act + (size_t)(2 * blockIdx.x + t) * kActWords;
  auto store_operands = [&](const bf16x8 (&op)[2][4], int at) {
    const bf16x8 e0 = identity16(0), e1 = identity16(16);
#pragma unroll
    for (int t = 0; t < 2; ++t)
      if (base + 32 * t < n)  // the tile exists
        store_tile_bf16(act[t] + at, mfma16(op[t][1], e1, mfma16(op[t][0], e0, zero16())),
                        mfma16(op[t][3], e1, mfma16(op[t][2], e0, zero16())));
  };
  auto store_through_lds = [&](const bf16x8 (&op)[2][4], int at) {
    uint16_t(*rows)[kHbStride] = reinterpret_cast<uint16_t(*)[kHbStride]>(pool);
#pragma unroll
    for (int t = 0; t < 2; ++t) {
      __syncthreads();  // pool is no longer read
#pragma unroll
      for (int s = 0; s < 4; ++s) lds_put8(&rows[c][16 * s + 8 * (int)(threadIdx.x >> 5)], op[t][s]);
      __syncthreads();
      if (base + 32 * t >= n) continue;
#pragma unroll
      for (int k = 0; k < 4; ++k) act[t][at + k * 64 + threadIdx.x] = lds_column(rows, 32 * (k >> 1) + c, k & 1);
    }
  };
  bool finite = true;
  bf16x8 op[2][4], om[2][4];  // H, M: tile, K step
#pragma unroll
  for (int t = 0; t < 2; ++t)
#pragma unroll
    for (int y = 0; y < 2; ++y) k_operands(h[t][y], op[t][2 * y], op[t][2 * y + 1]);
  if (TRAIN) store_operands(op, 0);
  // output half y of a layer for both tiles
  auto dense = [&](const uint16_t *W, int y, const bf16x8 (&in)[2][4], floatx16 &z0, floatx16 &z1) {
    z0 = zero16(), z1 = zero16();
#pragma unroll
    for (int s = 0; s < 4; ++s) {
      const bf16x8 w = load_wb16(W, kHid, 32 * y, 16 * s);
      z0 = mfma16(w, in[0][s], z0);
      z1 = mfma16(w, in[1][s], z1);
    }
  };
  // M = W2 H + n b2, kept as BF16
#pragma unroll
  for (int y = 0; y < 2; ++y) {
    floatx16 z0, z1;
    dense(m.w2b, y, op, z0, z1);
    if (y == 0) finite = finite && __builtin_isfinite(z0[0]) && __builtin_isfinite(z1[0]);
    const floatx16 b2 = by_row(prm + kOffB2 + 32 * y);
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      z0[r] += __uint_as_float(cnt[0]) * b2[r];
      z1[r] += __uint_as_float(cnt[1]) * b2[r];
    }
    k_operands(z0, om[0][2 * y], om[0][2 * y + 1]);
    k_operands(z1, om[1][2 * y], om[1][2 * y + 1]);
  }
  if (TRAIN) {
    store_operands(om, 4 * 64);
#pragma unroll
    for (int t = 0; t < 2; ++t) {
      if (base + 32 * t >= n) continue;
      floatx16 lo = zero16(), hi = zero16();
#pragma unroll
      for (int s = 0; s < 4; ++s) {
        lo = mfma16(om[t][s], load_wb16(m.w3b, kHid, 0, 16 * s), lo);
        hi = mfma16(om[t][s], load_wb16(m.w3b, kHid, 32, 16 * s), hi);
      }
      const float b3lo = prm[kOffB3 + c], b3hi = prm[kOffB3 + 32 + c];
#pragma unroll
      for (int r = 0; r < 16; ++r) lo[r] = relu(lo[r] + b3lo), hi[r] = relu(hi[r] + b3hi);
      store_tile_f32(reinterpret_cast<float4 *>(act[t] + 8 * 64), (int)threadIdx.x, lo, hi);
    }
  }
  // G = relu(W3 M + b3), FP32; then o = W4 G + b4
  float2 o = make_float2(prm[kOffB4], prm[kOffB4 + 1]);
#pragma unroll
  for (int y = 0; y < 2; ++y) {
    floatx16 z0, z1;
    dense(m.w3b, y, om, z0, z1);
    if (y == 0) finite = finite && __builtin_isfinite(z0[0]) && __builtin_isfinite(z1[0]);
    const floatx16 b3 = by_row(prm + kOffB3 + 32 * y);
    floatx16 g[2];  // rows c_row(r, 0), c_row(r, 1) of the lane's own particle
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      const auto q = __builtin_amdgcn_permlane32_swap(__float_as_uint(relu(z0[r] + b3[r])),
                                                      __float_as_uint(relu(z1[r] + b3[r])), false, false);
      g[0][r] = __uint_as_float(q[0]);
      g[1][r] = __uint_as_float(q[1]);
    }
#pragma unroll
    for (int k = 0; k < 32; ++k) {
      const float v = g[(k >> 2) & 1][4 * (k >> 3) + (k & 3)];
      o.x = __builtin_fmaf(prm[kOffW4 + 32 * y + k], v, o.x);
      o.y = __builtin_fmaf(prm[kOffW4 + kHid + 32 * y + k], v, o.y);
    }
    asm volatile("" : "+v"(o.x), "+v"(o.y));  // a half of W4 in scalar registers at a time: both would spill
  }
  if (TRAIN && __ballot(!finite) != 0ull) {  // again, over the first stores
    store_through_lds(op, 0);
    store_through_lds(om, 4 * 64);
  }
  return o;
}

// One wave takes 64 particles; every iteration of the walk adds one pair of each
// through the matrix cores.  Bound by the issue of an iteration's about 180
// vector instructions (relu and packing 64, features 40; its 12 products take
// two thirds of that time beside them) and by the start of each wave's walk.
// Two waves per SIMD: for three the compiler spills inside the walk (80 us at
// 262,144 particles, 46 without).
template <bool MULTI, bool TRAIN>
__global__ __launch_bounds__(64, 2) void k_sur_forward(Buffers b, DevParams p, DevScene s0, int n, SurrogateBufs m,
                                                       int mode) {
  __shared__ __align__(16) unsigned char pool[kStageBytes];
  const int lane = threadIdx.x;
  const int base = (int)blockIdx.x * kWaveRows;
  const int me = base + lane;
  const float *norm = m.params + kOffNorm;
  const W1Operands w1 = load_w1(m.w1b);
  const bf16x8 sel[2] = {selection(0), selection(1)};
  const PartRaw raw = part_raw(b, min(me, n - 1));  // a lane past n reads the last particle, unused
  TilePlan plan;
  DevScene scMe;
  int cx, cy;
  RowRange rr[3];
  open_block<MULTI, kTileCap, kWaveRows>(b, s0, b.startNext, base, n, raw.key, scMe, plan, cx, cy, rr);
  const PairSrc src = stage_pairs(b, p, norm, plan, pool);

  // 1. pair layer: H_i = sum_j relu(W1 f_ij), each term rounded to BF16
  const PartInfo q = part_info(p, norm, raw);
  const bool near = wave_near(p, q.xi);
  Cursor cu{0u, 0u, 0u, 0, me >= n, 0u, 0u, 0u, 0u, 0u, 0u, rr[0], rr[1], rr[2]};
  floatx16 h[2][2] = {{zero16(), zero16()}, {zero16(), zero16()}};  // tile, hidden half
  auto add = [&](bf16x8 z, int s, floatx16 &acc) { acc = mfma16(z, sel[s], acc); };
  auto add_tile = [&](bf16x8 a, floatx16 (&acc)[2]) {
    floatx16 zlo, zhi;
    pair_layer(a, w1, zlo, zhi);
    add(relu_rows(zlo, 0), 0, acc[0]);  // K steps 0 and 1 of each hidden half
    add(relu_rows(zhi, 0), 0, acc[1]);
    add(relu_rows(zlo, 1), 1, acc[0]);
    add(relu_rows(zhi, 1), 1, acc[1]);
  };
  uint32_t np = 0;
  auto walk = [&](const PairSrc &sp, auto rows) {
    for (;;) {
      uint32_t t = 0;
      float2 xj = make_float2(0.0f, 0.0f);
      float Rx = 0.0f, Ry = 0.0f, r2 = 0.0f;
      const bool have = next_pair(cu, p, sp, q, me, rows(), t, xj, Rx, Ry, r2);
      if (__ballot(have) == 0ull) break;  // wave-uniform
      uint32_t w[8] = {0u, 0u, 0u, 0u, 0u, 0u, 0u, 0u};
      if (have) {
        pair_words(w, sp, p, norm, q, t, xj, Rx, Ry, r2, near);
        ++np;
      }
      const PairA a = pair_operands(w);
      add_tile(a.t0, h[0]);
      add_tile(a.t1, h[1]);
    }
  };
  pair_pass(src, pool, b, p, q, rr, me, n, cu, walk);

  // 2. head
  if (TRAIN && me < n) m.cnt[me] = (float)np;
  const float2 o = head_output<TRAIN>(h, np, m, base, n, pool);
  if (m.pairPart) {
    uint32_t tot = np;
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) tot += (uint32_t)__shfl_xor((int)tot, off, 64);
    if (lane == 0) m.pairPart[blockIdx.x] = tot;
  }
  // 3. the network's output, and the state after the relaxation and the
  // boundary collisions
  const bool live = me < n;
  if (live && m.out) reinterpret_cast<float2 *>(m.out)[me] = o;
  if (!(mode & kFwdState)) return;
  DevScene sc = s0;
  float x = 0.0f, y = 0.0f;
  if (live) {
    sc = scene_of_slot<MULTI>(b, s0, b.keys[me]);
    const float2 xi = b.x1[me];
    x = xi.x + o.x * norm[5];
    y = xi.y + o.y * norm[5];
  }
  collide_wave<MULTI>(b, p, sc, x, y, live);                                   // demo4.cpp:411-444
  if (live) {
    if (mode & kFwdPressure) {
      const float2 d = b.dens[me];
      b.pres[me] = make_float2(p.k * (d.x - p.rho0), p.kn * d.y);              // sph.h:478-481
    }
    const float2 pv = b.prev[me];
    b.x0[me] = make_float2(x, y);
    b.v[me] = make_float2((x - pv.x) * p.invDt, (y - pv.y) * p.invDt);         // demo4.cpp:446-450
  }
}

// ---------------------------------------------------------------------------
// Backward
// ---------------------------------------------------------------------------
// Head backward and the gradients of W2..W4 and the biases, on the matrix core.
// Wave q takes the 16-particle blocks q, q + parts, ... and everything stays in
// the C layout (lane = hidden column, registers 0 .. 7 = the block's rows): dO
// and dG = (dO W4) . [G > 0] (FP32); dM = dG W3 and dH = dM W2 as K = 16 BF16
// MFMAs, their A operands through LDS (rows 16 .. 31 of those tiles repeat the
// block and their results are not used); dW3 += dG^T M, dW2 += dM^T H, dW4 +=
// dO^T G with K = the 16 particles, whose operands are a lane's registers after
// one exchange between the wave's halves (k_order).  The wave's sums stay in
// registers and are written once, as partial q; only dH is written per
// particle, for the pair backward.  Partials and the order of every sum depend
// on n alone, so training reproduces its results bit for bit.
// Bound by memory: 512 bytes of activations read and 256 of dH written per
// particle, the next block's loads in flight.  Storing dG and dM and reading
// them again in three outer-product kernels moved 2.5 KB per particle (327,680
// particles: head 74 us + products 132 us, now 68 us, 4.7 TB/s with the
// partials).  One wave per SIMD: 160 accumulator registers and two blocks'
// values (bounded to 256 registers for two waves it spills, 238 us); the
// weights come from LDS.
constexpr int kHeadWaves = 4;
constexpr int kGradParts = 2048;
constexpr int kHeadRows = 16;                    // particles per block
constexpr int kHeadPart = kNumWeights - kOffW2;  // a partial: the gradient from kOffW2 on
constexpr int kWtStride = kHid + 8;  // 144 bytes: 16-byte reads of 32 rows fall into different banks

__device__ __forceinline__ bf16x8 as_bf8(uint4 w) { return bf8(w.x, w.y, w.z, w.w); }
__device__ __forceinline__ bf16x8 pack_rows(const float (&z)[8]) {
  return bf8(pack2(z[0], z[1]), pack2(z[2], z[3]), pack2(z[4], z[5]), pack2(z[6], z[7]));
}
__device__ __forceinline__ void k_order8(float (&z)[8]) {
#pragma unroll
  for (int t = 0; t < 4; ++t) {
    const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(z[t]), __float_as_uint(z[4 + t]), false, false);
    z[t] = __uint_as_float(r[0]);
    z[4 + t] = __uint_as_float(r[1]);
  }
}

__global__ __launch_bounds__(kHeadWaves * 64, 1) void k_sur_back_head(int n, SurrogateBufs m, float invN, int parts) {
  __shared__ __align__(16) uint16_t tb[kHeadWaves][kHeadRows][kHbStride];  // dG, then dM, of a block (A operands)
  __shared__ float4 shD[kHeadWaves][kHeadRows];              // the rows' dO and pair counts
  __shared__ __align__(16) uint16_t wt[2][kHid][kWtStride];  // W3, W2 transposed (B operands)
  const int w = threadIdx.x >> 6, lane = threadIdx.x & 63, c = lane & 31, g = lane >> 5, row = lane & 15;
  const int blocks = (n + kHeadRows - 1) / kHeadRows;
  const float *prm = m.params;
  const float os = prm[kOffNorm + 5];
  const float wa0 = prm[kOffW4 + c], wa1 = prm[kOffW4 + 32 + c];
  const float wb0 = prm[kOffW4 + kHid + c], wb1 = prm[kOffW4 + kHid + 32 + c];
  for (int e = (int)threadIdx.x; e < kHid * kHid / 8; e += kHeadWaves * 64) {
    const int r = e / (kHid / 8), k = 8 * (e % (kHid / 8));
    *reinterpret_cast<uint4 *>(&wt[0][r][k]) = reinterpret_cast<const uint4 *>(m.w3t)[e];
    *reinterpret_cast<uint4 *>(&wt[1][r][k]) = reinterpret_cast<const uint4 *>(m.w2t)[e];
  }
  __syncthreads();
  const int first = (int)blockIdx.x * kHeadWaves + w;
  if (first >= parts) return;  // whole wave, after the last workgroup barrier
  floatx16 a3[2][2], a2[2][2], a4[2];  // dW3, dW2 [row half][column half]; dW4: rows 0, 1
#pragma unroll
  for (int y = 0; y < 2; ++y) {
    a4[y] = zero16();
#pragma unroll
    for (int x = 0; x < 2; ++x) a3[x][y] = zero16(), a2[x][y] = zero16();
  }
  float b3[2] = {0.0f, 0.0f}, b2[2] = {0.0f, 0.0f}, b4[2] = {0.0f, 0.0f}, err = 0.0f, ref = 0.0f;
  struct Block {
    uint4 h[2], m[2];
    float4 g[4];
    float2 o, t;
    float cnt;
  };
  auto load = [&](int block) {  // clamped: a block past the end reads the last one, unused
    Block q;
    const int b = min(block, blocks - 1), s = b & 1, i = min(b * kHeadRows + row, n - 1);
    const uint4 *act = m.act + (size_t)(b >> 1) * kActWords + lane;
#pragma unroll
    for (int k = 0; k < 4; ++k) q.g[k] = reinterpret_cast<const float4 *>(act)[(8 + 4 * s + k) * 64];
#pragma unroll
    for (int y = 0; y < 2; ++y) q.m[y] = act[(4 + 2 * y + s) * 64], q.h[y] = act[(2 * y + s) * 64];
    q.o = reinterpret_cast<const float2 *>(m.out)[i];
    q.t = m.target[i];
    q.cnt = m.cnt[i];
    return q;
  };
  // LDS hand-overs within the wave
  auto wave_sync = [] {
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_wave_barrier();
  };
  // the rows in tb times the transposed weights
  auto times_weights = [&](int which, float (&lo)[8], float (&hi)[8]) {
    wave_sync();
    floatx16 zlo = zero16(), zhi = zero16();
#pragma unroll
    for (int s = 0; s < 4; ++s) {
      const bf16x8 a = lds_bf8(&tb[w][row][16 * s + 8 * g]);
      zlo = mfma16(a, as_bf8(*reinterpret_cast<const uint4 *>(&wt[which][c][16 * s + 8 * g])), zlo);
      zhi = mfma16(a, as_bf8(*reinterpret_cast<const uint4 *>(&wt[which][32 + c][16 * s + 8 * g])), zhi);
    }
    wave_sync();  // the operands have been read
#pragma unroll
    for (int k = 0; k < 8; ++k) lo[k] = zlo[k], hi[k] = zhi[k];
  };
  Block cur = load(first);
  for (int b = first; b < blocks; b += parts) {
    const Block nxt = load(b + parts);
    const int i = b * kHeadRows + row;
    float d0 = 0.0f, d1 = 0.0f;
    if (i < n) {
      const float t0 = cur.t.x / os, t1 = cur.t.y / os;
      const float e0 = cur.o.x - t0, e1 = cur.o.y - t1;
      d0 = 2.0f * invN * e0;
      d1 = 2.0f * invN * e1;
      if (lane < kHeadRows) {
        err += e0 * e0 + e1 * e1;
        ref += t0 * t0 + t1 * t1;
      }
    }
    if (lane < kHeadRows) shD[w][row] = make_float4(d0, d1, i < n ? cur.cnt : 0.0f, 0.0f);
    wave_sync();
    float lo[8], hi[8];  // dG, then dM, then dH
    {
      float glo[8], ghi[8];
#pragma unroll
      for (int k = 0; k < 8; ++k) {
        const float4 q = cur.g[k >> 1], d = shD[w][c_row(k, g)];
        glo[k] = (k & 1) ? q.z : q.x;
        ghi[k] = (k & 1) ? q.w : q.y;
        const float x0 = __builtin_fmaf(wa0, d.x, wb0 * d.y), x1 = __builtin_fmaf(wa1, d.x, wb1 * d.y);
        lo[k] = glo[k] > 0.0f ? x0 : 0.0f;
        hi[k] = ghi[k] > 0.0f ? x1 : 0.0f;
        tb[w][c_row(k, g)][c] = f2bf(lo[k]);
        tb[w][c_row(k, g)][32 + c] = f2bf(hi[k]);
      }
      k_order8(lo), k_order8(hi), k_order8(glo), k_order8(ghi);
      float od[8];  // dO, component c of the lane's rows (lanes c < 2, else 0)
#pragma unroll
      for (int u = 0; u < 8; ++u) {
        const float4 d = shD[w][8 * g + u];
        od[u] = c == 0 ? d.x : (c == 1 ? d.y : 0.0f);
        b4[0] = b4[0] + d.x;
        b4[1] = b4[1] + d.y;
        b3[0] = b3[0] + lo[u];
        b3[1] = b3[1] + hi[u];
      }
      const bf16x8 xo = pack_rows(od), x0 = pack_rows(lo), x1 = pack_rows(hi);
      a4[0] = mfma16(xo, pack_rows(glo), a4[0]);
      a4[1] = mfma16(xo, pack_rows(ghi), a4[1]);
#pragma unroll
      for (int y = 0; y < 2; ++y) {
        a3[0][y] = mfma16(x0, as_bf8(cur.m[y]), a3[0][y]);
        a3[1][y] = mfma16(x1, as_bf8(cur.m[y]), a3[1][y]);
      }
    }
    times_weights(0, lo, hi);  // dM
#pragma unroll
    for (int k = 0; k < 8; ++k) {
      tb[w][c_row(k, g)][c] = f2bf(lo[k]);
      tb[w][c_row(k, g)][32 + c] = f2bf(hi[k]);
    }
    k_order8(lo), k_order8(hi);
#pragma unroll
    for (int u = 0; u < 8; ++u) {
      const float nc = shD[w][8 * g + u].z;
      b2[0] = __builtin_fmaf(lo[u], nc, b2[0]);
      b2[1] = __builtin_fmaf(hi[u], nc, b2[1]);
    }
    const bf16x8 z0 = pack_rows(lo), z1 = pack_rows(hi);
#pragma unroll
    for (int y = 0; y < 2; ++y) {
      a2[0][y] = mfma16(z0, as_bf8(cur.h[y]), a2[0][y]);
      a2[1][y] = mfma16(z1, as_bf8(cur.h[y]), a2[1][y]);
    }
    times_weights(1, lo, hi);  // dH
    float4 *dh = m.dH + (size_t)(b >> 1) * kGradWords + (b & 1) * 4 * 64 + lane;
#pragma unroll
    for (int q = 0; q < 4; ++q) dh[q * 64] = make_float4(lo[2 * q], hi[2 * q], lo[2 * q + 1], hi[2 * q + 1]);
    wave_sync();  // dO has been read
    cur = nxt;
  }
  for (int off = 8; off > 0; off >>= 1) {
    err += __shfl_xor(err, off, 64);
    ref += __shfl_xor(ref, off, 64);
  }
  if (lane == 0) {
    m.lossPart[2 * first] = err;
    m.lossPart[2 * first + 1] = ref;
  }
  float *out = m.part + (size_t)first * kHeadPart - kOffW2;
#pragma unroll
  for (int y = 0; y < 2; ++y) {
#pragma unroll
    for (int x = 0; x < 2; ++x)
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const int at = (32 * x + c_row(r, g)) * kHid + 32 * y + c;
        out[kOffW3 + at] = a3[x][y][r];
        out[kOffW2 + at] = a2[x][y][r];
      }
    const float s3 = b3[y] + __shfl_xor(b3[y], 32, 64), s2 = b2[y] + __shfl_xor(b2[y], 32, 64);
    const float s4 = b4[y] + __shfl_xor(b4[y], 32, 64);
    if (g == 0) {
      out[kOffW4 + 32 * y + c] = a4[y][0];
      out[kOffW4 + kHid + 32 * y + c] = a4[y][1];
      out[kOffB3 + 32 * y + c] = s3;
      out[kOffB2 + 32 * y + c] = s2;
      if (c == 0) out[kOffB4 + y] = s4;
    }
  }
}

// Sums the partials into the gradient (the first kOffW2 entries from the pair
// backward's rows, the others from the head's), the losses, and with adam.t >
// 0 one Adam step (Kingma & Ba 2015) on the FP32 master weights and their BF16
// copies, in one launch.  A workgroup takes 64 columns: its wave u adds rows u,
// u + 8, ... one after another, 32 loads in flight, and the eight sums are
// added in pairs (rows past the last multiple of 8 all go to the first), a
// fixed order that no split changes: 86 MB in 22 us at 2,048 rows.  One thread
// per column, with all eight sums, left 17 workgroups walking the rows: 77 us
// for each of four products.  The last workgroup reduces the losses: loss[0] = mean squared error, loss[1] =
// sum |e|^2 / sum |target/os|^2.
constexpr int kUpdateWaves = 8, kUpdateBlock = 64 * kUpdateWaves;
static_assert(kOffW2 % 64 == 0, "a workgroup's columns come from one set of partials");
__global__ __launch_bounds__(kUpdateBlock) void k_grad_update(const float *pairPart, int pairRows,
                                                              const float *headPart, int headRows, float *grad,
                                                              const float *lossPart, int lossRows, float invN,
                                                              float *loss, AdamStep adam, float c1, float c2) {
  __shared__ float red[kUpdateWaves][64];
  const int w = threadIdx.x >> 6, lane = threadIdx.x & 63;
  constexpr int kU = 32;
  if (blockIdx.x == gridDim.x - 1) {
    float e = 0.0f, r = 0.0f;
    for (int q = (int)threadIdx.x; q < lossRows; q += kUpdateBlock) e += lossPart[2 * q], r += lossPart[2 * q + 1];
    for (int off = 32; off > 0; off >>= 1) {
      e += __shfl_xor(e, off, 64);
      r += __shfl_xor(r, off, 64);
    }
    if (lane == 0) red[w][0] = e, red[w][1] = r;
    __syncthreads();
    if (threadIdx.x == 0) {
      for (int q = 1; q < kUpdateWaves; ++q) e += red[q][0], r += red[q][1];
      loss[0] = e * invN;
      loss[1] = r > 0.0f ? e / r : 0.0f;
    }
    return;
  }
  const int col = (int)blockIdx.x * 64 + lane, at = min(col, kNumWeights - 1);
  const bool pair = (int)blockIdx.x * 64 < kOffW2;  // uniform
  const float *src = pair ? pairPart + at : headPart + (at - kOffW2);
  const int rows = pair ? pairRows : headRows, width = pair ? kOffW2 : kHeadPart, whole = rows & ~7;
  float s = 0.0f;
  int q = w;
  for (; q + (kU - 1) * kUpdateWaves < whole; q += kU * kUpdateWaves) {
    float v[kU];
#pragma unroll
    for (int u = 0; u < kU; ++u) v[u] = src[(size_t)(q + u * kUpdateWaves) * width];
#pragma unroll
    for (int u = 0; u < kU; ++u) s += v[u];
  }
  for (; q < whole; q += kUpdateWaves) s += src[(size_t)q * width];
  if (w == 0)
    for (q = whole; q < rows; ++q) s += src[(size_t)q * width];
  red[w][lane] = s;
  __syncthreads();
  if (w != 0 || col >= kNumWeights) return;
  s = ((red[0][lane] + red[1][lane]) + (red[2][lane] + red[3][lane])) +
      ((red[4][lane] + red[5][lane]) + (red[6][lane] + red[7][lane]));
  grad[col] = s;
  if (adam.t <= 0) return;
  const float m1 = adam.b1 * adam.m[col] + (1.0f - adam.b1) * s;
  const float v1 = adam.b2 * adam.v[col] + (1.0f - adam.b2) * s * s;
  adam.m[col] = m1;
  adam.v[col] = v1;
  const float x = adam.params[col] - adam.lr * (m1 / c1) / (sqrtf(v1 / c2) + adam.eps);
  adam.params[col] = x;
  if (col < kOffW2) {
    adam.w1b[col] = f2bf(x);
  } else if (col < kOffB2) {
    const int t = col - kOffW2;
    adam.w2b[t] = f2bf(x);
    adam.w2t[(t % kHid) * kHid + t / kHid] = f2bf(x);
  } else if (col >= kOffW3 && col < kOffB3) {
    const int t = col - kOffW3;
    adam.w3b[t] = f2bf(x);
    adam.w3t[(t % kHid) * kHid + t / kHid] = f2bf(x);
  }
}

// B operand (16 rows x 32 features, 16 used) of K step st of the row tile from
// row0: K index 8g + u is row c_row(8 st + u, g).
__device__ __forceinline__ bf16x8 lds_features(const uint32_t (*fw)[kFeat / 2], int row0, int st) {
  const int c = threadIdx.x & 31, g = (threadIdx.x >> 5) & 1;
  uint32_t w[4];
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    uint32_t v[2];
#pragma unroll
    for (int e = 0; e < 2; ++e) {
      const uint32_t word = fw[row0 + c_row(8 * st + 2 * q + e, g)][(c & 15) >> 1];
      v[e] = c < kFeat ? ((c & 1) ? word >> 16 : word & 0xffffu) : 0u;
    }
    w[q] = v[0] | (v[1] << 16);
  }
  return bf8(w[0], w[1], w[2], w[3]);
}

// dW1 = sum_i sum_j (dH_i . [z_ij > 0]) f_ij^T, with the pair walk of the
// forward pass.  For row tile t the pair layer's pre-activations (C layout:
// lane = hidden unit, register r = tile row c_row(r, g)), masked and scaled by
// the rows' dH, are the A operand (hidden x 16 rows) of K step s (registers
// 8s .. 8s + 7); the same rows' features are the B operand (16 rows x 32
// features, 16 used): the features times the identity, on the matrix core, have
// the pre-activations' layout, so they need no transposition through LDS (by 16
// words read per tile and lane and taken apart, a 327,680-particle launch took
// 135 us instead of 63).  Each wave accumulates over its particles and writes
// one 64 x 16 partial.
// The product passes a row on only if all its features are finite: a NaN or an
// infinity times the identity's zeros makes the whole row NaN.  The 16 unused
// columns, zero otherwise, show it in the sums, and such a wave starts again
// with the features through LDS, each of which reaches its own column alone.
template <bool MULTI>
__global__ __launch_bounds__(64, 2) void k_sur_back_pairs(Buffers b, DevParams p, DevScene s0, int n, SurrogateBufs m,
                                                          float *pairPart) {
  __shared__ __align__(16) unsigned char pool[kStageBytes];
  __shared__ uint32_t fw[kWaveRows][kFeat / 2];  // the pairs' features, when they are not finite
  const int lane = threadIdx.x, c = lane & 31, g = lane >> 5;
  const float *norm = m.params + kOffNorm;
  const W1Operands w1 = load_w1(m.w1b);
  const bf16x8 unit = identity16(0);
  floatx16 glo, ghi;
  bool exact = false;  // wave-uniform
again:
  glo = zero16(), ghi = zero16();
  for (int base = (int)blockIdx.x * kWaveRows; base < n; base += (int)gridDim.x * kWaveRows) {
    const int me = base + lane;
    __syncthreads();  // the previous group's tile is no longer read
    const PartRaw raw = part_raw(b, min(me, n - 1));  // a lane past n reads the last particle, unused
    TilePlan plan;
    DevScene sc;
    int cx, cy;
    RowRange rr[3];
    open_block<MULTI, kTileCap, kWaveRows>(b, s0, b.startNext, base, n, raw.key, sc, plan, cx, cy, rr);
    const PairSrc src = stage_pairs(b, p, norm, plan, pool);
    // dH of the rows this lane's accumulator registers hold (the second tile
    // may lie past the last particle: its lanes have no pairs)
    floatx16 d00, d01, d10, d11;  // tile, hidden half
    const float4 *dh0 = m.dH + (size_t)(base / kSurRows) * kGradWords + lane;
    const float4 *dh1 = base + kSurRows < n ? dh0 + kGradWords : dh0;
#pragma unroll
    for (int k = 0; k < 8; ++k) {
      const float4 u = dh0[k * 64], v = dh1[k * 64];
      d00[2 * k] = u.x, d01[2 * k] = u.y, d00[2 * k + 1] = u.z, d01[2 * k + 1] = u.w;
      d10[2 * k] = v.x, d11[2 * k] = v.y, d10[2 * k + 1] = v.z, d11[2 * k + 1] = v.w;
    }
    const PartInfo q = part_info(p, norm, raw);
    const bool near = wave_near(p, q.xi);
    Cursor cu{0u, 0u, 0u, 0, me >= n, 0u, 0u, 0u, 0u, 0u, 0u, rr[0], rr[1], rr[2]};
    auto masked = [&](const floatx16 &z, const floatx16 &d, int st) {
      float v[8];
#pragma unroll
      for (int u = 0; u < 8; ++u) v[u] = z[8 * st + u] > 0.0f ? d[8 * st + u] : 0.0f;
      return pack_rows(v);
    };
    auto add_tile = [&](int t, bf16x8 a, const floatx16 &dlo, const floatx16 &dhi, auto viaLds) {
      floatx16 zlo, zhi;
      pair_layer(a, w1, zlo, zhi);
      const floatx16 f = mfma16(a, unit, zero16());
#pragma unroll
      for (int st = 0; st < 2; ++st) {
        const int r = 8 * st;
        const bf16x8 bf = viaLds() ? lds_features(fw, 32 * t, st)
                                   : bf8(pack2(f[r], f[r + 1]), pack2(f[r + 2], f[r + 3]), pack2(f[r + 4], f[r + 5]),
                                         pack2(f[r + 6], f[r + 7]));
        glo = mfma16(masked(zlo, dlo, st), bf, glo);
        ghi = mfma16(masked(zhi, dhi, st), bf, ghi);
      }
    };
    auto pairs = [&](const PairSrc &sp, auto rows, auto viaLds) {
      for (;;) {
        uint32_t t = 0;
        float2 xj = make_float2(0.0f, 0.0f);
        float Rx = 0.0f, Ry = 0.0f, r2 = 0.0f;
        const bool have = next_pair(cu, p, sp, q, me, rows(), t, xj, Rx, Ry, r2);
        if (__ballot(have) == 0ull) break;  // wave-uniform
        uint32_t w[8] = {0u, 0u, 0u, 0u, 0u, 0u, 0u, 0u};
        if (have) pair_words(w, sp, p, norm, q, t, xj, Rx, Ry, r2, near);
        if (viaLds()) {
          __syncthreads();  // the last iteration's features have been read
#pragma unroll
          for (int k = 0; k < kFeat / 2; ++k) fw[lane][k] = w[k];
          __syncthreads();
        }
        const PairA a = pair_operands(w);
        add_tile(0, a.t0, d00, d01, viaLds);
        add_tile(1, a.t1, d10, d11, viaLds);
      }
    };
    if (exact)  // one copy of the walk for all
      pairs(slot_src(src, b), std::false_type(), std::true_type());
    else
      pair_pass(src, pool, b, p, q, rr, me, n, cu,
                [&](const PairSrc &sp, auto rows) { pairs(sp, rows, std::false_type()); });
  }
  if (!exact) {
    float unused = 0.0f;
#pragma unroll
    for (int k = 0; k < 16; ++k) unused += glo[k] + ghi[k];
    if (__ballot(c >= kFeat && unused != 0.0f) != 0ull) {  // NaN
      exact = true;
      goto again;
    }
  }
  float *out = pairPart + (size_t)blockIdx.x * (kHid * kFeat);
  if (c < kFeat) {
#pragma unroll
    for (int k = 0; k < 16; ++k) {
      const int hid = c_row(k, g);
      out[hid * kFeat + c] = glo[k];
      out[(32 + hid) * kFeat + c] = ghi[k];
    }
  }
}

// BF16 copies of W1..W3 and the transposes of W2, W3 (w2t[n][k] = W2[k][n]) for
// the backward pass's B operands.
__global__ __launch_bounds__(kBlock) void k_bf16_weights(const float *params, uint16_t *w1b, uint16_t *w2b,
                                                         uint16_t *w3b, uint16_t *w2t, uint16_t *w3t) {
  const int t = (int)(blockIdx.x * kBlock + threadIdx.x);
  if (t < kHid * kFeat) w1b[t] = f2bf(params[kOffW1 + t]);
  if (t < kHid * kHid) {
    w2b[t] = f2bf(params[kOffW2 + t]);
    w3b[t] = f2bf(params[kOffW3 + t]);
    const int r = t / kHid, k = t % kHid;
    w2t[k * kHid + r] = f2bf(params[kOffW2 + t]);
    w3t[k * kHid + r] = f2bf(params[kOffW3 + t]);
  }
}

// FP64 sums for the density check: sum |a.x - b.x| and sum b.x.
constexpr int kErrItems = 8;
__global__ __launch_bounds__(kBlock) void k_dens_err_partial(const float2 *a, const float2 *bb, int n,
                                                             double *partials) {
  __shared__ double red[2][kBlock / 64];
  double s0 = 0.0, s1 = 0.0;
  const int base = (int)blockIdx.x * kBlock * kErrItems;
  for (int k = 0; k < kErrItems; ++k) {
    const int i = base + k * kBlock + (int)threadIdx.x;
    if (i >= n) break;
    const double x = a[i].x, y = bb[i].x;
    s0 += fabs(x - y);
    s1 += y;
  }
  for (int off = 32; off > 0; off >>= 1) {
    s0 += __shfl_xor(s0, off, 64);
    s1 += __shfl_xor(s1, off, 64);
  }
  if ((threadIdx.x & 63) == 0) {
    red[0][threadIdx.x >> 6] = s0;
    red[1][threadIdx.x >> 6] = s1;
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    double t0 = 0.0, t1 = 0.0;
    for (int w = 0; w < kBlock / 64; ++w) t0 += red[0][w], t1 += red[1][w];
    partials[2 * blockIdx.x] = t0;
    partials[2 * blockIdx.x + 1] = t1;
  }
}

// Per-scene sums of |a.x - b.x| and b.x into out[2 s], out[2 s + 1] (zeroed
// beforehand).  A scene's particles occupy consecutive slots.  A workgroup
// covers kErrItems * kBlock consecutive slots; when they all belong to one
// scene (the first and last slot share it) it reduces and adds once, else each
// wave adds per 64-slot group (once when the group shares a scene, per lane
// otherwise).
__global__ __launch_bounds__(kBlock) void k_dens_err_scenes(const float2 *a, const float2 *bb, const uint32_t *keys,
                                                            const uint32_t *sceneBase, int nScenes, int n,
                                                            double *out) {
  __shared__ double red[2][kBlock / 64];
  const int base = (int)blockIdx.x * kBlock * kErrItems;
  const int last = min(n, base + kBlock * kErrItems) - 1;
  const int s0 = scene_of_key(sceneBase, nScenes, keys[base]);
  const bool one = scene_of_key(sceneBase, nScenes, keys[last]) == s0;
  double e = 0.0, r = 0.0;
  for (int k = 0; k < kErrItems; ++k) {
    const int i = base + k * kBlock + (int)threadIdx.x;
    const bool valid = i < n;
    double ei = 0.0, ri = 0.0;
    if (valid) {
      ei = fabs((double)a[i].x - (double)bb[i].x);
      ri = (double)bb[i].x;
    }
    if (one) {
      e += ei;
      r += ri;
      continue;
    }
    const int sc = valid ? scene_of_key(sceneBase, nScenes, keys[i]) : -1;
    const int first = __shfl(sc, 0, 64);
    if (__ballot(valid && sc != first) == 0ull) {
      for (int off = 32; off > 0; off >>= 1) {
        ei += __shfl_xor(ei, off, 64);
        ri += __shfl_xor(ri, off, 64);
      }
      if ((threadIdx.x & 63) == 0 && first >= 0) {
        atomicAdd(&out[2 * first], ei);
        atomicAdd(&out[2 * first + 1], ri);
      }
    } else if (valid) {
      atomicAdd(&out[2 * sc], ei);
      atomicAdd(&out[2 * sc + 1], ri);
    }
  }
  if (!one) return;  // uniform across the workgroup
  for (int off = 32; off > 0; off >>= 1) {
    e += __shfl_xor(e, off, 64);
    r += __shfl_xor(r, off, 64);
  }
  if ((threadIdx.x & 63) == 0) red[0][threadIdx.x >> 6] = e, red[1][threadIdx.x >> 6] = r;
  __syncthreads();
  if (threadIdx.x == 0) {
    double t0 = 0.0, t1 = 0.0;
    for (int w = 0; w < kBlock / 64; ++w) t0 += red[0][w], t1 += red[1][w];
    atomicAdd(&out[2 * s0], t0);
    atomicAdd(&out[2 * s0 + 1], t1);
  }
}

__global__ __launch_bounds__(kBlock) void k_fill_f64(double *p, int count) {
  const int i = (int)(blockIdx.x * kBlock + threadIdx.x);
  if (i < count) p[i] = 0.0;
}

// Sums the partials in a fixed order: thread t adds partials t, t + 1024, ...,
// then a tree over the threads.
__global__ __launch_bounds__(1024) void k_dens_err_final(const double *partials, int nb, double *out) {
  __shared__ double red[2][1024 / 64];
  double t0 = 0.0, t1 = 0.0;
  for (int k = (int)threadIdx.x; k < nb; k += 1024) t0 += partials[2 * k], t1 += partials[2 * k + 1];
  for (int off = 32; off > 0; off >>= 1) {
    t0 += __shfl_xor(t0, off, 64);
    t1 += __shfl_xor(t1, off, 64);
  }
  if ((threadIdx.x & 63) == 0) red[0][threadIdx.x >> 6] = t0, red[1][threadIdx.x >> 6] = t1;
  __syncthreads();
  if (threadIdx.x == 0) {
    double s0 = 0.0, s1 = 0.0;
    for (int w = 0; w < 1024 / 64; ++w) s0 += red[0][w], s1 += red[1][w];
    out[0] = s0;
    out[1] = s1;
  }
}

// MFMA layout self-test (see the file header).
__global__ __launch_bounds__(64) void k_mfma_probe(const float *A, const float *B, float *C) {
  const int lane = threadIdx.x & 63, c = lane & 31, g = lane >> 5;
  bf16x4 a, bb;
#pragma unroll
  for (int t = 0; t < 4; ++t) {
    a[t] = (short)f2bf(A[c * 8 + 4 * g + t]);
    bb[t] = (short)f2bf(B[(4 * g + t) * 32 + c]);
  }
  const floatx16 r = mfma(a, bb, zero16());
#pragma unroll
  for (int k = 0; k < 16; ++k) C[c_row(k, g) * 32 + c] = r[k];
}

// K = 16 layout self-test: C (32 x 32) = A (32 x 16) B (16 x 32).
__global__ __launch_bounds__(64) void k_mfma16_probe(const float *A, const float *B, float *C) {
  const int lane = threadIdx.x & 63, c = lane & 31, g = lane >> 5;
  float a[8], bb[8];
#pragma unroll
  for (int t = 0; t < 8; ++t) {
    a[t] = A[c * 16 + 8 * g + t];
    bb[t] = B[(8 * g + t) * 32 + c];
  }
  const floatx16 r = mfma16(bf8(pack2(a[0], a[1]), pack2(a[2], a[3]), pack2(a[4], a[5]), pack2(a[6], a[7])),
                            bf8(pack2(bb[0], bb[1]), pack2(bb[2], bb[3]), pack2(bb[4], bb[5]), pack2(bb[6], bb[7])),
                            zero16());
#pragma unroll
  for (int k = 0; k < 16; ++k) C[c_row(k, g) * 32 + c] = r[k];
}

// ---------------------------------------------------------------------------
// Launchers
// ---------------------------------------------------------------------------
static unsigned waves_for(int n) { return (unsigned)((n + kWaveRows - 1) / kWaveRows); }
static unsigned back_pair_waves(int n) { return std::min(waves_for(n), 4096u); }
// partial gradients of the head's backward pass: one per 16 particles, at most kGradParts
static int head_parts(int n) { return std::max(1, std::min((n + kHeadRows - 1) / kHeadRows, kGradParts)); }

// the head's partials, then the pair backward's
size_t surrogate_part_floats(int n) {
  return (size_t)head_parts(n) * kHeadPart + std::max<size_t>(back_pair_waves(n), 1) * kHid * kFeat;
}

int surrogate_head_waves(int n) { return head_parts(n); }
int surrogate_forward_waves(int n) { return std::max(1, (int)waves_for(n)); }

void launch_surrogate_forward(const Buffers &b, const DevParams &p, const DevScene &s0, int n,
                              const SurrogateBufs &m, int mode, hipStream_t s) {
  if (n <= 0) return;
  const dim3 grid(waves_for(n));
  const bool train = (mode & kFwdTrain) != 0;
  if (b.nScenes > 1)
    hipLaunchKernelGGL((train ? k_sur_forward<true, true> : k_sur_forward<true, false>), grid, dim3(64), 0, s, b, p,
                       s0, n, m, mode);
  else
    hipLaunchKernelGGL((train ? k_sur_forward<false, true> : k_sur_forward<false, false>), grid, dim3(64), 0, s, b, p,
                       s0, n, m, mode);
}

void launch_surrogate_backward(const Buffers &b, const DevParams &p, const DevScene &s0, int n,
                               const SurrogateBufs &m, const AdamStep *adam, hipStream_t s) {
  if (n <= 0) return;
  const float invN = 1.0f / (float)n;
  const int parts = head_parts(n);
  const unsigned waves = back_pair_waves(n);
  float *pairPart = m.part + (size_t)parts * kHeadPart;
  hipLaunchKernelGGL(k_sur_back_head, dim3((parts + kHeadWaves - 1) / kHeadWaves), dim3(kHeadWaves * 64), 0, s, n,
                     m, invN, parts);
  if (b.nScenes > 1)
    hipLaunchKernelGGL(k_sur_back_pairs<true>, dim3(waves), dim3(64), 0, s, b, p, s0, n, m, pairPart);
  else
    hipLaunchKernelGGL(k_sur_back_pairs<false>, dim3(waves), dim3(64), 0, s, b, p, s0, n, m, pairPart);
  AdamStep a{};
  float c1 = 1.0f, c2 = 1.0f;
  if (adam) {
    a = *adam;
    c1 = 1.0f - std::pow(a.b1, (float)a.t), c2 = 1.0f - std::pow(a.b2, (float)a.t);
  }
  hipLaunchKernelGGL(k_grad_update, dim3((kNumWeights + 63) / 64 + 1), dim3(kUpdateBlock), 0, s,
                     (const float *)pairPart, (int)waves, (const float *)m.part, parts, m.grad,
                     (const float *)m.lossPart, parts, invN, m.loss + 2 * (size_t)m.lossIndex, a, c1,
                     c2);
}

void launch_bf16_weights(const float *params, uint16_t *w1b, uint16_t *w2b, uint16_t *w3b, uint16_t *w2t,
                         uint16_t *w3t, hipStream_t s) {
  hipLaunchKernelGGL(k_bf16_weights, dim3((kHid * kHid + kBlock - 1) / kBlock), dim3(kBlock), 0, s, params, w1b, w2b,
                     w3b, w2t, w3t);
}

void launch_density_error(const float2 *a, const float2 *bb, int n, double *partials, double *out, hipStream_t s) {
  const int nb = std::max(1, (n + kBlock * kErrItems - 1) / (kBlock * kErrItems));
  if (n > 0) hipLaunchKernelGGL(k_dens_err_partial, dim3(nb), dim3(kBlock), 0, s, a, bb, n, partials);
  hipLaunchKernelGGL(k_dens_err_final, dim3(1), dim3(1024), 0, s, (const double *)partials, n > 0 ? nb : 0, out);
}

void launch_density_error_scenes(const float2 *a, const float2 *bb, const uint32_t *keys, const uint32_t *sceneBase,
                                 int nScenes, int n, double *out, hipStream_t s) {
  hipLaunchKernelGGL(k_fill_f64, dim3((2 * nScenes + kBlock - 1) / kBlock), dim3(kBlock), 0, s, out, 2 * nScenes);
  if (n > 0)
    hipLaunchKernelGGL(k_dens_err_scenes, dim3((n + kBlock * kErrItems - 1) / (kBlock * kErrItems)), dim3(kBlock), 0,
                       s, a, bb, keys, sceneBase, nScenes, n, out);
}

void launch_mfma_probe(const float *a, const float *b, float *c, hipStream_t s) {
  hipLaunchKernelGGL(k_mfma_probe, dim3(1), dim3(64), 0, s, a, b, c);
}

void launch_mfma16_probe(const float *a, const float *b, float *c, hipStream_t s) {
  hipLaunchKernelGGL(k_mfma16_probe, dim3(1), dim3(64), 0, s, a, b, c);
}

}  // namespace nbs
