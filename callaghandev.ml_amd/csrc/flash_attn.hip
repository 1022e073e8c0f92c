// Fused flash-style fp32 attention forward for gfx950 (ScaledDotProductAttention
// and MultiHeadAttentionForward of the reference, AccelerationCPU.cs:1647-1956).
//
// One 256-thread workgroup owns 128 queries of one (sequence, head); each of
// its four waves owns 32 queries for the whole key loop.  All products run on
// the bf16 matrix cores from three bf16 pieces per fp32 value (common.h): K and V
// are split on their way into LDS, Q once into registers, the probabilities in
// registers.  Per key tile of BN keys (double-buffered LDS, next tile prefetched
// into registers while the current one is consumed):
//
//   S^T = K Q^T     A = K rows from LDS, B = the wave's Q pieces held in
//                   registers for the whole loop.  Computing S transposed puts
//                   one query per lane (lane % 32) and 16 keys per lane in the
//                   accumulator, so the softmax row reductions are in-lane plus
//                   one swap between the two half-waves.
//   online softmax  running max / sum per query in the exp2 domain
//                   (scale * log2 e folded into Q), masked keys -inf.
//   O^T += V^T P^T  accumulators 8 s .. 8 s + 7 of a lane hold the keys 16 s +
//                   {4 h .. 4 h + 3, 8 + 4 h .. 8 + 4 h + 3} (h = lane / 32): V is
//                   staged transposed with its keys in that order, so the
//                   probabilities are consumed in place.  V carries the split's
//                   scale (common.h), the probabilities do not (16 more VALU
//                   instructions per sub-block, 1-5% of the kernel): one below
//                   2^-110 loses at most 2^-134, where exp2 itself drops those
//                   below 2^-126.
//
// Causal: tiles entirely above the diagonal are never loaded; a wave skips
// MFMA work for its 32-key sub-blocks that lie wholly in its future; heavy
// query tiles are dispatched first.  A row whose keys are all masked ends
// with sum 0 and is written as 0 (AccelerationCPU.cs:1908-1911).
//
// What bounds it: at head dim 64 a 32 x 32 sub-block costs a wave 48 MFMAs
// (1536 cycles of the matrix pipe) and some 290 other VALU instructions, half of
// them the splits (5.96 per MFMA at 4 x 4096); at head dim 32 half the MFMAs and 280
// (11.8 per MFMA): the vector units there.  Measured on MI355X at 4 x 4096, 16 heads
// of 64: 0.69 ms (1.05 ms on the fp32 MFMA), matrix pipes 57% busy; 256 x 512, 8 heads
// of 32: 0.25 ms, 39%.  LDS bank conflicts take 11% of the active cycles at 4 x 4096.
#include <cfloat>

#include "common.h"

namespace cdml {
namespace {

constexpr int FA_THREADS = 256;
constexpr int FA_BM = 128;  // queries per workgroup (32 per wave)
constexpr float kLog2e = 1.4426950408889634f;

// Division by a launch-constant divisor d >= 1 for dividends 0 <= x < 2^31:
// x / d = (x * m) >> l with l = 31 + ceil(log2 d) and m = ceil(2^l / d) < 2^32
// (the error m * d - 2^l is below d, so x * error < 2^l for every such x).
// Block-uniform dividends keep the division on the scalar unit.
struct UDiv {
  uint32_t m;
  int l;
  static UDiv make(uint32_t d) {
    if (d == 0) d = 1;  // no launch divides by it
    int s = 0;
    while ((1ull << s) < d) ++s;
    const int l = 31 + s;
    return {(uint32_t)(((1ull << l) + d - 1) / d), l};
  }
  __device__ __forceinline__ int div(int x) const { return (int)(((uint64_t)(uint32_t)x * m) >> l); }
};

struct FlashArgs {
  const float *q, *k, *v;
  float *o;
  float *lse;  // optional [batch * heads][lq]: log2 of each row's softmax normaliser
  const uint8_t *mask;
  int ldq, ldk, ldv, ldo;
  int lq, lk, heads, hd;
  float scale_log2;
  int n_qt, n_bh, n_items;  // query tiles per sequence, (sequence, head) pairs, n_bh * n_qt
  UDiv by_bh, by_heads;     // division by n_bh and by heads
};

// Stages one tile of BN keys: K rows [k0, k0 + BN) and V transposed, of head
// column block `col0`, from global memory into registers and then, split into
// three bf16 pieces, into LDS (one plane per piece, rows of 16 values = 32
// bytes, as the GEMM's operand tiles).  The upper half of the workgroup's
// waves stages K, the lower half V, eight values per unit pair and unit.
//   K: slab s holds dims 16 s .. 16 s + 15 of every key: rows are keys, even
//      and odd ones in two clusters.  A unit is four dims of one key.
//   V: slab s holds keys 16 s .. 16 s + 15 of every dim: rows are dims, in four
//      clusters by d % 4, odd dims negated (common.h; the output undoes it).  A
//      unit is four dims of two keys; key k of a slab sits at place
//      8 (k / 4 % 2) + 4 (k / 8) + k % 4, the order the P.V product reads.
// Each thread's offsets inside a tile are fixed.  Rows past lk (the sequence
// end) are clamped to row lk - 1: their scores are masked to -inf and their
// probabilities are exactly 0.  Without VEC (head dims other than HD, unaligned
// rows) columns at or past hd read as zero.
template <int HD, int BN, bool VEC>
struct KvStage {
  static constexpr int HALF = FA_THREADS / 2;
  static constexpr int KROWB = BN / 2 * 32, VROWB = HD / 4 * 32;  // bytes of one row cluster
  static constexpr int KSLAB = 2 * KROWB + 128, VSLAB = 4 * VROWB + 256;
  static constexpr int KPLANE = HD / 16 * KSLAB, VPLANE = BN / 16 * VSLAB;
  static constexpr int BYTES = 3 * (KPLANE + VPLANE);  // K planes, then V planes
  static constexpr int VU = (HD / 4) * (BN / 2) / HALF;  // V units per thread; twice as many K units
  static constexpr int NV = 2 * VU;                      // loads of either
  static_assert(VU >= 1 && (HD / 4) * (BN / 2) % HALF == 0 && HALF / 8 % 16 == 0, "tile units");
  static __device__ __forceinline__ constexpr int kcluster(int c) { return c * (KROWB + 16); }
  static __device__ __forceinline__ constexpr int vcluster(int c) {
    return c * VROWB + (c & 1) * 16 + (c >> 1) * 128;
  }
  // What a thread's further units add to its first: K unit i is KSTEP keys
  // further down; V unit i is VG groups of four dims and whole slabs further.
  static constexpr int CH = HD / 4, KSTEP = HALF / CH;
  static __device__ __forceinline__ constexpr int vgroups(int i) { return HALF / 8 * i % CH; }
  static __device__ __forceinline__ constexpr int vslabs(int i) { return HALF / 8 * i / CH; }
  vf4 r[NV];
  uint32_t off;  // byte offset of the first load in a tile
  int col;       // its first column
  int dst;       // LDS byte offset of the first unit
  bool kside;

  __device__ __forceinline__ void init(int ldk, int ldv) {
    kside = __builtin_amdgcn_readfirstlane(threadIdx.x) >= HALF;
    const int t = threadIdx.x & (HALF - 1);
    // K: the P keys of one load instruction share a cluster
    constexpr int P = 64 / CH;
    const int c = t % CH, j = t / CH, kkey = (j & ~(2 * P - 1)) | ((j & (P - 1)) << 1) | ((j / P) & 1);
    const int sb = t & 7, g = (t >> 3) % CH, slab = (t >> 3) / CH;
    const int place = ((sb >> 1) & 1) * 4 + (sb >> 2) * 2 + (sb & 1);  // of V's key pair
    col = kside ? 4 * c : 4 * g;
    off = 4u * (uint32_t)((kside ? kkey * ldk : (16 * slab + 2 * sb) * ldv) + col);
    dst = kside ? (c >> 2) * KSLAB + kcluster(kkey & 1) + (kkey >> 1) * 32 + (c & 3) * 8
                : 3 * KPLANE + slab * VSLAB + g * 32 + place * 4;
  }

  __device__ __forceinline__ void load(const float *__restrict__ kbase, const float *__restrict__ vbase, int ldk,
                                       int ldv, int k0, int lk, int hd) {
    // wave-uniform tile base plus a 32-bit per-lane byte offset (one
    // scalar-base global load per row, no 64-bit address arithmetic)
    const int ld = kside ? ldk : ldv;
    const char *tile = reinterpret_cast<const char *>((kside ? kbase : vbase) + (size_t)k0 * ld);
    const uint32_t last = 4u * (uint32_t)min(lk - 1 - k0, BN - 1) * (uint32_t)ld;
#pragma unroll
    for (int i = 0; i < NV; ++i) {
      const int dc = kside ? 0 : 4 * vgroups(i / 2);
      const int rows = kside ? KSTEP * i : 16 * vslabs(i / 2) + (i & 1);
      const char *p = tile + min(off + 4u * (uint32_t)(rows * ld + dc), last + 4u * (uint32_t)(col + dc));
      if constexpr (VEC) {
        r[i] = *reinterpret_cast<const vf4 *>(p);
      } else {
#pragma unroll
        for (int c = 0; c < 4; ++c) r[i][c] = col + dc + c < hd ? reinterpret_cast<const float *>(p)[c] : 0.f;
      }
    }
  }

  // vscale: the split's scale of V, negative where the workgroup's outputs are
  // computed negated.
  __device__ __forceinline__ void store(char *lds, float vscale) const {
    if (kside) {
#pragma unroll
      for (int i = 0; i < NV; ++i) {
        uint32_t h0, m0, l0, h1, m1, l1;
        split_bf16x3(r[i][0], r[i][1], h0, m0, l0);
        split_bf16x3(r[i][2], r[i][3], h1, m1, l1);
        char *d = lds + dst + KSTEP / 2 * 32 * i;
        *reinterpret_cast<vu2 *>(d) = vu2{h0, h1};
        *reinterpret_cast<vu2 *>(d + KPLANE) = vu2{m0, m1};
        *reinterpret_cast<vu2 *>(d + 2 * KPLANE) = vu2{l0, l1};
      }
    } else {
#pragma unroll
      for (int i = 0; i < VU; ++i)
#pragma unroll
        for (int c = 0; c < 4; ++c) {
          uint32_t h, m, l;
          const float x = r[2 * i][c], y = r[2 * i + 1][c];
          const float f = c & 1 ? -vscale : vscale;
          split_bf16x3(x * f, y * f, h, m, l);
          char *d = lds + dst + vslabs(i) * VSLAB + vgroups(i) * 32 + vcluster(c);
          *reinterpret_cast<uint32_t *>(d) = h;
          *reinterpret_cast<uint32_t *>(d + VPLANE) = m;
          *reinterpret_cast<uint32_t *>(d + 2 * VPLANE) = l;
        }
    }
  }

  // Byte offsets of a lane's operands in a plane: dims 16 s + 8 hf + 0..7 of key
  // row0 + li (row0 a multiple of 32), and eight keys of slab s for dim 32 db + li.
  static __device__ __forceinline__ int koperand(int li, int hf) {
    return kcluster(li & 1) + (li >> 1) * 32 + hf * 16;
  }
  static __device__ __forceinline__ int voperand(int li, int hf) {
    return 3 * KPLANE + vcluster(li & 3) + (li >> 2) * 32 + hf * 16;
  }
};

// max / sum of a value over the two half-waves (lanes l and l ^ 32) with
// v_permlane32_swap: both results hold the value of lane l % 32 and of lane
// l % 32 + 32.
__device__ __forceinline__ float halves_max(float x) {
#pragma float_control(precise, off)
  auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  return __builtin_fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1]));  // scores: no signalling NaN
}
__device__ __forceinline__ float halves_sum(float x) {
  auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}

// max of three scores.  The scores come from MFMA accumulators and are
// never signalling NaNs, so the IEEE quieting that fmaxf otherwise adds to
// each operand is dropped (one v_max3_f32 instead of five instructions).
__device__ __forceinline__ float max3_scores(float a, float b, float c) {
#pragma float_control(precise, off)
  return __builtin_fmaxf(__builtin_fmaxf(a, b), c);
}

// Growth of the running max (log2 units) tolerated before the output is
// rescaled: probabilities stay <= 2^8, far from fp32 overflow.
constexpr float kRescaleThreshold = 8.0f;

// Offset of accumulator register r's key inside its 32-key sub-block for a
// lane of half-wave h: 8 * (r / 4) + 4 * h + r % 4 (the 32x32 MFMA D layout).
__device__ __forceinline__ constexpr int acc_key(int r) { return 8 * (r >> 2) + (r & 3); }

// A sub-block whose per-lane probability sum stays at or below this bound is
// accumulated without looking at its maximum: no probability exceeds it, so
// nothing overflows (the running sums stay below 2^32 times the key count).
constexpr float kFastSumLimit = 4294967296.0f;  // 2^32

// Q^T operand of a wave: the three bf16 pieces of q[qi][16 s + 8 hf + 0..7] times
// scale_log2.  Rows past lq read row lq - 1: they are computed but never stored.
// Scores start from the row's reference, so neither Q nor K takes the split's scale:
// what a component below 2^-110 loses (2^-134) reaches a score only through a
// component of 2^100 and more on the other side.  Returns whether Q holds one or
// the other (wave-uniform); such rows are recomputed on the fp32 MFMA.
template <int HD, bool VEC>
__device__ __forceinline__ bool load_q(bf16x8 (&q)[HD / 16][3], const FlashArgs &a, int b, int col0, int qi, int hf) {
  const float *qrow = a.q + ((size_t)b * a.lq + min(qi, a.lq - 1)) * a.ldq + col0;
  uint32_t most = 0, least = ~0u;  // of |x|, and of 2 |x| - 1 as integers, which leaves zeros out
#pragma unroll
  for (int s = 0; s < HD / 16; ++s) {
    float x[8];
#pragma unroll
    for (int g = 0; g < 2; ++g) {
      const int d = 16 * s + 8 * hf + 4 * g;
      if constexpr (VEC) {
        const vf4 t4 = *reinterpret_cast<const vf4 *>(qrow + d);
#pragma unroll
        for (int r = 0; r < 4; ++r) x[4 * g + r] = t4[r] * a.scale_log2;
      } else {
#pragma unroll
        for (int r = 0; r < 4; ++r) x[4 * g + r] = d + r < a.hd ? qrow[d + r] * a.scale_log2 : 0.f;
      }
    }
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      most = max(most, __float_as_uint(x[e]) & 0x7fffffffu);
      least = min(least, (__float_as_uint(x[e]) << 1) - 1u);
    }
    split_operand(x, 1.f, q[s]);
  }
  return __builtin_amdgcn_ballot_w64(most >= (100u + 127u) << 23 || least < (17u << 24) - 1u) != 0;  // 2^100, 2^-110
}

// The online softmax of one wave's 32 query rows (one per lane % 32) over
// 32-key sub-blocks.
template <int HD, int BN, bool HAS_MASK, bool VEC>
struct OnlineRows {
  typedef KvStage<HD, BN, VEC> Tile;
  static constexpr int NDB = HD / 32;     // 32-wide head-dim blocks of O^T
  static constexpr int NS = HD / 16;      // MFMA k-steps of Q.K
  floatx16 oacc[NDB], ocor[NDB];          // hh, and its corrections (common.h)
  // The reference max of this lane's query (exp2 domain) is subtracted by
  // the MFMA itself: the first step of every S^T block starts from negm,
  // -m_run in all 16 entries (0 until the first visible key sets m_run), so
  // the scores come out relative to the reference and p = exp2(score).
  floatx16 negm;
  float m_run, thr;  // thr: rescale threshold, any visible key until m_run is set
  float l_a, l_b;    // running sums over this half-wave's keys
  bool warm;         // every lane of the wave has its reference (wave-uniform)

  __device__ __forceinline__ void init() {
#pragma unroll
    for (int db = 0; db < NDB; ++db)
#pragma unroll
      for (int r = 0; r < 16; ++r) oacc[db][r] = ocor[db][r] = 0.f;
#pragma unroll
    for (int r = 0; r < 16; ++r) negm[r] = 0.f;
    m_run = -INFINITY;
    thr = -INFINITY;
    l_a = l_b = 0.f;
    warm = false;
  }

  // Sets the scores of keys this lane may not attend to -inf: keys past
  // last_vis (offset within the sub-block for this lane's half), and with
  // HAS_MASK also keys whose mask byte mrow[min(kb0 + offset, key_cap)] is 0
  // or any key when !row_ok.
  __device__ __forceinline__ void apply_mask(floatx16 &sacc, int hf, int last_vis, const uint8_t *mrow, int kb0,
                                             int key_cap, bool row_ok) const {
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      bool ok = acc_key(r) <= last_vis;
      if (HAS_MASK) {
        const int key = min(kb0 + acc_key(r) + 4 * hf, key_cap);
        ok = ok && row_ok && mrow[key] != 0;
      }
      sacc[r] = ok ? sacc[r] : -INFINITY;
    }
  }

  // O^T += V^T P^T for the sub-block whose first V slab is at vt (this lane's
  // operand of plane 0, dim block 0).
  __device__ __forceinline__ void accumulate_pv(const floatx16 &p, const char *vt) {
#pragma unroll
    for (int s = 0; s < 2; ++s) {
      float x[8];
#pragma unroll
      for (int e = 0; e < 8; ++e) x[e] = p[8 * s + e];
      bf16x8 pp[3];
      split_operand(x, 1.f, pp);
#pragma unroll
      for (int db = 0; db < NDB; ++db) {
        bf16x8 v[3];
#pragma unroll
        for (int q = 0; q < 3; ++q)
          v[q] = *reinterpret_cast<const bf16x8 *>(vt + q * Tile::VPLANE + s * Tile::VSLAB + db * 256);
#pragma unroll
        for (int q = 0; q < kSplitProducts; ++q) {
          floatx16 &c = q == kSplitMain ? oacc[db] : ocor[db];
          c = mfma32x32x16(v[kSplitA[q]], pp[kSplitB[q]], c);
        }
      }
    }
  }

  // The common sub-block once every row has its reference: probabilities and
  // their per-lane sum first, and only if some lane's sum is above 2^32 (a
  // score far above the reference) or NaN does the caller take the full path
  // (consume) on recomputed scores.  sacc is turned into probabilities in
  // place; on false the running state is unchanged and sacc is garbage.
  __device__ __forceinline__ bool try_fast(floatx16 &sacc, const char *vt, int hf, bool masked, int last_vis,
                                           const uint8_t *mrow, int kb0, int key_cap, bool row_ok) {
    if (HAS_MASK || masked) apply_mask(sacc, hf, last_vis, mrow, kb0, key_cap, row_ok);
#pragma unroll
    for (int r = 0; r < 16; ++r) sacc[r] = fast_exp2(sacc[r]);
    // pairwise sum (a tree of depth 4)
    float s8[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) s8[i] = sacc[2 * i] + sacc[2 * i + 1];
    const float ps = ((s8[0] + s8[1]) + (s8[2] + s8[3])) + ((s8[4] + s8[5]) + (s8[6] + s8[7]));
    if (__builtin_amdgcn_ballot_w64(!(ps <= kFastSumLimit))) return false;
    l_a += ps;
    accumulate_pv(sacc, vt);
    return true;
  }

  // S^T = K Q^T for the 32 keys whose operands start at kt (this lane's operand
  // of plane 0, slab 0), relative to the reference.
  __device__ __forceinline__ floatx16 scores(const char *kt, const bf16x8 (&q)[NS][3]) const {
    floatx16 sacc = negm, cor = {};
#pragma unroll
    for (int s = 0; s < NS; ++s) {
      bf16x8 k[3];
#pragma unroll
      for (int p = 0; p < 3; ++p) k[p] = *reinterpret_cast<const bf16x8 *>(kt + p * Tile::KPLANE + s * Tile::KSLAB);
#pragma unroll
      for (int i = 0; i < kSplitProducts; ++i) {
        floatx16 &c = i == kSplitMain ? sacc : cor;
        c = mfma32x32x16(k[kSplitA[i]], q[s][kSplitB[i]], c);
      }
    }
#pragma unroll
    for (int r = 0; r < 16; ++r) sacc[r] += cor[r];
    return sacc;
  }

  // Softmax of one sub-block's scores and O^T += V^T P^T.  masked
  // (wave-uniform): some key of the sub-block may be invisible (see apply_mask).
  __device__ __forceinline__ void consume(floatx16 sacc, const char *vt, int hf, bool masked, int last_vis,
                                          const uint8_t *mrow, int kb0, int key_cap, bool row_ok) {
    softmax(sacc, hf, masked, last_vis, mrow, kb0, key_cap, row_ok);
    accumulate_pv(sacc, vt);
  }

  __device__ __forceinline__ void softmax(floatx16 &sacc, int hf, bool masked, int last_vis, const uint8_t *mrow,
                                          int kb0, int key_cap, bool row_ok) {
    if (HAS_MASK || masked) apply_mask(sacc, hf, last_vis, mrow, kb0, key_cap, row_ok);
    // tile max relative to the reference (-inf: no visible key)
    // (a tree of depth 3: eight v_max3 whose inputs do not wait on each other)
    const float m0 = max3_scores(sacc[0], sacc[1], sacc[2]);
    const float m1 = max3_scores(sacc[3], sacc[4], sacc[5]);
    const float m2 = max3_scores(sacc[6], sacc[7], sacc[8]);
    const float m3 = max3_scores(sacc[9], sacc[10], sacc[11]);
    const float m4 = max3_scores(sacc[12], sacc[13], sacc[14]);
    float smax = max3_scores(max3_scores(m0, m1, m2), max3_scores(m3, m4, sacc[15]), -INFINITY);
    smax = halves_max(smax);

    // Lazy rescale: the first visible key sets the reference, later only a
    // rise of more than the threshold moves it (the scores shift with it).
    const bool need = smax > thr;
    if (__builtin_amdgcn_ballot_w64(need)) {
      const bool first = m_run == -INFINITY;
      const float shift = need ? smax : 0.f;
      const float alpha = (need && !first) ? fast_exp2(-smax) : 1.0f;  // o and l are 0 before the first key
      m_run = need ? (first ? smax : m_run + smax) : m_run;
      thr = m_run == -INFINITY ? -INFINITY : kRescaleThreshold;
      const float nref = m_run == -INFINITY ? 0.f : -m_run;
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        sacc[r] -= shift;
        negm[r] = nref;
      }
      if (__builtin_amdgcn_ballot_w64(need && !first)) {  // not at a row's first visible key
        l_a *= alpha;
        l_b *= alpha;
#pragma unroll
        for (int db = 0; db < NDB; ++db)
#pragma unroll
          for (int r = 0; r < 16; ++r) {
            oacc[db][r] *= alpha;
            ocor[db][r] *= alpha;
          }
      }
    }
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      const float p = fast_exp2(sacc[r]);
      sacc[r] = p;
      if (r & 1) l_b += p;
      else l_a += p;
    }
    warm = !__builtin_amdgcn_ballot_w64(m_run == -INFINITY);
  }

  // Joins the two accumulators and undoes V's scale (unscale) and the sign of the
  // odd dims; whether some row came out non-finite (wave-uniform).
  __device__ __forceinline__ bool finish(float unscale) {
    float bad = (l_a + l_b) * 0.f;
#pragma unroll
    for (int db = 0; db < NDB; ++db) {
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        // (adding 0 keeps the zeros of a row without a key positive)
        oacc[db][r] = fmaf(oacc[db][r] + ocor[db][r], r & 1 ? -unscale : unscale, 0.f);
      }
      bad = nonfinite_sum(oacc[db], bad);
    }
    return any_nonfinite(bad);
  }

  // The wave's rows on the fp32 MFMA straight from memory: only for rows that
  // came out non-finite (common.h) or whose Q is out of the split's range (load_q),
  // so that they hold what the fp32 products give.
  __device__ __forceinline__ void recompute(const FlashArgs &a, int b, int col0, int qi, int li, int hf, int kend,
                                            int key_last, const uint8_t *mrow) {
    init();
    const float *qrow = a.q + ((size_t)b * a.lq + min(qi, a.lq - 1)) * a.ldq + col0;
    const float *kb = a.k + (size_t)b * a.lk * a.ldk + col0, *vb = a.v + (size_t)b * a.lk * a.ldv + col0;
#pragma unroll 1
    for (int kb0 = 0; kb0 < kend; kb0 += 32) {
      const float *krow = kb + (size_t)min(kb0 + li, a.lk - 1) * a.ldk;
      floatx16 sacc = negm;
#pragma unroll 1
      for (int d = 0; d < HD; d += 2) {
        const bool in = d + hf < a.hd;
        sacc = mfma32x32x2(in ? krow[d + hf] : 0.f, in ? qrow[d + hf] * a.scale_log2 : 0.f, sacc);
      }
      softmax(sacc, hf, true, key_last - kb0 - 4 * hf, mrow, kb0, a.lk - 1, qi < a.lq);
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const float *vrow = vb + (size_t)min(kb0 + acc_key(r) + 4 * hf, a.lk - 1) * a.ldv;
#pragma unroll
        for (int db = 0; db < NDB; ++db)
          oacc[db] = mfma32x32x2(db * 32 + li < a.hd ? vrow[db * 32 + li] : 0.f, sacc[r], oacc[db]);
      }
    }
  }

  // Normalise and store row qi of (sequence b, head bh): the lane holds dims
  // db*32 + 8*(r/4) + 4*hf + r%4.  For the backward pass the row statistic
  // lse = m + log2(l) recovers every probability as exp2(s * scale * log2 e
  // - lse) (+inf for a row with no visible key, whose p are all 0).
  __device__ __forceinline__ void store(const FlashArgs &a, int bh, int b, int qi, int col0, int hf) const {
    const float l_tot = halves_sum(l_a + l_b);
    const float inv = l_tot > 0.f ? 1.0f / l_tot : 0.f;
    if (a.lse && hf == 0 && qi < a.lq)
      a.lse[(size_t)bh * a.lq + qi] = l_tot > 0.f ? m_run + __log2f(l_tot) : INFINITY;
    if (qi < a.lq) {
      float *orow = a.o + ((size_t)b * a.lq + qi) * a.ldo + col0;
#pragma unroll
      for (int db = 0; db < NDB; ++db) {
#pragma unroll
        for (int g = 0; g < 4; ++g) {
          const int d = db * 32 + 8 * g + 4 * hf;
          if constexpr (VEC) {
            *reinterpret_cast<float4 *>(orow + d) =
                make_float4(oacc[db][4 * g] * inv, oacc[db][4 * g + 1] * inv,
                            oacc[db][4 * g + 2] * inv, oacc[db][4 * g + 3] * inv);
          } else {
#pragma unroll
            for (int r = 0; r < 4; ++r)
              if (d + r < a.hd) orow[d + r] = oacc[db][4 * g + r] * inv;
          }
        }
      }
    }
  }
};

// Workgroup i runs (sequence, head) i % n_bh and, under the causal rule, query
// tile n_qt - 1 - i / n_bh (heaviest rows first), else tile i / n_bh.  With
// workgroup i on XCD i % 8, all tiles of one (sequence, head) share an XCD and
// its L2 whenever n_bh is a multiple of 8, and every XCD receives the heaviest
// tiles first (a near-optimal greedy schedule for a launch of several rounds).
template <int HD, int BN, bool CAUSAL, bool HAS_MASK, bool VEC>
__global__ void __launch_bounds__(FA_THREADS, HD <= 32 ? 3 : (HD <= 64 ? 2 : 1)) flash_fwd_kernel(const FlashArgs a) {
  constexpr int NKB = BN / 32;   // 32-key sub-blocks per tile
  typedef KvStage<HD, BN, VEC> Stage;
  __shared__ __attribute__((aligned(16))) char lds[2][Stage::BYTES];

  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int li = lane & 31, hf = lane >> 5;
  const int slot = a.by_bh.div(blockIdx.x), bh = blockIdx.x - slot * a.n_bh;
  const int qt = CAUSAL ? a.n_qt - 1 - slot : slot;
  const int b = a.by_heads.div(bh), col0 = (bh - b * a.heads) * a.hd;
  const int q0 = qt * FA_BM;
  const int qw0 = q0 + wave * 32;   // first query of this wave (wave-uniform)
  const int qi = qw0 + li;          // this lane's query
  const float *__restrict__ kbase = a.k + (size_t)b * a.lk * a.ldk + col0;
  const float *__restrict__ vbase = a.v + (size_t)b * a.lk * a.ldv + col0;

  Stage st;
  st.init(a.ldk, a.ldv);
  st.load(kbase, vbase, a.ldk, a.ldv, 0, a.lk, a.hd);
  bf16x8 q[HD / 16][3];
  const bool wide = load_q<HD, VEC>(q, a, b, col0, qi, hf);
  // Every other workgroup along a head's rows computes its outputs negated (common.h).
  const float sign = (qt + b) & 1 ? -1.f : 1.f, vscale = sign * kSplitScale;
  st.store(lds[0], vscale);
  __syncthreads();

  const int kend = CAUSAL ? min(q0 + FA_BM, a.lk) : a.lk;
  const int n_kt = (kend + BN - 1) / BN;
  OnlineRows<HD, BN, HAS_MASK, VEC> rows;
  rows.init();
  // Last key this lane may attend (the causal diagonal and the sequence end).
  const int key_last = CAUSAL ? min(qi, a.lk - 1) : a.lk - 1;
  const uint8_t *mrow = HAS_MASK ? a.mask + (size_t)min(qi, a.lq - 1) * a.lk : nullptr;
  const int ko = Stage::koperand(li, hf), vo = Stage::voperand(li, hf);

  for (int kt = 0; kt < n_kt; ++kt) {
    const int cur = kt & 1;
    const int k0 = kt * BN;
    // Next tile into registers; the last iteration re-stages its own tile into
    // the idle buffer (nobody reads it again): an unconditional stage keeps the
    // staging registers out of scratch memory.
    st.load(kbase, vbase, a.ldk, a.ldv, kt + 1 < n_kt ? k0 + BN : k0, a.lk, a.hd);
#pragma unroll
    for (int kb = 0; kb < NKB; ++kb) {
      const int kb0 = k0 + kb * 32;
      // A sub-block wholly past the sequence end or in this wave's future
      // contributes nothing (every probability would be 0), and a wave
      // whose rows all lie past lq (the last tile of a ragged length) has
      // nothing to compute: skip.
      if (kb0 >= a.lk || qw0 >= a.lq || (CAUSAL && kb0 > qw0 + 31)) continue;
      const char *kop = lds[cur] + ko + kb * 512, *vop = lds[cur] + vo + 2 * kb * Stage::VSLAB;
      floatx16 sacc = rows.scores(kop, q);
      // masking is needed on the diagonal and at the sequence end (wave-uniform)
      const bool masked = kb0 + 31 > (CAUSAL ? min(qw0, a.lk - 1) : a.lk - 1);
      const int last_vis = key_last - kb0 - 4 * hf;
      // Once every row has its reference, a sub-block is accumulated without
      // its maximum unless its probabilities come out unbounded; then its
      // scores are recomputed (K is still in LDS) for the full path.  Explicit
      // masks keep the full path.
      bool done = false;
      if (!HAS_MASK && rows.warm) {
        done = rows.try_fast(sacc, vop, hf, masked, last_vis, mrow, kb0, a.lk - 1, qi < a.lq);
        if (!done) {
          // K is read from LDS again (the compiler may not keep the first
          // scores, which would hold them live through the fast path)
          asm volatile("" ::: "memory");
          sacc = rows.scores(kop, q);
        }
      }
      if (!done) rows.consume(sacc, vop, hf, masked, last_vis, mrow, kb0, a.lk - 1, qi < a.lq);
    }
    st.store(lds[cur ^ 1], vscale);
    __syncthreads();
  }
  if ((rows.finish(sign * kSplitUnscale) || wide) && qw0 < a.lq)
    rows.recompute(a, b, col0, qi, li, hf, CAUSAL ? min(qw0 + 32, a.lk) : a.lk, key_last, mrow);
  rows.store(a, bh, b, qi, col0, hf);
}

// Head dims above 128: one workgroup per (sequence, head, query), keys in
// chunks of 256 with an online softmax; correctness path only.
__global__ void __launch_bounds__(256) flash_generic_kernel(const FlashArgs a, int causal) {
  extern __shared__ float sm[];  // q[hd] | o[hd] | p[256] | red[8]
  float *qv = sm;
  float *ov = sm + a.hd;
  float *pv = ov + a.hd;
  float *red = pv + 256;
  const int row = blockIdx.x;  // b * lq + i
  const int b = row / a.lq, i = row % a.lq;
  const int h = blockIdx.y;
  const int col0 = h * a.hd;
  const int t = threadIdx.x;
  const float *qrow = a.q + ((size_t)b * a.lq + i) * a.ldq + col0;
  for (int d = t; d < a.hd; d += 256) {
    qv[d] = qrow[d];
    ov[d] = 0.f;
  }
  __syncthreads();
  const int usable = causal ? min(i + 1, a.lk) : a.lk;
  float m_run = -INFINITY, l_run = 0.f;
  for (int c0 = 0; c0 < usable; c0 += 256) {
    const int j = c0 + t;
    float s = -INFINITY;
    if (j < usable && (!a.mask || a.mask[(size_t)i * a.lk + j])) {
      const float *krow = a.k + ((size_t)b * a.lk + j) * a.ldk + col0;
      float acc = 0.f;
      for (int d = 0; d < a.hd; ++d) acc += qv[d] * krow[d];
      s = acc * a.scale_log2;
    }
    float mx = s;
    for (int off = 32; off > 0; off >>= 1) mx = fmaxf(mx, __shfl_xor(mx, off));
    if ((t & 63) == 0) red[t >> 6] = mx;
    __syncthreads();
    mx = fmaxf(fmaxf(red[0], red[1]), fmaxf(red[2], red[3]));
    __syncthreads();
    const float m_new = fmaxf(m_run, mx);
    const float m_use = m_new == -INFINITY ? 0.f : m_new;
    const float alpha = fast_exp2(m_run - m_use);
    const float p = fast_exp2(s - m_use);
    pv[t] = p;
    float ps = p;
    for (int off = 32; off > 0; off >>= 1) ps += __shfl_xor(ps, off);
    if ((t & 63) == 0) red[4 + (t >> 6)] = ps;
    __syncthreads();
    l_run = l_run * alpha + (red[4] + red[5] + red[6] + red[7]);
    m_run = m_new;
    const int n = min(256, usable - c0);
    for (int d = t; d < a.hd; d += 256) {
      float acc = ov[d] * alpha;
      for (int jj = 0; jj < n; ++jj)
        acc += pv[jj] * a.v[((size_t)b * a.lk + c0 + jj) * a.ldv + col0 + d];
      ov[d] = acc;
    }
    __syncthreads();
  }
  const float inv = l_run > 0.f ? 1.0f / l_run : 0.f;
  float *orow = a.o + ((size_t)b * a.lq + i) * a.ldo + col0;
  for (int d = t; d < a.hd; d += 256) orow[d] = ov[d] * inv;
}

template <int HD, int BN, bool CAUSAL, bool HAS_MASK>
void launch_tpl(const FlashArgs &a, bool vec, hipStream_t st) {
  const dim3 grid(a.n_items), block(FA_THREADS);
  if (vec) flash_fwd_kernel<HD, BN, CAUSAL, HAS_MASK, true><<<grid, block, 0, st>>>(a);
  else flash_fwd_kernel<HD, BN, CAUSAL, HAS_MASK, false><<<grid, block, 0, st>>>(a);
}

template <int HD, int BN>
void launch_hd(const FlashArgs &a, bool causal, bool vec, hipStream_t st) {
  const bool m = a.mask != nullptr;
  if (causal) {
    if (m) launch_tpl<HD, BN, true, true>(a, vec, st);
    else launch_tpl<HD, BN, true, false>(a, vec, st);
  } else {
    if (m) launch_tpl<HD, BN, false, true>(a, vec, st);
    else launch_tpl<HD, BN, false, false>(a, vec, st);
  }
}

}  // namespace
}  // namespace cdml

using namespace cdml;

namespace cdml {

// Launches the forward kernels; the arguments are validated by the caller.
// causal here admits lq != lk (key j visible to query i iff j <= i).
int flash_forward(const float *q, int ldq, const float *k, int ldk, const float *v, int ldv,
                  float *o, int ldo, float *lse, int batch, int lq, int lk, int dim, int num_heads,
                  float scale, bool causal, const uint8_t *mask, hipStream_t st) {
  FlashArgs a{};
  a.q = q;
  a.k = k;
  a.v = v;
  a.o = o;
  a.lse = lse;
  a.mask = mask;
  a.ldq = ldq;
  a.ldk = ldk;
  a.ldv = ldv;
  a.ldo = ldo;
  a.lq = lq;
  a.lk = lk;
  a.heads = num_heads;
  a.hd = dim / num_heads;
  a.scale_log2 = scale * kLog2e;

  const int hd = a.hd;
  if (hd > 128) {
    if (lse) return fail(CDML_E_INVALID, "flash_forward: no row statistics above head dim 128");
    a.n_qt = lq;
    size_t smem = sizeof(float) * (2 * (size_t)hd + 256 + 8);
    if (smem > 160 * 1024) return fail(CDML_E_INVALID, "cdml_sdpa_fwd: head dim %d too large", hd);
    flash_generic_kernel<<<dim3(batch * lq, num_heads), dim3(256), smem, st>>>(a, causal);
    return check_launch("flash_generic_kernel");
  }
  const int hd_pad = hd <= 32 ? 32 : (hd <= 64 ? 64 : 128);
  const bool vec = hd == hd_pad && ldq % 4 == 0 && ldk % 4 == 0 && ldv % 4 == 0 && ldo % 4 == 0 &&
                   aligned16(q) && aligned16(k) && aligned16(v) && aligned16(o);
  a.n_bh = batch * num_heads;
  a.n_qt = (lq + FA_BM - 1) / FA_BM;
  a.by_bh = UDiv::make((uint32_t)a.n_bh);
  a.by_heads = UDiv::make((uint32_t)num_heads);
  long long total = (long long)batch * num_heads * a.n_qt;
  if (total > (1LL << 30)) return fail(CDML_E_INVALID, "cdml_sdpa_fwd: problem too large");
  a.n_items = (int)total;
  if (hd_pad == 32) launch_hd<32, 32>(a, causal, vec, st);
  else if (hd_pad == 64) launch_hd<64, 32>(a, causal, vec, st);
  else launch_hd<128, 32>(a, causal, vec, st);
  return check_launch("flash_fwd_kernel");
}

}  // namespace cdml

namespace {

int sdpa_fwd_impl(const float *q, int ldq, const float *k, int ldk, const float *v, int ldv, float *o,
                  int ldo, float *lse, int batch, int lq, int lk, int dim, int num_heads, float scale,
                  int causal, const uint8_t *mask, cdml_stream stream) {
  if (batch < 0 || lq < 0 || lk < 0 || dim <= 0 || num_heads <= 0)
    return fail(CDML_E_INVALID, "cdml_sdpa_fwd: bad size (batch %d, lq %d, lk %d, dim %d, heads %d)",
                batch, lq, lk, dim, num_heads);
  if (dim % num_heads != 0)
    return fail(CDML_E_INVALID, "cdml_sdpa_fwd: dim %d not divisible by num_heads %d", dim, num_heads);
  if (causal && lq != lk)
    return fail(CDML_E_CAUSAL, "cdml_sdpa_fwd: causal attention requires lq == lk (got %d, %d)", lq, lk);
  if (ldq < dim || ldk < dim || ldv < dim || ldo < dim)
    return fail(CDML_E_INVALID, "cdml_sdpa_fwd: row stride smaller than dim");
  if ((long long)ldk * 128 > INT32_MAX || (long long)ldv * 128 > INT32_MAX)
    return fail(CDML_E_INVALID, "cdml_sdpa_fwd: row stride above %d elements", INT32_MAX / 128);
  if (batch == 0 || lq == 0) return CDML_OK;
  if (lk == 0) return fail(CDML_E_INVALID, "cdml_sdpa_fwd: lk must be >= 1");
  if (!q || !k || !v || !o) return fail(CDML_E_INVALID, "cdml_sdpa_fwd: NULL pointer");
  int rc = ensure_device();
  if (rc) return rc;
  return flash_forward(q, ldq, k, ldk, v, ldv, o, ldo, lse, batch, lq, lk, dim, num_heads, scale,
                       causal != 0, mask, as_hip(stream));
}

}  // namespace

extern "C" int cdml_sdpa_fwd(const float *q, int ldq, const float *k, int ldk, const float *v,
                             int ldv, float *o, int ldo, int batch, int lq, int lk, int dim,
                             int num_heads, float scale, int causal, const uint8_t *mask,
                             cdml_stream stream) {
  return sdpa_fwd_impl(q, ldq, k, ldk, v, ldv, o, ldo, nullptr, batch, lq, lk, dim, num_heads, scale,
                       causal, mask, stream);
}

extern "C" int cdml_sdpa_fwd_lse(const float *q, int ldq, const float *k, int ldk, const float *v,
                                 int ldv, float *o, int ldo, float *lse, int batch, int lq, int lk,
                                 int dim, int num_heads, float scale, int causal,
                                 const uint8_t *mask, cdml_stream stream) {
  if (!lse) return fail(CDML_E_INVALID, "cdml_sdpa_fwd_lse: lse is NULL");
  return sdpa_fwd_impl(q, ldq, k, ldk, v, ldv, o, ldo, lse, batch, lq, lk, dim, num_heads, scale, causal,
                       mask, stream);
}
