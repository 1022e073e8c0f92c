// Attention backward for gfx950: MultiHeadAttentionBackward of the reference
// (AccelerationCPU.cs:1011-1280).
//
// With P = softmax(S), S = scale * Q K^T per (sequence, head) under the
// causal rule (key j visible to query i iff j <= i) and/or a mask:
//   dV = P^T dO,  dP = dO V^T,  dS = P (dP - D) with D_i = sum_j P_ij dP_ij,
//   dQ = scale dS K,  dK = scale dS^T Q.
// D_i equals dO_i . O_i, so the pass runs in four launches:
//   1. the forward kernel with row statistics: O and lse_i (log2 of the
//      softmax normaliser), so that P_ij = exp2(s_ij * scale * log2 e - lse_i);
//   2. bwd_delta_kernel: D = rowsum(dO * O) per head;
//   3. dK and dV, key-block major: a workgroup owns 128 keys of one (sequence,
//      head), 32 to a wave or a pair of waves, whose K and V rows stay in
//      registers; Q, dO, lse and D tiles stream through double-buffered LDS.
//      Per 32-query sub-block: S = Q K^T and dP = dO V^T land with one key
//      per lane and 16 queries per lane in registers, exactly the B operand
//      layout that dV^T += dO^T P and dK^T += Q^T dS need, so P and dS are
//      consumed in place (flash_bwd_dkdv_split_kernel on bf16 pieces for head
//      dims up to 64, flash_bwd_dkdv_kernel on fp32 MFMA above);
//   4. dQ, query-block major like the forward: from dS blocks that step 3 stored
//      (flash_bwd_dq_ds_kernel, on bf16 pieces), or recomputed on fp32 MFMA
//      (flash_bwd_dq_kernel): S^T = K Q^T and dP^T = V dO^T put one query per
//      lane, dS^T is consumed in place by dQ^T += K^T dS^T.
// Every output element is written by one lane of one workgroup: no atomics,
// and the result is the same on every run.  Head dims below 128 other than
// 32 and 64, or rows that are not 16-byte aligned, run the same kernels at the
// next of 32 / 64 / 128 with zero-filled scalar loads (VEC false) and
// predicated stores; zero columns of Q, K, V and dO leave S, dP and every
// stored gradient column unchanged.  Head dims above 128 take
// flash_bwd_generic_kernel, which follows the reference's per-row loops.
#include "common.h"

namespace cdml {
namespace {

constexpr int BW_THREADS = 256;
constexpr int BW_TILE = 128;  // keys (dK/dV) or queries (dQ) per workgroup
constexpr int kBufferWord3 = 0x00020000;  // gfx9 buffer resource word 3: raw 32-bit dwords
constexpr int kCachePolicyNT = 2;         // buffer instruction cache policy: non-temporal
constexpr float kLog2e = 1.4426950408889634f;

struct BwdArgs {
  const float *q, *k, *v, *dout;
  float *dq, *dk, *dv;
  const float *o;      // forward output [batch * lq][dim] (row stride ldo)
  const float *lse;    // [batch * heads][lq]
  float *delta;        // [batch * heads][lq]
  float *ds;           // stored dS blocks (causal, lq == lk) or NULL
  long long ds_bh;     // floats of ds per (sequence, head)
  const uint8_t *mask; // [lq][lk] or NULL
  int ldq, ldk, ldv, lddo, lddq, lddk, lddv, ldo;
  int batch, lq, lk, dim, heads, hd;
  float scale, scale_log2;
  int n_tiles, total;
  // Inverse rotary embedding applied to dQ and dK as they are stored
  // (cdml_sdpa_bwd_saved_rope): rope_cs[pos * hd / 2 + p] holds (cos, sin) of
  // position pos for pair p, and a row's position is its index in its
  // sequence.  NULL: no rotation.
  const float2 *rope_cs;
};

// The inverse rotation of one pair (x0, x1) = dims (2p, 2p + 1) by (cos, sin)
// t, rounded as rope_qk_table_kernel rounds it (each product before the sum),
// so the fused form stores the same bits as a separate cdml_rope_qk_table.
__device__ __forceinline__ float2 rope_inverse_pair(float x0, float x1, float2 t) {
#pragma clang fp contract(off)
  const float s = -t.y;
  return make_float2(x0 * t.x - x1 * s, x0 * s + x1 * t.x);
}

// Offset of accumulator register r's row inside its 32-row block for a lane of
// half-wave h: 8 * (r / 4) + 4 * h + r % 4 (the 32x32 MFMA D layout).
__device__ __forceinline__ constexpr int acc_row(int r) { return 8 * (r >> 2) + (r & 3); }

// One ROWS x HD tile of a row-major matrix (rows [row0, row0 + ROWS) of the
// head's column block), global -> registers -> LDS.  Each thread's offsets
// inside a tile are fixed; rows past `nrows` are clamped to the last row
// (their contributions are masked or never stored).  Without VEC, columns at
// or past the head dim `hd` read as zero and the rest are scalar loads.
template <int HD, int ROWS, bool VEC>
struct RowStage {
  static constexpr int F4 = HD / 4;
  static constexpr int RPP = BW_THREADS / F4;
  static constexpr int NV = ROWS / RPP;
  static_assert(NV >= 1 && ROWS % RPP == 0, "tile shape");
  vf4 r[NV];
  uint32_t off[NV];
  int col;

  __device__ __forceinline__ void init(int ld) {
    const int t = threadIdx.x;
    col = (t % F4) * 4;
#pragma unroll
    for (int i = 0; i < NV; ++i) off[i] = (uint32_t)((t / F4 + RPP * i) * ld + col);
  }
  __device__ __forceinline__ void load(const float *__restrict__ base, int ld, int row0, int nrows,
                                       int hd) {
    const float *tile = base + (size_t)row0 * ld;
    const uint32_t lim = (uint32_t)(min(nrows - 1 - row0, ROWS - 1) * ld) + col;
#pragma unroll
    for (int i = 0; i < NV; ++i) {
      if constexpr (VEC) {
        r[i] = *reinterpret_cast<const vf4 *>(tile + min(off[i], lim));
      } else {
        const float *p = tile + min(off[i], lim);
#pragma unroll
        for (int c = 0; c < 4; ++c) r[i][c] = col + c < hd ? p[c] : 0.f;
      }
    }
  }
  __device__ __forceinline__ void store(float (*lds)[HD + 4]) const {
    const int t = threadIdx.x;
#pragma unroll
    for (int i = 0; i < NV; ++i) *reinterpret_cast<vf4 *>(&lds[t / F4 + RPP * i][col]) = r[i];
  }
};

// D[b, h, i] = dO_i . O_i over head h's columns; one thread per (row, head).
// D[b, h, i] = dO[b, i, head h] . O[b, i, head h].  Thread e owns float4 e of
// the flat [batch * lq, dim / 4] view, so a wave reads whole rows (coalesced);
// the HD / 4 consecutive lanes of one head sum their partials with xor
// shuffles (HD / 4 divides 64, so a head never straddles two waves).
template <int HD>
__global__ void __launch_bounds__(256) bwd_delta_kernel(const BwdArgs a) {
  constexpr int G = HD / 4;
  const int d4 = a.dim >> 2;
  const long long e = (long long)blockIdx.x * 256 + threadIdx.x;
  const long long n = (long long)a.batch * a.lq * d4;
  const long long ec = e < n ? e : n - 1;  // every lane joins the shuffles
  const long long row = ec / d4;
  const int c4 = (int)(ec % d4);
  const vf4 x = *reinterpret_cast<const vf4 *>(a.dout + row * a.lddo + 4 * c4);
  const vf4 y = *reinterpret_cast<const vf4 *>(a.o + row * a.ldo + 4 * c4);
  float s = (x[0] * y[0] + x[1] * y[1]) + (x[2] * y[2] + x[3] * y[3]);
#pragma unroll
  for (int off = G / 2; off >= 1; off >>= 1) s += __shfl_xor(s, off);
  if (e < n && c4 % G == 0) {
    const int h = c4 / G;
    const int b = (int)(row / a.lq), i = (int)(row % a.lq);
    a.delta[((size_t)b * a.heads + h) * a.lq + i] = s;
  }
}

// D for any head dim and stride: thread e owns (row e / heads, head e % heads).
__global__ void __launch_bounds__(256) bwd_delta_scalar_kernel(const BwdArgs a) {
  const long long e = (long long)blockIdx.x * 256 + threadIdx.x;
  if (e >= (long long)a.batch * a.lq * a.heads) return;
  const long long row = e / a.heads;
  const int h = (int)(e % a.heads);
  const float *x = a.dout + row * a.lddo + h * a.hd;
  const float *y = a.o + row * a.ldo + h * a.hd;
  float s = 0.f;
  for (int d = 0; d < a.hd; ++d) s += x[d] * y[d];
  const int b = (int)(row / a.lq), i = (int)(row % a.lq);
  a.delta[((size_t)b * a.heads + h) * a.lq + i] = s;
}

// Stores one row of a gradient: this lane's x (register 4g + c of block db is
// dimension db*32 + 8g + 4*hf + c) times scale, rotated back by the pairs of
// rope_cs when non-NULL (the table row of its position).
template <int HD, bool VEC>
__device__ __forceinline__ void store_column(const BwdArgs &a, const floatx16 (&x)[HD / 32], float *row, float scale,
                                             const float2 *rope_cs, int hf) {
  constexpr int NDB = HD / 32;
  // (cos, sin) of the row's pairs, loaded before any store (a load issued after
  // a store waits for it)
  float2 cs[NDB][4][2];
  if (rope_cs) {
#pragma unroll
    for (int db = 0; db < NDB; ++db)
#pragma unroll
      for (int g = 0; g < 4; ++g)
#pragma unroll
        for (int j = 0; j < 2; ++j) {
          const int d = db * 32 + 8 * g + 4 * hf + 2 * j;
          cs[db][g][j] = d < a.hd ? rope_cs[d >> 1] : make_float2(1.f, 0.f);
        }
  }
#pragma unroll
  for (int db = 0; db < NDB; ++db) {
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      const int d = db * 32 + 8 * g + 4 * hf;
      vf4 y;
#pragma unroll
      for (int c = 0; c < 4; ++c) y[c] = x[db][4 * g + c] * scale;
      if (rope_cs) {  // dims d + c and d + c + 1 are one pair, in this lane
#pragma unroll
        for (int c = 0; c < 4; c += 2) {
          const float2 r = rope_inverse_pair(y[c], y[c + 1], cs[db][g][c >> 1]);
          y[c] = r.x;
          y[c + 1] = r.y;
        }
      }
      if constexpr (VEC) {
        *reinterpret_cast<vf4 *>(row + d) = y;
      } else {
#pragma unroll
        for (int c = 0; c < 4; ++c)
          if (d + c < a.hd) row[d + c] = y[c];
      }
    }
  }
}

// dK and dV on fp32 MFMA, for head dims above 64: two tensors' pieces of a
// wave's keys need 384 registers there.  Workgroup i takes (sequence, head)
// i % n_bh and key tile i / n_bh: under the causal rule the first key tiles are
// seen by the most queries, so the heaviest tiles go out first on every XCD.
template <int HD, bool CAUSAL, bool HAS_MASK, bool VEC>
__global__ void __launch_bounds__(BW_THREADS, 1) flash_bwd_dkdv_kernel(const BwdArgs a) {
  constexpr int BQ = 32;
  constexpr int NQB = BQ / 32;  // 32-query sub-blocks per tile
  constexpr int NDB = HD / 32;  // 32-wide head-dim blocks of dK^T / dV^T
  constexpr int NKG = HD / 8;   // 8-dim groups of the Q.K and dO.V products
  __shared__ __attribute__((aligned(16))) float Qs[2][BQ][HD + 4];
  __shared__ __attribute__((aligned(16))) float Gs[2][BQ][HD + 4];  // dO
  __shared__ __attribute__((aligned(16))) float Ls[2][BQ];          // lse
  __shared__ __attribute__((aligned(16))) float Ds[2][BQ];          // D

  const int n_bh = a.batch * a.heads;
  const int bh = blockIdx.x % n_bh, kt = blockIdx.x / n_bh;
  const int b = bh / a.heads, h = bh % a.heads;
  const int t = threadIdx.x;
  const int lane = t & 63;
  const int wave = __builtin_amdgcn_readfirstlane(t >> 6);
  const int li = lane & 31, hf = lane >> 5;
  const int k0 = kt * BW_TILE;
  const int kw0 = k0 + wave * 32;  // first key of this wave
  const int key = kw0 + li;        // this lane's key
  const int col0 = h * (VEC ? HD : a.hd);

  // B operands of S = Q K^T and dP = dO V^T: register 4u + r holds
  // K[key][8u + 4*hf + r] (and likewise V), fixed for the whole loop.
  float kreg[HD / 2], vreg[HD / 2];
  {
    const int kr = min(key, a.lk - 1);
    const float *krow = a.k + ((size_t)b * a.lk + kr) * a.ldk + col0;
    const float *vrow = a.v + ((size_t)b * a.lk + kr) * a.ldv + col0;
#pragma unroll
    for (int u = 0; u < NKG; ++u) {
      const int d = 8 * u + 4 * hf;
      if constexpr (VEC) {
        const vf4 x = *reinterpret_cast<const vf4 *>(krow + d);
        const vf4 y = *reinterpret_cast<const vf4 *>(vrow + d);
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          kreg[4 * u + r] = x[r];
          vreg[4 * u + r] = y[r];
        }
      } else {
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          kreg[4 * u + r] = d + r < a.hd ? krow[d + r] : 0.f;
          vreg[4 * u + r] = d + r < a.hd ? vrow[d + r] : 0.f;
        }
      }
    }
  }

  const int q_begin = CAUSAL ? k0 : 0;  // queries before k0 see none of these keys
  const int n_it = q_begin < a.lq ? (a.lq - q_begin + BQ - 1) / BQ : 0;
  const float *__restrict__ qbase = a.q + (size_t)b * a.lq * a.ldq + col0;
  const float *__restrict__ gbase = a.dout + (size_t)b * a.lq * a.lddo + col0;
  const float *__restrict__ lse = a.lse + (size_t)bh * a.lq;
  const float *__restrict__ dlt = a.delta + (size_t)bh * a.lq;

  floatx16 dk[NDB], dv[NDB];
#pragma unroll
  for (int db = 0; db < NDB; ++db)
#pragma unroll
    for (int r = 0; r < 16; ++r) dk[db][r] = dv[db][r] = 0.f;
  const floatx16 zero = {};

  RowStage<HD, BQ, VEC> sq, sg;
  sq.init(a.ldq);
  sg.init(a.lddo);
  float lreg = 0.f, dreg = 0.f;
  if (n_it > 0) {
    sq.load(qbase, a.ldq, q_begin, a.lq, a.hd);
    sg.load(gbase, a.lddo, q_begin, a.lq, a.hd);
    if (t < BQ) {
      const int qq = min(q_begin + t, a.lq - 1);
      lreg = lse[qq];
      dreg = dlt[qq];
    }
    sq.store(Qs[0]);
    sg.store(Gs[0]);
    if (t < BQ) {
      Ls[0][t] = lreg;
      Ds[0][t] = dreg;
    }
  }
  __syncthreads();

  for (int it = 0; it < n_it; ++it) {
    const int cur = it & 1;
    const int qt0 = q_begin + it * BQ;
    // Next tile into registers; the last iteration re-stages its own tile
    // into the idle buffer (an unconditional stage keeps the registers out
    // of scratch memory).
    const int nxt = it + 1 < n_it ? qt0 + BQ : qt0;
    sq.load(qbase, a.ldq, nxt, a.lq, a.hd);
    sg.load(gbase, a.lddo, nxt, a.lq, a.hd);
    if (t < BQ) {
      const int qq = min(nxt + t, a.lq - 1);
      lreg = lse[qq];
      dreg = dlt[qq];
    }

#pragma unroll
    for (int qb = 0; qb < NQB; ++qb) {
      const int qb0 = qt0 + qb * 32;
      // Sub-blocks past the sequence end or wholly before this wave's keys
      // contribute nothing, and neither does a wave whose keys all lie past lk.
      if (qb0 >= a.lq || kw0 >= a.lk || (CAUSAL && qb0 + 31 < kw0)) continue;
      const float(*qrow)[HD + 4] = &Qs[cur][qb * 32];
      const float(*grow)[HD + 4] = &Gs[cur][qb * 32];

      // S = Q K^T and dP = dO V^T (two independent MFMA chains).
      floatx16 s, dp;
      vf4 qa = *reinterpret_cast<const vf4 *>(&qrow[li][4 * hf]);
      vf4 ga = *reinterpret_cast<const vf4 *>(&grow[li][4 * hf]);
#pragma unroll
      for (int u = 0; u < NKG; ++u) {
        vf4 qn, gn;
        if (u + 1 < NKG) {
          qn = *reinterpret_cast<const vf4 *>(&qrow[li][8 * (u + 1) + 4 * hf]);
          gn = *reinterpret_cast<const vf4 *>(&grow[li][8 * (u + 1) + 4 * hf]);
        }
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          s = mfma32x32x2(qa[r], kreg[4 * u + r], (u == 0 && r == 0) ? zero : s);
          dp = mfma32x32x2(ga[r], vreg[4 * u + r], (u == 0 && r == 0) ? zero : dp);
        }
        if (u + 1 < NKG) {
          qa = qn;
          ga = gn;
        }
      }

      // P = exp2(S * scale * log2 e - lse) and dS = P (dP - D), per query row
      // 8g + 4*hf + c of the sub-block (registers 4g + c).
      // (the masked and the unmasked forms are separate branches: a select
      // per element would run the mask arithmetic on every sub-block)
      const bool need = HAS_MASK || (CAUSAL && qb0 < kw0 + 31) || qb0 + 31 >= a.lq;
      if (need) {
#pragma unroll
        for (int g = 0; g < 4; ++g) {
          const vf4 l4 = *reinterpret_cast<const vf4 *>(&Ls[cur][qb * 32 + 8 * g + 4 * hf]);
          const vf4 d4 = *reinterpret_cast<const vf4 *>(&Ds[cur][qb * 32 + 8 * g + 4 * hf]);
#pragma unroll
          for (int c = 0; c < 4; ++c) {
            const int r = 4 * g + c;
            const int qq = qb0 + 8 * g + 4 * hf + c;
            bool ok = qq < a.lq;
            if (CAUSAL) ok = ok && key <= qq;
            if (HAS_MASK) ok = ok && key < a.lk && a.mask[(size_t)min(qq, a.lq - 1) * a.lk + min(key, a.lk - 1)];
            const float p = ok ? fast_exp2(fmaf(s[r], a.scale_log2, -l4[c])) : 0.f;
            s[r] = p;
            dp[r] = p * (dp[r] - d4[c]);
          }
        }
      } else {
#pragma unroll
        for (int g = 0; g < 4; ++g) {
          const vf4 l4 = *reinterpret_cast<const vf4 *>(&Ls[cur][qb * 32 + 8 * g + 4 * hf]);
          const vf4 d4 = *reinterpret_cast<const vf4 *>(&Ds[cur][qb * 32 + 8 * g + 4 * hf]);
#pragma unroll
          for (int c = 0; c < 4; ++c) {
            const int r = 4 * g + c;
            const float p = fast_exp2(fmaf(s[r], a.scale_log2, -l4[c]));
            s[r] = p;
            dp[r] = p * (dp[r] - d4[c]);
          }
        }
      }
      // dV^T += dO^T P and dK^T += Q^T dS: MFMA step st pairs query rows
      // acc_row(st) (half 0) and acc_row(st) + 4 (half 1), the rows held by
      // register st of P and dS.
#pragma unroll
      for (int st = 0; st < 16; ++st) {
        const int qr = acc_row(st) + 4 * hf;
#pragma unroll
        for (int db = 0; db < NDB; ++db) {
          dv[db] = mfma32x32x2(grow[qr][db * 32 + li], s[st], dv[db]);
          dk[db] = mfma32x32x2(qrow[qr][db * 32 + li], dp[st], dk[db]);
        }
      }
    }

    sq.store(Qs[cur ^ 1]);
    sg.store(Gs[cur ^ 1]);
    if (t < BQ) {
      Ls[cur ^ 1][t] = lreg;
      Ds[cur ^ 1][t] = dreg;
    }
    __syncthreads();
  }

  if (key < a.lk) {
    const size_t krow = (size_t)b * a.lk + key;
    store_column<HD, VEC>(a, dk, a.dk + krow * a.lddk + col0, a.scale,
                          a.rope_cs ? a.rope_cs + (size_t)key * (a.hd >> 1) : nullptr, hf);
    store_column<HD, VEC>(a, dv, a.dv + krow * a.lddv + col0, 1.f, nullptr, hf);
  }
}

// One tile of 32 query rows of Q and of dO for the split dK/dV kernel, split
// into three bf16 pieces on its way into LDS, each tensor in two layouts (rows of
// 16 values = 32 bytes, one plane per piece, as the GEMM's operand tiles):
//   rows:       slab s holds dims 16 s .. 16 s + 15 of every query (S and dP);
//               even and odd queries in two clusters;
//   transposed: slab s holds queries 16 s .. 16 s + 15 of every dim (dV and dK),
//               query k of a slab at place 8 (k / 4 % 2) + 4 (k / 8) + k % 4, the
//               order in which the score accumulators hold them; four clusters by
//               d % 4.
// Odd dims are negated in both (common.h); K and V carry the same sign in the
// wave's registers, and the stores undo it, as that of dO (gscale).  A unit is four
// dims of two queries: its pieces are packed along the queries as they are split and
// repacked along the dims by byte permutes.
template <int HD, bool VEC>
struct QgStage {
  static constexpr int CH = HD / 4;
  static constexpr int UNITS = CH * 16;                        // of one tensor
  static constexpr int NU = 2 * UNITS / BW_THREADS;            // per thread: 2 (Q and dO) or 1 (either)
  static constexpr int RSLAB = 2 * 512 + 128, TSLAB = 4 * (CH * 32) + 256;
  static constexpr int RPLANE = HD / 16 * RSLAB, TPLANE = 2 * TSLAB;
  static constexpr int TENSOR = 3 * (RPLANE + TPLANE);         // rows planes, then transposed planes
  static constexpr int BYTES = 2 * TENSOR;
  static_assert(NU == 1 || NU == 2, "tile units");
  static __device__ __forceinline__ constexpr int rcluster(int c) { return c * (512 + 16); }
  static __device__ __forceinline__ constexpr int tcluster(int c) { return c * CH * 32 + (c & 1) * 16 + (c >> 1) * 128; }
  vf4 r[NU][2];
  int row, col, rdst, tdst;  // first query and dim of the unit, its places in the two layouts
  bool gside;                // NU == 1: this thread stages dO

  __device__ __forceinline__ void init() {
    const int t = threadIdx.x;  // the staging waves are the first four
    gside = NU == 1 && __builtin_amdgcn_readfirstlane(t) >= UNITS;
    const int u = t % UNITS, sb = u & 7, g = (u >> 3) % CH, slab = (u >> 3) / CH;
    row = 16 * slab + 2 * sb;
    col = 4 * g;
    const int place = ((sb >> 1) & 1) * 4 + (sb >> 2) * 2 + (sb & 1);  // of the query pair
    rdst = (g >> 2) * RSLAB + (row >> 1) * 32 + (g & 3) * 8;
    tdst = 3 * RPLANE + slab * TSLAB + g * 32 + place * 4;
  }
  __device__ __forceinline__ void load(const float *__restrict__ qbase, const float *__restrict__ gbase, int ldq,
                                       int ldg, int row0, int nrows, int hd) {
#pragma unroll
    for (int i = 0; i < NU; ++i) {
      const bool g = NU == 1 ? gside : i == 1;
      const int ld = g ? ldg : ldq;
      const float *tile = (g ? gbase : qbase) + (size_t)row0 * ld;  // wave-uniform
#pragma unroll
      for (int x = 0; x < 2; ++x) {
        const float *p = tile + (uint32_t)(min(row + x, nrows - 1 - row0) * ld + col);
        if constexpr (VEC) {
          r[i][x] = *reinterpret_cast<const vf4 *>(p);
        } else {
#pragma unroll
          for (int c = 0; c < 4; ++c) r[i][x][c] = col + c < hd ? p[c] : 0.f;
        }
      }
    }
  }
  // Without VEC the scaling would be scheduled beside the guarded loads and wait for them:
  // the values pass through an empty asm here first (42 x 3528, one head of 40: 943 -> 832 us
  // causal, 1843 -> 1524 not).  Zeroing the padding through the factor instead takes as long
  // but holds a dozen registers more: 200 against 172 us, 8 x 1024 with four heads of 20 under
  // a mask, where it spilled.
  __device__ __forceinline__ void store(char *lds, float gscale) const {
#pragma unroll
    for (int i = 0; i < NU; ++i) {
      const float scale = (NU == 1 ? gside : i == 1) ? gscale : kSplitScale;
      char *base = lds + (NU == 1 ? (gside ? TENSOR : 0) : i * TENSOR);
      uint32_t w[3][4];  // [piece][dim]: query `row` in the low half, `row + 1` in the high half
#pragma unroll
      for (int c = 0; c < 4; ++c) {
        const float f = c & 1 ? -scale : scale;
        float r0 = r[i][0][c], r1 = r[i][1][c];
        if constexpr (!VEC) asm volatile("" : "+v"(r0), "+v"(r1));
        split_bf16x3(r0 * f, r1 * f, w[0][c], w[1][c], w[2][c]);
      }
#pragma unroll
      for (int q = 0; q < 3; ++q) {
#pragma unroll
        for (int c = 0; c < 4; ++c)
          *reinterpret_cast<uint32_t *>(base + tdst + q * TPLANE + tcluster(c)) = w[q][c];
        // low halves of two words, high halves of two words
        const vu2 even = {__builtin_amdgcn_perm(w[q][1], w[q][0], 0x05040100), __builtin_amdgcn_perm(w[q][3], w[q][2], 0x05040100)};
        const vu2 odd = {__builtin_amdgcn_perm(w[q][1], w[q][0], 0x07060302), __builtin_amdgcn_perm(w[q][3], w[q][2], 0x07060302)};
        *reinterpret_cast<vu2 *>(base + rdst + q * RPLANE) = even;
        *reinterpret_cast<vu2 *>(base + rdst + q * RPLANE + rcluster(1)) = odd;
      }
    }
  }
  // Byte offsets of a lane's operands in plane 0 of a tensor.
  static __device__ __forceinline__ int roperand(int li, int hf) {
    return rcluster(li & 1) + (li >> 1) * 32 + hf * 16;
  }
  static __device__ __forceinline__ int toperand(int li, int hf) {
    return 3 * RPLANE + tcluster(li & 3) + (li >> 2) * 32 + hf * 16;
  }
};

// dK and dV on three bf16 pieces per fp32 operand (common.h), head dims up to 64;
// workgroups over keys as flash_bwd_dkdv_kernel's.
//
// Head dim 64: a pair of waves owns 32 keys.  Wave w (0..3) holds K's pieces,
// forms S and P and sums dV; wave w + 4 holds V's, forms dP, takes P through LDS,
// forms and stores dS and sums dK.  A pair shares a SIMD, so one wave's
// exponentials and splits run under the other's products, and each needs 224
// registers (one wave for both needs 470 and is alone on its SIMD: 35% of the
// cycles in the matrix pipes, paired 45%).  Per 32-query tile, two barriers: P is
// written before the first, read after it.  Head dim 32: one wave does both in
// 250 registers, two workgroups to a CU; pairs took 31% longer there, half the
// products per barrier.
// Measured on MI355X: 4 x 4096, 16 heads of 64, 1.69 ms (2.19 on the fp32 MFMA); 256 x
// 511, 8 heads of 32, 0.65 ms (0.77).  Bound by the exponentials and splits between
// the products: 5.1 and 10.2 VALU instructions beside each MFMA, matrix pipes 45% and
// 30% busy.
//
// All operands but P carry the split's scale; a probability below 2^-110 loses at
// most 2^-134, where exp2 itself drops those below 2^-126.
//
// S and dP of odd keys are computed negated, so that the drift of the bf16 MFMA
// (common.h) cancels in a query's sum of dS over its keys, which has to be zero;
// dK and dV alternate their sign along the keys as well as the dims for the column
// sums that bias gradients take of them.
//
// With STORE_DS (causal, lq == lk) the kernel also writes every dS sub-block
// it forms, for flash_bwd_dq_ds_kernel: block (query block i, key block j),
// j <= i, holds 32 x 32 floats at ds + bh * ds_bh + (i (i + 1) / 2 + j) * 1024,
// query row r of the block at [32 r, 32 r + 32) with key 2s + c at 16 c + s,
// which is the operand order of the dQ product (16 contiguous floats per lane).
__host__ __device__ constexpr bool paired_keys(int hd) { return hd > 32; }
template <int HD, bool CAUSAL, bool HAS_MASK, bool VEC, bool STORE_DS>
__global__ void __launch_bounds__(paired_keys(HD) ? 2 * BW_THREADS : BW_THREADS, 2) flash_bwd_dkdv_split_kernel(const BwdArgs a) {
  constexpr int BQ = 32;
  constexpr int NDB = HD / 32;  // 32-wide head-dim blocks of dK^T / dV^T
  constexpr int NS = HD / 16;   // MFMA k-steps of Q.K and dO.V
  constexpr bool PAIRED = paired_keys(HD);
  constexpr int NT = PAIRED ? 1 : 2;  // gradients of a wave: dV or dK, or dV (0) and dK (1)
  typedef QgStage<HD, VEC> Stage;
  __shared__ __attribute__((aligned(16))) char lds[2][Stage::BYTES];
  __shared__ __attribute__((aligned(16))) vf4 Ps[PAIRED ? 4 : 1][4][64];  // P of a pair, as its lanes hold it
  __shared__ __attribute__((aligned(16))) float Ls[2][BQ];   // lse
  __shared__ __attribute__((aligned(16))) float Ds[2][BQ];   // D

  const int n_bh = a.batch * a.heads;
  const int bh = blockIdx.x % n_bh, kt = blockIdx.x / n_bh;
  const int b = bh / a.heads, h = bh % a.heads;
  const int t = threadIdx.x;
  const int lane = t & 63;
  const int wave = __builtin_amdgcn_readfirstlane(t >> 6);
  const int pair = wave & 3;
  const bool role_p = wave < 4;  // P and dV; else dS and dK
  const int li = lane & 31, hf = lane >> 5;
  const int k0 = kt * BW_TILE;
  const int kw0 = k0 + pair * 32;  // first key of this pair
  const int key = kw0 + li;        // this lane's key
  const int col0 = h * (VEC ? HD : a.hd);

  // B operands of S = Q K^T and / or dP = dO V^T: the pieces of K[key][16 s + 8 hf
  // + 0..7] and of V, odd dims negated as in the staged tiles, and odd keys.
  const float sgn = li & 1 ? -1.f : 1.f;
  bf16x8 kv[NT][NS][3];
#pragma unroll
  for (int x = 0; x < NT; ++x) {
    const size_t kr = (size_t)b * a.lk + min(key, a.lk - 1);
    const float *row = (PAIRED ? role_p : x == 0) ? a.k + kr * a.ldk + col0 : a.v + kr * a.ldv + col0;
#pragma unroll
    for (int s = 0; s < NS; ++s) {
      float f[8];
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        const int d = 16 * s + 8 * hf + e;
        const float v = VEC || d < a.hd ? row[d] : 0.f;
        f[e] = e & 1 ? -v : v;
      }
      split_operand(f, sgn * kSplitScale, kv[x][s]);
    }
  }

  const int q_begin = CAUSAL ? k0 : 0;  // queries before k0 see none of these keys
  const int n_it = q_begin < a.lq ? (a.lq - q_begin + BQ - 1) / BQ : 0;
  const float *__restrict__ qbase = a.q + (size_t)b * a.lq * a.ldq + col0;
  const float *__restrict__ gbase = a.dout + (size_t)b * a.lq * a.lddo + col0;
  const float *__restrict__ lse = a.lse + (size_t)bh * a.lq;
  const float *__restrict__ dlt = a.delta + (size_t)bh * a.lq;

  floatx16 acc[NT][NDB], cor[NT][NDB];  // hh, and its corrections
#pragma unroll
  for (int x = 0; x < NT; ++x)
#pragma unroll
    for (int db = 0; db < NDB; ++db)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[x][db][r] = cor[x][db][r] = 0.f;

  // P = exp2(S scale log2 e - lse) in place; scale_log2 carries the sign of an
  // odd key and undoes the split's scale.  l4(g): lse of query rows 8 g + 4 hf + 0..3 of the sub-block.
  auto probabilities = [&](floatx16 &s, float scale_log2, int qb0, auto l4) {
    // (the masked and the unmasked forms are separate branches: a select
    // per element would run the mask arithmetic on every sub-block)
    const bool need = HAS_MASK || (CAUSAL && qb0 < kw0 + 31) || qb0 + 31 >= a.lq;
    if (need) {
#pragma unroll
      for (int g = 0; g < 4; ++g) {
        const vf4 l = l4(g);
#pragma unroll
        for (int c = 0; c < 4; ++c) {
          const int r = 4 * g + c;
          const int qq = qb0 + 8 * g + 4 * hf + c;
          bool ok = qq < a.lq;
          if (CAUSAL) ok = ok && key <= qq;
          if (HAS_MASK) ok = ok && key < a.lk && a.mask[(size_t)min(qq, a.lq - 1) * a.lk + min(key, a.lk - 1)];
          s[r] = ok ? fast_exp2(fmaf(s[r], scale_log2, -l[c])) : 0.f;
        }
      }
    } else {
#pragma unroll
      for (int g = 0; g < 4; ++g) {
        const vf4 l = l4(g);
#pragma unroll
        for (int c = 0; c < 4; ++c) s[4 * g + c] = fast_exp2(fmaf(s[4 * g + c], scale_log2, -l[c]));
      }
    }
  };
  // dS = P (f dP - D) in place of dP, and the dS store.
  auto score_gradients = [&](const floatx16 &p, floatx16 &dp, float f, int qb0, auto d4) {
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      const vf4 d = d4(g);
#pragma unroll
      for (int c = 0; c < 4; ++c) dp[4 * g + c] = p[4 * g + c] * fmaf(f, dp[4 * g + c], -d[c]);
    }
    if constexpr (STORE_DS) {
      // The stored dS blocks of this (sequence, head) as a buffer resource (the
      // launch keeps ds_bh * 4 bytes within 2^31): the block's byte offset in a
      // scalar register, this lane's fixed offset plus the row's immediate (one
      // VGPR of address).  Non-temporal (the nt bit): the blocks stream to HBM
      // rather than sitting dirty in the caches, where the dQ pass's reads would
      // evict and write them back under its own traffic.
      const __amdgpu_buffer_rsrc_t ds_rsrc = __builtin_amdgcn_make_buffer_rsrc(a.ds + (size_t)bh * a.ds_bh, (short)0,
                                                                               (int)(a.ds_bh * 4), kBufferWord3);
      const int ds_lane = 4 * (4 * hf * 32 + (li & 1) * 16 + (li >> 1));
      const int qi = qb0 >> 5, kj = kw0 >> 5;
      const int boff = (qi * (qi + 1) / 2 + kj) * 4096;
#pragma unroll
      for (int r = 0; r < 16; ++r)
        __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(dp[r]), ds_rsrc, ds_lane + 128 * acc_row(r), boff,
                                              kCachePolicyNT);
    }
  };
  // The 32 x 32 product of the staged rows of one tensor with K's or V's pieces.
  const int ro = Stage::roperand(li, hf), to = Stage::toperand(li, hf);
  auto row_product = [&](const char *rows, const bf16x8 (&w)[NS][3]) {
    floatx16 m = {}, c = {};
#pragma unroll
    for (int u = 0; u < NS; ++u) {
      bf16x8 x[3];
#pragma unroll
      for (int p = 0; p < 3; ++p)
        x[p] = *reinterpret_cast<const bf16x8 *>(rows + ro + p * Stage::RPLANE + u * Stage::RSLAB);
#pragma unroll
      for (int i = 0; i < kSplitProducts; ++i) {
        floatx16 &z = i == kSplitMain ? m : c;
        z = mfma32x32x16(x[kSplitA[i]], w[u][kSplitB[i]], z);
      }
    }
#pragma unroll
    for (int r = 0; r < 16; ++r) m[r] += c[r];
    return m;
  };
  // acc[n] += (the staged transposed rows of one tensor) x w, w the 32 x 32 P or dS
  // times ws.
  auto column_product = [&](const char *cols, const floatx16 &w, float ws, int n) {
#pragma unroll
    for (int st = 0; st < 2; ++st) {
      float x[8];
#pragma unroll
      for (int e = 0; e < 8; ++e) x[e] = w[8 * st + e];
      bf16x8 wp[3];
      split_operand(x, ws, wp);
#pragma unroll
      for (int db = 0; db < NDB; ++db) {
        bf16x8 g[3];
#pragma unroll
        for (int p = 0; p < 3; ++p)
          g[p] = *reinterpret_cast<const bf16x8 *>(cols + to + p * Stage::TPLANE + st * Stage::TSLAB + db * 256);
#pragma unroll
        for (int i = 0; i < kSplitProducts; ++i) {
          floatx16 &z = i == kSplitMain ? acc[n][db] : cor[n][db];
          z = mfma32x32x16(g[kSplitA[i]], wp[kSplitB[i]], z);
        }
      }
    }
  };
  // Sub-blocks wholly before these keys contribute nothing, and keys that all
  // lie past lk take nothing.
  auto active = [&](int qb0) { return kw0 < a.lk && !(CAUSAL && qb0 + 31 < kw0); };
  // Both operands of S and dP carry the split's scale.  dK of odd keys, and dV of
  // every other workgroup along a head's rows (through dO), are summed negated.
  const float gsgn = (kt + b) & 1 ? -1.f : 1.f;
  const float s_scale = sgn * kSplitUnscale2 * a.scale_log2, dp_scale = sgn * gsgn * kSplitUnscale2;
  const float ds_scale = sgn * kSplitScale;
  constexpr float p_scale = 1.f;

  auto lse4 = [&](int buf) {
    return [&, buf](int g) { return *reinterpret_cast<const vf4 *>(&Ls[buf][8 * g + 4 * hf]); };
  };
  auto delta4 = [&](int buf) {
    return [&, buf](int g) { return *reinterpret_cast<const vf4 *>(&Ds[buf][8 * g + 4 * hf]); };
  };

  if (!PAIRED || role_p) {
    // Where waves are paired, the staging ones store nothing to memory, so that
    // waiting for a tile's loads never waits for the dS stores.
    Stage sg;
    sg.init();
    float lreg = 0.f, dreg = 0.f;
    auto fetch = [&](int it) {  // past the end: the last tile again, into a buffer that nothing reads
      const int row0 = q_begin + min(it, n_it - 1) * BQ;
      sg.load(qbase, gbase, a.ldq, a.lddo, row0, a.lq, a.hd);
      if (t < BQ) {
        const int qq = min(row0 + t, a.lq - 1);
        lreg = lse[qq];
        dreg = dlt[qq];
      }
    };
    auto stage = [&](int buf) {
      sg.store(lds[buf], gsgn * kSplitScale);
      if (t < BQ) {
        Ls[buf][t] = lreg;
        Ds[buf][t] = dreg;
      }
    };
    if (n_it > 0) {
      fetch(0);
      stage(0);
    }
    __syncthreads();
    for (int it = 0; it < n_it; ++it) {
      const int cur = it & 1, qb0 = q_begin + it * BQ;
      fetch(it + 1);
      floatx16 p;
      if (active(qb0)) {
        p = row_product(lds[cur], kv[0]);
        if constexpr (PAIRED) {
          probabilities(p, s_scale, qb0, lse4(cur));
#pragma unroll
          for (int g = 0; g < 4; ++g) Ps[pair][g][lane] = vf4{p[4 * g], p[4 * g + 1], p[4 * g + 2], p[4 * g + 3]};
        } else {
          floatx16 dp = row_product(lds[cur] + Stage::TENSOR, kv[NT - 1]);
          probabilities(p, s_scale, qb0, lse4(cur));
          column_product(lds[cur] + Stage::TENSOR, p, p_scale, 0);
          score_gradients(p, dp, dp_scale, qb0, delta4(cur));
          column_product(lds[cur], dp, ds_scale, NT - 1);
        }
      }
      if constexpr (PAIRED) {
        __syncthreads();
        if (active(qb0)) column_product(lds[cur] + Stage::TENSOR, p, p_scale, 0);  // dV^T += dO^T P
      }
      stage(cur ^ 1);
      __syncthreads();
    }
  } else {
    __syncthreads();
    for (int it = 0; it < n_it; ++it) {
      const int cur = it & 1, qb0 = q_begin + it * BQ;
      floatx16 dp;
      if (active(qb0)) dp = row_product(lds[cur] + Stage::TENSOR, kv[0]);
      __syncthreads();
      if (active(qb0)) {
        floatx16 p;
#pragma unroll
        for (int g = 0; g < 4; ++g) {
          const vf4 x = Ps[pair][g][lane];
#pragma unroll
          for (int c = 0; c < 4; ++c) p[4 * g + c] = x[c];
        }
        score_gradients(p, dp, dp_scale, qb0, delta4(cur));
        column_product(lds[cur], dp, ds_scale, 0);  // dK^T += Q^T dS
      }
      __syncthreads();
    }
  }

  // odd dims (registers of odd index) were negated
  float bad = 0.f;
#pragma unroll
  for (int n = 0; n < NT; ++n) {
    const bool of_v = PAIRED ? role_p : n == 0;
    const float f = of_v ? gsgn * kSplitUnscale : sgn * kSplitUnscale2;
#pragma unroll
    for (int db = 0; db < NDB; ++db) {
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[n][db][r] = (acc[n][db][r] + cor[n][db][r]) * (r & 1 ? -f : f);
      bad = nonfinite_sum(acc[n][db], bad);
    }
  }
  if (any_nonfinite(bad) && kw0 < a.lk) {
    // An infinity or a NaN reached these keys, or a product overflowed: the
    // whole column on the fp32 MFMA straight from memory, dS blocks included.
#pragma unroll
    for (int n = 0; n < NT; ++n)
#pragma unroll
      for (int db = 0; db < NDB; ++db)
#pragma unroll
        for (int r = 0; r < 16; ++r) acc[n][db][r] = 0.f;
    const size_t krow = (size_t)b * a.lk + min(key, a.lk - 1);
#pragma unroll 1
    for (int qb0 = CAUSAL ? kw0 : 0; qb0 < a.lq; qb0 += 32) {
      floatx16 s = {}, dp = {};
      const size_t qrow = min(qb0 + li, a.lq - 1);
#pragma unroll 1
      for (int d = hf; d < a.hd + hf; d += 2) {
        const bool in = d < a.hd;
        const int dc = in ? d : 0;
        s = mfma32x32x2(in ? qbase[qrow * a.ldq + dc] : 0.f, in ? a.k[krow * a.ldk + col0 + dc] : 0.f, s);
        dp = mfma32x32x2(in ? gbase[qrow * a.lddo + dc] : 0.f, in ? a.v[krow * a.ldv + col0 + dc] : 0.f, dp);
      }
      auto four = [&](const float *x, int g) {
        vf4 v;
#pragma unroll
        for (int c = 0; c < 4; ++c) v[c] = x[min(qb0 + 8 * g + 4 * hf + c, a.lq - 1)];
        return v;
      };
      probabilities(s, a.scale_log2, qb0, [&](int g) { return four(lse, g); });
      if (!PAIRED || !role_p) score_gradients(s, dp, 1.f, qb0, [&](int g) { return four(dlt, g); });
#pragma unroll
      for (int n = 0; n < NT; ++n) {
        const bool of_v = PAIRED ? role_p : n == 0;
        const float *base = of_v ? gbase : qbase;
        const int ld = of_v ? a.lddo : a.ldq;
#pragma unroll
        for (int st = 0; st < 16; ++st) {
          const size_t qr = min(qb0 + acc_row(st) + 4 * hf, a.lq - 1);
#pragma unroll
          for (int db = 0; db < NDB; ++db) {
            const int d = db * 32 + li;
            acc[n][db] = mfma32x32x2(d < a.hd ? base[qr * ld + d] : 0.f, of_v ? s[st] : dp[st], acc[n][db]);
          }
        }
      }
    }
  }
  if (key < a.lk) {
    const size_t krow = (size_t)b * a.lk + key;
#pragma unroll
    for (int n = 0; n < NT; ++n) {
      if (PAIRED ? role_p : n == 0) store_column<HD, VEC>(a, acc[n], a.dv + krow * a.lddv + col0, 1.f, nullptr, hf);
      else store_column<HD, VEC>(a, acc[n], a.dk + krow * a.lddk + col0, a.scale,
                                 a.rope_cs ? a.rope_cs + (size_t)key * (a.hd >> 1) : nullptr, hf);
    }
  }
}

// dQ.  Query-tile major with the heaviest causal tiles first, as the forward.
template <int HD, int BN, bool CAUSAL, bool HAS_MASK, bool VEC>
__global__ void __launch_bounds__(BW_THREADS, 2) flash_bwd_dq_kernel(const BwdArgs a) {
  constexpr int NKB = BN / 32;
  constexpr int NDB = HD / 32;
  constexpr int NKG = HD / 8;
  __shared__ __attribute__((aligned(16))) float Ks[2][BN][HD + 4];
  __shared__ __attribute__((aligned(16))) float Vs[2][BN][HD + 4];

  const int n_bh = a.batch * a.heads;
  const int bh = blockIdx.x % n_bh;
  int qt = blockIdx.x / n_bh;
  if (CAUSAL) qt = a.n_tiles - 1 - qt;
  const int b = bh / a.heads, h = bh % a.heads;
  const int t = threadIdx.x;
  const int lane = t & 63;
  const int wave = __builtin_amdgcn_readfirstlane(t >> 6);
  const int li = lane & 31, hf = lane >> 5;
  const int q0 = qt * BW_TILE;
  const int qw0 = q0 + wave * 32;
  const int qi = qw0 + li;
  const int qc = min(qi, a.lq - 1);
  const int col0 = h * (VEC ? HD : a.hd);

  // B operands of S^T = K Q^T and dP^T = V dO^T: register 4u + r holds
  // Q[qi][8u + 4*hf + r] (and likewise dO).
  float qreg[HD / 2], greg[HD / 2];
  {
    const float *qrow = a.q + ((size_t)b * a.lq + qc) * a.ldq + col0;
    const float *grow = a.dout + ((size_t)b * a.lq + qc) * a.lddo + col0;
#pragma unroll
    for (int u = 0; u < NKG; ++u) {
      const int d = 8 * u + 4 * hf;
      if constexpr (VEC) {
        const vf4 x = *reinterpret_cast<const vf4 *>(qrow + d);
        const vf4 y = *reinterpret_cast<const vf4 *>(grow + d);
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          qreg[4 * u + r] = x[r];
          greg[4 * u + r] = y[r];
        }
      } else {
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          qreg[4 * u + r] = d + r < a.hd ? qrow[d + r] : 0.f;
          greg[4 * u + r] = d + r < a.hd ? grow[d + r] : 0.f;
        }
      }
    }
  }
  const float lse_q = a.lse[(size_t)bh * a.lq + qc];
  const float d_q = a.delta[(size_t)bh * a.lq + qc];
  const int key_last = CAUSAL ? min(qi, a.lk - 1) : a.lk - 1;
  const uint8_t *mrow = HAS_MASK ? a.mask + (size_t)qc * a.lk : nullptr;

  const int kend = CAUSAL ? min(q0 + BW_TILE, a.lk) : a.lk;
  const int n_kt = (kend + BN - 1) / BN;
  const float *__restrict__ kbase = a.k + (size_t)b * a.lk * a.ldk + col0;
  const float *__restrict__ vbase = a.v + (size_t)b * a.lk * a.ldv + col0;

  floatx16 dq[NDB];
#pragma unroll
  for (int db = 0; db < NDB; ++db)
#pragma unroll
    for (int r = 0; r < 16; ++r) dq[db][r] = 0.f;
  const floatx16 zero = {};

  RowStage<HD, BN, VEC> sk, sv;
  sk.init(a.ldk);
  sv.init(a.ldv);
  sk.load(kbase, a.ldk, 0, a.lk, a.hd);
  sv.load(vbase, a.ldv, 0, a.lk, a.hd);
  sk.store(Ks[0]);
  sv.store(Vs[0]);
  __syncthreads();

  for (int kt = 0; kt < n_kt; ++kt) {
    const int cur = kt & 1;
    const int k0 = kt * BN;
    const int nxt = kt + 1 < n_kt ? k0 + BN : k0;
    sk.load(kbase, a.ldk, nxt, a.lk, a.hd);
    sv.load(vbase, a.ldv, nxt, a.lk, a.hd);

#pragma unroll
    for (int kb = 0; kb < NKB; ++kb) {
      const int kb0 = k0 + kb * 32;
      if (kb0 >= a.lk || qw0 >= a.lq || (CAUSAL && kb0 > qw0 + 31)) continue;  // nothing to add
      const float(*krow)[HD + 4] = &Ks[cur][kb * 32];
      const float(*vrow)[HD + 4] = &Vs[cur][kb * 32];

      // S^T = K Q^T and dP^T = V dO^T
      floatx16 s, dp;
      vf4 ka = *reinterpret_cast<const vf4 *>(&krow[li][4 * hf]);
      vf4 va = *reinterpret_cast<const vf4 *>(&vrow[li][4 * hf]);
#pragma unroll
      for (int u = 0; u < NKG; ++u) {
        vf4 kn, vn;
        if (u + 1 < NKG) {
          kn = *reinterpret_cast<const vf4 *>(&krow[li][8 * (u + 1) + 4 * hf]);
          vn = *reinterpret_cast<const vf4 *>(&vrow[li][8 * (u + 1) + 4 * hf]);
        }
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          s = mfma32x32x2(ka[r], qreg[4 * u + r], (u == 0 && r == 0) ? zero : s);
          dp = mfma32x32x2(va[r], greg[4 * u + r], (u == 0 && r == 0) ? zero : dp);
        }
        if (u + 1 < NKG) {
          ka = kn;
          va = vn;
        }
      }

      // dS^T = P^T (dP^T - D); register r holds key kb0 + acc_row(r) + 4*hf.
      const bool need = HAS_MASK || kb0 + 31 > (CAUSAL ? min(qw0, a.lk - 1) : a.lk - 1);
      const int thr = key_last - kb0 - 4 * hf;
      if (need) {  // separate branches, as in the dK/dV kernel
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          bool ok = acc_row(r) <= thr;
          if (HAS_MASK) ok = ok && mrow[min(kb0 + acc_row(r) + 4 * hf, a.lk - 1)] != 0;
          const float p = ok ? fast_exp2(fmaf(s[r], a.scale_log2, -lse_q)) : 0.f;
          dp[r] = p * (dp[r] - d_q);
        }
      } else {
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          const float p = fast_exp2(fmaf(s[r], a.scale_log2, -lse_q));
          dp[r] = p * (dp[r] - d_q);
        }
      }

      // dQ^T += K^T dS^T
#pragma unroll
      for (int st = 0; st < 16; ++st) {
        const int kr = acc_row(st) + 4 * hf;
#pragma unroll
        for (int db = 0; db < NDB; ++db) dq[db] = mfma32x32x2(krow[kr][db * 32 + li], dp[st], dq[db]);
      }
    }

    sk.store(Ks[cur ^ 1]);
    sv.store(Vs[cur ^ 1]);
    __syncthreads();
  }

  if (qi < a.lq)
    store_column<HD, VEC>(a, dq, a.dq + ((size_t)b * a.lq + qi) * a.lddq + col0, a.scale,
                          a.rope_cs ? a.rope_cs + (size_t)qi * (a.hd >> 1) : nullptr, hf);
}

// Stores a 32-row block of dQ from accumulators that hold dQ[q][d] with d in the
// lanes: register r of block db is row q0 + 8 (r / 4) + 4 hf + r % 4, column db * 32
// + li, so 32 lanes write 128 contiguous bytes (lanes that hold 16 bytes of 32
// different rows cost the pass 28 us of 320 at 256 x 511, 8 heads of 32).  x is
// multiplied by scale and rotated back by the rows' pairs of rope_cs when
// non-NULL; the partner of a column is in the neighbouring lane.
template <int HD>
struct RowStore {
  static constexpr int NDB = HD / 32;
  float2 cs[NDB][16];  // loaded before any store (a load issued after a store waits for it)
  __device__ __forceinline__ void load(const BwdArgs &a, int q0, int li, int hf) {
    if (!a.rope_cs) return;
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      const float2 *row = a.rope_cs + (size_t)min(q0 + acc_row(r) + 4 * hf, a.lq - 1) * (HD / 2) + (li >> 1);
#pragma unroll
      for (int db = 0; db < NDB; ++db) cs[db][r] = row[db * 16];
    }
  }
  __device__ __forceinline__ void store(const BwdArgs &a, const floatx16 (&x)[NDB], int b, int q0, int col0, int li,
                                        int hf) const {
#pragma clang fp contract(off)
    float *base = a.dq + ((size_t)b * a.lq + q0) * a.lddq + col0 + li;
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      const int row = acc_row(r) + 4 * hf;
#pragma unroll
      for (int db = 0; db < NDB; ++db) {
        float y = x[db][r] * a.scale;
        if (a.rope_cs) {  // rope_inverse_pair on (y, partner), in every lane
          const float z = __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(y), 0xB1, 0xF, 0xF, false));
          const float c = cs[db][r].x, s = -cs[db][r].y;
          y = li & 1 ? z * s + y * c : y * c - z * s;
        }
        if (q0 + row < a.lq) base[(size_t)row * a.lddq + db * 32] = y;
      }
    }
  }
};

// K^T tile of the stored-dS dQ kernel: BN keys of one head as 16-value rows of
// dims (slab s holds keys 16 s .. 16 s + 15, key k of a slab at place
// 8 (k % 2) + k / 2, the order of the stored dS operands), split into three bf16
// planes.  A unit is four dims of two keys of equal parity; clusters by d % 4.
template <int HD, int BN>
struct KtStage {
  static constexpr int CH = HD / 4;
  static constexpr int NU = CH * (BN / 2) / BW_THREADS;
  static constexpr int SLAB = 4 * (CH * 32) + 256, PLANE = BN / 16 * SLAB, BYTES = 3 * PLANE;
  static_assert(NU >= 1 && CH * (BN / 2) % BW_THREADS == 0 && (BW_THREADS / 8) % CH == 0, "tile units");
  static __device__ __forceinline__ constexpr int cluster(int c) { return c * CH * 32 + (c & 1) * 16 + (c >> 1) * 128; }
  // Keys row and row + 2 of unit (slab, dim group, sb), its place, and its pieces' stores.
  static __device__ __forceinline__ int unit_row(int slab, int sb) { return 16 * slab + 4 * (sb >> 1) + (sb & 1); }
  static __device__ __forceinline__ int unit_dst(int slab, int g, int sb) {
    return slab * SLAB + g * 32 + ((sb & 1) * 4 + (sb >> 1)) * 4;
  }
  static __device__ __forceinline__ void put(char *d, int plane, const vf4 &r0, const vf4 &r1) {
#pragma unroll
    for (int c = 0; c < 4; ++c) {
      uint32_t h, m, l;
      const float f = c & 1 ? -kSplitScale : kSplitScale;
      split_bf16x3(r0[c] * f, r1[c] * f, h, m, l);
      *reinterpret_cast<uint32_t *>(d + cluster(c)) = h;
      *reinterpret_cast<uint32_t *>(d + cluster(c) + plane) = m;
      *reinterpret_cast<uint32_t *>(d + cluster(c) + 2 * plane) = l;
    }
  }
  vf4 r[NU][2];
  int row, col, dst;
  __device__ __forceinline__ void init() {
    const int t = threadIdx.x, sb = t & 7, g = (t >> 3) % CH, slab = (t >> 3) / CH;
    row = unit_row(slab, sb);
    col = 4 * g;
    dst = unit_dst(slab, g, sb);
  }
  __device__ __forceinline__ void load(const float *__restrict__ base, int ld, int row0, int nrows) {
    const float *tile = base + (size_t)row0 * ld;
#pragma unroll
    for (int i = 0; i < NU; ++i)
#pragma unroll
      for (int x = 0; x < 2; ++x)
        r[i][x] = *reinterpret_cast<const vf4 *>(
            tile + (uint32_t)(min(row + 16 * (BW_THREADS / 8 / CH) * i + 2 * x, nrows - 1 - row0) * ld + col));
  }
  __device__ __forceinline__ void store(char *lds) const {
#pragma unroll
    for (int i = 0; i < NU; ++i) put(lds + dst + BW_THREADS / 8 / CH * SLAB * i, PLANE, r[i][0], r[i][1]);
  }
  static __device__ __forceinline__ int operand(int li, int hf) { return cluster(li & 3) + (li >> 2) * 32 + hf * 16; }
};

// One 32-key block of dQ = dS K: cur is this lane's dS operand, kt its K^T operand
// of plane 0, first slab of the block.  Odd queries and odd dims are computed
// negated (common.h).
template <int HD>
__device__ __forceinline__ void dq_block(const vf4 (&cur)[4], float ds_scale, const char *kt, int plane, int slab,
                                         floatx16 (&dq)[HD / 32], floatx16 (&dqc)[HD / 32]) {
#pragma unroll
  for (int st = 0; st < 2; ++st) {
    float x[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) x[e] = cur[2 * st + (e >> 2)][e & 3];
    bf16x8 ds[3];
    split_operand(x, ds_scale, ds);
#pragma unroll
    for (int db = 0; db < HD / 32; ++db) {
      bf16x8 k[3];
#pragma unroll
      for (int p = 0; p < 3; ++p) k[p] = *reinterpret_cast<const bf16x8 *>(kt + p * plane + st * slab + db * 256);
#pragma unroll
      for (int i = 0; i < kSplitProducts; ++i) {
        floatx16 &c = i == kSplitMain ? dq[db] : dqc[db];
        c = mfma32x32x16(ds[kSplitA[i]], k[kSplitB[i]], c);
      }
    }
  }
}

// Joins the two accumulators and undoes scale and signs (register r holds a query of
// r's parity, lane li a dim of li's); whether some row came out non-finite
// (wave-uniform).
template <int HD>
__device__ __forceinline__ bool dq_finish(floatx16 (&dq)[HD / 32], const floatx16 (&dqc)[HD / 32], int li) {
  const float f = li & 1 ? -kSplitUnscale2 : kSplitUnscale2;
  float bad = 0.f;
#pragma unroll
  for (int db = 0; db < HD / 32; ++db) {
#pragma unroll
    for (int r = 0; r < 16; ++r) dq[db][r] = (dq[db][r] + dqc[db][r]) * (r & 1 ? -f : f);
    bad = nonfinite_sum(dq[db], bad);
  }
  return any_nonfinite(bad);
}

// Query block qi on the fp32 MFMA straight from memory (see the dK/dV kernel); dsw:
// this lane's part of its dS blocks.
template <int HD>
__device__ __forceinline__ void dq_recompute(const BwdArgs &a, const float *kbase, const float *dsw, int qi, int li,
                                             int hf, floatx16 (&dq)[HD / 32]) {
#pragma unroll
  for (int db = 0; db < HD / 32; ++db)
#pragma unroll
    for (int r = 0; r < 16; ++r) dq[db][r] = 0.f;
#pragma unroll 1
  for (int j = 0; j <= qi; ++j)
#pragma unroll 1
    for (int s = 0; s < 16; ++s) {
      const float x = dsw[(size_t)j * 1024 + s];
      const float *krow = kbase + (size_t)min(32 * j + 2 * s + hf, a.lk - 1) * a.ldk;
#pragma unroll
      for (int db = 0; db < HD / 32; ++db) dq[db] = mfma32x32x2(x, krow[db * 32 + li], dq[db]);
    }
}

// dQ from the dS blocks that the dK/dV kernel stored (causal, lq == lk, 16-byte
// aligned rows): dQ = scale dS K, one product instead of recomputing S and dP, on
// three bf16 pieces per fp32 operand (common.h).  Query-tile major with
// the heaviest tiles first, as the forward.  Wave w owns query block i = q0 / 32 +
// w; for its key blocks j <= i the dS operand (dS[q][2s + c], s = 0..15, in lane
// (q, c)) is 16 contiguous floats per lane, loaded two blocks ahead, and K^T
// streams through double-buffered LDS as the other operand.  The blocks' bytes
// bound it: 2.1 GB in 0.60 ms at 4 x 4096, 16 heads of 64.
template <int HD, int BN>
__global__ void __launch_bounds__(BW_THREADS, 2) flash_bwd_dq_ds_kernel(const BwdArgs a) {
  constexpr int NKB = BN / 32;
  constexpr int NDB = HD / 32;
  typedef KtStage<HD, BN> Stage;
  __shared__ __attribute__((aligned(16))) char lds[2][Stage::BYTES];

  const int n_bh = a.batch * a.heads;
  const int bh = blockIdx.x % n_bh;
  const int qt = a.n_tiles - 1 - (int)(blockIdx.x / n_bh);
  const int b = bh / a.heads, h = bh % a.heads;
  const int t = threadIdx.x;
  const int lane = t & 63;
  const int wave = __builtin_amdgcn_readfirstlane(t >> 6);
  const int li = lane & 31, hf = lane >> 5;
  const int q0 = qt * BW_TILE;
  const int qw0 = q0 + wave * 32;
  const int qi = qw0 >> 5;                    // this wave's query block
  const int last = qw0 < a.lq ? qi : -1;      // its last key block (none past the end)
  const int col0 = h * HD;
  const float *__restrict__ kbase = a.k + (size_t)b * a.lk * a.ldk + col0;
  const float *__restrict__ dsw = a.ds + (size_t)bh * a.ds_bh + (size_t)qi * (qi + 1) / 2 * 1024 + li * 32 + hf * 16;

  floatx16 dq[NDB], dqc[NDB];  // hh, and its corrections
#pragma unroll
  for (int db = 0; db < NDB; ++db)
#pragma unroll
    for (int r = 0; r < 16; ++r) dq[db][r] = dqc[db][r] = 0.f;

  const int kend = min(q0 + BW_TILE, a.lk);
  const int n_kt = (kend + BN - 1) / BN;
  Stage sk;
  sk.init();
  sk.load(kbase, a.ldk, 0, a.lk);
  sk.store(lds[0]);
  // dS operands two blocks ahead: cur (block j), n1 (j + 1), n2 (j + 2)
  vf4 cur[4], n1[4], n2[4];
  if (last >= 0) {
#pragma unroll
    for (int i = 0; i < 4; ++i) cur[i] = *reinterpret_cast<const vf4 *>(dsw + 4 * i);
  }
  if (last >= 1) {
#pragma unroll
    for (int i = 0; i < 4; ++i) n1[i] = *reinterpret_cast<const vf4 *>(dsw + 1024 + 4 * i);
  }
  __syncthreads();

  const int ko = Stage::operand(li, hf);
  const float ds_scale = li & 1 ? -kSplitScale : kSplitScale;
  for (int kt = 0; kt < n_kt; ++kt) {
    const int lbuf = kt & 1;
    const int k0 = kt * BN;
    sk.load(kbase, a.ldk, kt + 1 < n_kt ? k0 + BN : k0, a.lk);
#pragma unroll
    for (int kb = 0; kb < NKB; ++kb) {
      const int j = kt * NKB + kb;  // key block
      if (j > last) continue;
      if (j + 2 <= last) {
#pragma unroll
        for (int i = 0; i < 4; ++i) n2[i] = *reinterpret_cast<const vf4 *>(dsw + (size_t)(j + 2) * 1024 + 4 * i);
      }
      dq_block<HD>(cur, ds_scale, lds[lbuf] + ko + 2 * kb * Stage::SLAB, Stage::PLANE, Stage::SLAB, dq, dqc);
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        cur[i] = n1[i];
        n1[i] = n2[i];
      }
    }
    sk.store(lds[lbuf ^ 1]);
    __syncthreads();
  }

  if (last < 0) return;
  if (dq_finish<HD>(dq, dqc, li)) dq_recompute<HD>(a, kbase, dsw, qi, li, hf, dq);
  RowStore<HD> out;
  out.load(a, qw0, li, hf);
  out.store(a, dq, b, qw0, col0, li, hf);
}

// The same product, in the same order, for sequences of head dim 32 up to 32 *
// kShortQB long: one workgroup per (sequence, head) stages the pieces of the head's
// whole K^T once (flash_bwd_dq_ds_kernel's workgroups read K 2.5 times over at 512
// queries: 1482 instead of 1276 MB for 2048 heads); wave w owns query blocks w and
// nqb - 1 - w, so every wave has nqb + 1 key blocks of work (the middle block of an
// odd count alone) and no barrier follows the staging.
constexpr int kShortQB = 16;
__global__ void __launch_bounds__(32 * kShortQB, 2) flash_bwd_dq_ds_short_kernel(const BwdArgs a) {
  constexpr int HD = 32;
  typedef KtStage<HD, 64> Stage;
  constexpr int NDB = HD / 32, CH = HD / 4, PLANE = 2 * kShortQB * Stage::SLAB;
  constexpr int PF = 4;
  __shared__ __attribute__((aligned(16))) char lds[3 * PLANE];
  const int bh = blockIdx.x;
  const int b = bh / a.heads, h = bh % a.heads;
  const int t = threadIdx.x;
  const int lane = t & 63;
  const int wave = __builtin_amdgcn_readfirstlane(t >> 6);
  const int li = lane & 31, hf = lane >> 5;
  const int nqb = (a.lq + 31) >> 5;
  const int col0 = h * HD;
  const float *__restrict__ kbase = a.k + (size_t)b * a.lk * a.ldk + col0;
  const float *__restrict__ dsbh = a.ds + (size_t)bh * a.ds_bh + li * 32 + hf * 16;
  // dS operands PF blocks ahead in a ring: block j lives in buf[j % PF] (the loop
  // is unrolled by PF, so every index is a constant and no load in flight is ever
  // copied), and the load of block j + PF goes into the buffer that block j has
  // just left.  The second query block's first loads go out before the first
  // one's stores.
  vf4 buf[PF][4];
  auto fetch = [&](vf4 (&x)[4], int qi, int j) {
    if (j <= qi) {
#pragma unroll
      for (int i = 0; i < 4; ++i)
        x[i] = *reinterpret_cast<const vf4 *>(dsbh + ((size_t)qi * (qi + 1) / 2 + j) * 1024 + 4 * i);
    }
  };
#pragma unroll
  for (int p = 0; p < PF; ++p) fetch(buf[p], nqb - 1 - wave, p);
  // K rows [0, 32 nqb) of the head, rows past lk clamped (their dS is 0)
  for (int e = t; e < nqb * 16 * CH; e += blockDim.x) {
    const int sb = e & 7, g = (e >> 3) % CH, slab = (e >> 3) / CH;
    const int row = Stage::unit_row(slab, sb);
    const vf4 r0 = *reinterpret_cast<const vf4 *>(kbase + (size_t)min(row, a.lk - 1) * a.ldk + 4 * g);
    const vf4 r1 = *reinterpret_cast<const vf4 *>(kbase + (size_t)min(row + 2, a.lk - 1) * a.ldk + 4 * g);
    Stage::put(lds + Stage::unit_dst(slab, g, sb), PLANE, r0, r1);
  }
  __syncthreads();
  const int ko = Stage::operand(li, hf);
  const float ds_scale = li & 1 ? -kSplitScale : kSplitScale;
#pragma unroll 1
  for (int pass = 0; pass < 2; ++pass) {
    const int qi = pass == 0 ? nqb - 1 - wave : wave;
    if (pass == 1 && qi >= nqb - 1 - wave) break;  // the middle block ran in pass 0
    floatx16 dq[NDB], dqc[NDB];                     // hh, and its corrections
#pragma unroll
    for (int db = 0; db < NDB; ++db)
#pragma unroll
      for (int r = 0; r < 16; ++r) dq[db][r] = dqc[db][r] = 0.f;
    for (int j0 = 0; j0 <= qi; j0 += PF) {
#pragma unroll
      for (int u = 0; u < PF; ++u) {
        const int j = j0 + u;
        if (j > qi) break;
        dq_block<HD>(buf[u], ds_scale, lds + ko + 2 * j * Stage::SLAB, PLANE, Stage::SLAB, dq, dqc);
        fetch(buf[u], qi, j + PF);
      }
    }
    RowStore<HD> out;
    out.load(a, 32 * qi, li, hf);
    if (pass == 0 && wave < nqb - 1 - wave) {
#pragma unroll
      for (int p = 0; p < PF; ++p) fetch(buf[p], wave, p);
    }
    if (dq_finish<HD>(dq, dqc, li)) dq_recompute<HD>(a, kbase, dsbh + (size_t)qi * (qi + 1) / 2 * 1024, qi, li, hf, dq);
    out.store(a, dq, b, 32 * qi, col0, li, hf);
  }
}

// Any head dim, any strides: one workgroup per (sequence, head) walks the
// queries in order, as AccelerationCPU.cs:1092-1268 does per head, with the
// keys spread over the threads.  scratch holds two floats per key.
__global__ void __launch_bounds__(256) flash_bwd_generic_kernel(const BwdArgs a, float *scratch,
                                                                 int causal) {
  extern __shared__ float sm[];  // q_i[hd] | dout_i[hd] | red[8]
  float *qv = sm, *gv = sm + a.hd, *red = sm + 2 * a.hd;
  const int bh = blockIdx.x;
  const int b = bh / a.heads, h = bh % a.heads;
  const int t = threadIdx.x, hd = a.hd, col0 = h * hd;
  float *w = scratch + (size_t)bh * 2 * a.lk;
  float *da = w + a.lk;
  const float *K = a.k + (size_t)b * a.lk * a.ldk + col0;
  const float *V = a.v + (size_t)b * a.lk * a.ldv + col0;
  float *dK = a.dk + (size_t)b * a.lk * a.lddk + col0;
  float *dV = a.dv + (size_t)b * a.lk * a.lddv + col0;
  for (int j = t; j < a.lk; j += 256)
    for (int d = 0; d < hd; ++d) dK[(size_t)j * a.lddk + d] = dV[(size_t)j * a.lddv + d] = 0.f;

  auto block_max = [&](float x) {
    for (int off = 32; off > 0; off >>= 1) x = fmaxf(x, __shfl_xor(x, off));
    __syncthreads();
    if ((t & 63) == 0) red[t >> 6] = x;
    __syncthreads();
    return fmaxf(fmaxf(red[0], red[1]), fmaxf(red[2], red[3]));
  };
  auto block_sum = [&](float x) {
    for (int off = 32; off > 0; off >>= 1) x += __shfl_xor(x, off);
    __syncthreads();
    if ((t & 63) == 0) red[t >> 6] = x;
    __syncthreads();
    return (red[0] + red[1]) + (red[2] + red[3]);
  };

  for (int i = 0; i < a.lq; ++i) {
    const float *qrow = a.q + ((size_t)b * a.lq + i) * a.ldq + col0;
    const float *grow = a.dout + ((size_t)b * a.lq + i) * a.lddo + col0;
    float *dqrow = a.dq + ((size_t)b * a.lq + i) * a.lddq + col0;
    __syncthreads();
    for (int d = t; d < hd; d += 256) {
      qv[d] = qrow[d];
      gv[d] = grow[d];
    }
    __syncthreads();
    const int visible = causal ? min(i + 1, a.lk) : a.lk;
    float mx = -INFINITY;
    for (int j = t; j < visible; j += 256) {
      float s = -INFINITY;
      if (!a.mask || a.mask[(size_t)i * a.lk + j]) {
        float acc = 0.f;
        for (int d = 0; d < hd; ++d) acc += qv[d] * K[(size_t)j * a.ldk + d];
        s = acc * a.scale;
      }
      w[j] = s;
      mx = fmaxf(mx, s);
    }
    mx = block_max(mx);
    float sum = 0.f;
    if (mx != -INFINITY) {
      for (int j = t; j < visible; j += 256) {
        const float e = w[j] == -INFINITY ? 0.f : expf(w[j] - mx);
        w[j] = e;
        sum += e;
      }
    }
    sum = block_sum(sum);
    if (!(mx != -INFINITY && sum > 0.f)) {  // the row contributes nothing
      for (int d = t; d < hd; d += 256) dqrow[d] = 0.f;
      continue;
    }
    const float inv = 1.0f / sum;
    float rd = 0.f;
    for (int j = t; j < visible; j += 256) {
      const float wj = w[j] * inv;
      float g = 0.f;
      for (int d = 0; d < hd; ++d) g += gv[d] * V[(size_t)j * a.ldv + d];
      w[j] = wj;
      da[j] = g;
      rd += wj * g;
    }
    rd = block_sum(rd);
    for (int j = t; j < visible; j += 256) {
      const float wj = w[j];
      const float dd = wj * (da[j] - rd) * a.scale;
      for (int d = 0; d < hd; ++d) {
        dV[(size_t)j * a.lddv + d] += wj * gv[d];
        if (dd != 0.f) dK[(size_t)j * a.lddk + d] += dd * qv[d];
      }
      da[j] = dd;
    }
    __syncthreads();
    for (int d = t; d < hd; d += 256) {
      float acc = 0.f;
      for (int j = 0; j < visible; ++j) acc += da[j] * K[(size_t)j * a.ldk + d];
      dqrow[d] = acc;
    }
  }
}

// rows x cols block (row stride ld) set to zero.
__global__ void __launch_bounds__(256) zero_rows_kernel(float *p, long long rows, int cols, int ld) {
  const long long n = rows * cols;
  for (long long e = (long long)blockIdx.x * 256 + threadIdx.x; e < n; e += (long long)gridDim.x * 256)
    p[(e / cols) * ld + e % cols] = 0.f;
}

int zero_rows(float *p, long long rows, int cols, int ld, hipStream_t st) {
  if (rows <= 0 || cols <= 0) return CDML_OK;
  const long long n = rows * cols;
  zero_rows_kernel<<<dim3((unsigned)std::min<long long>((n + 255) / 256, 16384)), dim3(256), 0, st>>>(
      p, rows, cols, ld);
  return check_launch("zero_rows_kernel");
}

size_t align256(size_t n) { return (n + 255) / 256 * 256; }

template <int HD, int BN, bool CAUSAL, bool HAS_MASK, bool VEC>
void launch_bwd(BwdArgs &a, hipStream_t st) {
  const int n_bh = a.batch * a.heads;
  const int kt = (a.lk + BW_TILE - 1) / BW_TILE;
  a.n_tiles = (a.lq + BW_TILE - 1) / BW_TILE;
  const dim3 kgrid(n_bh * kt), qgrid(n_bh * a.n_tiles), block(BW_THREADS);
  if constexpr (HD <= 64) {
    const dim3 kblock(paired_keys(HD) ? 2 * BW_THREADS : BW_THREADS);
    if constexpr (CAUSAL && !HAS_MASK && VEC) {
      if (a.ds) {  // dQ from the stored dS blocks
        flash_bwd_dkdv_split_kernel<HD, true, false, true, true><<<kgrid, kblock, 0, st>>>(a);
        // Whole K^T per (sequence, head) where that fills the device: us at 8 heads
        // of 32, short / not: 256 x 511 313 / 358, 128 x 512 160 / 176, 64 x 512 81 /
        // 86, 32 x 512 37 / 37, 64 x 400 58 / 60; at 384 keys and below the staged
        // tile is half empty (128 x 300 79 / 74).
        if (HD == 32 && a.lq > 384 && a.lq <= 32 * kShortQB && n_bh >= 2 * num_cus())
          flash_bwd_dq_ds_short_kernel<<<dim3(n_bh), dim3(64 * ((a.lq + 63) / 64)), 0, st>>>(a);
        else
          flash_bwd_dq_ds_kernel<HD, 64><<<qgrid, block, 0, st>>>(a);
        return;
      }
    }
    flash_bwd_dkdv_split_kernel<HD, CAUSAL, HAS_MASK, VEC, false><<<kgrid, kblock, 0, st>>>(a);
  } else {
    flash_bwd_dkdv_kernel<HD, CAUSAL, HAS_MASK, VEC><<<kgrid, block, 0, st>>>(a);
  }
  flash_bwd_dq_kernel<HD, BN, CAUSAL, HAS_MASK, VEC><<<qgrid, block, 0, st>>>(a);
}

template <int HD, int BN, bool VEC>
void launch_bwd_mode(BwdArgs &a, bool causal, hipStream_t st) {
  if (causal) {
    if (a.mask) launch_bwd<HD, BN, true, true, VEC>(a, st);
    else launch_bwd<HD, BN, true, false, VEC>(a, st);
  } else if (a.mask) {
    launch_bwd<HD, BN, false, true, VEC>(a, st);
  } else {
    launch_bwd<HD, BN, false, false, VEC>(a, st);
  }
}

template <int HD, int BN>
void launch_bwd_hd(BwdArgs &a, bool causal, bool vec, hipStream_t st) {
  if (vec) launch_bwd_mode<HD, BN, true>(a, causal, st);
  else launch_bwd_mode<HD, BN, false>(a, causal, st);
}

}  // namespace
}  // namespace cdml

using namespace cdml;

extern "C" int cdml_sdpa_bwd_workspace_size(int batch, int lq, int lk, int dim, int num_heads,
                                            size_t *bytes) {
  if (!bytes) return fail(CDML_E_INVALID, "cdml_sdpa_bwd_workspace_size: bytes is NULL");
  if (batch < 0 || lq < 0 || lk < 0 || dim <= 0 || num_heads <= 0 || dim % num_heads)
    return fail(CDML_E_INVALID, "cdml_sdpa_bwd_workspace_size: bad size");
  const size_t f = sizeof(float), bh = (size_t)batch * num_heads;
  // O | lse | D | two floats per key for the generic kernel
  *bytes = align256(f * (size_t)batch * lq * dim) + 2 * align256(f * bh * lq) + align256(f * 2 * bh * lk);
  return CDML_OK;
}

namespace cdml {
namespace {

// Bytes of the stored-dS workspace of cdml_sdpa_bwd_saved (after D), or 0 when
// the shape does not take that path: causal, lq == lk, head dim 32 or 64.
size_t ds_bytes(int batch, int lq, int lk, int dim, int num_heads, bool causal) {
  const int hd = dim / num_heads;
  if (!causal || lq != lk || (hd != 32 && hd != 64) || lq == 0) return 0;
  const size_t nb = ((size_t)lq + 31) / 32;
  return (size_t)batch * num_heads * (nb * (nb + 1) / 2) * 1024 * sizeof(float);
}

}  // namespace
}  // namespace cdml

extern "C" int cdml_sdpa_bwd_stored_ds_workspace_size(int batch, int lq, int lk, int dim, int num_heads,
                                                      int causal, size_t *bytes) {
  int rc = cdml_sdpa_bwd_workspace_size(batch, lq, lk, dim, num_heads, bytes);
  if (rc) return rc;
  *bytes = align256(*bytes) + ds_bytes(batch, lq, lk, dim, num_heads, causal != 0);
  return CDML_OK;
}

extern "C" int cdml_sdpa_bwd_saved_workspace_size(int batch, int lq, int lk, int dim, int num_heads,
                                                  int causal, size_t *bytes) {
  if (!bytes) return fail(CDML_E_INVALID, "cdml_sdpa_bwd_saved_workspace_size: bytes is NULL");
  if (batch < 0 || lq < 0 || lk < 0 || dim <= 0 || num_heads <= 0 || dim % num_heads)
    return fail(CDML_E_INVALID, "cdml_sdpa_bwd_saved_workspace_size: bad size");
  const size_t d = sizeof(float) * (size_t)batch * num_heads * lq;
  const size_t extra = ds_bytes(batch, lq, lk, dim, num_heads, causal != 0);
  *bytes = extra ? align256(d) + extra : d;
  return CDML_OK;
}

namespace cdml {
namespace {

// cdml_sdpa_bwd, and with o_saved / lse_saved the backward from the forward's
// saved output and row statistics (cdml_sdpa_bwd_saved): no forward pass.
int sdpa_bwd_impl(const float *q, int ldq, const float *k, int ldk, const float *v, int ldv,
                  const float *o_saved, int ldo_saved, const float *lse_saved, const float *dout,
                  int lddo, float *dq, int lddq, float *dk, int lddk, float *dv, int lddv, int batch,
                  int lq, int lk, int dim, int num_heads, float scale, int causal,
                  const uint8_t *mask, void *workspace, size_t workspace_bytes, cdml_stream stream,
                  const char *what, const float *rope_cs = nullptr) {
  const bool saved = o_saved != nullptr;
  size_t need = 0;
  int rc = cdml_sdpa_bwd_workspace_size(batch, lq, lk, dim, num_heads, &need);
  if (rc) return rc;
  if (saved) {
    need = sizeof(float) * (size_t)batch * num_heads * lq;
    if (!lse_saved || ldo_saved < dim)
      return fail(CDML_E_INVALID, "%s: saved output needs the row statistics and a row stride of at "
                  "least dim", what);
  }
  if (ldq < dim || ldk < dim || ldv < dim || lddo < dim || lddq < dim || lddk < dim || lddv < dim)
    return fail(CDML_E_INVALID, "%s: row stride smaller than dim", what);
  if ((long long)ldq * 128 > INT32_MAX || (long long)ldk * 128 > INT32_MAX ||
      (long long)ldv * 128 > INT32_MAX || (long long)lddo * 128 > INT32_MAX)
    return fail(CDML_E_INVALID, "%s: row stride above %d elements", what, INT32_MAX / 128);
  if (batch == 0 || (lq == 0 && lk == 0)) return CDML_OK;
  if ((lq && (!dq || !q || !dout)) || (lk && (!dk || !dv || !k || !v)))
    return fail(CDML_E_INVALID, "%s: NULL pointer", what);
  rc = ensure_device();
  if (rc) return rc;
  hipStream_t st = as_hip(stream);
  if (lq == 0 || lk == 0) {  // nothing attends: every gradient is 0
    rc = zero_rows(dq, (long long)batch * lq, dim, lddq, st);
    if (!rc) rc = zero_rows(dk, (long long)batch * lk, dim, lddk, st);
    if (!rc) rc = zero_rows(dv, (long long)batch * lk, dim, lddv, st);
    return rc;
  }
  if (!workspace || workspace_bytes < need)
    return fail(CDML_E_INVALID, "%s: workspace of %zu bytes needed, %zu given", what, need,
                workspace_bytes);
  if ((long long)batch * num_heads * ((std::max(lq, lk) + BW_TILE - 1) / BW_TILE) > (1LL << 30))
    return fail(CDML_E_INVALID, "%s: problem too large", what);

  BwdArgs a{};
  a.q = q;
  a.k = k;
  a.v = v;
  a.dout = dout;
  a.dq = dq;
  a.dk = dk;
  a.dv = dv;
  a.mask = mask;
  a.ldq = ldq;
  a.ldk = ldk;
  a.ldv = ldv;
  a.lddo = lddo;
  a.lddq = lddq;
  a.lddk = lddk;
  a.lddv = lddv;
  a.batch = batch;
  a.lq = lq;
  a.lk = lk;
  a.dim = dim;
  a.heads = num_heads;
  a.hd = dim / num_heads;
  a.scale = scale;
  a.scale_log2 = scale * kLog2e;
  a.rope_cs = reinterpret_cast<const float2 *>(rope_cs);
  char *ws = static_cast<char *>(workspace);
  const size_t f = sizeof(float), bh = (size_t)batch * num_heads;
  float *o = reinterpret_cast<float *>(ws);
  float *lse = reinterpret_cast<float *>(ws + align256(f * (size_t)batch * lq * dim));
  float *delta = reinterpret_cast<float *>(reinterpret_cast<char *>(lse) + align256(f * bh * lq));
  float *scratch = reinterpret_cast<float *>(reinterpret_cast<char *>(delta) + align256(f * bh * lq));
  a.o = o;
  a.ldo = dim;
  a.lse = lse;
  a.delta = delta;
  if (saved) {  // workspace holds D only
    a.o = o_saved;
    a.ldo = ldo_saved;
    a.lse = lse_saved;
    a.delta = reinterpret_cast<float *>(ws);
  }

  const int hd = a.hd;
  if (hd > 128 && saved)
    return fail(CDML_E_INVALID, "%s: saved statistics need head dim <= 128; use cdml_sdpa_bwd", what);
  if (hd > 128) {
    const size_t smem = f * (2 * (size_t)hd + 8);
    if (smem > 64 * 1024) return fail(CDML_E_INVALID, "%s: head dim %d too large", what, hd);
    flash_bwd_generic_kernel<<<dim3((unsigned)bh), dim3(256), smem, st>>>(a, scratch, causal ? 1 : 0);
    return check_launch("flash_bwd_generic_kernel");
  }
  // 1. O and the row statistics (unless the caller saved them)
  if (!saved) {
    rc = flash_forward(q, ldq, k, ldk, v, ldv, o, dim, lse, batch, lq, lk, dim, num_heads, scale,
                       causal != 0, mask, st);
    if (rc) return rc;
  }
  // 2. D = rowsum(dO * O)
  const int hd_pad = hd <= 32 ? 32 : (hd <= 64 ? 64 : 128);
  const bool vec = hd == hd_pad && ldq % 4 == 0 && ldk % 4 == 0 && ldv % 4 == 0 && lddo % 4 == 0 &&
                   lddq % 4 == 0 && lddk % 4 == 0 && lddv % 4 == 0 && aligned16(q) && aligned16(k) &&
                   aligned16(v) && aligned16(dout) && aligned16(dq) && aligned16(dk) && aligned16(dv);
  if (vec && a.ldo % 4 == 0 && aligned16(a.o)) {
    const long long n = (long long)batch * lq * (dim / 4);
    const dim3 grid((unsigned)((n + 255) / 256));
    if (hd == 32) bwd_delta_kernel<32><<<grid, dim3(256), 0, st>>>(a);
    else if (hd == 64) bwd_delta_kernel<64><<<grid, dim3(256), 0, st>>>(a);
    else bwd_delta_kernel<128><<<grid, dim3(256), 0, st>>>(a);
  } else {
    const long long n = (long long)batch * lq * num_heads;
    bwd_delta_scalar_kernel<<<dim3((unsigned)((n + 255) / 256)), dim3(256), 0, st>>>(a);
  }
  rc = check_launch("bwd_delta_kernel");
  if (rc) return rc;
  // 3. dK, dV and 4. dQ; with room for the dS blocks after the required
  // workspace, dQ is one product over them
  if (vec && !mask) {
    const size_t extra = ds_bytes(batch, lq, lk, dim, num_heads, causal != 0);
    const size_t off = align256(need);  // the dS blocks follow the required workspace
    // (a (sequence, head)'s blocks must fit a buffer resource's 31-bit range)
    if (extra && workspace_bytes >= off + extra && extra / bh <= (size_t)INT32_MAX) {
      a.ds = reinterpret_cast<float *>(ws + off);
      a.ds_bh = (long long)(extra / sizeof(float) / bh);
    }
  }
  if (hd_pad == 32) launch_bwd_hd<32, 64>(a, causal != 0, vec, st);
  else if (hd_pad == 64) launch_bwd_hd<64, 32>(a, causal != 0, vec, st);
  else launch_bwd_hd<128, 32>(a, causal != 0, vec, st);
  return check_launch("flash_bwd_dkdv_kernel / flash_bwd_dq_kernel");
}

}  // namespace
}  // namespace cdml

extern "C" int cdml_sdpa_bwd(const float *q, int ldq, const float *k, int ldk, const float *v, int ldv,
                             const float *dout, int lddo, float *dq, int lddq, float *dk, int lddk,
                             float *dv, int lddv, int batch, int lq, int lk, int dim, int num_heads,
                             float scale, int causal, const uint8_t *mask, void *workspace,
                             size_t workspace_bytes, cdml_stream stream) {
  return sdpa_bwd_impl(q, ldq, k, ldk, v, ldv, nullptr, 0, nullptr, dout, lddo, dq, lddq, dk, lddk, dv,
                       lddv, batch, lq, lk, dim, num_heads, scale, causal, mask, workspace,
                       workspace_bytes, stream, "cdml_sdpa_bwd");
}

extern "C" int cdml_sdpa_bwd_saved(const float *q, int ldq, const float *k, int ldk, const float *v,
                                   int ldv, const float *o, int ldo, const float *lse,
                                   const float *dout, int lddo, float *dq, int lddq, float *dk,
                                   int lddk, float *dv, int lddv, int batch, int lq, int lk, int dim,
                                   int num_heads, float scale, int causal, const uint8_t *mask,
                                   void *workspace, size_t workspace_bytes, cdml_stream stream) {
  if (!o) return fail(CDML_E_INVALID, "cdml_sdpa_bwd_saved: o is NULL");
  return sdpa_bwd_impl(q, ldq, k, ldk, v, ldv, o, ldo, lse, dout, lddo, dq, lddq, dk, lddk, dv, lddv,
                       batch, lq, lk, dim, num_heads, scale, causal, mask, workspace, workspace_bytes,
                       stream, "cdml_sdpa_bwd_saved");
}

extern "C" int cdml_sdpa_bwd_saved_rope(const float *q, int ldq, const float *k, int ldk, const float *v,
                                        int ldv, const float *o, int ldo, const float *lse,
                                        const float *dout, int lddo, float *dq, int lddq, float *dk,
                                        int lddk, float *dv, int lddv, int batch, int lq, int lk, int dim,
                                        int num_heads, float scale, int causal, const uint8_t *mask,
                                        const float *rope_cs, int n_pos, void *workspace,
                                        size_t workspace_bytes, cdml_stream stream) {
  const char *what = "cdml_sdpa_bwd_saved_rope";
  if (!o) return fail(CDML_E_INVALID, "%s: o is NULL", what);
  if (num_heads > 0 && dim > 0 && dim % num_heads == 0 && ((dim / num_heads) & 1))
    return fail(CDML_E_INVALID, "%s: RoPE requires an even head dimension", what);
  if (!rope_cs) return fail(CDML_E_INVALID, "%s: rope_cs is NULL", what);
  if (reinterpret_cast<uintptr_t>(rope_cs) % 8)
    return fail(CDML_E_INVALID, "%s: rope_cs must be 8-byte aligned", what);
  if (n_pos < std::max(lq, lk))
    return fail(CDML_E_INVALID, "%s: a %d-row table does not cover %d positions", what, n_pos, std::max(lq, lk));
  return sdpa_bwd_impl(q, ldq, k, ldk, v, ldv, o, ldo, lse, dout, lddo, dq, lddq, dk, lddk, dv, lddv,
                       batch, lq, lk, dim, num_heads, scale, causal, mask, workspace, workspace_bytes,
                       stream, what, rope_cs);
}
