// fp32 GEMM on the matrix cores for the projections of the attention path and
// their gradients:
//   C[m, n] = act(sum_k opA[m, k] * opB[k, n] + bias[n])  (+ C[m, n] when beta)
// opA is A [M, K] (row stride lda) or, transposed, A stored [K, M]; opB is the
// weight W [N, K] ([out, in], the reference's layout: y = x W^T) or, for
// gradients, B stored [K, N].  Up to three problems with the same shape run in
// one launch (the fused Q/K/V projection and its weight gradients).
//
// Forward (A [M, K], W [N, K]):                  y = x W^T    ProjectQKV, linear
// Input gradient (A = dY [M, K], B = W [K, N]):  dX = dY W    BackpropQKV, ...
// Weight gradient (A = dY stored [K, M], B = X [K, N]): dW += dY^T X, with the
//   bias gradient (row sums of opA = column sums of dY) folded into the
//   staging of opA.
//
// The main kernel (gemm_tile_kernel) multiplies three bf16 pieces per operand
// (common.h) and is the same for every layout; a transposed operand is
// transposed on its way into LDS.  Small and odd shapes have kernels of their
// own, and gemm_f32_kernel keeps the fp32 MFMA for the pre-activations of ReLU
// layers.
#include <algorithm>
#include <type_traits>

#include "common.h"

namespace cdml {
namespace {

constexpr int BM = 128, BN = 128, BK = 32, LDSK = BK + 4;
constexpr int NTHREADS = 256;
constexpr int GROUP_M = 8;

struct GemmProblem {
  const float *a;     // opA source
  const float *w;     // opB source
  const float *bias;  // [N] or NULL
  float *c;
  float *bgrad;       // [M] += row sums of opA (transposed-A launches only), or NULL
};

struct GemmArgs {
  GemmProblem p[3];
  int lda, ldb, ldc;
  int M, N, K;
  int nprob;
  int tiles_m, tiles_n;  // tiles_n counts the tiles of one problem
  int total, padded;
  int act;
  int beta;  // 1: add the result to C
  // Split-K weight gradient with a ragged K: the tiled chunks cover rows
  // [0, ktail0) and splitk_reduce_kernel adds rows [ktail0, K) of opA^T opB
  // (and of opA's row sums) itself; 0 when K % 16 == 0.  (It fills the
  // padding before rope_cs.)
  int ktail0;
  // Rotary position embedding applied to problems 0 and 1 (Q and K) in the
  // epilogue when rope_cs is set: rope_cs[pos * rope_hd / 2 + p] holds
  // (cos, sin) of position pos for pair p; row m has position
  // rope_pos0 + (rope_seg > 0 ? m % rope_seg : m), below rope_npos.
  const float2 *rope_cs;
  int rope_hd, rope_npos, rope_pos0, rope_seg;
  // Split-K of the weight-gradient GEMMs (transposed-A launches): ksplit
  // chunks of kchunk k-tiles each; chunk c of problem p writes its partial
  // C to ws + (c * nprob + p) * M * N ([M][N], row stride N) and its partial
  // bias-gradient row sums to wsb + (c * nprob + p) * M; splitk_reduce_kernel
  // adds the chunks, in chunk order, to C and bgrad.  tiles counts the
  // output tiles of all problems (total = tiles * ksplit).
  int ksplit, kchunk, tiles;
  float *ws, *wsb;
  int small;  // split-K by wgrad_small_kernel (kchunk counts rows, not k-tiles)
  // K segments of an input-gradient launch (opB stored [K, N], one problem):
  // when kseg > 0, k-tiles [s * kseg, (s + 1) * kseg) read opA from p[s].a
  // and opB from p[s].w (s < 3), so dX = dQ WQ + dK WK + dV WV is one
  // product with K = 3 * out.  (It fills the padding before `pre`.)
  int kseg;
  // Single-problem epilogue options (store_elem): pre receives the
  // pre-activation acc + bias (forward layers whose backward needs it); dz
  // multiplies the result by act'(dz) with act = dact (the hidden deltas of
  // NeuralNetwork.ComputeInputGradientBatch); add is added last (a residual
  // gradient, MatrixAddInPlace).
  float *pre;
  const float *dz, *add;
  int ldpre, lddz, ldadd, dact;
  int f32;  // forward: keep the fp32 MFMA (gemm_f32_kernel)
};

// The value of lane l ^ 1 (a DPP quad permutation [1, 0, 3, 2]).
__device__ __forceinline__ float swap_pair(float y) {
  return __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(y), 0xB1, 0xF, 0xF, false));
}

// Epilogue of the fallback forward kernel (gemm_nt_kernel) with the rotary embedding
// of AccelerationCPU.cs:4947-4975 folded in.  A lane holds column n of rows
// mrow0 + 32 i + 8 (r / 4) + 4 hf + r % 4, so the pair partner of column n
// (n ^ 1; head dims are even) sits in lane li ^ 1 of the same register: one
// lane swap gives each lane both halves of its pair.  The swap runs in every
// lane; only the store is predicated.
template <int BI, int BJ>
__device__ __forceinline__ void store_rope(const GemmArgs &args, const GemmProblem &P,
                                           const floatx16 (&acc)[BI][BJ], int mrow0, int ncol0,
                                           int li, int hf) {
  // each rotation product rounded before the sum, as the reference and the
  // in-place rope kernels evaluate it: no fused multiply-add
#pragma clang fp contract(off)
  const int pairs = args.rope_hd >> 1;
  int n[BJ], pidx[BJ];
  bool odd[BJ];
  float bias[BJ];
#pragma unroll
  for (int j = 0; j < BJ; ++j) {
    n[j] = ncol0 + j * 32 + li;
    const int c = n[j] % args.rope_hd;
    pidx[j] = c >> 1;
    odd[j] = c & 1;
    bias[j] = (P.bias && n[j] < args.N) ? P.bias[n[j]] : 0.f;
  }
  // rows of block i: mb + dr(r), dr = 8 (r / 4) + 4 hf + r % 4
  auto block = [&](int i, int mb, auto position) {
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      const int dr = 8 * (r >> 2) + 4 * hf + (r & 3);
      const int m = mb + dr;
      const int pos = min(position(m, dr), args.rope_npos - 1);  // rows past M are never stored
      const float2 *cs = args.rope_cs + (size_t)pos * pairs;
#pragma unroll
      for (int j = 0; j < BJ; ++j) {
        const float y = acc[i][j][r] + bias[j];
        const float yp = swap_pair(y);
        const float2 t = cs[pidx[j]];
        const float out = odd[j] ? yp * t.y + y * t.x : y * t.x - yp * t.y;
        if (m < args.M && n[j] < args.N) P.c[(size_t)m * args.ldc + n[j]] = out;
      }
    }
  };
  const int seg = args.rope_seg;
  // every row and column of this wave's blocks exists (wave-uniform)
  const bool full = mrow0 + 32 * BI <= args.M && ncol0 + 32 * BJ <= args.N;
#pragma unroll
  for (int i = 0; i < BI; ++i) {
    const int mb = mrow0 + i * 32;             // wave-uniform
    const int pb = seg > 0 ? mb % seg : mb;    // position of row mb in its segment
    if (seg <= 0 || pb + 31 < seg) {
      if (full) {
        // A whole block inside one segment: positions pos0 + pb + dr (every one inside
        // the table, which the entry point checks), no predicates, and per row only
        // wave-uniform offsets from the lane's bases.  The table entries of four rows
        // are loaded before any of their stores: a load issued after a store waits
        // for it (the memory counter covers both).
        const float2 *__restrict__ csb = args.rope_cs + (size_t)(args.rope_pos0 + pb + 4 * hf) * pairs;
        float *__restrict__ cb = P.c + (size_t)(mb + 4 * hf) * args.ldc;
#pragma unroll
        for (int g = 0; g < 4; ++g) {
          float2 t[4][BJ];
#pragma unroll
          for (int rr = 0; rr < 4; ++rr)
#pragma unroll
            for (int j = 0; j < BJ; ++j) t[rr][j] = csb[(8 * g + rr) * pairs + pidx[j]];
#pragma unroll
          for (int rr = 0; rr < 4; ++rr) {
            const int r = 4 * g + rr;
            float *c = cb + (size_t)(8 * g + rr) * args.ldc;
#pragma unroll
            for (int j = 0; j < BJ; ++j) {
              const float y = acc[i][j][r] + bias[j];
              const float yp = swap_pair(y);
              c[n[j]] = odd[j] ? yp * t[rr][j].y + y * t[rr][j].x : y * t[rr][j].x - yp * t[rr][j].y;
            }
          }
        }
      } else {
        block(i, mb, [&](int, int dr) { return args.rope_pos0 + pb + dr; });
      }
    } else {
      // a block across a segment boundary divides per row
      block(i, mb, [&](int m, int) { return args.rope_pos0 + m % seg; });
    }
  }
}

// 1 / (1 + e^-x) for x >= 0, e^x / (1 + e^x) below, without a branch.
__device__ __forceinline__ float stable_sigmoid(float x) {
  const float z = expf(-fabsf(x));
  return (x >= 0.f ? 1.f : z) / (1.f + z);
}

// Activation and derivative codes of the derivative-from-output form
// (cdml_linear_preact without z, CDML_ACT_FROM_OUTPUT): ReLU whose zero output
// is -0 where z < 0 or z is NaN, and ReLU's derivative read from that sign.
// Leaky ReLU needs neither: its output has the sign of z, so act'(y) equals
// act'(z) with the same expression.
constexpr int kActReluMarked = 6;
constexpr int kDerivReluOut = 7;

// Activation derivative at the pre-activation z, as FillActivationAndDerivative
// (Neural Network/NeuralNetwork.cs:885-944) defines it, including its ReLU
// derivative of 1 at z = 0 and leaky-ReLU slope 0.1 for z <= 0.
__device__ __forceinline__ float act_deriv(float z, int act) {
  switch (act) {
    case CDML_ACT_SIGMOID: {
      const float s = stable_sigmoid(z);
      return s * (1.f - s);
    }
    case CDML_ACT_TANH: {
      const float t = tanhf(z);
      return 1.f - t * t;
    }
    case CDML_ACT_RELU:
      return z >= 0.f ? 1.f : 0.f;
    case CDML_ACT_LEAKYRELU:
      return z <= 0.f ? 0.1f : 1.f;
    case kDerivReluOut:  // z >= 0 exactly where the marked output is not -0
      return __float_as_int(z) < 0 ? 0.f : 1.f;
    case CDML_ACT_SWISH: {
      const float s = stable_sigmoid(z);
      return s + z * s * (1.f - s);
    }
    default:
      return 1.f;
  }
}

__device__ __forceinline__ float activate(float x, int act) {
  switch (act) {
    case CDML_ACT_SIGMOID:
      return stable_sigmoid(x);
    case CDML_ACT_TANH:
      return tanhf(x);
    case CDML_ACT_RELU:
      return x > 0.f ? x : 0.f;
    case kActReluMarked:
      return x > 0.f ? x : (x >= 0.f ? 0.f : -0.f);
    case CDML_ACT_LEAKYRELU:
      return x > 0.f ? x : 0.01f * x;
    case CDML_ACT_SWISH:
      return x * stable_sigmoid(x);
    default:
      return x;
  }
}

// Stores output (m, n) of problem P from z = acc + bias: pre <- z,
// v = act(z), v *= act'(dz) and v += add when those options are set, then
// C = v (or C + v with beta).
// The options are a compile-time switch (EPI) so that launches without them
// keep the plain epilogue.
template <bool EPI>
__device__ __forceinline__ void store_elem(const GemmArgs &args, const GemmProblem &P, int m, int n,
                                           float z, int act) {
  float v;
  if constexpr (EPI) {
    if (args.pre) args.pre[(size_t)m * args.ldpre + n] = z;
    v = activate(z, act);
    if (args.dz) v *= act_deriv(args.dz[(size_t)m * args.lddz + n], args.dact);
    if (args.add) v += args.add[(size_t)m * args.ldadd + n];
  } else {
    v = activate(z, act);
  }
  float *pc = P.c + (size_t)m * args.ldc + n;
  *pc = args.beta ? *pc + v : v;
}

inline bool has_epi(const GemmArgs &g) { return g.pre || g.dz || g.add; }

// Global -> register staging of one 128x32 tile of a row-major [rows, K]
// matrix.  VEC: K % 4 == 0 and 16-byte aligned rows, four float4 per thread;
// otherwise sixteen guarded scalars per thread.
template <bool VEC>
struct TileStage {
  float4 r[4];
  float s[16];

  __device__ __forceinline__ void load(const float *__restrict__ src, int ld, int row0, int rows,
                                       int k0, int K) {
    const int t = threadIdx.x;
    if constexpr (VEC) {
      const int c = (t & 7) * 4;
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int row = row0 + (t >> 3) + 32 * i;
        if (row < rows && k0 + c < K)
          r[i] = *reinterpret_cast<const float4 *>(src + (size_t)row * ld + k0 + c);
        else
          r[i] = make_float4(0.f, 0.f, 0.f, 0.f);
      }
    } else {
      const int c = t & 31;
#pragma unroll
      for (int i = 0; i < 16; ++i) {
        const int row = row0 + (t >> 5) + 8 * i;
        s[i] = (row < rows && k0 + c < K) ? src[(size_t)row * ld + k0 + c] : 0.f;
      }
    }
  }

  __device__ __forceinline__ void store(float (*lds)[LDSK]) {
    const int t = threadIdx.x;
    if constexpr (VEC) {
      const int c = (t & 7) * 4;
#pragma unroll
      for (int i = 0; i < 4; ++i) *reinterpret_cast<float4 *>(&lds[(t >> 3) + 32 * i][c]) = r[i];
    } else {
      const int c = t & 31;
#pragma unroll
      for (int i = 0; i < 16; ++i) lds[(t >> 5) + 8 * i][c] = s[i];
    }
  }
};

// Guarded fallback of the forward layout (any K, any alignment) on the fp32
// MFMA: operand tiles in LDS as [rows][k] with row pitch BK + 4 floats, every
// lane's operands 16-byte LDS reads that feed four v_mfma_f32_32x32x2_f32 each,
// k in the permuted order kappa(s, h) = 8*(s/4) + 4*h + s%4 on both operands.
template <bool VEC, bool EPI>
__global__ void __launch_bounds__(NTHREADS) gemm_nt_kernel(const GemmArgs args) {
  __shared__ __attribute__((aligned(16))) float As[2][BM][LDSK];
  __shared__ __attribute__((aligned(16))) float Bs[2][BN][LDSK];

  const int lid = xcd_remap(blockIdx.x, args.padded);
  if (lid >= args.total) return;

  // Grouped ordering over (tiles_m, nprob * tiles_n): GROUP_M tile-rows share
  // each weight panel while it is hot in L2.
  const int tiles_n_all = args.tiles_n * args.nprob;
  const int in_group = GROUP_M * tiles_n_all;
  const int group = lid / in_group;
  const int first_m = group * GROUP_M;
  const int gsize = min(args.tiles_m - first_m, GROUP_M);
  const int tm = first_m + (lid % in_group) % gsize;
  const int tn_all = (lid % in_group) / gsize;
  const int prob = tn_all / args.tiles_n;
  const int tn = tn_all % args.tiles_n;

  const GemmProblem P = args.p[prob];
  const int m0 = tm * BM, n0 = tn * BN;
  const int M = args.M, N = args.N, K = args.K;

  const int lane = threadIdx.x & 63;
  const int wave = threadIdx.x >> 6;
  const int wm = wave >> 1, wn = wave & 1;
  const int li = lane & 31, hf = lane >> 5;

  floatx16 acc[2][2];
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[i][j][r] = 0.f;

  TileStage<VEC> sa, sb;
  const int nk = (K + BK - 1) / BK;
  sa.load(P.a, args.lda, m0, M, 0, K);
  sb.load(P.w, args.ldb, n0, N, 0, K);
  sa.store(As[0]);
  sb.store(Bs[0]);
  __syncthreads();

  for (int kt = 0; kt < nk; ++kt) {
    const int cur = kt & 1;
    const bool more = kt + 1 < nk;
    if (more) {
      sa.load(P.a, args.lda, m0, M, (kt + 1) * BK, K);
      sb.load(P.w, args.ldb, n0, N, (kt + 1) * BK, K);
    }
#pragma unroll
    for (int u = 0; u < BK / 8; ++u) {
      float4 a4[2], b4[2];
#pragma unroll
      for (int i = 0; i < 2; ++i)
        a4[i] = *reinterpret_cast<const float4 *>(&As[cur][wm * 64 + i * 32 + li][u * 8 + hf * 4]);
#pragma unroll
      for (int j = 0; j < 2; ++j)
        b4[j] = *reinterpret_cast<const float4 *>(&Bs[cur][wn * 64 + j * 32 + li][u * 8 + hf * 4]);
      const float av[2][4] = {{a4[0].x, a4[0].y, a4[0].z, a4[0].w},
                              {a4[1].x, a4[1].y, a4[1].z, a4[1].w}};
      const float bv[2][4] = {{b4[0].x, b4[0].y, b4[0].z, b4[0].w},
                              {b4[1].x, b4[1].y, b4[1].z, b4[1].w}};
#pragma unroll
      for (int r = 0; r < 4; ++r)
#pragma unroll
        for (int i = 0; i < 2; ++i)
#pragma unroll
          for (int j = 0; j < 2; ++j) acc[i][j] = mfma32x32x2(av[i][r], bv[j][r], acc[i][j]);
    }
    if (more) {
      sa.store(As[cur ^ 1]);
      sb.store(Bs[cur ^ 1]);
    }
    __syncthreads();
  }

  if (args.rope_cs && prob < 2) {
    store_rope<2, 2>(args, P, acc, m0 + wm * 64, n0 + wn * 64, li, hf);
    return;
  }
  // Epilogue: D[i][j] of block (bi, bj) sits at row 8*(r/4) + 4*hf + r%4,
  // column li; 32 lanes store 32 consecutive columns of one row.
#pragma unroll
  for (int j = 0; j < 2; ++j) {
    const int n = n0 + wn * 64 + j * 32 + li;
    if (n >= N) continue;
    const float bias = P.bias ? P.bias[n] : 0.f;
#pragma unroll
    for (int i = 0; i < 2; ++i) {
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const int m = m0 + wm * 64 + i * 32 + 8 * (r >> 2) + 4 * hf + (r & 3);
        if (m < M) store_elem<EPI>(args, P, m, n, acc[i][j][r] + bias, args.act);
      }
    }
  }
}

// Global -> LDS staging of one ROWS x 16 operand tile of the tiled kernel,
// split on the way into its three bf16 pieces (split_bf16x3), one LDS plane
// each; a row's 16 k-values are 32 contiguous bytes of a plane.
// Row r of the tile sits in cluster r % NC at place r / NC; odd clusters hold
// their rows negated (see common.h).
//   T = false: the source is [rows][K] (k contiguous, row stride ld): a unit
//     is four k of one row, one 16-byte load and an 8-byte store per plane; a
//     thread's units come in pairs of neighbouring rows, one in each of NC = 2
//     clusters, so the stores of a wave cover 512 contiguous bytes (with one unit
//     per thread, NP = 1, a wave's rows fall in both clusters).
//   T = true:  the source is [K][rows] (rows contiguous, k-row stride ld): a
//     unit is four rows of two k, two 16-byte loads and per row (NC = 4) a
//     4-byte store per plane, 256 contiguous bytes for eight units.  Where a
//     tile has fewer units than threads, the first UNITS threads stage it.
// The clusters start 16, 128 and 144 bytes past a multiple of 256, so that
// the 16-byte pieces of sixteen lanes of an operand read fall in different
// banks.  Each thread's offsets are fixed for the whole K loop; rows past the
// end are clamped to the last row (T: the last four rows; rows % 4 == 0), so
// loads need no predication and clamped rows only feed results that are never
// stored.
template <int ROWS, int NT, bool T>
struct OpStage {
  static constexpr int NC = T ? 4 : 2;
  static constexpr int ROWB = ROWS / NC * 32;              // bytes of one row cluster
  // Byte offset of cluster c in a plane: 16, 128 and 144 past a multiple of 256.
  static __device__ __forceinline__ constexpr int cluster(int c) {
    return c * ROWB + (c & 1) * 16 + (c >> 1) * 128;
  }
  static constexpr int PLANE = NC * ROWB + (T ? 256 : 64);  // bytes of one piece
  static constexpr int BYTES = 3 * PLANE;
  static constexpr int BLOCK = 32 / NC * 32;               // bytes between 32-row blocks
  static constexpr int UNITS = ROWS * (T ? 2 : 4);
  static constexpr int NP = UNITS < NT ? 1 : UNITS / NT;   // units per thread, of the first UNITS threads
  static constexpr int NV = T ? 2 * NP : NP;               // their loads
  static constexpr int SPLITS = 2 * NV;                    // split_bf16x3 calls
  static constexpr int STORES = T ? 12 * NP : 3 * NP;
  static_assert(UNITS < NT ? T && UNITS % 64 == 0 : UNITS % NT == 0 && (T || NP % 2 == 0 || NP == 1), "staging shape");
  uint32_t off[NP];
  vf4 v[NV];
  int sa, sb;  // T = false: (row pair, first k / 4); T = true: (row group, k / 2)
  int ldk;     // T = true: row stride of the source

  // First tile row of unit i.
  __device__ __forceinline__ int unit_row(int i) const {
    if (T) return 4 * (sa + NT / 8 * i);
    return NP == 1 ? sa : 2 * sa + (i & 1) + NT / 2 * (i >> 1);
  }
  __device__ __forceinline__ void init(int row0, int rows, int ld) {
    const int t = threadIdx.x;
    sa = T ? t / 8 : t / 4;
    sb = T ? t % 8 : t % 4;
    ldk = ld;
#pragma unroll
    for (int i = 0; i < NP; ++i) {
      if constexpr (T)
        off[i] = (uint32_t)(2 * sb) * (uint32_t)ld + (uint32_t)min(row0 + unit_row(i), rows - 4);
      else
        off[i] = (uint32_t)min(row0 + unit_row(i), rows - 1) * (uint32_t)ld + 4 * sb;
    }
  }
  // Whether this wave has units.  One without loads rows past the tile (clamped) and
  // stores nothing: a conditional load would put the staging registers into scratch.
  static __device__ __forceinline__ bool staging() {
    return UNITS >= NT || __builtin_amdgcn_readfirstlane(threadIdx.x) < UNITS;
  }
  // First element of k-tile kt.
  static __device__ __forceinline__ const float *tile(const float *x, int kt, int ld) {
    return T ? x + (size_t)kt * 16 * ld : x + (size_t)kt * 16;
  }
  __device__ __forceinline__ void load(const float *__restrict__ base) {
#pragma unroll
    for (int i = 0; i < NP; ++i) {
      if constexpr (T) {
        v[2 * i] = *reinterpret_cast<const vf4 *>(base + off[i]);
        v[2 * i + 1] = *reinterpret_cast<const vf4 *>(base + off[i] + ldk);
      } else {
        v[i] = *reinterpret_cast<const vf4 *>(base + off[i]);
      }
    }
  }
  // The last, ragged k-tile: k at or past kvalid are not read, they count as zero.
  __device__ __forceinline__ void load_tail(const float *__restrict__ base, int kvalid) {
    const vf4 zero = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int i = 0; i < NP; ++i) {
      if constexpr (T) {
        v[2 * i] = v[2 * i + 1] = zero;
        if (2 * sb < kvalid) v[2 * i] = *reinterpret_cast<const vf4 *>(base + off[i]);
        if (2 * sb + 1 < kvalid) v[2 * i + 1] = *reinterpret_cast<const vf4 *>(base + off[i] + ldk);
      } else {
        v[i] = zero;
        if (4 * sb + 3 < kvalid) {
          v[i] = *reinterpret_cast<const vf4 *>(base + off[i]);
        } else {
#pragma unroll
          for (int c = 0; c < 3; ++c)
            if (4 * sb + c < kvalid) v[i][c] = base[off[i] + c];
        }
      }
    }
  }
  // scale: kSplitScale or its negative.
  __device__ __forceinline__ void store(char *lds, float scale) const {
    auto scaled = [&](float x, bool neg) { return x * (neg ? -scale : scale); };
    if (!staging()) return;
#pragma unroll
    for (int i = 0; i < NP; ++i) {
      if constexpr (T) {
        char *d = lds + (sa + NT / 8 * i) * 32 + sb * 4;
#pragma unroll
        for (int c = 0; c < 4; ++c) {
          uint32_t h, m, l;
          split_bf16x3(scaled(v[2 * i][c], c & 1), scaled(v[2 * i + 1][c], c & 1), h, m, l);
          *reinterpret_cast<uint32_t *>(d + cluster(c)) = h;
          *reinterpret_cast<uint32_t *>(d + cluster(c) + PLANE) = m;
          *reinterpret_cast<uint32_t *>(d + cluster(c) + 2 * PLANE) = l;
        }
      } else {
        const bool odd = NP == 1 ? sa & 1 : i & 1;
        const int place = NP == 1 ? sa >> 1 : sa + NT / 4 * (i >> 1);
        char *d = lds + cluster(odd) + place * 32 + sb * 8;
        const float f = odd ? -scale : scale;
        uint32_t h0, m0, l0, h1, m1, l1;
        split_bf16x3(v[i][0] * f, v[i][1] * f, h0, m0, l0);
        split_bf16x3(v[i][2] * f, v[i][3] * f, h1, m1, l1);
        *reinterpret_cast<vu2 *>(d) = vu2{h0, h1};
        *reinterpret_cast<vu2 *>(d + PLANE) = vu2{m0, m1};
        *reinterpret_cast<vu2 *>(d + 2 * PLANE) = vu2{l0, l1};
      }
    }
  }
  // Byte offset of a lane's operand (eight k of row row0 + li) in a plane.
  static __device__ __forceinline__ int operand(int row0, int li, int hf) {
    return cluster(li % NC) + (row0 / NC + li / NC) * 32 + hf * 16;
  }
};

// A wave's BI x BJ blocks recomputed on the fp32 MFMA straight from memory,
// one block after the other: only for blocks whose split products came out
// non-finite (common.h), so that they hold what the fp32 sum gives.  k runs over
// [k0, k1) of each of nseg operand pairs.
template <int BI, int BJ, bool TA, bool TB>
__device__ __forceinline__ void recompute_blocks(const GemmArgs &args, int prob, int nseg, int k0, int k1, int mw,
                                                 int nw, int li, int hf, floatx16 (&acc)[BI][BJ]) {
#pragma unroll
  for (int i = 0; i < BI; ++i) {
    const size_t m = min(mw + i * 32 + li, args.M - 1);
#pragma unroll
    for (int j = 0; j < BJ; ++j) {
      const size_t n = min(nw + j * 32 + li, args.N - 1);
      floatx16 c = {};
#pragma unroll 1
      for (int s = 0; s < nseg; ++s) {
        const float *A = args.p[prob + s].a, *W = args.p[prob + s].w;
#pragma unroll 1
        for (int k = k0; k < k1; k += 2) {
          const size_t kk = min(k + hf, k1 - 1);
          const float av = A[TA ? kk * args.lda + m : m * args.lda + kk];
          const float bv = W[TB ? kk * args.ldb + n : n * args.ldb + kk];
          const bool in = k + hf < k1;
          c = mfma32x32x2(in ? av : 0.f, in ? bv : 0.f, c);
        }
      }
      acc[i][j] = c;
    }
  }
}

// Orders the LDS accesses of a wave's lanes where they pass values to each other
// without a workgroup barrier: the hardware keeps a wave's LDS accesses in order, and
// this keeps the compiler from moving them past each other.  It emits no instruction.
__device__ __forceinline__ void lds_handover() {
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  __builtin_amdgcn_wave_barrier();
}

// Where a wave's blocks go: C (or a split-K partial, which takes neither bias
// nor activation nor beta).
struct TileOut {
  float *c;
  int ldc;
  const float *bias;
  int act, beta;
  bool rope;
};

// Epilogue of a wave's BI x BJ blocks through `lds` (32 * (32 * BJ + 4) floats
// of the wave's own; the k-loop has ended on a barrier, so the operand tiles
// are free): one 32-row band at a time is laid down as the MFMA holds it and
// read back as rows, so that a lane has four consecutive columns: bias,
// activation, training options (EPI) and stores take 16-byte accesses where
// the strides allow them, and both halves of a rotary pair are in one lane.
// The operands of four rows are loaded before any of their stores (a load
// issued after a store waits for it).  The loop over rows is rolled, so the
// activations cost no code per register (unrolled over the accumulators they
// took the kernels into scratch memory).
template <int BI, int BJ, bool EPI, bool ROPE>
__device__ __forceinline__ void store_tile(const GemmArgs &args, const TileOut &out,
                                           const floatx16 (&acc)[BI][BJ], int mw, int nw, int lane, float *lds) {
#pragma clang fp contract(off)
  constexpr int PITCH = 32 * BJ + 4;
  constexpr int RPI = 8 / BJ;  // rows per step of the wave (8 BJ lanes hold a row)
  constexpr int GROUP = 4;     // steps whose loads run ahead of their stores
  static_assert(8 % BJ == 0 && 32 % (GROUP * RPI) == 0, "epilogue shape");
  const int M = args.M, N = args.N;
  const int li = lane & 31, hf = lane >> 5;
  const int n = nw + 4 * (lane % (8 * BJ)), r0 = lane / (8 * BJ);
  bool vec = N % 4 == 0 && out.ldc % 4 == 0 && (reinterpret_cast<uintptr_t>(out.c) & 15) == 0;
  if (EPI) {
    if (args.pre) vec = vec && args.ldpre % 4 == 0 && (reinterpret_cast<uintptr_t>(args.pre) & 15) == 0;
    if (args.dz) vec = vec && args.lddz % 4 == 0 && (reinterpret_cast<uintptr_t>(args.dz) & 15) == 0;
    if (args.add) vec = vec && args.ldadd % 4 == 0 && (reinterpret_cast<uintptr_t>(args.add) & 15) == 0;
  }
  auto get = [&](auto full, const float *p) {  // four columns from n, zero past N
    vf4 x = {0.f, 0.f, 0.f, 0.f};
    if constexpr (decltype(full)::value) {
      x = *reinterpret_cast<const vf4 *>(p);
    } else if (vec) {
      if (n < N) x = *reinterpret_cast<const vf4 *>(p);
    } else {
#pragma unroll
      for (int c = 0; c < 4; ++c)
        if (n + c < N) x[c] = p[c];
    }
    return x;
  };
  auto put = [&](auto full, float *p, vf4 x) {
    if constexpr (decltype(full)::value) {
      *reinterpret_cast<vf4 *>(p) = x;
    } else if (vec) {
      if (n < N) *reinterpret_cast<vf4 *>(p) = x;
    } else {
#pragma unroll
      for (int c = 0; c < 4; ++c)
        if (n + c < N) p[c] = x[c];
    }
  };
  vf4 bias = {0.f, 0.f, 0.f, 0.f};
  if (out.bias) {
#pragma unroll
    for (int c = 0; c < 4; ++c)
      if (n + c < N) bias[c] = out.bias[n + c];
  }
  // rotary pairs of columns n, n + 1 and n + 2, n + 3 in their heads
  const bool rope = ROPE && out.rope;
  int p0 = 0, p1 = 0, pairs = 0;
  if (rope) {
    pairs = args.rope_hd >> 1;
    p0 = (n % args.rope_hd) >> 1;
    p1 = ((n + 2) % args.rope_hd) >> 1;
  }
#pragma unroll 1
  for (int i = 0; i < BI; ++i) {
    if (i > 0) lds_handover();  // the band's last reads
#pragma unroll
    for (int ii = 0; ii < BI; ++ii)
      if (ii == i) {  // the accumulators need constant indices, the loop's body only one copy
#pragma unroll
        for (int j = 0; j < BJ; ++j)
#pragma unroll
          for (int r = 0; r < 16; ++r) lds[(8 * (r >> 2) + 4 * hf + (r & 3)) * PITCH + j * 32 + li] = acc[ii][j][r];
      }
    lds_handover();
    auto rows = [&](auto full) {
      constexpr bool FULL = decltype(full)::value;  // every row and column exists, 16-byte accesses
#pragma unroll 1
    for (int g = 0; g < 32; g += GROUP * RPI) {
      vf4 z[GROUP], zv[GROUP], av[GROUP], old[GROUP];
      float2 t0[GROUP], t1[GROUP];
#pragma unroll
      for (int u = 0; u < GROUP; ++u) {
        const int row = g + u * RPI + r0, m = mw + i * 32 + row;
        z[u] = *reinterpret_cast<const vf4 *>(&lds[row * PITCH + (n - nw)]);
        if (FULL || m < M) {
          if (EPI && args.dz) zv[u] = get(full, args.dz + (size_t)m * args.lddz + n);
          if (EPI && args.add) av[u] = get(full, args.add + (size_t)m * args.ldadd + n);
          if (out.beta) old[u] = get(full, out.c + (size_t)m * out.ldc + n);
          if (ROPE && rope && (FULL || n < N)) {
            const int pos = args.rope_pos0 + (args.rope_seg > 0 ? m % args.rope_seg : m);
            const float2 *cs = args.rope_cs + (size_t)pos * pairs;
            t0[u] = cs[p0];
            t1[u] = cs[p1];
          }
        }
      }
#pragma unroll
      for (int u = 0; u < GROUP; ++u) {
        const int row = g + u * RPI + r0, m = mw + i * 32 + row;
        if (!FULL && m >= M) continue;
        vf4 v;
#pragma unroll
        for (int c = 0; c < 4; ++c) v[c] = z[u][c] + bias[c];
        if (EPI && args.pre) put(full, args.pre + (size_t)m * args.ldpre + n, v);
        if (!ROPE && out.act != CDML_ACT_NONE) {
#pragma unroll
          for (int c = 0; c < 4; ++c) v[c] = activate(v[c], out.act);
        }
        if (EPI && args.dz) {
#pragma unroll
          for (int c = 0; c < 4; ++c) v[c] *= act_deriv(zv[u][c], args.dact);
        }
        if (EPI && args.add) {
#pragma unroll
          for (int c = 0; c < 4; ++c) v[c] += av[u][c];
        }
        if (ROPE && rope) {
          // each rotation product rounded before the sum, as the reference
          // (AccelerationCPU.cs:4947-4975) and the in-place rope kernels
          // evaluate it: no fused multiply-add
          v = vf4{v[0] * t0[u].x - v[1] * t0[u].y, v[0] * t0[u].y + v[1] * t0[u].x,
                  v[2] * t1[u].x - v[3] * t1[u].y, v[2] * t1[u].y + v[3] * t1[u].x};
        }
        if (out.beta) {
#pragma unroll
          for (int c = 0; c < 4; ++c) v[c] = old[u][c] + v[c];
        }
        put(full, out.c + (size_t)m * out.ldc + n, v);
      }
    }
    };
    if (vec && mw + (i + 1) * 32 <= M && nw + 32 * BJ <= N) rows(std::true_type{});
    else rows(std::false_type{});
  }
}

// Tiled kernel (16-byte aligned rows, element offsets below 2^32; rows % 4 == 0
// where an operand is [K][rows]).  A
// workgroup of WM x WN waves computes a TM x TN tile of C, each wave a
// (TM/WM) x (TN/WN) block of 32x32 tiles on the bf16 MFMA, both operands split
// into three bf16 pieces on their way into LDS (common.h).  K advances by 16
// through NB LDS buffers; the k-tile after the last staged one is fetched into
// registers while the current one is multiplied.
//
// With NB = 3 the next k-tile is complete in LDS while the current one is
// multiplied, so the operands of its first product are read before the
// barrier, and the split (VALU) and LDS instructions are spread between the
// MFMAs by scheduling groups; with NB = 2 (small tiles) several workgroups per
// CU hide each other's staging.  Measured on MI355X (fp32-equivalent TFLOP/s,
// forward, dX and dW of 16384 x 4096 x 1024): 199, 183 and 193, where the fp32 MFMA form that this replaces had 138, 128 and 131.  The
// library's own bf16 product reaches 1170-1340 TFLOP/s, a sixth of which is
// 195-223: the power of the matrix cores bounds both (a loop of MFMAs alone on
// random data runs at 1.8 of 2.4 GHz); matrix pipes 60-64% busy forward, 4.3-4.5
// VALU instructions beside each MFMA (128 x 128 tiles 58-63%, 5.4-5.6).  256 x 256 tiles would take 208-229 with one
// accumulator (see common.h); the registers do not hold two.
//
// With TA and a bias-gradient pointer, the workgroups of the first column
// tile also sum the opA values that they stage (every k once) and add the row
// sums to bgrad: the bias gradient of a weight-gradient GEMM costs no extra
// pass over dY.  Each thread sums its own k pair of its rows; the eight k pairs
// of a row sit in neighbouring lanes.
template <int TM, int TN, int WM, int WN, int MINB, int NB, bool ROPE, bool TA, bool TB, bool EPI>
__global__ void __launch_bounds__(64 * WM * WN, MINB) gemm_tile_kernel(const GemmArgs args) {
  constexpr int NT = 64 * WM * WN;
  constexpr int BI = TM / WM / 32, BJ = TN / WN / 32;
  static_assert(BI >= 1 && BJ >= 1 && (NB == 2 || NB == 3), "tile shape");
  typedef OpStage<TM, NT, TA> StageA;
  typedef OpStage<TN, NT, TB> StageB;
  __shared__ __attribute__((aligned(16))) char smem[NB * (StageA::BYTES + StageB::BYTES)];
  char *const As = smem, *const Bs = smem + NB * StageA::BYTES;

  int lid = xcd_remap(blockIdx.x, args.padded);
  if (lid >= args.total) return;
  // Split-K: chunk-major, so the workgroups of one chunk (which share its
  // k-range of both operands) sit together on an XCD.
  int chunk = 0;
  if (args.ksplit > 1) {
    chunk = lid / args.tiles;
    lid -= chunk * args.tiles;
  }
  // Grouped ordering over (tiles_m, nprob * tiles_n): GROUP_M tile-rows share
  // each weight panel while it is hot in L2.
  const int tiles_n_all = args.tiles_n * args.nprob;
  const int in_group = GROUP_M * tiles_n_all;
  const int group = lid / in_group;
  const int first_m = group * GROUP_M;
  const int gsize = min(args.tiles_m - first_m, GROUP_M);
  const int tm = first_m + (lid % in_group) % gsize;
  const int tn_all = (lid % in_group) / gsize;
  const int prob = __builtin_amdgcn_readfirstlane(tn_all / args.tiles_n);
  const int tn = tn_all % args.tiles_n;

  const GemmProblem P = args.p[prob];
  const int m0 = tm * TM, n0 = tn * TN;
  const int M = args.M, N = args.N, K = args.K;

  const int t = threadIdx.x;
  const int lane = t & 63;
  const int wave = __builtin_amdgcn_readfirstlane(t >> 6);
  const int wm = wave / WN, wn = wave % WN;
  const int li = lane & 31, hf = lane >> 5;
  const int mw = m0 + wm * (TM / WM), nw = n0 + wn * (TN / WN);

  StageA sa;
  StageB sb;
  sa.init(m0, M, args.lda);
  sb.init(n0, N, args.ldb);
  floatx16 acc[BI][BJ], cor[BI][BJ];  // hh, and the five corrections
#pragma unroll
  for (int i = 0; i < BI; ++i)
#pragma unroll
    for (int j = 0; j < BJ; ++j)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[i][j][r] = cor[i][j][r] = 0.f;
  const int kt0 = chunk * args.kchunk;
  const int nk = args.ksplit > 1 ? min(args.kchunk, K / 16 - kt0) : K / 16;
  const int ktail = args.ksplit > 1 ? 0 : K % 16;  // split-K: the reduce adds the ragged rows
  const float *__restrict__ A = StageA::tile(P.a, kt0, args.lda);
  const float *__restrict__ W = StageB::tile(P.w, kt0, args.ldb);
  // K segments exist only in the plain input-gradient instance; the segment of
  // k-tile kt is wave-uniform, so choosing it takes scalar selects only.
  constexpr bool SEG = TB && !TA && !EPI;
  auto load = [&](int kt) {
    if (SEG && args.kseg > 0) {
      const int sg = (kt >= args.kseg) + (kt >= 2 * args.kseg);
      const int kl = kt - sg * args.kseg;
      sa.load(StageA::tile(sg == 0 ? args.p[0].a : sg == 1 ? args.p[1].a : args.p[2].a, kl, args.lda));
      sb.load(StageB::tile(sg == 0 ? args.p[0].w : sg == 1 ? args.p[1].w : args.p[2].w, kl, args.ldb));
    } else {
      sa.load(StageA::tile(A, kt, args.lda));
      sb.load(StageB::tile(W, kt, args.ldb));
    }
  };
  const bool bsum = TA && P.bgrad && tn == 0;
  float bpart[TA ? 4 * StageA::NP : 1];
  if constexpr (TA) {
#pragma unroll
    for (int i = 0; i < 4 * StageA::NP; ++i) bpart[i] = 0.f;
  }
  auto add_bias = [&]() {
    if constexpr (TA) {
#pragma unroll
      for (int i = 0; i < StageA::NP; ++i)
#pragma unroll
        for (int c = 0; c < 4; ++c) bpart[4 * i + c] += sa.v[2 * i][c] + sa.v[2 * i + 1][c];
    }
  };
  // Split-K chunks take turns in the sign of opA: the drift of the partial
  // sums (common.h) would otherwise add up over the chunks.
  const float scale_a = TA && TB && (chunk & 1) ? -kSplitScale : kSplitScale;
  auto stage = [&](int buf) {
    sa.store(As + buf * StageA::BYTES, scale_a);
    sb.store(Bs + buf * StageB::BYTES, kSplitScale);
  };
  const int ao = StageA::operand(wm * (TM / WM), li, hf), bo = StageB::operand(wn * (TN / WN), li, hf);
  bf16x8 a[3][BI], b[3][BJ];
  auto read_a = [&](int p, int buf) {
#pragma unroll
    for (int i = 0; i < BI; ++i)
      a[p][i] = *reinterpret_cast<const bf16x8 *>(As + buf * StageA::BYTES + p * StageA::PLANE + ao +
                                                  i * StageA::BLOCK);
  };
  auto read_b = [&](int p, int buf) {
#pragma unroll
    for (int j = 0; j < BJ; ++j)
      b[p][j] = *reinterpret_cast<const bf16x8 *>(Bs + buf * StageB::BYTES + p * StageB::PLANE + bo +
                                                  j * StageB::BLOCK);
  };
  auto product = [&](int q) {
#pragma unroll
    for (int i = 0; i < BI; ++i)
#pragma unroll
      for (int j = 0; j < BJ; ++j) {
        floatx16 &c = q == kSplitMain ? acc[i][j] : cor[i][j];
        c = mfma32x32x16(a[kSplitA[q]][i], b[kSplitB[q]][j], c);
      }
  };

  if (nk > 0) {
    // k-tiles 0 .. NB - 2 -> LDS, k-tile NB - 1 -> registers.  Past the end
    // (here and in the loop) loads and stages repeat the last tile into a
    // buffer that nothing reads again: unconditional, they keep the staging
    // registers out of scratch memory.
#pragma unroll
    for (int i = 0; i < NB; ++i) {
      load(min(i, nk - 1));
      if (i < NB - 1) {
        if (TA && bsum && i < nk) add_bias();
        stage(i);
      }
    }
    __syncthreads();
    if constexpr (NB == 3) {
      read_a(2, 0);
      read_b(0, 0);
    }
    int cur = 0;
#pragma unroll 1
    for (int kt = 0; kt < nk; ++kt) {
      const int nxt = cur + 1 < NB ? cur + 1 : 0;
      const int st = NB == 2 ? nxt : (nxt + 1 < NB ? nxt + 1 : 0);  // the buffer k-tile kt - 1 has left
      if (TA && bsum && kt + NB - 1 < nk) add_bias();
      if constexpr (NB == 2) {
        read_a(2, cur);
        read_b(0, cur);
      }
      read_a(0, cur);
      read_b(2, cur);
      read_a(1, cur);
      read_b(1, cur);
      product(0);
      product(1);
      stage(st);
      load(min(kt + NB, nk - 1));
      product(2);
      product(3);
      product(4);
      product(5);
      if constexpr (NB == 3) {
        read_a(2, nxt);
        read_b(0, nxt);
        constexpr int NM = kSplitProducts * BI * BJ;
        constexpr int NR = 2 * (BI + BJ);  // reads between the first MFMAs, then the stores
// Spreads a k-tile's VALU instructions (104 of the splits) over its 24 MFMAs; us with
        // 4 / 6 of them per MFMA: forward 16384 x 4096 -> 1024 702 / 710, its dW 737 / 727.
        constexpr int VALU = TA || TB ? 6 : 4;
        constexpr int STORES = StageA::STORES + StageB::STORES;
        constexpr int AT_ONCE = (STORES + NM - NR - 1) / (NM - NR);
        constexpr int EVERY = STORES > (NM - NR) / 2 ? 1 : 2;
#pragma unroll
        for (int q = 0; q < NM; ++q) {
          __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);     // MFMA
          __builtin_amdgcn_sched_group_barrier(0x002, VALU, 0);  // VALU
          if (q < NR) __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);                             // LDS read
          else if (q % EVERY == EVERY - 1) __builtin_amdgcn_sched_group_barrier(0x200, AT_ONCE, 0);  // LDS write
        }
      }
      __syncthreads();
      cur = nxt;
    }
  }
  if (ktail) {  // uniform over the workgroup
    sa.load_tail(StageA::tile(A, nk, args.lda), ktail);
    sb.load_tail(StageB::tile(W, nk, args.ldb), ktail);
    if (TA && bsum) add_bias();
    stage(0);
    __syncthreads();
#pragma unroll
    for (int p = 0; p < 3; ++p) {
      read_a(p, 0);
      read_b(p, 0);
    }
#pragma unroll
    for (int q = 0; q < kSplitProducts; ++q) product(q);
    __syncthreads();
  }
  {
    // rows and columns of odd index were negated (rows 8 (r / 4) + 4 hf + r % 4)
    const float s0 = (li & 1) != (scale_a < 0.f) ? -kSplitUnscale2 : kSplitUnscale2;
    float bad = 0.f;
#pragma unroll
    for (int i = 0; i < BI; ++i)
#pragma unroll
      for (int j = 0; j < BJ; ++j) {
#pragma unroll
        for (int r = 0; r < 16; ++r) acc[i][j][r] = (acc[i][j][r] + cor[i][j][r]) * (r & 1 ? -s0 : s0);
        bad = nonfinite_sum(acc[i][j], bad);
      }
    if (any_nonfinite(bad)) {
      const bool seg = SEG && args.kseg > 0;
      recompute_blocks<BI, BJ, TA, TB>(args, seg ? 0 : prob, seg ? 3 : 1, seg ? 0 : kt0 * 16,
                                       seg ? args.kseg * 16 : kt0 * 16 + nk * 16 + ktail, mw, nw, li, hf, acc);
    }
  }

  if constexpr (TA) {
    if (bsum) {
      // the eight k pairs of four rows are lanes 8 g .. 8 g + 7
#pragma unroll
      for (int i = 0; i < StageA::NP; ++i)
#pragma unroll
        for (int c = 0; c < 4; ++c) {
          float s = bpart[4 * i + c];
#pragma unroll
          for (int off = 4; off > 0; off >>= 1) s += __shfl_xor(s, off);
          const int m = m0 + sa.unit_row(i) + c;
          if (sa.sb == 0 && m < M) {
            if (args.ksplit > 1)
              args.wsb[((size_t)chunk * args.nprob + prob) * M + m] = s;
            else
              P.bgrad[m] += s;
          }
        }
    }
  }
  float *band = reinterpret_cast<float *>(smem) + wave * 32 * (32 * BJ + 4);
  static_assert(sizeof(smem) >= sizeof(float) * WM * WN * 32 * (32 * BJ + 4), "epilogue bands");
  TileOut out{P.c, args.ldc, P.bias, args.act, args.beta, ROPE && prob < 2};
  if (TA && args.ksplit > 1)  // the partial product of this chunk, reduced later
    out = TileOut{args.ws + ((size_t)chunk * args.nprob + prob) * (size_t)M * N, N, nullptr, CDML_ACT_NONE, 0, false};
  store_tile<BI, BJ, EPI, ROPE>(args, out, acc, mw, nw, lane, band);
}

// Forward product on the fp32 MFMA (K % 16 == 0, 16-byte aligned rows, element
// offsets below 2^32), for the pre-activations of ReLU and leaky ReLU layers
// that train (GemmArgs::f32): the sign of z picks the derivative, so a z within
// rounding of 0 moves a whole row of the layer below's gradient by up to a
// tenth of its rms when its last bits change; above 16 rows these products keep
// the bits they have always had.  fp32-equivalent TFLOP/s with z / without:
// 130816 x 256 -> 1024 118 / 127, 16380 x 1024 -> 4096 137 / 138 (the split
// kernel has 147-195).
//
// Both operand tiles sit in LDS as [rows][16] with pitch 20 floats, double
// buffered; lanes read 16-byte operands that feed four v_mfma_f32_32x32x2_f32
// each, so k is visited in the order 8 (s / 4) + 4 h + s % 4.  The operands of
// the second half of a k-tile are read while the MFMAs of the first run.  The
// rows of a wave's 16 are stored in the order 0, 4, 8, 12, 1, 5, ..., whose
// 64-byte pieces fall in disjoint banks.  The activation is a template argument
// and the epilogue stores from the accumulators, whole wave blocks without a
// predicate: with a run-time activation behind store_tile, and without the
// read-ahead, the kernel took 697 instead of 541 us for 130816 x 256 -> 1024 and 90
// instead of 78 us for 16384 x 512 -> 512.
template <int TM, int TN, int WM, int WN, int ACT, bool EPI>
__global__ void __launch_bounds__(64 * WM * WN, 2) gemm_f32_kernel(const GemmArgs args) {
  constexpr int NT = 64 * WM * WN, BKK = 16, LD = BKK + 4;
  constexpr int BI = TM / WM / 32, BJ = TN / WN / 32;
  constexpr int RPP = NT / 4, NA = TM / RPP, NB = TN / RPP;
  __shared__ __attribute__((aligned(16))) float As[2][TM][LD];
  __shared__ __attribute__((aligned(16))) float Bs[2][TN][LD];

  const int lid = xcd_remap(blockIdx.x, args.padded);
  if (lid >= args.total) return;
  const int in_group = GROUP_M * args.tiles_n;
  const int group = lid / in_group;
  const int first_m = group * GROUP_M;
  const int gsize = min(args.tiles_m - first_m, GROUP_M);
  const int tm = first_m + (lid % in_group) % gsize;
  const int tn = (lid % in_group) / gsize;
  const GemmProblem P = args.p[0];
  const int M = args.M, N = args.N;
  const int m0 = tm * TM, n0 = tn * TN;
  const int t = threadIdx.x, lane = t & 63;
  const int wave = __builtin_amdgcn_readfirstlane(t >> 6);
  const int wm = wave / WN, wn = wave % WN;
  const int li = lane & 31, hf = lane >> 5;

  const int q = t / 4, row = (q & ~15) | ((q & 3) << 2) | ((q >> 2) & 3), col = (t % 4) * 4;
  uint32_t offa[NA], offb[NB];
  vf4 va[NA], vb[NB];
#pragma unroll
  for (int i = 0; i < NA; ++i) offa[i] = (uint32_t)min(m0 + row + RPP * i, M - 1) * (uint32_t)args.lda + col;
#pragma unroll
  for (int i = 0; i < NB; ++i) offb[i] = (uint32_t)min(n0 + row + RPP * i, N - 1) * (uint32_t)args.ldb + col;
  auto load = [&](int kt) {
#pragma unroll
    for (int i = 0; i < NA; ++i) va[i] = *reinterpret_cast<const vf4 *>(P.a + (size_t)kt * BKK + offa[i]);
#pragma unroll
    for (int i = 0; i < NB; ++i) vb[i] = *reinterpret_cast<const vf4 *>(P.w + (size_t)kt * BKK + offb[i]);
  };
  auto stage = [&](int buf) {
#pragma unroll
    for (int i = 0; i < NA; ++i) *reinterpret_cast<vf4 *>(&As[buf][row + RPP * i][col]) = va[i];
#pragma unroll
    for (int i = 0; i < NB; ++i) *reinterpret_cast<vf4 *>(&Bs[buf][row + RPP * i][col]) = vb[i];
  };
  floatx16 acc[BI][BJ];
#pragma unroll
  for (int i = 0; i < BI; ++i)
#pragma unroll
    for (int j = 0; j < BJ; ++j)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[i][j][r] = 0.f;
  const int nk = args.K / BKK;
  load(0);
  stage(0);
  load(min(1, nk - 1));
  __syncthreads();
  for (int kt = 0; kt < nk; ++kt) {
    const int cur = kt & 1;
    const float(*as)[LD] = &As[cur][wm * (TM / WM) + li];
    const float(*bs)[LD] = &Bs[cur][wn * (TN / WN) + li];
    vf4 a4[2][BI], b4[2][BJ];  // operands of the two halves of the k-tile
    auto read = [&](int u) {
#pragma unroll
      for (int i = 0; i < BI; ++i) a4[u][i] = *reinterpret_cast<const vf4 *>(&as[i * 32][u * 8 + hf * 4]);
#pragma unroll
      for (int j = 0; j < BJ; ++j) b4[u][j] = *reinterpret_cast<const vf4 *>(&bs[j * 32][u * 8 + hf * 4]);
    };
    read(0);
#pragma unroll
    for (int u = 0; u < BKK / 8; ++u) {
      if (u == 0) read(1);
#pragma unroll
      for (int r = 0; r < 4; ++r)
#pragma unroll
        for (int i = 0; i < BI; ++i)
#pragma unroll
          for (int j = 0; j < BJ; ++j) acc[i][j] = mfma32x32x2(a4[u][i][r], b4[u][j][r], acc[i][j]);
    }
    // past the end both repeat the last tile into the idle buffer
    stage(cur ^ 1);
    load(min(kt + 2, nk - 1));
    __syncthreads();
  }

  const int mw = m0 + wm * (TM / WM), nw = n0 + wn * (TN / WN);
  float bias[BJ];
#pragma unroll
  for (int j = 0; j < BJ; ++j) {
    const int n = nw + j * 32 + li;
    bias[j] = P.bias && n < N ? P.bias[n] : 0.f;
  }
  // D[i][j] of a block sits at row 8 (r / 4) + 4 hf + r % 4, column li: 32 lanes
  // store 32 consecutive columns of one row.  A launch here has no option but
  // the pre-activation (cdml_linear_preact).
  float *cb = P.c + (size_t)(mw + 4 * hf) * args.ldc + nw + li;
  float *pb = EPI ? args.pre + (size_t)(mw + 4 * hf) * args.ldpre + nw + li : nullptr;
  auto store = [&](auto whole) {
#pragma unroll
    for (int i = 0; i < BI; ++i)
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const int d = i * 32 + 8 * (r >> 2) + (r & 3);
#pragma unroll
        for (int j = 0; j < BJ; ++j) {
          if (!decltype(whole)::value && (mw + 4 * hf + d >= M || nw + j * 32 + li >= N)) continue;
          const float z = acc[i][j][r] + bias[j];
          if (EPI) pb[(size_t)d * args.ldpre + j * 32] = z;
          cb[(size_t)d * args.ldc + j * 32] = activate(z, ACT);
        }
      }
  };
  if (mw + TM / WM <= M && nw + TN / WN <= N) store(std::true_type{});  // wave-uniform
  else store(std::false_type{});
}

// Few rows (decode steps, short batches: M <= MR), non-transposed operands,
// 16-byte aligned rows with K % 4 == 0.  W is read once and bounds the kernel,
// so what counts is how much of it is in flight: a wave owns a pair of output
// columns (n, n + 1), its lanes stride over K in float4 steps, and the W loads
// of four steps are issued before the first product.  Rows past M repeat the
// last one (a load in place of a branch per row and step) and are not stored.
// The pair is also the rotation pair of the fused RoPE epilogue (head dims are
// even).
//   KS = 1: the workgroup's four waves take four column pairs.
//   KS = 4: they share one pair, wave w taking every fourth step from w on, and
//     wave 0 adds the four sums in that order: four times the workgroups for
//     launches that would leave CUs idle (see launch_rows).
// The 2 * MR sums of a lane are reduced by halving: a step of the xor tree
// leaves each lane half of the values, 17 shuffles at MR = 8 instead of 96,
// with the tree's additions.
// Measured on MI355X: a decoder layer's step for 8 sequences (D 1024, FF 4096,
// 2048 keys, 12.6 M weights) took 133.7 us with one float4 of each column in
// flight, a branch per row and one pair per wave throughout, and takes 82.1 us.
template <int MR, int KS, bool EPI>
__global__ void __launch_bounds__(256) gemm_rows_kernel(const GemmArgs args) {
  static_assert(KS == 1 || KS == 4, "waves per column pair");
  constexpr int U = 4;  // steps whose W loads are in flight together
  // x of the next step is loaded before this one's products: us without / with
  // at KS = 1, 8 rows, 1024 -> 4096 9.3 / 7.5, 1024 -> 16384 24.1 / 21.1; one row
  // gains nothing (4096 -> 2040 8.0 / 9.2), and at KS = 4 the registers cost more
  // where K is short (1024 -> 1536 5.2 / 6.5).
  constexpr bool AHEAD = KS == 1 && (MR == 4 || MR == 8);
  const int prob = blockIdx.y;
  const GemmProblem P = args.p[prob];
  const int M = args.M, N = args.N, K = args.K;
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int n0 = 2 * (KS == 1 ? (int)blockIdx.x * 4 + wave : (int)blockIdx.x);
  if (n0 >= N) return;  // KS = 4: the whole workgroup or none of it
  const int n1 = min(n0 + 1, N - 1);
  const float *__restrict__ w0 = P.w + (size_t)n0 * args.ldb;
  const float *__restrict__ w1 = P.w + (size_t)n1 * args.ldb;
  const float *x[MR];
#pragma unroll
  for (int m = 0; m < MR; ++m) x[m] = P.a + (size_t)min(m, M - 1) * args.lda;
  float s[2 * MR];  // (row m, column n0 + c) at 2 m + c
#pragma unroll
  for (int i = 0; i < 2 * MR; ++i) s[i] = 0.f;
  auto load_x = [&](int k, float4 (&v)[MR]) {
#pragma unroll
    for (int m = 0; m < MR; ++m) v[m] = *reinterpret_cast<const float4 *>(x[m] + k);
  };
  auto step = [&](const float4 (&v)[MR], const float4 &a, const float4 &b) {
#pragma unroll
    for (int m = 0; m < MR; ++m) {
      s[2 * m] += (v[m].x * a.x + v[m].y * a.y) + (v[m].z * a.z + v[m].w * a.w);
      s[2 * m + 1] += (v[m].x * b.x + v[m].y * b.y) + (v[m].z * b.z + v[m].w * b.w);
    }
  };
  constexpr int KSTEP = 256 * KS;
  int kb = KS == 1 ? 0 : 256 * wave;  // wave-uniform; the lane's k is kb + 4 lane
  for (; kb + (U - 1) * KSTEP + 256 <= K; kb += U * KSTEP) {
    float4 a[U], b[U];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      a[u] = *reinterpret_cast<const float4 *>(w0 + kb + u * KSTEP + 4 * lane);
      b[u] = *reinterpret_cast<const float4 *>(w1 + kb + u * KSTEP + 4 * lane);
    }
    float4 v[AHEAD ? 2 : 1][MR];
    if (AHEAD) load_x(kb + 4 * lane, v[0]);
#pragma unroll
    for (int u = 0; u < U; ++u) {
      if (!AHEAD) {
        load_x(kb + u * KSTEP + 4 * lane, v[0]);
      } else {
        if (u + 1 < U) load_x(kb + (u + 1) * KSTEP + 4 * lane, v[(u + 1) & 1]);
        __builtin_amdgcn_sched_barrier(0);  // keeps them ahead of this step's products
      }
      step(v[AHEAD ? u & 1 : 0], a[u], b[u]);
    }
  }
  for (int k = kb + 4 * lane; k < K; k += KSTEP) {
    float4 v[MR];
    load_x(k, v);
    step(v, *reinterpret_cast<const float4 *>(w0 + k), *reinterpret_cast<const float4 *>(w1 + k));
  }
  // After the halving steps, lane l holds value l / (32 / MR).
#pragma unroll
  for (int half = MR, off = 32; off > 0; off >>= 1, half >>= 1) {
    if (half > 0) {
      const bool up = (lane & off) != 0;
#pragma unroll
      for (int i = 0; i < half; ++i) {
        const float keep = up ? s[i + half] : s[i], give = up ? s[i] : s[i + half];
        s[i] = keep + __shfl_xor(give, off);
      }
    } else {
      s[0] += __shfl_xor(s[0], off);
    }
  }
  float z0 = s[0], z1 = __shfl_xor(s[0], 32 / MR);  // of row m, in its first lane
  constexpr int LPR = 64 / MR;                      // lanes per row
  const int m = lane / LPR;
  if constexpr (KS > 1) {
    __shared__ float2 part[KS][MR];
    if (lane % LPR == 0) part[wave][m] = make_float2(z0, z1);
    __syncthreads();
    if (wave > 0) return;
    z0 = z1 = 0.f;
#pragma unroll
    for (int w = 0; w < KS; ++w) {
      z0 += part[w][m].x;
      z1 += part[w][m].y;
    }
  }
  if (lane % LPR != 0 || m >= M) return;
  const bool has1 = n0 + 1 < N;
  z0 += P.bias ? P.bias[n0] : 0.f;
  if (has1) z1 += P.bias ? P.bias[n0 + 1] : 0.f;
  if (args.rope_cs && prob < 2) {  // AccelerationCPU.cs:4947-4975 on the pair (n0, n0 + 1)
#pragma clang fp contract(off)
    int pos = args.rope_pos0 + (args.rope_seg > 0 ? m % args.rope_seg : m);
    pos = min(pos, args.rope_npos - 1);
    const float2 t = args.rope_cs[(size_t)pos * (args.rope_hd >> 1) + ((n0 % args.rope_hd) >> 1)];
    float *c = P.c + (size_t)m * args.ldc + n0;
    c[0] = z0 * t.x - z1 * t.y;
    if (has1) c[1] = z1 * t.x + z0 * t.y;
    return;
  }
  store_elem<EPI>(args, P, m, n0, z0, args.act);
  if (has1) store_elem<EPI>(args, P, m, n0 + 1, z1, args.act);
}

// A short reduction (K <= 16: the input projection of a time-series model,
// F features -> D), non-transposed operands, N <= 1024: thread t owns the
// four columns 4 (t % n4) .. + 3 (n4 = ceil(N / 4)) of rows t / n4,
// t / n4 + 256 / n4, ..., and keeps their K x 4 weights and biases in
// registers.  The threads of one row read the same K inputs (broadcast
// loads) and the four results leave as one float4 when the row layout
// allows it.  Every output sums its K products in k order.  TB: W is read as
// [K, N] (the input gradient dX = dY W of a layer with few outputs).
template <bool EPI, bool TB = false>
__global__ void __launch_bounds__(256) gemm_smallk_kernel(const GemmArgs args) {
  const GemmProblem P = args.p[blockIdx.y];
  const int M = args.M, N = args.N, K = args.K;
  const int n4 = (N + 3) / 4;
  const int rpp = 256 / n4;  // rows per pass of the workgroup (n4 <= 256)
  const int r = threadIdx.x / n4, n0 = (threadIdx.x % n4) * 4;
  if (r >= rpp) return;      // threads past the last whole row group
  float w[16][4], bias[4];
#pragma unroll
  for (int k = 0; k < 16; ++k)
#pragma unroll
    for (int c = 0; c < 4; ++c) {
      const int n = min(n0 + c, N - 1);
      w[k][c] = k < K ? P.w[TB ? (size_t)k * args.ldb + n : (size_t)n * args.ldb + k] : 0.f;
    }
#pragma unroll
  for (int c = 0; c < 4; ++c) bias[c] = P.bias && n0 + c < N ? P.bias[n0 + c] : 0.f;
  for (int m = blockIdx.x * rpp + r; m < M; m += gridDim.x * rpp) {
    const float *__restrict__ x = P.a + (size_t)m * args.lda;
    float z[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int k = 0; k < 16; ++k) {
      if (k < K) {
        const float xv = x[k];
#pragma unroll
        for (int c = 0; c < 4; ++c) z[c] += xv * w[k][c];
      }
    }
    float *crow = P.c + (size_t)m * args.ldc;
    if (!EPI && !args.beta && n0 + 3 < N && ((reinterpret_cast<uintptr_t>(crow + n0) & 15) == 0)) {
      vf4 y;
#pragma unroll
      for (int c = 0; c < 4; ++c) y[c] = activate(z[c] + bias[c], args.act);
      *reinterpret_cast<vf4 *>(crow + n0) = y;
      continue;
    }
#pragma unroll
    for (int c = 0; c < 4; ++c)
      if (n0 + c < N) store_elem<EPI>(args, P, m, n0 + c, z[c] + bias[c], args.act);
  }
}

// Few output columns (N <= 4: a regression head, D -> 1), non-transposed
// operands, K % 4 == 0 with 16-byte aligned rows: the 16 lanes of a group
// take every 16th float4 of one row, their partial dot products meet through
// four xor shuffles inside the group, and its first lane stores the N
// outputs.  (The tiled kernel would run a 128 x 128 MFMA tile for one live
// column.)
constexpr int kNarrowN = 4;
template <bool EPI>
__global__ void __launch_bounds__(256) gemm_narrow_n_kernel(const GemmArgs args) {
  const GemmProblem P = args.p[blockIdx.y];
  const int M = args.M, N = args.N, K4 = args.K / 4;
  const int g = threadIdx.x & 15;
  for (int m = (blockIdx.x * 256 + threadIdx.x) >> 4; m < M; m += gridDim.x * 16) {
    const float *__restrict__ x = P.a + (size_t)m * args.lda;
    float z[kNarrowN] = {0.f, 0.f, 0.f, 0.f};
    for (int i = g; i < K4; i += 16) {
      const vf4 xv = *reinterpret_cast<const vf4 *>(x + 4 * i);
#pragma unroll
      for (int n = 0; n < kNarrowN; ++n)
        if (n < N) {
          const vf4 wv = *reinterpret_cast<const vf4 *>(P.w + (size_t)n * args.ldb + 4 * i);
          z[n] += (xv[0] * wv[0] + xv[1] * wv[1]) + (xv[2] * wv[2] + xv[3] * wv[3]);
        }
    }
#pragma unroll
    for (int n = 0; n < kNarrowN; ++n)
#pragma unroll
      for (int off = 8; off > 0; off >>= 1) z[n] += __shfl_xor(z[n], off, 16);
    if (g == 0) {
#pragma unroll
      for (int n = 0; n < kNarrowN; ++n)
        if (n < N) store_elem<EPI>(args, P, m, n, z[n] + (P.bias ? P.bias[n] : 0.f), args.act);
    }
  }
}

// Any layout, any shape (the gradient GEMMs whose sizes miss the tiled
// kernel's conditions): a 64 x 64 tile of C per 256-thread workgroup, 4 x 4
// outputs per thread, K in steps of 16 through LDS with guarded loads that
// walk each source along its contiguous dimension.
template <bool TA, bool TB, bool EPI>
__global__ void __launch_bounds__(256) gemm_any_kernel(const GemmArgs args) {
  __shared__ float As[16][65], Bs[16][65];  // [k][m], [k][n]
  const GemmProblem P = args.p[blockIdx.z];
  const int m0 = blockIdx.y * 64, n0 = blockIdx.x * 64;
  const int M = args.M, N = args.N, K = args.K;
  const int t = threadIdx.x, tx = t & 15, ty = t >> 4;
  float acc[4][4] = {};
  for (int k0 = 0; k0 < K; k0 += 16) {
    for (int e = t; e < 1024; e += 256) {
      const int kk = TA ? e / 64 : e % 16, mm = TA ? e % 64 : e / 16;
      const int m = m0 + mm, k = k0 + kk;
      As[kk][mm] = (m < M && k < K) ? (TA ? P.a[(size_t)k * args.lda + m] : P.a[(size_t)m * args.lda + k]) : 0.f;
      const int kb = TB ? e / 64 : e % 16, nn = TB ? e % 64 : e / 16;
      const int n = n0 + nn, kq = k0 + kb;
      Bs[kb][nn] = (n < N && kq < K) ? (TB ? P.w[(size_t)kq * args.ldb + n] : P.w[(size_t)n * args.ldb + kq]) : 0.f;
    }
    __syncthreads();
#pragma unroll
    for (int kk = 0; kk < 16; ++kk) {
      float a[4], b[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) a[i] = As[kk][ty * 4 + i];
#pragma unroll
      for (int j = 0; j < 4; ++j) b[j] = Bs[kk][tx * 4 + j];
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j) acc[i][j] += a[i] * b[j];
    }
    __syncthreads();
  }
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int m = m0 + ty * 4 + i;
    if (m >= M) continue;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int n = n0 + tx * 4 + j;
      if (n >= N) continue;
      store_elem<EPI>(args, P, m, n, acc[i][j] + (P.bias ? P.bias[n] : 0.f), args.act);
    }
  }
}

// bgrad[m] += sum_k opA[m, k] for the problems of a gemm_any_kernel launch.
template <bool TA>
__global__ void __launch_bounds__(256) op_rowsum_kernel(const GemmArgs args) {
  const GemmProblem P = args.p[blockIdx.y];
  const int m = blockIdx.x * 256 + threadIdx.x;
  if (!P.bgrad || m >= args.M) return;
  float s = 0.f;
  for (int k = 0; k < args.K; ++k) s += TA ? P.a[(size_t)k * args.lda + m] : P.a[(size_t)m * args.lda + k];
  P.bgrad[m] += s;
}

// Sum of the split-K partials: C (+)= sum_c ws[c], bgrad += sum_c wsb[c].
// N % 4 == 0 (the tiled path's transposed staging of opB needs it), so an
// output is four consecutive columns.  LANES consecutive lanes share an
// output: lane g adds chunks g, g + LANES, ... in order, and a fixed
// xor-shuffle tree joins the sums, so the order of every addition is fixed
// (the same bits on every run) while the chunk loads of the group are in
// flight together.  The group of output e also sums bias row e.  Eight
// lanes pay off from 32 chunks on; below that one lane walks the chunks.
template <int LANES>
__global__ void __launch_bounds__(256) splitk_reduce_kernel(const GemmArgs args) {
  constexpr int kReduceLanes = LANES;
  const int prob = blockIdx.y;
  const GemmProblem P = args.p[prob];
  const int M = args.M, N = args.N, n4 = N >> 2;
  const size_t plane = (size_t)args.nprob * M * N;
  const size_t e = ((size_t)blockIdx.x * 256 + threadIdx.x) / kReduceLanes;
  const int g = threadIdx.x % kReduceLanes;
  const size_t n_out = (size_t)M * n4;
  if (e < n_out) {
    const int m = (int)(e / n4), n = (int)(e % n4) * 4;
    const float *src = args.ws + (size_t)prob * M * N + (size_t)m * N + n;
    vf4 s = {0.f, 0.f, 0.f, 0.f};
    for (int c = g; c < args.ksplit; c += kReduceLanes) {
      const vf4 x = *reinterpret_cast<const vf4 *>(src + c * plane);
      s[0] += x[0];
      s[1] += x[1];
      s[2] += x[2];
      s[3] += x[3];
    }
    // the ragged last rows: opA stored [K, M], opB [K, N] (16-byte rows)
    for (int k = args.ktail0 + g; args.ktail0 > 0 && k < args.K; k += kReduceLanes) {
      const float av = P.a[(size_t)k * args.lda + m];
      const vf4 bv = *reinterpret_cast<const vf4 *>(P.w + (size_t)k * args.ldb + n);
#pragma unroll
      for (int q = 0; q < 4; ++q) s[q] += av * bv[q];
    }
#pragma unroll
    for (int off = kReduceLanes / 2; off > 0; off >>= 1)
#pragma unroll
      for (int q = 0; q < 4; ++q) s[q] += __shfl_xor(s[q], off);
    if (g == 0) {
      float *dst = P.c + (size_t)m * args.ldc + n;
#pragma unroll
      for (int q = 0; q < 4; ++q) dst[q] = args.beta ? dst[q] + s[q] : s[q];
    }
  }
  // every lane of a group runs the shuffles together (e is uniform in a group)
  if (P.bgrad && e < (size_t)M) {
    float s = 0.f;
    for (int c = g; c < args.ksplit; c += kReduceLanes)
      s += args.wsb[((size_t)c * args.nprob + prob) * M + e];
    for (int k = args.ktail0 + g; args.ktail0 > 0 && k < args.K; k += kReduceLanes)
      s += P.a[(size_t)k * args.lda + e];
#pragma unroll
    for (int off = kReduceLanes / 2; off > 0; off >>= 1) s += __shfl_xor(s, off);
    if (g == 0) P.bgrad[e] += s;
  }
}

// Split-K plan of a weight-gradient GEMM (M = out, N = in, K = rows): enough
// chunks to give every CU two resident workgroups when the output alone has
// too few tiles, at least eight k-tiles (128 rows) per chunk (two for small
// outputs).
struct SplitPlan {
  int ksplit = 1, kchunk = 0;
  bool small = false;  // small output: wgrad_small_kernel, kchunk in rows
  size_t bytes = 0;    // workspace: ksplit * nprob * (M * N + M) floats
};

// Weight gradients whose output is too small or too oddly shaped for the
// tiled kernel (an input projection [D, 5], a regression head [1, D]) but
// whose row reduction is long: block c sums rows [c * kchunk, (c + 1) *
// kchunk) of opA^T opB (opA stored [K, M], opB [K, N]) and of opA's row
// sums into its own partial; wgrad_small_reduce_kernel adds the partials in
// block order.  Each thread owns up to kSmallPer outputs.
constexpr int kSmallPer = 16;
constexpr int kSmallOut = 256 * kSmallPer;

__global__ void __launch_bounds__(256) wgrad_small_kernel(const GemmArgs args) {
  const int chunk = blockIdx.x, prob = blockIdx.y, t = threadIdx.x;
  const GemmProblem P = args.p[prob];
  const int M = args.M, N = args.N, MN = M * N;
  const int k0 = chunk * args.kchunk, k1 = min(args.K, k0 + args.kchunk);
  float acc[kSmallPer], bacc[kSmallPer];
  int am[kSmallPer], bn[kSmallPer];
#pragma unroll
  for (int i = 0; i < kSmallPer; ++i) {
    const int e = min(t + 256 * i, MN - 1);
    am[i] = e / N;
    bn[i] = e % N;
    acc[i] = bacc[i] = 0.f;
  }
  const bool bsum = P.bgrad != nullptr;
  for (int k = k0; k < k1; ++k) {
    const float *ar = P.a + (size_t)k * args.lda;
    const float *br = P.w + (size_t)k * args.ldb;
#pragma unroll
    for (int i = 0; i < kSmallPer; ++i)
      if (t + 256 * i < MN) acc[i] += ar[am[i]] * br[bn[i]];
    if (bsum) {
#pragma unroll
      for (int i = 0; i < kSmallPer; ++i)
        if (t + 256 * i < M) bacc[i] += ar[t + 256 * i];
    }
  }
  float *out = args.ws + ((size_t)chunk * args.nprob + prob) * MN;
#pragma unroll
  for (int i = 0; i < kSmallPer; ++i)
    if (t + 256 * i < MN) out[t + 256 * i] = acc[i];
  if (bsum) {
    float *ob = args.wsb + ((size_t)chunk * args.nprob + prob) * M;
#pragma unroll
    for (int i = 0; i < kSmallPer; ++i)
      if (t + 256 * i < M) ob[t + 256 * i] = bacc[i];
  }
}

// The same weight gradients when one side is narrow (at most kNarrow): the
// input projection [D, F] (F = 5) and a regression head [O, D] (O <= 16).
// Threads run along the wide side, so each row of that operand is one
// coalesced load and the narrow side's few values of the row are broadcast
// loads; a thread keeps the narrow side's sums (and the bias row sums) in
// registers over its chunk of rows, in row order, four rows per iteration.
// OVER_M: the output rows m are wide (thread m, columns n < N narrow);
// otherwise the columns n are wide and the rows m < M narrow.
constexpr int kNarrow = 16;
template <bool OVER_M>
__global__ void __launch_bounds__(256) wgrad_narrow_kernel(const GemmArgs args) {
  const int chunk = blockIdx.x, prob = blockIdx.z;
  const GemmProblem P = args.p[prob];
  const int M = args.M, N = args.N, MN = M * N;
  const int wide = OVER_M ? M : N, narrow = OVER_M ? N : M;
  const int i = blockIdx.y * 256 + threadIdx.x;
  const int ic = min(i, wide - 1);
  const int k0 = chunk * args.kchunk, k1 = min(args.K, k0 + args.kchunk);
  const bool bsum = P.bgrad != nullptr;
  float acc[kNarrow], bacc[kNarrow];
#pragma unroll
  for (int j = 0; j < kNarrow; ++j) acc[j] = bacc[j] = 0.f;
  auto row = [&](int k) {
    const float *ar = P.a + (size_t)k * args.lda;
    const float *br = P.w + (size_t)k * args.ldb;
    if constexpr (OVER_M) {
      const float x = ar[ic];
#pragma unroll
      for (int j = 0; j < kNarrow; ++j)
        if (j < narrow) acc[j] += x * br[j];
      bacc[0] += x;
    } else {
      const float y = br[ic];
#pragma unroll
      for (int j = 0; j < kNarrow; ++j)
        if (j < narrow) {
          const float x = ar[j];
          acc[j] += x * y;
          bacc[j] += x;
        }
    }
  };
  int k = k0;
  for (; k + 4 <= k1; k += 4) {
    row(k);
    row(k + 1);
    row(k + 2);
    row(k + 3);
  }
  for (; k < k1; ++k) row(k);
  if (i >= wide) return;
  float *out = args.ws + ((size_t)chunk * args.nprob + prob) * MN;
#pragma unroll
  for (int j = 0; j < kNarrow; ++j)
    if (j < narrow) out[OVER_M ? (size_t)i * N + j : (size_t)j * N + i] = acc[j];
  if (bsum) {
    float *ob = args.wsb + ((size_t)chunk * args.nprob + prob) * M;
    if constexpr (OVER_M) {
      ob[i] = bacc[0];
    } else if (i == 0) {
#pragma unroll
      for (int j = 0; j < kNarrow; ++j)
        if (j < narrow) ob[j] = bacc[j];
    }
  }
}

// Sum of the small-output partials, kSmallLanes lanes per output: lane g adds
// chunks g, g + kSmallLanes, ... in order and a fixed xor-shuffle tree joins
// them (the same bits on every run); the group of output e also sums bias
// row e.
constexpr int kSmallLanes = 64;
__global__ void __launch_bounds__(256) wgrad_small_reduce_kernel(const GemmArgs args) {
  const int prob = blockIdx.y;
  const GemmProblem P = args.p[prob];
  const int M = args.M, N = args.N, MN = M * N;
  const int e = (blockIdx.x * 256 + threadIdx.x) / kSmallLanes;
  const int g = threadIdx.x % kSmallLanes;
  if (e < MN) {
    float s = 0.f;
    for (int c = g; c < args.ksplit; c += kSmallLanes) s += args.ws[((size_t)c * args.nprob + prob) * MN + e];
#pragma unroll
    for (int off = kSmallLanes / 2; off > 0; off >>= 1) s += __shfl_xor(s, off);
    if (g == 0) {
      float *dst = P.c + (size_t)(e / N) * args.ldc + e % N;
      *dst = args.beta ? *dst + s : s;
    }
  }
  if (P.bgrad && e < M) {
    float s = 0.f;
    for (int c = g; c < args.ksplit; c += kSmallLanes) s += args.wsb[((size_t)c * args.nprob + prob) * M + e];
#pragma unroll
    for (int off = kSmallLanes / 2; off > 0; off >>= 1) s += __shfl_xor(s, off);
    if (g == 0) P.bgrad[e] += s;
  }
}

SplitPlan splitk_plan(int M, int N, int K, int nprob) {
  SplitPlan sp;
  const int nk = K / 16;  // whole k-tiles; the reduce or a tail launch adds a ragged tail
  sp.kchunk = nk;
  if (M <= 0 || N <= 0) return sp;
  if (nk < 1 || N % 4 || M % 4) {  // not the tiled kernel's shape
    if ((long long)M * N > kSmallOut || K < 2048) return sp;
    sp.small = true;
    // chunks of 64 rows (at most 4096 chunks): each workgroup's row loop is
    // short, so the launch is not bound by one loop's load latency
    const int bound = std::min(4096, (K + 63) / 64);
    sp.ksplit = bound;
    sp.kchunk = (K + sp.ksplit - 1) / sp.ksplit;
    sp.ksplit = (K + sp.kchunk - 1) / sp.kchunk;
    // sized for the bound, which never decreases with K: a workspace sized
    // for a caller's largest row count covers every smaller one
    sp.bytes = (size_t)bound * nprob * ((size_t)M * N + M) * sizeof(float);
    return sp;
  }
  const int tiles = ((M + 127) / 128) * ((N + 127) / 128) * nprob;
  const int slots = 512;  // two 128 x 128 workgroups per CU
  // at least eight k-tiles per chunk, or two for a small output (at most
  // 64 K elements, so a chunk's partial is at most 256 KB): a short
  // reduction into a few tiles is otherwise one workgroup's serial k-loop
  const int min_kt = (long long)M * N * nprob <= 65536 ? 2 : 8;
  const int s = std::min(slots / tiles, nk / min_kt);
  if (s <= 1) return sp;
  sp.kchunk = (nk + s - 1) / s;
  sp.ksplit = (nk + sp.kchunk - 1) / sp.kchunk;
  if (sp.ksplit <= 1) {
    sp = SplitPlan{};
    sp.kchunk = nk;
    return sp;
  }
  // sized for s (at least ksplit, and never decreasing with K, unlike
  // ksplit itself: 75 k-tiles in 3-tile chunks take 25, 74 in 2-tile chunks
  // 37), so a workspace sized for a caller's largest row count covers every
  // smaller one
  sp.bytes = (size_t)s * nprob * ((size_t)M * N + M) * sizeof(float);
  return sp;
}

template <int TM, int TN, int WM, int WN, int MINB, int NB, bool TA, bool TB>
int launch_tile(GemmArgs g, hipStream_t stream) {
  g.tiles_m = (g.M + TM - 1) / TM;
  g.tiles_n = (g.N + TN - 1) / TN;
  g.tiles = g.tiles_m * g.tiles_n * g.nprob;
  if (g.ksplit < 1) g.ksplit = 1;
  g.total = g.tiles * g.ksplit;
  g.padded = pad_to_xcd(g.total);
  const dim3 grid(g.padded), block(64 * WM * WN);
  if (!TA && !TB && g.rope_cs)
    gemm_tile_kernel<TM, TN, WM, WN, MINB, NB, !TA && !TB, TA, TB, false><<<grid, block, 0, stream>>>(g);
  else if (!(TA && TB) && has_epi(g))
    gemm_tile_kernel<TM, TN, WM, WN, MINB, NB, false, TA, TB, !(TA && TB)><<<grid, block, 0, stream>>>(g);
  else
    gemm_tile_kernel<TM, TN, WM, WN, MINB, NB, false, TA, TB, false><<<grid, block, 0, stream>>>(g);
  if (TA && TB && g.ksplit > 1) {
    const size_t outs = std::max((size_t)g.M * (g.N / 4), (size_t)g.M);
    if (g.ksplit >= 32)
      splitk_reduce_kernel<8><<<dim3((unsigned)((outs * 8 + 255) / 256), g.nprob), dim3(256), 0, stream>>>(g);
    else
      splitk_reduce_kernel<1><<<dim3((unsigned)((outs + 255) / 256), g.nprob), dim3(256), 0, stream>>>(g);
  }
  return CDML_OK;
}

// Whether a [rows, K] (T = false) or [K, rows] (T = true) operand with row
// stride ld and base p suits the tiled kernel's staging.
bool stage_ok(const float *p, int rows, int ld, bool T) {
  if (!aligned16(p) || ld % 4) return false;
  if (T) return rows % 4 == 0 && 16ull * (unsigned long long)ld + (unsigned long long)rows < (1ull << 32);
  return (unsigned long long)rows * ld < (1ull << 32);
}

// Forward products of many rows take 256 x 128 tiles (eight waves, one workgroup per
// CU), which split a quarter less per product: us against 128 x 128, 16384 x 1024 ->
// 4096 690 / 726, 16384 x 512 -> 512 50.6 / 53.7, 130816 x 256 -> 1024 453 / 459.  A last
// round that is less than three quarters full costs more than that until it is one
// of seven (5000 x 1000 -> 2000, 1.25 rounds: 148 / 133).  Both gradients are 2-8%
// slower so: their short k-loops and long epilogues want another workgroup beside.
inline bool wide_tiles(const GemmArgs &g) {
  const int cus = num_cus();
  const long long tiles = (long long)((g.M + 255) / 256) * ((g.N + 127) / 128) * g.nprob, rest = tiles % cus;
  return g.M >= 2048 && tiles > 0 && (rest == 0 || 4 * rest >= 3LL * cus || tiles >= 6LL * cus);
}

// Else 128 x 128 tiles (two workgroups per CU) where they give three quarters of the
// CUs one, 64 x 64 otherwise, four times as many (dX, us): 4096 x 1024 x 1024, 256 tiles
// of 128 x 128: 64 against 69; 2048 x 1024 x 1024, 128 tiles: 62 against 54; 512 x 1024 x
// 1024: 54 against 44.
template <bool TA, bool TB>
int launch_tiled(GemmArgs &g, hipStream_t stream) {
  const long long tiles = (long long)((g.M + 127) / 128) * ((g.N + 127) / 128) * g.nprob * std::max(g.ksplit, 1);
  if constexpr (!TA && !TB)
    if (wide_tiles(g)) return launch_tile<256, 128, 4, 2, 2, 3, TA, TB>(g, stream);
  if (4 * tiles >= 3LL * num_cus()) return launch_tile<128, 128, 2, 2, 2, 3, TA, TB>(g, stream);
  // Four waves where A runs along K: a launch of few workgroups is bound by the splits
  // between a wave's products (520 x 512 -> 512 forward 21.5 -> 16.3 us, dX 24.8 -> 19.8;
  // 200 x 1024 -> 1024 37.4 -> 27.6 and 44 -> 34).  A transposed operand has units for two
  // of them only.
  if constexpr (!TA) return launch_tile<64, 64, 2, 2, 3, 2, TA, TB>(g, stream);
  return launch_tile<64, 64, 2, 1, 3, 2, TA, TB>(g, stream);
}

// 256 x 128 tiles unless they would not fill one round of two workgroups per
// CU: then 128 x 128 tiles spread the same work over twice as many workgroups
// (16384 x 512 -> 512: 81 -> 78 us, same bits).
template <int TM, int TN, int WM, int WN>
void launch_f32_tile(GemmArgs &g, hipStream_t stream) {
  g.tiles_m = (g.M + TM - 1) / TM;
  g.tiles_n = (g.N + TN - 1) / TN;
  g.total = g.tiles_m * g.tiles_n;
  g.padded = pad_to_xcd(g.total);
  const dim3 grid(g.padded), block(64 * WM * WN);
  const bool relu = g.act != CDML_ACT_LEAKYRELU;
  if (g.pre)
    relu ? gemm_f32_kernel<TM, TN, WM, WN, CDML_ACT_RELU, true><<<grid, block, 0, stream>>>(g)
         : gemm_f32_kernel<TM, TN, WM, WN, CDML_ACT_LEAKYRELU, true><<<grid, block, 0, stream>>>(g);
  else
    relu ? gemm_f32_kernel<TM, TN, WM, WN, kActReluMarked, false><<<grid, block, 0, stream>>>(g)
         : gemm_f32_kernel<TM, TN, WM, WN, CDML_ACT_LEAKYRELU, false><<<grid, block, 0, stream>>>(g);
}
void launch_f32(GemmArgs &g, hipStream_t stream) {
  const long long big = (long long)((g.M + 255) / 256) * ((g.N + 127) / 128);
  if (g.M >= 1024 && big >= 2 * num_cus()) launch_f32_tile<256, 128, 4, 2>(g, stream);
  else launch_f32_tile<128, 128, 2, 2>(g, stream);
}

template <bool TA, bool TB>
int launch_any(GemmArgs &g, hipStream_t stream) {
  const dim3 grid((g.N + 63) / 64, (g.M + 63) / 64, g.nprob);
  if (has_epi(g)) gemm_any_kernel<TA, TB, true><<<grid, dim3(256), 0, stream>>>(g);
  else gemm_any_kernel<TA, TB, false><<<grid, dim3(256), 0, stream>>>(g);
  bool bgrad = false;
  for (int i = 0; i < g.nprob; ++i) bgrad = bgrad || g.p[i].bgrad;
  if (bgrad && g.K > 0) op_rowsum_kernel<TA><<<dim3((g.M + 255) / 256, g.nprob), dim3(256), 0, stream>>>(g);
  return CDML_OK;
}

// The four waves of a workgroup share a column pair (KS = 4) where one pair per
// wave would give workgroups to fewer than three CUs in four and K has more than
// one step.  us with KS = 1 / 4, 8 rows: 1024 -> 1024 5.3 / 4.9, 4096 -> 1024
// 11.8 / 9.6, 512 -> 512 4.6 / 4.2; from 1536 outputs on (192 workgroups of 256
// CUs) 1024 -> 1536 5.2 / 5.2, 1024 -> 2040 5.3 / 5.8, 4096 -> 2040 13.2 / 14.7.
template <int MR>
void launch_rows(const GemmArgs &g, hipStream_t stream) {
  const int pairs = (g.N + 1) / 2, wgs = (pairs + 3) / 4;
  const bool epi = has_epi(g), split = 4LL * wgs * g.nprob < 3 * num_cus() && g.K > 256;
  const dim3 grid((unsigned)(split ? pairs : wgs), (unsigned)g.nprob), block(256);
  if (split)
    epi ? gemm_rows_kernel<MR, 4, true><<<grid, block, 0, stream>>>(g)
        : gemm_rows_kernel<MR, 4, false><<<grid, block, 0, stream>>>(g);
  else
    epi ? gemm_rows_kernel<MR, 1, true><<<grid, block, 0, stream>>>(g)
        : gemm_rows_kernel<MR, 1, false><<<grid, block, 0, stream>>>(g);
}

// ta / tb: opA / opB stored transposed ([K, M] / [K, N]).
int launch_gemm(GemmArgs &g, bool ta, bool tb, hipStream_t stream, const char *what) {
  if (g.M == 0 || g.N == 0) return CDML_OK;
  if ((ta || tb) && (g.M > 65535 * 64 || g.N > 65535 * 64))
    return fail(CDML_E_INVALID, "%s: matrix too large", what);
  bool fast = g.K > 0;
  for (int i = 0; i < g.nprob; ++i)
    fast = fast && stage_ok(g.p[i].a, g.M, g.lda, ta) && stage_ok(g.p[i].w, g.N, g.ldb, tb);
  if (g.kseg) {  // only the tiled input-gradient kernel reads K segments
    bool ok = !ta && tb && !has_epi(g) && g.nprob == 1 && g.ksplit <= 1 && g.kseg * 16 * 3 == g.K;
    for (int i = 0; ok && i < 3; ++i)
      ok = stage_ok(g.p[i].a, g.M, g.lda, false) && stage_ok(g.p[i].w, g.N, g.ldb, true);
    if (!ok) return fail(CDML_E_INVALID, "%s: K segments need the tiled input-gradient kernel", what);
    fast = true;
  }
  if (ta || tb) {
    if (!ta && tb && g.K <= 16 && g.K > 0 && g.M > 16 && g.N <= 1024) {  // few layer outputs
      const int rpp = 256 / ((g.N + 3) / 4);
      const dim3 grid((unsigned)std::min((g.M + rpp - 1) / rpp, 2048), (unsigned)g.nprob), block(256);
      has_epi(g) ? gemm_smallk_kernel<true, true><<<grid, block, 0, stream>>>(g)
                 : gemm_smallk_kernel<false, true><<<grid, block, 0, stream>>>(g);
      return check_launch(what);
    }
    if (ta && tb && g.small && g.ksplit > 1) {  // small output, long reduction
      if (g.N <= kNarrow)
        wgrad_narrow_kernel<true><<<dim3(g.ksplit, (g.M + 255) / 256, g.nprob), dim3(256), 0, stream>>>(g);
      else if (g.M <= kNarrow)
        wgrad_narrow_kernel<false><<<dim3(g.ksplit, (g.N + 255) / 256, g.nprob), dim3(256), 0, stream>>>(g);
      else
        wgrad_small_kernel<<<dim3(g.ksplit, g.nprob), dim3(256), 0, stream>>>(g);
      const int n = std::max(g.M * g.N, g.M) * kSmallLanes;
      wgrad_small_reduce_kernel<<<dim3((n + 255) / 256, g.nprob), dim3(256), 0, stream>>>(g);
      return check_launch(what);
    }
    if (fast && ta && tb) {
      if (g.ksplit > 1) g.ktail0 = g.K % 16 ? g.K - g.K % 16 : 0;  // the reduce adds the last K % 16 rows
      launch_tiled<true, true>(g, stream);
    } else if (fast && tb) {
      launch_tiled<false, true>(g, stream);
    } else {
      g.ksplit = 1;
      if (ta && tb) launch_any<true, true>(g, stream);
      else if (tb) launch_any<false, true>(g, stream);
      else launch_any<true, false>(g, stream);
    }
    return check_launch(what);
  }
  g.tiles_m = (g.M + BM - 1) / BM;
  g.tiles_n = (g.N + BN - 1) / BN;
  g.total = g.tiles_m * g.tiles_n * g.nprob;
  g.padded = pad_to_xcd(g.total);
  bool vec = (g.K % 4 == 0) && (g.lda % 4 == 0) && (g.ldb % 4 == 0);
  for (int i = 0; i < g.nprob; ++i) vec = vec && aligned16(g.p[i].a) && aligned16(g.p[i].w);
  if (g.K <= 16 && g.K > 0 && g.M > 16 && !g.rope_cs && g.N <= 1024) {
    const int rpp = 256 / ((g.N + 3) / 4);
    const dim3 grid((unsigned)std::min((g.M + rpp - 1) / rpp, 2048), (unsigned)g.nprob), block(256);
    has_epi(g) ? gemm_smallk_kernel<true><<<grid, block, 0, stream>>>(g)
               : gemm_smallk_kernel<false><<<grid, block, 0, stream>>>(g);
    return check_launch(what);
  }
  if (vec && g.N <= kNarrowN && g.K > 16 && g.M > 16 && !g.rope_cs) {
    const dim3 grid((unsigned)std::min((g.M + 15) / 16, 4096), (unsigned)g.nprob), block(256);
    has_epi(g) ? gemm_narrow_n_kernel<true><<<grid, block, 0, stream>>>(g)
               : gemm_narrow_n_kernel<false><<<grid, block, 0, stream>>>(g);
    return check_launch(what);
  }
  if (vec && g.M <= 16 && g.K > 0 && (g.rope_cs == nullptr || g.rope_hd % 2 == 0)) {
    if (g.M <= 1)
      launch_rows<1>(g, stream);
    else if (g.M <= 2)
      launch_rows<2>(g, stream);
    else if (g.M <= 4)
      launch_rows<4>(g, stream);
    else if (g.M <= 8)
      launch_rows<8>(g, stream);
    else
      launch_rows<16>(g, stream);
    return check_launch(what);
  }
  if (fast && g.f32 && g.K % 16 == 0) {
    launch_f32(g, stream);
  } else if (fast && !g.f32) {
    launch_tiled<false, false>(g, stream);
  } else if (vec)
    has_epi(g) ? gemm_nt_kernel<true, true><<<dim3(g.padded), dim3(NTHREADS), 0, stream>>>(g)
               : gemm_nt_kernel<true, false><<<dim3(g.padded), dim3(NTHREADS), 0, stream>>>(g);
  else
    has_epi(g) ? gemm_nt_kernel<false, true><<<dim3(g.padded), dim3(NTHREADS), 0, stream>>>(g)
               : gemm_nt_kernel<false, false><<<dim3(g.padded), dim3(NTHREADS), 0, stream>>>(g);
  return check_launch(what);
}

// Attaches the split-K workspace of a weight-gradient launch (M = out, N =
// in, K = rows) to g; fails when the caller's workspace is smaller than
// splitk_plan asks for.
int attach_split(GemmArgs &g, void *workspace, size_t workspace_bytes, const char *what) {
  const SplitPlan sp = splitk_plan(g.M, g.N, g.K, g.nprob);
  if (sp.ksplit <= 1) return CDML_OK;
  if (!workspace || workspace_bytes < sp.bytes)
    return fail(CDML_E_INVALID, "%s: workspace of %zu bytes needed, %zu given", what, sp.bytes,
                workspace ? workspace_bytes : (size_t)0);
  if (!aligned16(workspace)) return fail(CDML_E_INVALID, "%s: workspace must be 16-byte aligned", what);
  g.ksplit = sp.ksplit;
  g.kchunk = sp.kchunk;
  g.small = sp.small ? 1 : 0;
  g.ws = static_cast<float *>(workspace);
  g.wsb = g.ws + (size_t)sp.ksplit * g.nprob * g.M * g.N;
  return CDML_OK;
}

}  // namespace
}  // namespace cdml

using namespace cdml;

extern "C" int cdml_linear_backward_workspace_size(int rows, int in_dim, int out_dim, size_t *bytes) {
  if (!bytes) return fail(CDML_E_INVALID, "cdml_linear_backward_workspace_size: NULL pointer");
  if (rows < 0 || in_dim < 0 || out_dim < 0)
    return fail(CDML_E_INVALID, "cdml_linear_backward_workspace_size: negative size");
  *bytes = splitk_plan(out_dim, in_dim, rows, 1).bytes;
  return CDML_OK;
}

extern "C" int cdml_backprop_qkv_workspace_size(int rows, int in_dim, int out_dim, size_t *bytes) {
  if (!bytes) return fail(CDML_E_INVALID, "cdml_backprop_qkv_workspace_size: NULL pointer");
  if (rows < 0 || in_dim < 0 || out_dim < 0)
    return fail(CDML_E_INVALID, "cdml_backprop_qkv_workspace_size: negative size");
  *bytes = splitk_plan(out_dim, in_dim, rows, 3).bytes;
  return CDML_OK;
}

extern "C" int cdml_project_qkv(const float *x, const float *wq, const float *bq, const float *wk,
                                const float *bk, const float *wv, const float *bv, float *q,
                                float *k, float *v, int rows, int in_dim, int out_dim,
                                cdml_stream stream) {
  if (rows < 0 || in_dim < 0 || out_dim < 0)
    return fail(CDML_E_INVALID, "cdml_project_qkv: negative size");
  if (rows == 0 || out_dim == 0) return CDML_OK;
  if (!x || !wq || !wk || !wv || !q || !k || !v)
    return fail(CDML_E_INVALID, "cdml_project_qkv: NULL pointer");
  int rc = ensure_device();
  if (rc) return rc;
  // in_dim == 0: a K of zero leaves the accumulators at 0 and y = bias.
  GemmArgs g{};
  g.lda = in_dim;
  g.ldb = in_dim;
  g.ldc = out_dim;
  g.M = rows;
  g.N = out_dim;
  g.K = in_dim;
  g.nprob = 3;
  g.p[0] = {x, wq, bq, q, nullptr};
  g.p[1] = {x, wk, bk, k, nullptr};
  g.p[2] = {x, wv, bv, v, nullptr};
  g.act = CDML_ACT_NONE;
  return launch_gemm(g, false, false, as_hip(stream), "cdml_project_qkv");
}

extern "C" int cdml_project_qkv_rope(const float *x, const float *wq, const float *bq,
                                     const float *wk, const float *bk, const float *wv,
                                     const float *bv, float *q, float *k, float *v, int rows,
                                     int in_dim, int out_dim, int head_dim, const float *rope_cs,
                                     int n_pos, int pos_offset, int seg_len, cdml_stream stream) {
  if (rows < 0 || in_dim < 0 || out_dim < 0 || n_pos < 0 || pos_offset < 0 || seg_len < 0)
    return fail(CDML_E_INVALID, "cdml_project_qkv_rope: negative size");
  if (head_dim <= 0 || (head_dim & 1) || out_dim % head_dim)
    return fail(CDML_E_INVALID,
                "cdml_project_qkv_rope: head_dim must be even, positive and divide out_dim");
  if (rows == 0 || out_dim == 0) return CDML_OK;
  if (!x || !wq || !wk || !wv || !q || !k || !v || !rope_cs)
    return fail(CDML_E_INVALID, "cdml_project_qkv_rope: NULL pointer");
  if (reinterpret_cast<uintptr_t>(rope_cs) % 8)
    return fail(CDML_E_INVALID, "cdml_project_qkv_rope: rope_cs must be 8-byte aligned");
  const long long last_pos = (long long)pos_offset + (seg_len > 0 ? std::min(rows, seg_len) : rows) - 1;
  if (last_pos >= n_pos)
    return fail(CDML_E_INVALID, "cdml_project_qkv_rope: position %lld outside the %d-row table",
                last_pos, n_pos);
  int rc = ensure_device();
  if (rc) return rc;
  GemmArgs g{};
  g.lda = in_dim;
  g.ldb = in_dim;
  g.ldc = out_dim;
  g.M = rows;
  g.N = out_dim;
  g.K = in_dim;
  g.nprob = 3;
  g.p[0] = {x, wq, bq, q, nullptr};
  g.p[1] = {x, wk, bk, k, nullptr};
  g.p[2] = {x, wv, bv, v, nullptr};
  g.act = CDML_ACT_NONE;
  g.rope_cs = reinterpret_cast<const float2 *>(rope_cs);
  g.rope_hd = head_dim;
  g.rope_npos = n_pos;
  g.rope_pos0 = pos_offset;
  g.rope_seg = seg_len;
  return launch_gemm(g, false, false, as_hip(stream), "cdml_project_qkv_rope");
}

extern "C" int cdml_linear(const float *x, int ldx, const float *w, const float *b, float *y,
                           int ldy, int rows, int in_dim, int out_dim, int activation,
                           cdml_stream stream) {
  if (rows < 0 || in_dim < 0 || out_dim < 0)
    return fail(CDML_E_INVALID, "cdml_linear: negative size");
  if (activation < CDML_ACT_NONE || activation > CDML_ACT_SWISH)
    return fail(CDML_E_INVALID, "cdml_linear: unknown activation %d", activation);
  if (rows == 0 || out_dim == 0) return CDML_OK;
  if (!x || !w || !y) return fail(CDML_E_INVALID, "cdml_linear: NULL pointer");
  if (ldx < in_dim || ldy < out_dim)
    return fail(CDML_E_INVALID, "cdml_linear: row stride smaller than the row");
  int rc = ensure_device();
  if (rc) return rc;
  GemmArgs g{};
  g.lda = ldx;
  g.ldb = in_dim;
  g.ldc = ldy;
  g.M = rows;
  g.N = out_dim;
  g.K = in_dim;
  g.nprob = 1;
  g.p[0] = {x, w, b, y, nullptr};
  g.act = activation;
  return launch_gemm(g, false, false, as_hip(stream), "cdml_linear");
}

namespace {

// cdml_linear_backward with the epilogue options of the input gradient:
// dx = (dY W) * act'(dz) + add (dz / add NULL: not applied; both use row
// stride lddx), or dx += dY W with accumulate_dx.
int linear_backward_impl(const float *x, int ldx, const float *dy, int lddy, const float *w,
                         const float *dz, int dact, const float *add, float *dx, int lddx,
                         float *wgrad, float *bgrad, int rows, int in_dim, int out_dim,
                         int accumulate_dx, void *workspace, size_t workspace_bytes,
                         cdml_stream stream, const char *what) {
  if (rows < 0 || in_dim < 0 || out_dim < 0) return fail(CDML_E_INVALID, "%s: negative size", what);
  if (lddy < out_dim || (dx && lddx < in_dim) || (wgrad && ldx < in_dim))
    return fail(CDML_E_INVALID, "%s: row stride smaller than the row", what);
  if (rows == 0) return CDML_OK;
  if (!dy || (dx && !w) || (wgrad && !x)) return fail(CDML_E_INVALID, "%s: NULL pointer", what);
  int rc = ensure_device();
  if (rc) return rc;
  hipStream_t st = as_hip(stream);
  if (dx && in_dim > 0) {
    // dX (+)= dY W: opA = dY [rows, out], opB = W read as [out, in]
    GemmArgs g{};
    g.lda = lddy;
    g.ldb = in_dim;
    g.ldc = lddx;
    g.M = rows;
    g.N = in_dim;
    g.K = out_dim;
    g.nprob = 1;
    g.p[0] = {dy, w, nullptr, dx, nullptr};
    g.beta = accumulate_dx ? 1 : 0;
    g.dz = dz;
    g.lddz = lddx;
    g.dact = dact;
    g.add = add;
    g.ldadd = lddx;
    rc = launch_gemm(g, false, true, st, what);
    if (rc) return rc;
  }
  if ((wgrad || bgrad) && out_dim > 0) {
    // W_grad += dY^T X: opA = dY read as [out, rows], opB = X read as
    // [rows, in]; the bias gradient rides on the staging of opA.
    GemmArgs g{};
    g.lda = lddy;
    g.ldb = ldx;
    g.ldc = in_dim;
    g.M = out_dim;
    g.N = in_dim;
    g.K = rows;
    g.nprob = 1;
    g.p[0] = {dy, x, nullptr, wgrad, bgrad};
    g.beta = 1;
    if (wgrad && in_dim > 0) {
      rc = attach_split(g, workspace, workspace_bytes, what);
      if (rc) return rc;
      rc = launch_gemm(g, true, true, st, what);
    } else if (bgrad) {
      op_rowsum_kernel<true><<<dim3((out_dim + 255) / 256, 1), dim3(256), 0, st>>>(g);
      rc = check_launch(what);
    }
    if (rc) return rc;
  }
  return CDML_OK;
}

}  // namespace

extern "C" int cdml_linear_backward(const float *x, int ldx, const float *dy, int lddy,
                                    const float *w, float *dx, int lddx, float *wgrad,
                                    float *bgrad, int rows, int in_dim, int out_dim,
                                    int accumulate_dx, void *workspace, size_t workspace_bytes,
                                    cdml_stream stream) {
  return linear_backward_impl(x, ldx, dy, lddy, w, nullptr, CDML_ACT_NONE, nullptr, dx, lddx, wgrad,
                              bgrad, rows, in_dim, out_dim, accumulate_dx, workspace, workspace_bytes,
                              stream, "cdml_linear_backward");
}

extern "C" int cdml_linear_backward_act(const float *x, int ldx, const float *dy, int lddy,
                                        const float *w, const float *dz, int activation,
                                        const float *add, float *dx, int lddx, float *wgrad,
                                        float *bgrad, int rows, int in_dim, int out_dim,
                                        void *workspace, size_t workspace_bytes,
                                        cdml_stream stream) {
  const int base = activation & ~CDML_ACT_FROM_OUTPUT;
  if (base < CDML_ACT_NONE || base > CDML_ACT_SWISH)
    return fail(CDML_E_INVALID, "cdml_linear_backward_act: unknown activation %d", activation);
  const bool from_out = (activation & CDML_ACT_FROM_OUTPUT) != 0;
  if (from_out && base != CDML_ACT_RELU && base != CDML_ACT_LEAKYRELU)
    return fail(CDML_E_INVALID, "cdml_linear_backward_act: CDML_ACT_FROM_OUTPUT needs ReLU or leaky ReLU");
  const int dact = from_out && base == CDML_ACT_RELU ? kDerivReluOut : base;
  return linear_backward_impl(x, ldx, dy, lddy, w, dz, dact, add, dx, lddx, wgrad, bgrad,
                              rows, in_dim, out_dim, 0, workspace, workspace_bytes, stream,
                              "cdml_linear_backward_act");
}

extern "C" int cdml_matmul(const float *a, int lda, const float *b, int ldb, float *c, int ldc, int m,
                           int k, int n, cdml_stream stream) {
  if (m < 0 || k < 0 || n < 0) return fail(CDML_E_INVALID, "cdml_matmul: negative size");
  if (m == 0 || n == 0) return CDML_OK;
  if (!a || !b || !c) return fail(CDML_E_INVALID, "cdml_matmul: NULL pointer");
  if (lda < k || ldb < n || ldc < n) return fail(CDML_E_INVALID, "cdml_matmul: row stride smaller than the row");
  int rc = ensure_device();
  if (rc) return rc;
  GemmArgs g{};  // k == 0: the generic kernel stores zeros
  g.lda = lda;
  g.ldb = ldb;
  g.ldc = ldc;
  g.M = m;
  g.N = n;
  g.K = k;
  g.nprob = 1;
  g.p[0] = {a, b, nullptr, c, nullptr};
  return launch_gemm(g, false, true, as_hip(stream), "cdml_matmul");
}

extern "C" int cdml_linear_preact(const float *x, int ldx, const float *w, const float *b, float *z,
                                  float *y, int ldy, int rows, int in_dim, int out_dim,
                                  int activation, cdml_stream stream) {
  if (rows < 0 || in_dim < 0 || out_dim < 0)
    return fail(CDML_E_INVALID, "cdml_linear_preact: negative size");
  if (activation < CDML_ACT_NONE || activation > CDML_ACT_SWISH)
    return fail(CDML_E_INVALID, "cdml_linear_preact: unknown activation %d", activation);
  if (!z && activation != CDML_ACT_RELU && activation != CDML_ACT_LEAKYRELU)
    return fail(CDML_E_INVALID, "cdml_linear_preact: z may be NULL only with ReLU or leaky ReLU");
  if (rows == 0 || out_dim == 0) return CDML_OK;
  if (!x || !w || !y) return fail(CDML_E_INVALID, "cdml_linear_preact: NULL pointer");
  if (ldx < in_dim || ldy < out_dim)
    return fail(CDML_E_INVALID, "cdml_linear_preact: row stride smaller than the row");
  int rc = ensure_device();
  if (rc) return rc;
  GemmArgs g{};
  g.lda = ldx;
  g.ldb = in_dim;
  g.ldc = ldy;
  g.M = rows;
  g.N = out_dim;
  g.K = in_dim;
  g.nprob = 1;
  g.p[0] = {x, w, b, y, nullptr};
  g.act = !z && activation == CDML_ACT_RELU ? kActReluMarked : activation;
  g.pre = z;
  g.ldpre = ldy;
  g.f32 = activation == CDML_ACT_RELU || activation == CDML_ACT_LEAKYRELU;
  return launch_gemm(g, false, false, as_hip(stream), "cdml_linear_preact");
}

extern "C" int cdml_backprop_qkv(const float *x, const float *dq, const float *dk, const float *dv,
                                 const float *wq, const float *wk, const float *wv, float *wq_grad,
                                 float *bq_grad, float *wk_grad, float *bk_grad, float *wv_grad,
                                 float *bv_grad, float *dx, int rows, int in_dim, int out_dim,
                                 void *workspace, size_t workspace_bytes, cdml_stream stream) {
  if (rows < 0 || in_dim < 0 || out_dim < 0)
    return fail(CDML_E_INVALID, "cdml_backprop_qkv: negative size");
  if (rows == 0) return CDML_OK;
  if (!x || !dq || !dk || !dv || !wq || !wk || !wv || !wq_grad || !bq_grad || !wk_grad ||
      !bk_grad || !wv_grad || !bv_grad || !dx)
    return fail(CDML_E_INVALID, "cdml_backprop_qkv: NULL pointer");
  int rc = ensure_device();
  if (rc) return rc;
  hipStream_t st = as_hip(stream);
  if (out_dim > 0) {
    // W*_grad += d*^T X and b*_grad += column sums of d*, three problems in
    // one launch
    GemmArgs g{};
    g.lda = out_dim;
    g.ldb = in_dim;
    g.ldc = in_dim;
    g.M = out_dim;
    g.N = in_dim;
    g.K = rows;
    g.nprob = 3;
    g.p[0] = {dq, x, nullptr, wq_grad, bq_grad};
    g.p[1] = {dk, x, nullptr, wk_grad, bk_grad};
    g.p[2] = {dv, x, nullptr, wv_grad, bv_grad};
    g.beta = 1;
    if (in_dim > 0) {
      rc = attach_split(g, workspace, workspace_bytes, "cdml_backprop_qkv");
      if (rc) return rc;
      rc = launch_gemm(g, true, true, st, "cdml_backprop_qkv (weight gradients)");
    } else {
      op_rowsum_kernel<true><<<dim3((out_dim + 255) / 256, 3), dim3(256), 0, st>>>(g);
      rc = check_launch("cdml_backprop_qkv (bias gradients)");
    }
    if (rc) return rc;
  }
  if (in_dim > 0) {
    // dX = dQ WQ + dK WK + dV WV: one product over K = 3 * out_dim when the
    // tiled kernel can stage all three operand pairs (the k-loop switches
    // source at each third), else the three products accumulated in turn
    // (out_dim == 0: dX = 0)
    const float *d[3] = {dq, dk, dv};
    const float *w[3] = {wq, wk, wv};
    bool fused = out_dim > 0 && out_dim % 16 == 0 && (long long)3 * out_dim <= INT32_MAX;
    for (int s = 0; fused && s < 3; ++s)
      fused = stage_ok(d[s], rows, out_dim, false) && stage_ok(w[s], in_dim, in_dim, true);
    if (fused) {
      GemmArgs g{};
      g.lda = out_dim;
      g.ldb = in_dim;
      g.ldc = in_dim;
      g.M = rows;
      g.N = in_dim;
      g.K = 3 * out_dim;
      g.nprob = 1;
      for (int s = 0; s < 3; ++s) g.p[s] = {d[s], w[s], nullptr, dx, nullptr};
      g.kseg = out_dim / 16;
      return launch_gemm(g, false, true, st, "cdml_backprop_qkv (input gradient)");
    }
    for (int s = 0; s < 3; ++s) {
      GemmArgs g{};
      g.lda = out_dim;
      g.ldb = in_dim;
      g.ldc = in_dim;
      g.M = rows;
      g.N = in_dim;
      g.K = out_dim;
      g.nprob = 1;
      g.p[0] = {d[s], w[s], nullptr, dx, nullptr};
      g.beta = s > 0;
      rc = launch_gemm(g, false, true, st, "cdml_backprop_qkv (input gradient)");
      if (rc) return rc;
    }
  }
  return CDML_OK;
}
