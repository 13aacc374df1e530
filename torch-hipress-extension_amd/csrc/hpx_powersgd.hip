// PowerSGD rank-r phases over a batch of row-major fp32 matrices.
//
// Semantics are the ones the reference's comments state (powersgd_body.h:20-29,
// :41-50, :64-76); its literal copy_ calls have source and destination
// swapped:
//   encode1  M.flat[:N] = grad + residual ;  P = M Q        (n x m)(m x r)
//   encode2  P <- orthonormal columns     ;  Q = M^T P      (m x n)(n x r)
//   decode   M = P Q^T ; residual = grad - M.flat[:N] ; grad = M.flat[:N]
//
// Every phase is one streaming pass over the n x m data, so all three are bound
// by HBM; the rank-r contractions ride along on the matrix cores with
// v_mfma_f32_4x4x1_16b_f32: sixteen independent 4x4 outer-product blocks per
// instruction, so four columns of a rank-4 factor fill the N dimension exactly.
// Operand layout of that instruction: A[blk][i] in lane 4*blk+i, B[blk][j] in
// lane 4*blk+j, D[blk][i][j] in lane 4*blk+j, register i.
//
// Ranks up to 16 are handled as up to four column groups of four in one pass over the data.  Larger ranks
// (the reference takes any, powersgd_body.h:28,49,69) go sixteen columns at a time: every pass names a block
// of columns of P and Q by an offset pointer, the block's width `r` and the factors' row stride `ld`; encode1
// stores M in its first pass and reads it back in the others, decode builds M up over its passes and writes the
// residual and the gradient in the last.
#include <type_traits>

#include "hpx_common.h"

namespace {
using namespace hpx;

typedef float f32x4 __attribute__((ext_vector_type(4)));

constexpr int kThreads = 256;
constexpr int kWaves = kThreads / kWave;
// Matrices per launch.  A launch that follows another waits for the last workgroup of it: ResNet-50's 54 matrices in
// two launches a phase (tables of 40) took 73 + 34 + 73 us for encode1, encode2's product and decode, in one 62 + 25 + 65.
// A smaller table is searched faster: up to 16 entries by the scalar unit, up to 64 with one load per lane.
constexpr int kSegSmall = 16, kSegMiddle = 64, kSegLarge = 160;
#define PSGD_BY_COUNT(LAUNCHES, ...)                               \
  (count <= kSegSmall    ? LAUNCHES<kSegSmall>(count, __VA_ARGS__)  \
   : count <= kSegMiddle ? LAUNCHES<kSegMiddle>(count, __VA_ARGS__) \
                         : LAUNCHES<kSegLarge>(count, __VA_ARGS__))
constexpr int kMaxCG = 4;                 // column groups of 4 -> rank <= 16
// Decode is three write streams against one read stream; with 8 rows per wave instead of 32 the
// stores of a workgroup stay close together in time and address and the pass runs 10 % faster.
constexpr int64_t kDecTiles = 256;        // fewer than this many tiles are halved
constexpr int kDecRowsPerBlock = 32;      // rows of a decode tile 256 columns wide (narrower tiles are as much taller)

// encode2 and decode cut a matrix into strips of 4 * lanes columns; a wave lays kWave / lanes row groups of a strip
// side by side.  256 columns unless the lanes past the last column would be more than a quarter of those before it, then
// 128, then 64.  30 ragged matrices of up to 1500 x 1001: 163 us a pass at a quarter, 170 at an eighth, 181 at a
// sixteenth: narrow strips touch more lines per byte; wide ones leave lanes idle.
inline int strip_lanes(int m) {
  for (int lanes = kWave; lanes > 16; lanes /= 2) {
    const int64_t w = 4 * lanes;
    if ((m + w - 1) / w * w - m <= m / 4) return lanes;
  }
  return 16;
}

struct Seg {
  const float* grad;   // encode1: in.  decode: in/out (as float*)
  const float* res;    // encode1: in.  decode: out
  const float* Q;
  float* M;
  float* P;
  float* Qout;         // encode2: Q to write;  partials live in the workspace
  int64_t numel;
  int32_t n, m, r;
  int32_t part_off;    // encode2: offset (in floats / 4) of this matrix's partials
  int32_t ld;          // row stride of P and Q (the full rank; r is the width of the block of columns at hand)
  int32_t mode;        // kFromM | kOntoM | kKeepGrad, for the passes of a rank above 16
  int32_t split;       // encode1: waves that share four rows.  encode2: q_lanes.  decode: strip_lanes
  int32_t rows;        // encode2: rows folded into one partial of Q (of a strip 256 columns wide)
};
constexpr int32_t kFromM = 1;    // encode1: M has been stored by an earlier pass: read it instead of grad + residual
constexpr int32_t kOntoM = 2;    // decode: add this block's P Q^T to what M holds instead of starting from zero
constexpr int32_t kKeepGrad = 4; // decode: more blocks follow: write M only, leave residual and gradient alone
template <int CAP>
struct Args {
  int32_t nseg;
  int32_t rows;        // decode: rows of a tile (of a strip 256 columns wide)
  int32_t keep;        // encode1: a Keep
  int32_t tile_start[CAP + 1];
  Seg seg[CAP];
  float* partials;
};
static_assert(sizeof(Args<kSegLarge>) <= 18000, "kernel-argument budget");

// What a pass keeps in the 256 MB Infinity Cache from one phase to the next, by the bytes of M in the call.  Streaming
// accesses leave nothing there, plain ones do.  encode1 reads the gradient, which decode reads again, and writes M, which
// encode2 reads and decode writes; decode's three outputs are streamed, array after array.  us of a pass (encode1, encode2
// and decode of matrices of 4096 columns, three sets of buffers in turn) with encode1 streaming everything / keeping the
// gradient and M / keeping the gradient: 8 MB 36.9 / 38.0 / 38.6, 17 MB 49.1 / 48.4 / 52.5, 34 MB 82.4 / 76.7 / 79.5, 67 MB
// 123 / 112 / 117, 117 MB 191 / 177 / 182, 168 MB 263 / 251 / 251, 201 MB 306 / 294 / 291, 235 MB 351 / 339 / 335; ResNet-50's
// 94 MB 168 / 151 / 153, the layer set's 1208 MB 1562 / 1581 / 1556.
constexpr int64_t kKeepFrom = 10 << 20;        // below, everything stays in the caches anyway
constexpr int64_t kKeepBothTo = 192 << 20;     // gradient and M together 384 MB: the first third of each is lost
enum Keep : int32_t { kKeepNone, kKeepGradM, kKeepGradOnly };
inline Keep keep_rule(int64_t m_bytes) { return m_bytes < kKeepFrom ? kKeepNone : m_bytes < kKeepBothTo ? kKeepGradM : kKeepGradOnly; }
template <bool STREAM>
__device__ __forceinline__ float4 ld4_as(const float* p) { return STREAM ? ld4_stream(p) : ld4(p); }
template <bool STREAM>
__device__ __forceinline__ void st4_as(float* p, float4 v) {
  if (STREAM) st4_stream(p, v); else st4(p, v);
}
// Whether rows of m elements from these addresses on all start on a cache line.  Where they do not, the pieces of a row that
// successive instructions move share lines: streaming accesses, which keep nothing in the caches, then fetch and write such a
// line twice, and plain ones are the faster.  encode1 / decode of 1200 x 601 matrices 30.8 / 36.1 us streaming, 26.4 / 29.9
// plain, of 2049 columns 25.4 / 28.1 and 20.4 / 23.0.
__device__ __forceinline__ bool rows_on_lines(int m, const void* a, const void* b, const void* c) {
  return ((uintptr_t(a) | uintptr_t(b) | uintptr_t(c) | uintptr_t(uint32_t(m)) * 4) & 127) == 0;
}

__device__ __forceinline__ f32x4 mfma4(float a, float b, f32x4 c) {
  return __builtin_amdgcn_mfma_f32_4x4x1f32(a, b, c, 0, 0, 0);
}

// ---- encode1: M = G + R (flat prefix), P = M Q -------------------------------
// Lane 4b+i of a wave owns row i of four and the 4 columns k0+4b..k0+4b+3 of each 64-column step, which is one
// 128-bit load of G and of R and one store of M.  Bound by HBM (12 bytes an element).  A workgroup takes four rows
// with all its waves where rows are long; of shorter rows it takes eight or sixteen, two or one wave to four rows
// (split_rows below): otherwise the waves past the end of the row idle and a workgroup is gone before the next
// has started.
template <int CG, int CAP>
__global__ __launch_bounds__(kThreads) void psgd_encode1_kernel(const Args<CAP> a) {
  const int tile = blockIdx.x;
  const int s = find_segment<CAP>(a.tile_start, a.nseg, tile);
  const Seg& sg = a.seg[s];
  const float* __restrict__ G = sg.grad;
  const float* __restrict__ R = sg.res;
  const float* __restrict__ Q = sg.Q;
  float* __restrict__ M = sg.M;
  const int n = sg.n, m = sg.m, r = sg.r, ld = sg.ld;
  const bool from_m = (sg.mode & kFromM) != 0;
  const int64_t N = sg.numel;
  const int lane = threadIdx.x & (kWave - 1), wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
  const int split = sg.split, groups = kWaves / split;
  const int part = wave % split;  // of the waves that share four rows
  const int64_t tile_row = int64_t(tile - a.tile_start[s]) * 4 * groups;
  const int64_t row0 = tile_row + wave / split * 4;
  const int i = lane & 3, b = lane >> 2;
  const int64_t row = row0 + i;
  // Columns: the waves walk the rows in chunks of split * 256 columns, wave w taking the w-th 256 of each
  // chunk, so that at any time they read neighbouring pieces of the same four rows (a contiguous
  // quarter of the row per wave ran 9 % slower); what is left past the last whole 256 goes round the waves in
  // 64-column steps.
  constexpr int kUnroll = 4;
  constexpr int kChunk = 64 * kUnroll;
  const int mfull = m / kChunk * kChunk;

  f32x4 acc[CG];
#pragma unroll
  for (int c = 0; c < CG; c++) acc[c] = f32x4{0.f, 0.f, 0.f, 0.f};

  const bool rows_full = (row0 + 3 < n) && ((row0 + 4) * m <= N);
  const float* __restrict__ A = from_m ? M : G;
  const int64_t lane_at = row * m + 4 * b;
  struct Chunk { float4 g[kUnroll], r[kUnroll]; float q[kUnroll][4][CG]; };
  auto chunks = [&](auto stream_g, auto stream_r, auto stream_m) {
    constexpr bool G_STREAM = decltype(stream_g)::value, R_STREAM = decltype(stream_r)::value, M_STREAM = decltype(stream_m)::value;
    // kUnroll 64-column steps at a time, every load issued before the first use
    auto load = [&](Chunk& h, int k0) {
#pragma unroll
      for (int u = 0; u < kUnroll; u++) {
        h.g[u] = ld4_as<G_STREAM>(A + lane_at + k0 + 64 * u);
        h.r[u] = from_m ? make_float4(0.f, 0.f, 0.f, 0.f) : ld4_as<R_STREAM>(R + lane_at + k0 + 64 * u);
      }
#pragma unroll
      for (int u = 0; u < kUnroll; u++)
#pragma unroll
        for (int t = 0; t < 4; t++)
#pragma unroll
          for (int c = 0; c < CG; c++) {
            const int col = c * 4 + i;  // B operand: lane 4b+j holds Q[k][j]
            h.q[u][t][c] = col < r ? Q[int64_t(k0 + 64 * u + 4 * b + t) * ld + col] : 0.f;
          }
    };
    // Of each half of a chunk, added to the rest afterwards: shorter chains of fp32 sums.  (P's distance from the exact
    // product 1.00e-7 of its norm for 4096 x 4096, 9.1e-8 for 200 x 600; in one chain 1.09e-7 and 1.11e-7; time alike.)
    auto use = [&](const Chunk& h, int k0) {
      f32x4 sum[2][CG];
#pragma unroll
      for (int c = 0; c < CG; c++) sum[0][c] = sum[1][c] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int u = 0; u < kUnroll; u++) {
        const float4 m4 = make_float4(h.g[u].x + h.r[u].x, h.g[u].y + h.r[u].y, h.g[u].z + h.r[u].z, h.g[u].w + h.r[u].w);
        if (!from_m) st4_as<M_STREAM>(M + lane_at + k0 + 64 * u, m4);
        const float v[4] = {m4.x, m4.y, m4.z, m4.w};
#pragma unroll
        for (int t = 0; t < 4; t++)
#pragma unroll
          for (int c = 0; c < CG; c++) sum[u & 1][c] = mfma4(v[t], h.q[u][t][c], sum[u & 1][c]);
      }
#pragma unroll
      for (int c = 0; c < CG; c++) acc[c] += sum[0][c] + sum[1][c];
    };
    // Two chunks in turn, the next one's loads under way while one is used: 2048 x 1024 alone 37.7 us for all three phases
    // (one chunk after the other 38.8), the layer set 1563 (1572).
    const int step = split * kChunk;
    int k0 = part * kChunk;
    if (k0 >= mfull) return;
    Chunk x, y;
    if constexpr (CG > 1) {  // (their Q takes the registers: rank 8 with two chunks in turn 36 matrices 566, so 560)
#pragma unroll 1
      for (; k0 < mfull; k0 += step) {
        load(x, k0);
        use(x, k0);
      }
      return;
    }
    load(x, k0);
#pragma unroll 1
    for (;;) {
      const int k1 = k0 + step;
      if (k1 < mfull) load(y, k1);
      use(x, k0);
      if (k1 >= mfull) return;
      k0 = k1 + step;
      if (k0 < mfull) load(x, k0);
      use(y, k1);
      if (k0 >= mfull) return;
    }
  };
  if (rows_full) {  // (a loop for each choice: of one loop with a choice at each access the compiler makes plain ones)
    constexpr auto kPlain = std::false_type{};
    constexpr auto kStream = std::true_type{};
    if (!rows_on_lines(m, G, R, M)) chunks(kPlain, kPlain, kPlain);
    else if (a.keep == kKeepNone) chunks(kStream, kStream, kStream);
    else if (a.keep == kKeepGradM) chunks(kPlain, kStream, kPlain);
    else chunks(kPlain, kStream, kStream);
  }
  // What is left of the columns (or everything, of rows that are not full), two steps' loads in flight together where the
  // wave has several (four: as fast, but the registers they take slow the loop above): one step after the other, each
  // waits for memory (encode1 of 1200 x 147 matrices 44 us, now 33).
  const int rest = (rows_full ? mfull : 0) + part * 64;
  auto steps = [&](auto unroll) {
    constexpr int kSteps = decltype(unroll)::value;
    for (int k0 = rest; k0 < m; k0 += split * 64 * kSteps) {
      float4 g4[kSteps], r4[kSteps];
      float q[kSteps][4][CG];
      bool whole[kSteps];
#pragma unroll
      for (int u = 0; u < kSteps; u++) {
        const int64_t kk = int64_t(k0) + u * split * 64 + 4 * b, f0 = row * m + kk;
        whole[u] = row < n && kk + 4 <= m && f0 + 4 <= N;
        if (whole[u]) {
          g4[u] = from_m ? ld4(M + f0) : ld4(G + f0);
          r4[u] = from_m ? make_float4(0.f, 0.f, 0.f, 0.f) : ld4(R + f0);
        }
#pragma unroll
        for (int t = 0; t < 4; t++)
#pragma unroll
          for (int c = 0; c < CG; c++) {
            const int col = c * 4 + i;  // B operand: lane 4b+j holds Q[k][j]
            q[u][t][c] = (kk + t < m && col < r) ? Q[(kk + t) * ld + col] : 0.f;
          }
      }
#pragma unroll
      for (int u = 0; u < kSteps; u++) {
        const int64_t kk = int64_t(k0) + u * split * 64 + 4 * b, f0 = row * m + kk;
        float v[4];
        f32x4 sum[CG];
#pragma unroll
        for (int c = 0; c < CG; c++) sum[c] = f32x4{0.f, 0.f, 0.f, 0.f};
        if (whole[u]) {
          const float4 m4 = make_float4(g4[u].x + r4[u].x, g4[u].y + r4[u].y, g4[u].z + r4[u].z, g4[u].w + r4[u].w);
          if (!from_m) st4(M + f0, m4);
          v[0] = m4.x; v[1] = m4.y; v[2] = m4.z; v[3] = m4.w;
        } else {
#pragma unroll
          for (int t = 0; t < 4; t++) {
            const int64_t f = f0 + t;
            float x = 0.f;
            if (row < n && kk + t < m) {
              if (f < N && !from_m) {
                x = G[f] + R[f];
                M[f] = x;
              } else {
                x = M[f];  // beyond the gradient: whatever the caller left in M takes part in P = M Q
              }
            }
            v[t] = x;
          }
        }
#pragma unroll
        for (int t = 0; t < 4; t++)
#pragma unroll
          for (int c = 0; c < CG; c++) sum[c] = mfma4(v[t], q[u][t][c], sum[c]);
#pragma unroll
        for (int c = 0; c < CG; c++) acc[c] += sum[c];
      }
    }
  };
  if (rest + split * 64 >= m) steps(std::integral_constant<int, 1>{}); else steps(std::integral_constant<int, 2>{});
  // acc[c][ii] in lane 4b+j is the part of P[row0+ii][4c+j] from this lane's columns: fold the 16 blocks
  __shared__ float s_p[kWaves][CG][4][4];
#pragma unroll
  for (int c = 0; c < CG; c++)
#pragma unroll
    for (int ii = 0; ii < 4; ii++) {
      float x = acc[c][ii];
#pragma unroll
      for (int o = 4; o < kWave; o <<= 1) x += __shfl_xor(x, o, kWave);
      if (lane < 4) s_p[wave][c][ii][lane] = x;
    }
  __syncthreads();
  if (threadIdx.x < groups * CG * 16) {
    const int grp = threadIdx.x / (CG * 16), e = threadIdx.x % (CG * 16);
    const int c = e / 16, ii = (e / 4) & 3, j = e & 3;
    const int64_t prow = tile_row + grp * 4 + ii;
    const int col = c * 4 + j;
    if (prow < n && col < r) {
      float x = s_p[grp * split][c][ii][j];
      for (int w = 1; w < split; w++) x += s_p[grp * split + w][c][ii][j];
      sg.P[prow * ld + col] = x;
    }
  }
}

// ---- encode2, step 1: orthonormalise the columns of P -------------------------
// One workgroup per matrix.  The factor is small (64 KB at 4096 x 4) and the launch is a chain of workgroup-wide
// reductions, so what counts is how many there are: up to kGramCols columns need ONE, of all products of two columns
// at once (gram_orth below); modified Gram-Schmidt, r + r(r-1)/2 reductions a sweep and two sweeps, is for wider
// factors and for columns that nearly depend on each other.
constexpr int kOrthThreads = 1024;
constexpr int kOrthWaves = kOrthThreads / kWave;
constexpr int kGramCols = 8;

__device__ __forceinline__ double block_sum(double v, double* s_red) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, kWave);
  const int w = threadIdx.x / kWave;
  __syncthreads();
  if ((threadIdx.x & (kWave - 1)) == 0) s_red[w] = v;
  __syncthreads();
  double t = 0;
#pragma unroll
  for (int k = 0; k < kOrthThreads / kWave; k++) t += s_red[k];
  return t;
}

// P[row][c] of the matrix being orthonormalised: either the caller's row-major
// array in global memory or a column-major copy in LDS (conflict-free for the
// row-strided sweeps below).
template <bool LDS>
struct PView {
  float* p;
  int n, r;
  __device__ __forceinline__ float& at(int row, int c) const { return LDS ? p[c * n + row] : p[int64_t(row) * r + c]; }
};

template <bool LDS>
__device__ __forceinline__ void gram_schmidt(const PView<LDS> P, double* s_red) {
  const int n = P.n, r = P.r;
  for (int sweep = 0; sweep < 2; sweep++) {
    for (int c = 0; c < r; c++) {
      double ss = 0;
      for (int row = threadIdx.x; row < n; row += kOrthThreads) {
        const double x = P.at(row, c);
        ss += x * x;
      }
      ss = block_sum(ss, s_red);
      const float inv = ss > 0 ? static_cast<float>(1.0 / sqrt(ss)) : 0.f;
      for (int row = threadIdx.x; row < n; row += kOrthThreads) P.at(row, c) *= inv;
      for (int c2 = c + 1; c2 < r; c2++) {
        double d = 0;
        for (int row = threadIdx.x; row < n; row += kOrthThreads) d += double(P.at(row, c)) * double(P.at(row, c2));
        d = block_sum(d, s_red);
        const float df = static_cast<float>(d);
        for (int row = threadIdx.x; row < n; row += kOrthThreads) P.at(row, c2) -= df * P.at(row, c);
      }
    }
  }
}

// Row `row` of a factor of r columns, r <= C; zeros behind them and for rows past the end.
template <int C>
__device__ __forceinline__ void load_row(float (&x)[C], const float* P, int64_t row, int n, int r) {
  if (r == C) {
#pragma unroll
    for (int c = 0; c < C; c += 4) {
      const float4 v = row < n ? ld4(P + row * C + c) : make_float4(0.f, 0.f, 0.f, 0.f);
      x[c] = v.x; x[c + 1] = v.y; x[c + 2] = v.z; x[c + 3] = v.w;
    }
  } else {
#pragma unroll
    for (int c = 0; c < C; c++) x[c] = c < r && row < n ? P[row * r + c] : 0.f;
  }
}
template <int C>
__device__ __forceinline__ void store_row(const float (&y)[C], float* P, int64_t row, int n, int r) {
  if (row >= n) return;
  if (r == C) {
#pragma unroll
    for (int c = 0; c < C; c += 4) st4(P + row * C + c, make_float4(y[c], y[c + 1], y[c + 2], y[c + 3]));
  } else {
#pragma unroll
    for (int c = 0; c < C; c++)
      if (c < r) P[row * r + c] = y[c];
  }
}

// Orthonormalises the columns by way of their Gram matrix: G = P^T P in fp64 (the products of fp32 values are exact
// there), G = R^T R, P <- P R^-1 in fp64 with one rounding to fp32 at the end: one pass over P for the sums and one for
// the result.  What the sums, the elimination and the product round away is at most k 2^-53 sqrt(G_ii G_jj) in the entries
// of G and comes out multiplied by R^-1 from both sides: with s_c = sum over l of |R^-1_lc| sqrt(G_ll) the columns are
// orthonormal to k 2^-53 s_c^2, k the length of the longest chain of sums (the n / 256 rows of one accumulator, the fold over
// accumulators, blocks and waves, the elimination: 36 for all but the first).  s_c is about 1 for columns that have little to do with each other
// and grows with the product of what the columns before lose to each other, not only with each one's own loss: a chain
// c_1 = u_1, c_k+1 = u_k + 0.05 u_k+1 of eight columns keeps every R_cc^2 above 2^-10 G_cc, and its P R^-1 is no
// orthonormal matrix at all.  Where k s_c^2 exceeds 2^27 (2^-26 in the products of columns, a quarter of fp32's own rounding), or is no number,
// nothing is written and the answer is false.  A column of zeros stays zero.
// The sums ride on v_mfma_f64_4x4x4_4b_f64, four blocks of 4 x 4 products summed over four rows each: A[blk][i][k] and
// B[blk][k][i] are lane 16k + 4blk + i alike, so one register of sixteen rows by four columns is both operands, and D[blk][i][j]
// (lane 16i + 4blk + j) is left to be added up over the blocks alone.  (As fp64 products in every lane the sums had to be
// folded over 64 lanes, ten or 36 of them: for eight columns that was most of the launch.)
// Up to four columns are loaded a row to a lane and turned round within four lanes: with an element to a lane, as of more
// columns, a wave made four times as many requests.  What a thread has loaded it still holds when the result is worked out, its
// rows being the same, in factors of up to 4096 rows.
// us of the launch, folded over the lanes / an element to a lane / so: 36 factors of 2048 x 8 23.5 / 8.3, one of 30000 x 8 164 / 61;
// the 36 of the layer set (4 columns) 10.5 / 13.1 / 5.6, 36 of 8192 x 4 18.3 / 23.6 / 9.4, of 8192 x 2 11.3 / 23.5 / 9.9, of 4096 x 3
// 9.2 / 14.2 / 6.0, one of 30000 x 4 47 / 56 / 24; 512 x 512 of rank 4, all three phases, 27.7 / 26.2 / 25.3.
__device__ __forceinline__ float quad_xor(float x, int one_or_two) {   // of the lane across, within four
  return __int_as_float(one_or_two == 1 ? __builtin_amdgcn_update_dpp(0, __float_as_int(x), 0xB1, 0xF, 0xF, false)
                                        : __builtin_amdgcn_update_dpp(0, __float_as_int(x), 0x4E, 0xF, 0xF, false));
}
// Four rows, one to a lane of each four, to four registers of one row each with a column to a lane.
__device__ __forceinline__ float4 quad_transpose(float4 v, int lane) {
  const bool odd = lane & 1, high = lane & 2;
  const float a = quad_xor(odd ? v.x : v.y, 1), b = quad_xor(odd ? v.z : v.w, 1);
  const float x = odd ? a : v.x, y = odd ? v.y : a, z = odd ? b : v.z, w = odd ? v.w : b;
  const float c = quad_xor(high ? x : z, 2), d = quad_xor(high ? y : w, 2);
  return make_float4(high ? c : x, high ? d : y, high ? z : c, high ? w : d);
}
template <int C>
__device__ __forceinline__ bool gram_orth(float* __restrict__ P, int n, int r) {
  constexpr int H = C / 4, kBlocks = H * (H + 1) / 2;   // 4 x 4 blocks of the Gram matrix: (0, 0), and (0, 1), (1, 1)
  constexpr int kPairs = C * (C + 1) / 2;
  static_assert(C % 4 == 0 && C <= kGramCols, "columns in fours");
  __shared__ double s_part[kOrthWaves][kBlocks][16];
  __shared__ double s_gram[C][C];
  __shared__ double s_T[C][C];
  __shared__ double s_norm[C];
  const int lane = threadIdx.x & (kWave - 1), wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
  constexpr int kAcc = 4;              // independent sums
  constexpr int kGroups = 16 / H;      // of sixteen rows, loaded together; the groups go round the waves
  double acc[kBlocks][kAcc];
#pragma unroll
  for (int k = 0; k < kBlocks; k++)
#pragma unroll
    for (int u = 0; u < kAcc; u++) acc[k][u] = 0;
  const int col = lane & 3;
  constexpr int kRows = 16 / C;  // loaded together, a row to a lane
  float own[kRows][C];           // up to four columns: the thread's rows, all of them where held
  bool held = false;
  if constexpr (C == 4) {
    held = n <= kRows * kOrthThreads;
    auto sums = [&](auto columns) {
      constexpr int R = decltype(columns)::value;
      for (int64_t row0 = int64_t(wave) * kWave; row0 < n; row0 += kRows * kOrthThreads) {
#pragma unroll
        for (int u = 0; u < kRows; u++) {
          const int64_t row = row0 + u * kOrthThreads + lane;
          const float* at = P + (row < n ? row : n - 1) * R;   // (no branch between the loads)
          if constexpr (R == C) {
            const float4 v = ld4(at);
            own[u][0] = v.x; own[u][1] = v.y; own[u][2] = v.z; own[u][3] = v.w;
          } else {
#pragma unroll
            for (int c = 0; c < C; c++) own[u][c] = c < R ? at[c] : 0.f;
          }
        }
#pragma unroll
        for (int u = 0; u < kRows; u++) {
#pragma unroll
          for (int c = 0; c < R; c++) own[u][c] = row0 + u * kOrthThreads + lane < n ? own[u][c] : 0.f;
          const float4 t = quad_transpose(make_float4(own[u][0], own[u][1], own[u][2], own[u][3]), lane);
          acc[0][0] = __builtin_amdgcn_mfma_f64_4x4x4f64(t.x, t.x, acc[0][0], 0, 0, 0);
          acc[0][1] = __builtin_amdgcn_mfma_f64_4x4x4f64(t.y, t.y, acc[0][1], 0, 0, 0);
          acc[0][2] = __builtin_amdgcn_mfma_f64_4x4x4f64(t.z, t.z, acc[0][2], 0, 0, 0);
          acc[0][3] = __builtin_amdgcn_mfma_f64_4x4x4f64(t.w, t.w, acc[0][3], 0, 0, 0);
        }
      }
    };
    if (r == 4) sums(std::integral_constant<int, 4>{});
    else if (r == 3) sums(std::integral_constant<int, 3>{});
    else if (r == 2) sums(std::integral_constant<int, 2>{});
    else sums(std::integral_constant<int, 1>{});
  } else for (int64_t row0 = int64_t(wave) * 16; row0 < n; row0 += kGroups * kOrthWaves * 16) {
    float x[kGroups][H];
#pragma unroll
    for (int u = 0; u < kGroups; u++) {
      const int64_t row = row0 + u * (kOrthWaves * 16) + lane / 4;
      const float* at = P + (row < n ? row : n - 1) * r;   // (no branch between the loads)
#pragma unroll
      for (int h = 0; h < H; h++) x[u][h] = at[4 * h + col < r ? 4 * h + col : 0];
    }
#pragma unroll
    for (int u = 0; u < kGroups; u++)
#pragma unroll
      for (int h = 0; h < H; h++)
        x[u][h] = row0 + u * (kOrthWaves * 16) + lane / 4 < n && 4 * h + col < r ? x[u][h] : 0.f;
#pragma unroll
    for (int u = 0; u < kGroups; u++) {
      if (row0 + u * (kOrthWaves * 16) >= n) break;   // wave-uniform
      acc[0][u % kAcc] = __builtin_amdgcn_mfma_f64_4x4x4f64(x[u][0], x[u][0], acc[0][u % kAcc], 0, 0, 0);
      if constexpr (H == 2) {
        acc[1][u % kAcc] = __builtin_amdgcn_mfma_f64_4x4x4f64(x[u][0], x[u][1], acc[1][u % kAcc], 0, 0, 0);
        acc[2][u % kAcc] = __builtin_amdgcn_mfma_f64_4x4x4f64(x[u][1], x[u][1], acc[2][u % kAcc], 0, 0, 0);
      }
    }
  }
#pragma unroll
  for (int k = 0; k < kBlocks; k++) {
    double x = (acc[k][0] + acc[k][1]) + (acc[k][2] + acc[k][3]);
    x += __shfl_xor(x, 4, kWave);
    x += __shfl_xor(x, 8, kWave);
    if ((lane & 12) == 0) s_part[wave][k][lane / 16 * 4 + col] = x;   // [i][j]
  }
  __syncthreads();
  if (threadIdx.x < kBlocks * 16) {
    const int k = threadIdx.x / 16, i = threadIdx.x / 4 % 4, j = threadIdx.x % 4;
    double x[kOrthWaves];
#pragma unroll
    for (int w = 0; w < kOrthWaves; w++) x[w] = s_part[w][k][threadIdx.x % 16];
#pragma unroll
    for (int o = kOrthWaves / 2; o > 0; o /= 2)
#pragma unroll
      for (int w = 0; w < o; w++) x[w] += x[w + o];
    const int gi = i + (k == 2 ? 4 : 0), gj = j + (k != 0 ? 4 : 0);
    s_gram[gi][gj] = x[0];
    s_gram[gj][gi] = x[0];
  }
  __syncthreads();
  // Cholesky's factor of G and the inverse of it by elimination on [G | I], lane j of the first wave with column j of both
  // halves.  Row k of the left half ends as R's, column l of the right half as R^-1's row l.
  if (wave == 0) {
    const int own = lane < C ? lane : C - 1;
    double A[C], Y[C];
#pragma unroll
    for (int k = 0; k < C; k++) {
      A[k] = s_gram[k][own];
      Y[k] = k == own ? 1.0 : 0.0;
    }
#pragma unroll
    for (int k = 0; k < C; k++) {
      const double d = __shfl(A[k], k, kWave);
      const double inv = s_gram[k][k] != 0 ? rsqrt(d) : 0;  // of what is not above zero: no number, or infinite
      A[k] *= inv;
      Y[k] *= inv;
#pragma unroll
      for (int i = k + 1; i < C; i++) {
        const double f = __shfl(A[k], i, kWave);
        A[i] = fma(-f, A[k], A[i]);
        Y[i] = fma(-f, Y[k], Y[i]);
      }
    }
    if (lane < C) {
#pragma unroll
      for (int k = 0; k < C; k++) s_T[lane][k] = Y[k];
      s_norm[lane] = sqrt(s_gram[lane][lane]);
    }
  }
  __syncthreads();
  double T[kPairs];
  bool ok = true;
  const double limit = 0x1p27 / (36 + (n - 1) / 256 + 1);
#pragma unroll
  for (int c = 0; c < C; c++) {
    double s = 0;
#pragma unroll
    for (int l = 0; l <= c; l++) {
      T[c * (c + 1) / 2 + l] = s_T[l][c];
      s = fma(fabs(T[c * (c + 1) / 2 + l]), s_norm[l], s);
    }
    ok = ok && s * s <= limit;
  }
  if (!ok) return false;  // the same in every thread
  for (int64_t row0 = threadIdx.x; row0 < n; row0 += kRows * kOrthThreads) {
    float x[kRows][C];
#pragma unroll
    for (int u = 0; u < kRows; u++) {
      if (held) {
#pragma unroll
        for (int c = 0; c < C; c++) x[u][c] = own[u][c];
      } else {
        load_row<C>(x[u], P, row0 + u * kOrthThreads, n, r);
      }
    }
#pragma unroll
    for (int u = 0; u < kRows; u++) {
      float out[C];
#pragma unroll
      for (int c = 0; c < C; c++) {
        double y = 0;
#pragma unroll
        for (int l = 0; l <= c; l++) y = fma(double(x[u][l]), T[c * (c + 1) / 2 + l], y);
        out[c] = float(y);
      }
      store_row<C>(out, P, row0 + u * kOrthThreads, n, r);
    }
  }
  return true;
}

// WIDE: the call has factors of more than four columns that gram_orth takes.  LDS: every factor of the call (at most
// kOrthLdsFloats values) fits dynamic shared memory, where Gram-Schmidt then works.
constexpr int kOrthLdsFloats = 36 * 1024;  // 144 KiB of the 160 KiB LDS
template <bool WIDE, bool LDS, int CAP>
__global__ __launch_bounds__(kOrthThreads) void psgd_orth_kernel(const Args<CAP> a) {
  __shared__ double s_red[kOrthWaves];
  extern __shared__ float s_p[];
  const Seg& sg = a.seg[blockIdx.x];
  float* __restrict__ Pg = sg.P;
  const int n = sg.n, r = sg.r;
  if (r <= 4) {
    if (gram_orth<4>(Pg, n, r)) return;
  } else if (WIDE && r <= kGramCols) {
    if (gram_orth<kGramCols>(Pg, n, r)) return;
  }
  if constexpr (LDS) {
    for (int e = threadIdx.x; e < n * r; e += kOrthThreads) s_p[(e % r) * n + e / r] = Pg[e];
    __syncthreads();
    gram_schmidt(PView<true>{s_p, n, r}, s_red);
    __syncthreads();
    for (int e = threadIdx.x; e < n * r; e += kOrthThreads) Pg[e] = s_p[(e % r) * n + e / r];
  } else {
    gram_schmidt(PView<false>{Pg, n, r}, s_red);
  }
}

// ---- encode2, step 2: Q = M^T P ------------------------------------------------
// A workgroup takes a strip of columns (256, or 128 or 64 with two or four rows side by side in a wave: q_lanes)
// and sg.rows rows of it (two or four times that), in blocks of 32 rows (64, 128) that the workgroups of a strip take in
// turn: what is being read at any time is one stretch of the matrix, not a place every sg.rows rows (the layer set 210 us
// with each workgroup's rows in one piece, 188 so).  The rows of a block go round the waves.  Per row a
// lane loads its 4 columns of M with one 128-bit load; register t of that load
// is the A operand of MFMA t, whose block b / row-of-block i' is column
// k0 + 16b + 4i' + t; the B operand is P[row][j] in every block.  The waves (and the rows side by side) meet
// in LDS and the workgroup writes one partial of Q; a second kernel adds the
// partials in a fixed order.  (Ranks up to four are held to the registers of four waves per SIMD: ResNet-50's matrices 149.7 us
// for all three phases, 151.4 with three.)
template <int CG, int CAP>
__global__ __launch_bounds__(kThreads, CG == 1 ? 4 : 1) void psgd_mtp_kernel(const Args<CAP> a) {
  const int tile = blockIdx.x;
  const int s = find_segment<CAP>(a.tile_start, a.nseg, tile);
  const Seg& sg = a.seg[s];
  const float* __restrict__ M = sg.M;
  const float* __restrict__ P = sg.P;
  const int n = sg.n, m = sg.m, r = sg.r, ld = sg.ld;
  const int lanes = sg.split, side = kWave / lanes, width = 4 * lanes;
  const int strips = (m + width - 1) / width;
  const int t_in = tile - a.tile_start[s];
  const int strip = t_in % strips, rblk = t_in / strips;
  const int lane = threadIdx.x & (kWave - 1), wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
  const int k0 = strip * width;
  const int kk = k0 + 4 * (lane & (lanes - 1));
  const int step = kWaves * side;  // rows of the workgroup per round
  const int64_t per = int64_t(sg.rows) * side, parts = (n + per - 1) / per;

  f32x4 acc[CG][4];
#pragma unroll
  for (int c = 0; c < CG; c++)
#pragma unroll
    for (int t = 0; t < 4; t++) acc[c][t] = f32x4{0.f, 0.f, 0.f, 0.f};

  const int j = lane & 3;
  const int mine = lane / lanes;  // which of the rows side by side
  constexpr int kRows = 8;
  // K rounds' rows, summed on their own in two chains and added to what there is
  auto add_up = [&](const auto& m4, const auto& p) {
    constexpr int K = sizeof(m4) / sizeof(m4[0]);
#pragma unroll
    for (int c = 0; c < CG; c++) {
      f32x4 sum[2][4];
#pragma unroll
      for (int t = 0; t < 4; t++) sum[0][t] = sum[1][t] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int u = 0; u < K; u++) {
        const float v[4] = {m4[u].x, m4[u].y, m4[u].z, m4[u].w};
#pragma unroll
        for (int t = 0; t < 4; t++) sum[u & 1][t] = mfma4(v[t], p[u][c], sum[u & 1][t]);
      }
#pragma unroll
      for (int t = 0; t < 4; t++) acc[c][t] += sum[0][t] + sum[1][t];
    }
  };
  const int64_t block = kRows * step;
  int64_t row0 = rblk * block + wave * side;  // the first of the wave's rows in a round
  // Rounds `from` ... `from` + K - 1 of the rows from row0 on; every load is issued before the first use, and only the lane that
  // holds the row's end and those past it take the element-wise way.  WHOLE: all of these rows are the matrix's.
  auto load = [&](auto whole, int64_t row0, int from, auto& m4, auto& p) {
    constexpr bool WHOLE = decltype(whole)::value;
    constexpr int K = sizeof(m4) / sizeof(m4[0]);
    auto row_of = [&](int u) {
      const int64_t row = row0 + (from + u) * step + mine;
      return WHOLE || row < n ? row : int64_t(n) - 1;
    };
    if (kk + 4 <= m) {
#pragma unroll
      for (int u = 0; u < K; u++) m4[u] = ld4_stream(M + row_of(u) * m + kk);
    } else {
#pragma unroll
      for (int u = 0; u < K; u++) {
        const float* q = M + row_of(u) * m + kk;
        m4[u] = make_float4(kk < m ? q[0] : 0.f, kk + 1 < m ? q[1] : 0.f, kk + 2 < m ? q[2] : 0.f, 0.f);
      }
    }
#pragma unroll
    for (int u = 0; u < K; u++)
#pragma unroll
      for (int c = 0; c < CG; c++) p[u][c] = (c * 4 + j) < r ? P[row_of(u) * ld + c * 4 + j] : 0.f;
  };
  auto clear_past = [&](int64_t row0, int from, auto& m4) {
    constexpr int K = sizeof(m4) / sizeof(m4[0]);
#pragma unroll
    for (int u = 0; u < K; u++) {
      const bool any = row0 + (from + u) * step + mine < n;
      m4[u] = make_float4(any ? m4[u].x : 0.f, any ? m4[u].y : 0.f, any ? m4[u].z : 0.f, any ? m4[u].w : 0.f);
    }
  };
  constexpr auto kWhole = std::true_type{};
  constexpr auto kRagged = std::false_type{};
  if (parts == 1 && n > block && n <= block + kRows / 2 * step) {
    // One partial of a block and at most half of another: both are loaded together (one after the other 192 x 192 20.4 us for
    // all three phases, 30 of up to 250 x 1220 56.5; now 19.6 and 55.3).
    float4 m4[kRows], rest4[kRows / 2];
    float p[kRows][CG], rest_p[kRows / 2][CG];
    load(kWhole, row0, 0, m4, p);
    load(kRagged, row0, kRows, rest4, rest_p);
    add_up(m4, p);
    clear_past(row0, kRows, rest4);
    add_up(rest4, rest_p);
    row0 = n;
  }
  // Main loop: a block at a time, summed on their own in two chains and added to
  // what there is (one chain of fp32 sums down all rows of a partial of 512 left Q half as far again from the exact product;
  // two chains of four instead of one of eight 8.24e-8 of its norm for 4096 x 4096 and 7.5e-8 for 200 x 600, from
  // 8.46e-8 and 7.7e-8).
  for (; row0 + (kRows - 1) * step + side <= n; row0 += parts * block) {
    float4 m4[kRows];
    float p[kRows][CG];
    load(kWhole, row0, 0, m4, p);
    add_up(m4, p);
  }
  // The matrix's last block, where this wave's rows of it are not whole: all their loads in flight together, no branch between
  // them (one round after the other 12 of 1200 x 601 took 57.7 us for all three phases, together with a branch each 56.5, now 55.2).
  const int64_t after = row0 - wave * side + block;
  for (const int64_t rend = after < n ? after : n; row0 < rend; row0 += kRows * step) {
    float4 m4[kRows];
    float p[kRows][CG];
    load(kRagged, row0, 0, m4, p);
    clear_past(row0, 0, m4);
    add_up(m4, p);
  }
  // acc[c][t][i'] in lane 4b+j  ->  Q[k0 + (16b + 4i' + t) % width][4c + j], part (16b + 4i' + t) / width of the wave
  __shared__ float s_q[kWaves][CG][4 * kWave][4];
#pragma unroll
  for (int c = 0; c < CG; c++)
#pragma unroll
    for (int t = 0; t < 4; t++)
#pragma unroll
      for (int ii = 0; ii < 4; ii++) s_q[wave][c][16 * (lane >> 2) + 4 * ii + t][j] = acc[c][t][ii];
  __syncthreads();
  // the one partial of a matrix of few rows is Q itself
  const bool whole = parts == 1;
  float* part = whole ? sg.Qout : a.partials + (int64_t(sg.part_off) * 4) + int64_t(rblk) * m * r;
  const int stride = whole ? ld : r;
  for (int e = threadIdx.x; e < CG * width * 4; e += kThreads) {
    const int c = e / (width * 4), kl = (e / 4) & (width - 1), jj = e & 3;
    const int k = k0 + kl, col = c * 4 + jj;
    if (k < m && col < r) {
      static_assert(kWaves == 4, "summed in pairs");
      auto rows_beside = [&](int h) {
        const int l = h * width + kl;
        return (s_q[0][c][l][jj] + s_q[1][c][l][jj]) + (s_q[2][c][l][jj] + s_q[3][c][l][jj]);
      };
      const float x = side == 1 ? rows_beside(0) : side == 2 ? rows_beside(0) + rows_beside(1)
                                                             : (rows_beside(0) + rows_beside(1)) + (rows_beside(2) + rows_beside(3));
      part[int64_t(k) * stride + col] = x;
    }
  }
}

template <int CAP>
__global__ __launch_bounds__(kThreads) void psgd_qreduce_kernel(const Args<CAP> a) {
  const int tile = blockIdx.x;
  const int s = find_segment<CAP>(a.tile_start, a.nseg, tile);
  const Seg& sg = a.seg[s];
  const int64_t mr = int64_t(sg.m) * sg.r;
  const int64_t per = int64_t(sg.rows) * (kWave / sg.split);
  const int nparts = int((sg.n + per - 1) / per);
  const float* part = a.partials + int64_t(sg.part_off) * 4;
  const int64_t e = int64_t(tile - a.tile_start[s]) * kThreads + threadIdx.x;
  if (e < mr) {
    float x = 0.f;
    int p = 0;
    for (; p + 8 <= nparts; p += 8) {  // eight loads under way, added in pairs (a chain over all partials is less exact)
      float y[8];
#pragma unroll
      for (int u = 0; u < 8; u++) y[u] = part[int64_t(p + u) * mr + e];
      x += ((y[0] + y[1]) + (y[2] + y[3])) + ((y[4] + y[5]) + (y[6] + y[7]));
    }
    for (; p < nparts; p++) x += part[int64_t(p) * mr + e];
    sg.Qout[(e / sg.r) * sg.ld + e % sg.r] = x;
  }
}

// ---- decode: M = P Q^T, residual = grad - M, grad = M ---------------------------
// A workgroup takes a strip of 256 columns and kDecRowsPerBlock rows (8 per wave), or 128 or 64 columns and two or
// four times the rows, two or four groups of four rows side by side in a wave (strip_lanes).  MFMA
// (t, j) has A = P[row0+i'][j] and B = Q[k0+4*lane+t][j], so after the sum over
// j register i' of accumulator t is M[row0+i'][k0+4*lane+t]: the four
// accumulators give each lane 4 consecutive columns of 4 rows, i.e. 128-bit
// loads of grad and 128-bit stores of M, residual and grad.
template <int CG, int CAP>
__global__ __launch_bounds__(kThreads) void psgd_decode_kernel(const Args<CAP> a) {
  const int tile = blockIdx.x;
  const int s = find_segment<CAP>(a.tile_start, a.nseg, tile);
  const Seg& sg = a.seg[s];
  const float* __restrict__ P = sg.P;
  const float* __restrict__ Q = sg.Q;
  float* __restrict__ M = sg.M;
  float* __restrict__ G = const_cast<float*>(sg.grad);
  float* __restrict__ R = const_cast<float*>(sg.res);
  const int n = sg.n, m = sg.m, r = sg.r, ld = sg.ld;
  const bool onto_m = (sg.mode & kOntoM) != 0, keep_grad = (sg.mode & kKeepGrad) != 0;
  const int64_t N = sg.numel;
  const int lanes = sg.split, side = kWave / lanes, width = 4 * lanes;
  const int strips = (m + width - 1) / width;
  const int t_in = tile - a.tile_start[s];
  const int strip = t_in % strips, rblk = t_in / strips;
  const int lane = threadIdx.x & (kWave - 1), wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
  const int kk = strip * width + 4 * (lane & (lanes - 1));
  const int per_wave = a.rows / kWaves * side;
  const int64_t rbeg = (int64_t(rblk) * kWaves + wave) * per_wave;
  const int64_t rend = rbeg + per_wave < n ? rbeg + per_wave : n;
  const int i = lane & 3;

  float q[4][CG * 4];  // Q[kk+t][col]
#pragma unroll
  for (int t = 0; t < 4; t++)
#pragma unroll
    for (int col = 0; col < CG * 4; col++) q[t][col] = (kk + t < m && col < r) ? Q[int64_t(kk + t) * ld + col] : 0.f;

  // (two loops: of one loop with a choice at each store the compiler makes plain stores)
  auto rows = [&](auto stream) {
    constexpr bool STREAM = decltype(stream)::value;
    for (int64_t at = rbeg; at < rend; at += 4 * side) {
      const int64_t row0 = at + 4 * (lane / lanes);
      const bool full4 = kk + 4 <= m && row0 + 4 <= rend && (row0 + 3) * m + kk + 4 <= N;
      float4 g4[4];
      if (full4) {
#pragma unroll
        for (int ii = 0; ii < 4; ii++) g4[ii] = ld4_as<STREAM>(G + (row0 + ii) * m + kk);
      }
      f32x4 acc[4];
#pragma unroll
      for (int t = 0; t < 4; t++) acc[t] = f32x4{0.f, 0.f, 0.f, 0.f};
      if (onto_m) {  // a later block of columns of a rank above 16: go on from what the earlier blocks left in M
#pragma unroll
        for (int ii = 0; ii < 4; ii++)
#pragma unroll
          for (int t = 0; t < 4; t++)
            if (row0 + ii < rend && kk + t < m) acc[t][ii] = M[(row0 + ii) * m + kk + t];
      }
#pragma unroll
      for (int col = 0; col < CG * 4; col++) {
        const float p = (row0 + i < n && col < r) ? P[(row0 + i) * ld + col] : 0.f;
#pragma unroll
        for (int t = 0; t < 4; t++) acc[t] = mfma4(p, q[t][col], acc[t]);
      }
      if (full4) {
        float4 m4[4], r4[4];
#pragma unroll
        for (int ii = 0; ii < 4; ii++) {
          m4[ii] = make_float4(acc[0][ii], acc[1][ii], acc[2][ii], acc[3][ii]);
          r4[ii] = make_float4(g4[ii].x - m4[ii].x, g4[ii].y - m4[ii].y, g4[ii].z - m4[ii].z, g4[ii].w - m4[ii].w);
        }
        // array after array (the layer set: 765 us; row after row 794)
        if (!keep_grad) {
#pragma unroll
          for (int ii = 0; ii < 4; ii++) st4_as<STREAM>(R + (row0 + ii) * m + kk, r4[ii]);
#pragma unroll
          for (int ii = 0; ii < 4; ii++) st4_as<STREAM>(G + (row0 + ii) * m + kk, m4[ii]);  // in place over the line just read
        }
#pragma unroll
        for (int ii = 0; ii < 4; ii++) st4_as<STREAM>(M + (row0 + ii) * m + kk, m4[ii]);
        continue;
      }
#pragma unroll
      for (int ii = 0; ii < 4; ii++) {
        const int64_t row = row0 + ii;
        if (row >= rend) break;
        const int64_t f = row * m + kk;
        const float mv[4] = {acc[0][ii], acc[1][ii], acc[2][ii], acc[3][ii]};
#pragma unroll
        for (int t = 0; t < 4; t++) {
          if (kk + t < m) {
            if (f + t < N && !keep_grad) {
              R[f + t] = G[f + t] - mv[t];
              G[f + t] = mv[t];
            }
            M[f + t] = mv[t];
          }
        }
      }
    }
  };
  if (rows_on_lines(m, G, R, M)) rows(std::true_type{}); else rows(std::false_type{});
}

inline int32_t cdiv(int64_t x, int64_t y) { return static_cast<int32_t>((x + y - 1) / y); }

struct Batch {
  int count;
  const int32_t *ns, *ms, *rs;
};

constexpr int kPassCols = 4 * kMaxCG;  // columns of the factors one pass over the data handles

int check_dims(const char* who, const Batch& b, int* max_rank) {
  *max_rank = 1;
  for (int i = 0; i < b.count; i++) {
    HPX_ARG(b.ns[i] > 0 && b.ms[i] > 0 && b.rs[i] > 0, "%s: matrix %d has dims %d x %d rank %d", who, i, b.ns[i], b.ms[i],
            b.rs[i]);
    if (b.rs[i] > *max_rank) *max_rank = b.rs[i];
  }
  return HPX_OK;
}
// The block of columns [c0, c0 + kPassCols) of a rank-r factor: its width (0: the matrix has no such block) and
// the column groups of four it needs.
inline int block_cols(int r, int c0) { return r <= c0 ? 0 : (r - c0 < kPassCols ? r - c0 : kPassCols); }

// encode1: waves that share four rows of an n x m matrix.  A wave keeps 256 columns in flight, so a row of fewer than
// 768 is one wave's work and one of fewer than 1536 two waves' (ResNet-50's matrices: 61 us with this rule; all
// rows to four waves 64, to one or two 73).  A matrix of fewer than 128 rows spreads them over as many workgroups as it can
// (64 x 147, all three phases: 21.9 us, 22.9 by the other rule).  The sums that make up an entry of P are cut at the waves,
// so the choice rests on the matrix alone and not on what else is in the call: a matrix has one P.
inline int split_rows(int n, int m) { return n < 128 || m >= 1536 ? kWaves : m >= 768 ? kWaves / 2 : 1; }

#define PSGD_LAUNCH_CG_LDS(KERNEL, cg, grid, lds, st, args)                                                             \
  switch (cg) {                                                                                                         \
    case 1: HPX_LAUNCH_LDS(#KERNEL, hpx::g_prof_on, (KERNEL<1, CAP>), dim3(grid), dim3(kThreads), lds, st, args); break;  \
    case 2: HPX_LAUNCH_LDS(#KERNEL, hpx::g_prof_on, (KERNEL<2, CAP>), dim3(grid), dim3(kThreads), lds, st, args); break;  \
    case 3: HPX_LAUNCH_LDS(#KERNEL, hpx::g_prof_on, (KERNEL<3, CAP>), dim3(grid), dim3(kThreads), lds, st, args); break;  \
    default: HPX_LAUNCH_LDS(#KERNEL, hpx::g_prof_on, (KERNEL<4, CAP>), dim3(grid), dim3(kThreads), lds, st, args); break; \
  }
#define PSGD_LAUNCH_CG(KERNEL, cg, grid, st, args) PSGD_LAUNCH_CG_LDS(KERNEL, cg, grid, 0, st, args)

template <int CAP>
int encode1_launches(int count, int max_rank, const float* const* grads, const int64_t* numels, const float* const* residuals,
                     const float* const* Qs, float* const* Ms, float* const* Ps, const int32_t* ns, const int32_t* ms,
                     const int32_t* rs, hipStream_t st) {
  Args<CAP> a;
  int64_t m_bytes = 0;
  for (int k = 0; k < count; k++) m_bytes += int64_t(ns[k]) * ms[k] * int64_t(sizeof(float));
  a.keep = keep_rule(m_bytes);
  a.partials = nullptr;
  for (int c0 = 0; c0 < max_rank; c0 += kPassCols) {
    int i = 0;
    while (i < count) {
      a.nseg = 0;
      a.tile_start[0] = 0;
      int cg = 1;
      while (i < count && a.nseg < CAP) {
        const int rb = block_cols(rs[i], c0);
        if (rb == 0) { i++; continue; }
        const int split = split_rows(ns[i], ms[i]);
        const int32_t t = cdiv(ns[i], 4 * (kWaves / split));
        if (int64_t(a.tile_start[a.nseg]) + t > INT32_MAX) break;
        a.seg[a.nseg] = Seg{grads[i], residuals[i], Qs[i] + c0, Ms[i], Ps[i] + c0, nullptr, numels[i], ns[i], ms[i], rb, 0,
                            rs[i], c0 ? kFromM : 0, split, 0};
        if ((rb + 3) / 4 > cg) cg = (rb + 3) / 4;
        a.tile_start[a.nseg + 1] = a.tile_start[a.nseg] + t;
        a.nseg++;
        i++;
      }
      if (a.nseg == 0) continue;
      // Two read streams and a write stream: held to four workgroups per CU (LDS the kernel never touches).  Ranks up to
      // four are held to three by their registers; without either limit the layer set's 36 matrices took 618 us, at four 598.
      PSGD_LAUNCH_CG_LDS(psgd_encode1_kernel, cg, a.tile_start[a.nseg], hpx::kWriteStreamPadLds4, st, a);
      HPX_HIP(hipGetLastError());
    }
  }
  return HPX_OK;
}

template <bool WIDE, bool LDS, int CAP>
int orth_launch(const Args<CAP>& a, size_t lds, hipStream_t st) {
  if (lds)
    HPX_HIP(hipFuncSetAttribute(reinterpret_cast<const void*>(psgd_orth_kernel<WIDE, LDS, CAP>),
                                hipFuncAttributeMaxDynamicSharedMemorySize, int(lds)));
  HPX_LAUNCH_LDS("psgd_orth_kernel", hpx::g_prof_on, (psgd_orth_kernel<WIDE, LDS, CAP>), dim3(a.nseg), dim3(kOrthThreads), lds, st, a);
  HPX_HIP(hipGetLastError());
  return HPX_OK;
}

// A matrix of up to kQWholeRows rows, one block and a half of the narrowest strips, takes the product in one partial, which is Q
// itself: a call of such matrices needs no launch to add partials up.  us of a pass, by the strips of other matrices / so:
// 128 x 128 20.3 / 17.5, 192 x 192 23.1 / 19.6, 190 x 4000 34.5 / 30.0, 30 of up to 150 x 220 29.5 / 25.4, of up to 190 x 800
// 42.8 / 39.4, 10 of up to 64 x 2000 30.8 / 25.8; among taller matrices, where the launch is there anyway, 30 of up to 250 x 1220
// 54.8 / 55.3, of up to 400 x 600 47.2 / 47.2, of up to 600 x 300 44.5 / 45.4, 12 of up to 256 x 2000 42.6 / 43.2 (56.5, 48.8, 45.8
// and 44.5 with the half block loaded behind the block), 10 of up to 512 x 512 36.5 / 35.7; at 256 rows these 39.7.
constexpr int kQWholeRows = 192;
inline int q_lanes(int n, int m) { return n <= kQWholeRows ? 16 : strip_lanes(m); }
// Partials of a matrix: of `rows` rows each, as many times more as strips side by side in a wave.
inline int32_t q_parts(int n, int m, int rows) { return cdiv(n, int64_t(rows) * (kWave / q_lanes(n, m))); }

// Rows per partial: as many as leave the matrix kQTiles workgroups, since every partial is written and read back; 64 at
// least, or 32 where 64 would leave fewer than kQTilesSmall.  Like split_rows by the matrix alone: Q is the sum of the
// partials, and what a matrix's Q is must not depend on what else is in the call.  A pass over all three phases in us, with the rows
// chosen so that the call had 1024 workgroups / with this rule / with at most 256 rows: layer set of 36 matrices 1566 /
// 1574 / 1588, 4 of 2000 x 1000 74 / 70 / 70, ResNet-50's 54 157.6 / 157.5 / 157.5
// (with 32 rows for all of those 160.5); with kQTiles 64 and 32 4096 x 1024 alone is at 59 and 68 instead of 56.
constexpr int kQRowsMin = 32, kQRowsMax = 512;
// A matrix of 2^24 elements and more is given kQTilesLarge workgroups.  us of a pass with 128 / 256: 4096 x 4096 alone 113.1 / 107.2, of
// rank 8 152 / 142.5, 16384 x 1024 131 / 126.5, 5000 x 3500 166 / 157, 30000 x 600 184 / 177, 4 of 4100 x 4099 285 / 273; from 2^25
// elements 512 rows a partial leave as many anyway; the layer set, which twelve such matrices are part of, pays 2.5 of
// 1550 for their partials.
constexpr int64_t kQTiles = 128, kQTilesSmall = 32, kQTilesLarge = 256;
inline int q_rows(int n, int m) {
  static_assert(kQWholeRows <= 2 * kQRowsMin * (kWave / 16), "rows of one partial of the narrowest strips");
  if (n <= kQWholeRows) return 2 * kQRowsMin;
  auto tiles = [=](int rows) { return int64_t(cdiv(m, 4 * q_lanes(n, m))) * q_parts(n, m, rows); };
  int rows = kQRowsMax;
  const int64_t enough = int64_t(n) * m >= (1 << 24) ? kQTilesLarge : kQTiles;
  while (rows > 2 * kQRowsMin && tiles(rows) < enough) rows /= 2;
  return rows == 2 * kQRowsMin && tiles(rows) < kQTilesSmall ? kQRowsMin : rows;
}

template <int CAP>
int encode2_launches(int count, int max_rank, float* partials, float* const* Ps, const float* const* Ms, float* const* Qs,
                     const int32_t* ns, const int32_t* ms, const int32_t* rs, hipStream_t st) {
  Args<CAP> a;
  a.rows = 0;
  a.partials = partials;
  // step 1: orthonormalise every P over all of its columns
  for (int i = 0; i < count;) {
    a.nseg = 0;
    int64_t max_nr = 0;
    bool wide = false;
    for (; i < count && a.nseg < CAP; i++) {
      a.seg[a.nseg++] = Seg{nullptr, nullptr, nullptr, nullptr, Ps[i], nullptr, 0, ns[i], ms[i], rs[i], 0, rs[i], 0, 0, 0};
      if (int64_t(ns[i]) * rs[i] > max_nr) max_nr = int64_t(ns[i]) * rs[i];
      wide = wide || (rs[i] > 4 && rs[i] <= kGramCols);
    }
    const bool fits = max_nr <= kOrthLdsFloats;
    const size_t lds = fits ? size_t(max_nr) * sizeof(float) : 0;
    const int rc = wide ? (fits ? orth_launch<true, true>(a, lds, st) : orth_launch<true, false>(a, lds, st))
                        : (fits ? orth_launch<false, true>(a, lds, st) : orth_launch<false, false>(a, lds, st));
    if (rc != HPX_OK) return rc;
  }
  // step 2: Q = M^T P, sixteen columns per pass over M
  for (int c0 = 0; c0 < max_rank; c0 += kPassCols) {
    int i = 0;
    int64_t poff = 0;
    while (i < count) {
      a.nseg = 0;
      a.tile_start[0] = 0;
      int32_t red_start[CAP + 1];
      red_start[0] = 0;
      int cg = 1;
      while (i < count && a.nseg < CAP) {
        const int rb = block_cols(rs[i], c0);
        if (rb == 0) { i++; continue; }
        const int lanes = q_lanes(ns[i], ms[i]);
        const int rows = q_rows(ns[i], ms[i]);
        const int32_t parts = q_parts(ns[i], ms[i], rows);
        const int64_t t = int64_t(cdiv(ms[i], 4 * lanes)) * parts;
        const int32_t tr = parts > 1 ? cdiv(int64_t(ms[i]) * rb, kThreads) : 0;
        if (a.tile_start[a.nseg] + t > INT32_MAX || int64_t(red_start[a.nseg]) + tr > INT32_MAX) {
          HPX_ARG(a.nseg > 0, "hpx_powersgd_encode2: matrix %d is too large", i);
          break;
        }
        a.seg[a.nseg] = Seg{nullptr, nullptr, nullptr, const_cast<float*>(Ms[i]), Ps[i] + c0, Qs[i] + c0, 0, ns[i], ms[i], rb,
                            static_cast<int32_t>(poff), rs[i], 0, lanes, rows};
        poff += (int64_t(parts) * ms[i] * rb + 3) / 4;
        if ((rb + 3) / 4 > cg) cg = (rb + 3) / 4;
        a.tile_start[a.nseg + 1] = a.tile_start[a.nseg] + int32_t(t);
        red_start[a.nseg + 1] = red_start[a.nseg] + tr;
        a.nseg++;
        i++;
      }
      if (a.nseg == 0) continue;
      PSGD_LAUNCH_CG(psgd_mtp_kernel, cg, a.tile_start[a.nseg], st, a);
      HPX_HIP(hipGetLastError());
      for (int k = 0; k <= a.nseg; k++) a.tile_start[k] = red_start[k];
      if (a.tile_start[a.nseg] == 0) continue;
      HPX_LAUNCH("psgd_qreduce_kernel", psgd_qreduce_kernel<CAP>, dim3(a.tile_start[a.nseg]), dim3(kThreads), st, a);
      HPX_HIP(hipGetLastError());
    }
  }
  return HPX_OK;
}

template <int CAP>
int decode_launches(int count, int max_rank, const float* const* Ps, const float* const* Qs, float* const* Ms, float* const* residuals,
                    float* const* grads, const int64_t* numels, const int32_t* ns, const int32_t* ms, const int32_t* rs, hipStream_t st) {
  auto tiles_of = [&](int i, int rows) {
    const int lanes = strip_lanes(ms[i]);
    return int64_t(cdiv(ms[i], 4 * lanes)) * cdiv(ns[i], int64_t(rows) * (kWave / lanes));
  };
  int64_t tiles = 0;
  for (int i = 0; i < count; i++) tiles += tiles_of(i, kDecRowsPerBlock);
  Args<CAP> a;
  a.partials = nullptr;
  // Where the chip takes the whole call at once a wave has one group of rows, not one after the other.
  a.rows = tiles < kDecTiles ? kDecRowsPerBlock / 2 : kDecRowsPerBlock;
  for (int c0 = 0; c0 < max_rank; c0 += kPassCols) {
    int i = 0;
    while (i < count) {
      a.nseg = 0;
      a.tile_start[0] = 0;
      int cg = 1;
      while (i < count && a.nseg < CAP) {
        const int rb = block_cols(rs[i], c0);
        if (rb == 0) { i++; continue; }
        const int lanes = strip_lanes(ms[i]);
        const int64_t t = tiles_of(i, a.rows);
        if (a.tile_start[a.nseg] + t > INT32_MAX) {
          HPX_ARG(a.nseg > 0, "hpx_powersgd_decode: matrix %d is too large", i);
          break;
        }
        const int32_t mode = (c0 ? kOntoM : 0) | (c0 + kPassCols < rs[i] ? kKeepGrad : 0);
        a.seg[a.nseg] = Seg{grads[i], residuals[i], Qs[i] + c0, Ms[i], const_cast<float*>(Ps[i]) + c0, nullptr, numels[i], ns[i],
                            ms[i], rb, 0, rs[i], mode, lanes, 0};
        if ((rb + 3) / 4 > cg) cg = (rb + 3) / 4;
        a.tile_start[a.nseg + 1] = a.tile_start[a.nseg] + int32_t(t);
        a.nseg++;
        i++;
      }
      if (a.nseg == 0) continue;
      // One read and three writes per element: held to two workgroups per CU (LDS the kernel never touches,
      // hpx_common.h), the 36 matrices of the configuration decode in 765 us instead of 784 with three or four (a
      // pass over three such sets of buffers in turn; 755 in another process, with buffers at other addresses, and a launch
      // between 744 and 831).
      PSGD_LAUNCH_CG_LDS(psgd_decode_kernel, cg, a.tile_start[a.nseg], hpx::kWriteStreamPadLds2, st, a);
      HPX_HIP(hipGetLastError());
    }
  }
  return HPX_OK;
}

}  // namespace

HPX_API int hpx_powersgd_encode1(int count, const float* const* grads, const int64_t* numels,
                                 const float* const* residuals, const float* const* Qs, float* const* Ms,
                                 float* const* Ps, const int32_t* ns, const int32_t* ms, const int32_t* rs,
                                 hpx_stream_t stream) {
  hpx::clear_error();
  HPX_ARG(count >= 0, "hpx_powersgd_encode1: negative count");
  if (count == 0) return HPX_OK;
  HPX_ARG(grads && numels && residuals && Qs && Ms && Ps && ns && ms && rs, "hpx_powersgd_encode1: null argument array");
  int max_rank = 1;
  int rc = check_dims("hpx_powersgd_encode1", Batch{count, ns, ms, rs}, &max_rank);
  if (rc != HPX_OK) return rc;
  for (int i = 0; i < count; i++) {
    HPX_ARG(grads[i] && residuals[i] && Qs[i] && Ms[i] && Ps[i], "hpx_powersgd_encode1: matrix %d has a null pointer", i);
    HPX_ARG(numels[i] >= 0 && numels[i] <= int64_t(ns[i]) * ms[i], "hpx_powersgd_encode1: matrix %d: numel %lld exceeds n*m", i,
            static_cast<long long>(numels[i]));
  }
  hipStream_t st = static_cast<hipStream_t>(stream);
  return PSGD_BY_COUNT(encode1_launches, max_rank, grads, numels, residuals, Qs, Ms, Ps, ns, ms, rs, st);
}

HPX_API int hpx_powersgd_encode2(int count, float* const* Ps, const float* const* Ms, float* const* Qs,
                                 const int32_t* ns, const int32_t* ms, const int32_t* rs, hpx_stream_t stream) {
  hpx::clear_error();
  HPX_ARG(count >= 0, "hpx_powersgd_encode2: negative count");
  if (count == 0) return HPX_OK;
  HPX_ARG(Ps && Ms && Qs && ns && ms && rs, "hpx_powersgd_encode2: null argument array");
  int max_rank = 1;
  int rc = check_dims("hpx_powersgd_encode2", Batch{count, ns, ms, rs}, &max_rank);
  if (rc != HPX_OK) return rc;
  for (int i = 0; i < count; i++) HPX_ARG(Ps[i] && Ms[i] && Qs[i], "hpx_powersgd_encode2: matrix %d has a null pointer", i);
  int64_t part_quads = 0;  // partial storage in units of 4 floats (one pass at a time uses it)
  for (int i = 0; i < count; i++) part_quads += (int64_t(q_parts(ns[i], ms[i], q_rows(ns[i], ms[i]))) * ms[i] * block_cols(rs[i], 0) + 3) / 4;
  HPX_ARG(part_quads <= INT32_MAX, "hpx_powersgd_encode2: batch too large for one call");
  hipStream_t st = static_cast<hipStream_t>(stream);
  hpx::Workspace* ws = hpx::workspace_record(st);
  if (!ws) return HPX_ERR_HIP;
  std::lock_guard<std::mutex> lock(ws->mu);
  rc = hpx::ensure_workspace(ws, size_t(part_quads) * 16);
  if (rc != HPX_OK) return rc;
  float* partials = reinterpret_cast<float*>(ws->dev);
  return PSGD_BY_COUNT(encode2_launches, max_rank, partials, Ps, Ms, Qs, ns, ms, rs, st);
}

HPX_API int hpx_powersgd_decode(int count, const float* const* Ps, const float* const* Qs, float* const* Ms,
                                float* const* residuals, float* const* grads, const int64_t* numels,
                                const int32_t* ns, const int32_t* ms, const int32_t* rs, hpx_stream_t stream) {
  hpx::clear_error();
  HPX_ARG(count >= 0, "hpx_powersgd_decode: negative count");
  if (count == 0) return HPX_OK;
  HPX_ARG(Ps && Qs && Ms && residuals && grads && numels && ns && ms && rs, "hpx_powersgd_decode: null argument array");
  int max_rank = 1;
  int rc = check_dims("hpx_powersgd_decode", Batch{count, ns, ms, rs}, &max_rank);
  if (rc != HPX_OK) return rc;
  for (int i = 0; i < count; i++) {
    HPX_ARG(Ps[i] && Qs[i] && Ms[i] && residuals[i] && grads[i], "hpx_powersgd_decode: matrix %d has a null pointer", i);
    HPX_ARG(numels[i] >= 0 && numels[i] <= int64_t(ns[i]) * ms[i], "hpx_powersgd_decode: matrix %d: numel %lld exceeds n*m", i,
            static_cast<long long>(numels[i]));
  }
  hipStream_t st = static_cast<hipStream_t>(stream);
  return PSGD_BY_COUNT(decode_launches, max_rank, Ps, Qs, Ms, residuals, grads, numels, ns, ms, rs, st);
}
