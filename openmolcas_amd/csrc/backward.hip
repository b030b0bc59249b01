// Backward of the closed-shell energy functional of the J/K build.
//
//   E(C, L) = tr(P h) + 1/2 sum_J V_J^2 - 1/4 sum_J tr(P L^J P L^J),
//   P = 2 C C^T,  V_J = tr(P L^J),  F = h + J[P] - 1/2 K[P]
//   dE/dC   = 4 F C
//   dE/dL^J = V_J P - 1/2 P L^J P = V_J P - 2 C Z^J C^T,  Z^J = C^T L^J C
// with the packed-parameter rule: off-diagonal entries of dE/dL_packed carry
// a factor 2 (L_ab and L_ba are the same parameter).
//
// The energy expression is that of src/scf/eneclc.F90:58,77,104 with the
// Fock matrix of src/fock_util/cho_fscf.F90 (DECO convention, ExFac = 1/2 on
// V = sqrt(2) C); the gradient has no counterpart in the reference, which only
// evaluates the Fock matrix.
//
// Kernels: with Z kept by the forward, k_grad_rows forms W = C Z in registers and
// the packed lower triangle of W C^T in one launch; without it X^J = C^T L^J is
// recomputed chunk by chunk (the chunk size follows the context's X budget) and
// Z = X C comes from k_zsym.  Above 128 orbitals W and the packed product go
// through one batched FP64-MFMA GEMM whose epilogue writes packed storage.
#include <type_traits>

#include "mjk_internal.h"

namespace mjk {
namespace {

constexpr int kThreads = 256;
constexpr int kTM = 64;  // output tile
constexpr int kBK = 16;  // contraction chunk

__device__ inline v4d mfma64(double a, double b, v4d c) {
  return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
}
__device__ inline int64_t tri0(int64_t a) { return a * (a + 1) / 2; }

struct GemmBatch {
  const double *A;  // A[b][i][k] at A + b*sA + i*lda + k
  const float *A32; // the same for an FP32 A operand (k_gemm<..., float>)
  int64_t sA, lda;
  const double *B;  // NN: B[b][k][j] at B + b*sB + k*ldb + j;  NT: B[b][j][k] at ... j*ldb + k
  int64_t sB, ldb;
  double *O;        // dense: O[b][i][j] at O + b*sO + i*ldo + j
  int64_t sO, ldo;
  int m, n, k;
  double alpha;
  // packed-gradient epilogue (EPI == 1), only for i >= j:
  // G[b*ldg + tri0(i) + j] = (i == j ? 1 : 2) * (gv*V[b] * Pl[tri0(i)+j] + alpha*acc)
  double *G;
  int64_t ldg;
  const double *V;
  const double *Pl;
  double gv;
  // launch shape, set by gemm(): output tiles per product (EPI == 1: the
  // lower-triangle tiles only) and tiles x batch work items
  int tiles;
  int64_t items;
};

// grid.x = round_up(tiles * batch, 8).  O = alpha * A B (NN) or A B^T (NT).
// Work item l = b * tiles + t (product b, output tile t); the block id is
// remapped so that consecutive items run on one XCD (the hardware deals
// blocks to the eight XCDs in turn): the tiles of one product then share
// that XCD's L2 for their common operand rows instead of each XCD fetching
// them from HBM.
// Double-buffered LDS with one barrier per kBK chunk: chunk c is multiplied
// out of buffer c&1 while chunk c+1 is stored from registers into the other
// buffer and chunk c+2 is fetched.  TA: element type of A (an FP32 A is
// widened to FP64 on load; the products and sums are FP64).
template <bool BT, int EPI, typename TA = double>
__global__ __launch_bounds__(kThreads) void k_gemm(GemmBatch g) {
  __shared__ double sA[2][kTM][kBK + 1];
  __shared__ double sB[2][kBK][kTM + 1];
  const int64_t nblk = gridDim.x;  // multiple of 8
  const int64_t l = (int64_t(blockIdx.x) & 7) * (nblk >> 3) + (int64_t(blockIdx.x) >> 3);
  if (l >= g.items) return;
  const int64_t b = l / g.tiles;
  const int t = int(l - b * g.tiles);
  int ti, tj;
  if constexpr (EPI == 1) {  // lower-triangle tile t = ti (ti + 1) / 2 + tj
    ti = int((sqrt(8.0 * t + 1.0) - 1.0) * 0.5);
    while (ti * (ti + 1) / 2 > t) --ti;
    while ((ti + 1) * (ti + 2) / 2 <= t) ++ti;
    tj = t - ti * (ti + 1) / 2;
  } else {
    const int ntj = (g.n + kTM - 1) / kTM;
    ti = t / ntj;
    tj = t - ti * ntj;
  }
  const int i0 = ti * kTM, j0 = tj * kTM;
  const TA *__restrict__ A;
  if constexpr (std::is_same<TA, float>::value) A = g.A32 + b * g.sA;
  else A = g.A + b * g.sA;
  const double *__restrict__ B = g.B + b * g.sB;
  const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
  const int wm = w >> 1, wn = w & 1;
  v4d acc[2][2];
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j) acc[i][j] = v4d{0.0, 0.0, 0.0, 0.0};

  constexpr int PN = kTM * kBK / kThreads;
  static_assert(2 * PN <= 32, "element mask");
  double ra[PN], rb[PN];
  // Element it of a thread sits at a fixed (row, contraction column) of every
  // chunk, so its offset inside the product's operand is computed once and a
  // chunk adds only its first contraction index (32-bit byte offsets from the
  // product's base: every operand is below 2^28 elements, checked by gemm()).
  // Out-of-range elements load element 0 and are zeroed when stashed (bit it
  // of the mask for A, bit PN + it for B), so a chunk's loads stay in flight
  // across the multiply of the previous chunk.
  uint32_t aoff[PN], boff[PN];
  int akk[PN], bkk[PN];
  uint32_t rowok = 0;  // bit it: A row inside m; bit PN + it: B row / column inside n
#pragma unroll
  for (int it = 0; it < PN; ++it) {
    const int e = tid + kThreads * it;
    const int r = e / kBK, kk = e % kBK;  // A: row r, column kk
    const int gi = i0 + r;
    aoff[it] = uint32_t(gi) * uint32_t(g.lda) + uint32_t(kk);
    akk[it] = kk;
    rowok |= gi < g.m ? 1u << it : 0u;
    if (BT) {  // B stored [j][k]: row r of the j tile
      const int gj = j0 + r;
      boff[it] = uint32_t(gj) * uint32_t(g.ldb) + uint32_t(kk);
      bkk[it] = kk;
      rowok |= gj < g.n ? 1u << (PN + it) : 0u;
    } else {  // B stored [k][j]
      const int kr = e / kTM, jj = e % kTM, gj = j0 + jj;
      boff[it] = uint32_t(kr) * uint32_t(g.ldb) + uint32_t(gj);
      bkk[it] = kr;
      rowok |= gj < g.n ? 1u << (PN + it) : 0u;
    }
  }
  const char *__restrict__ Ab = reinterpret_cast<const char *>(A);
  const char *__restrict__ Bb = reinterpret_cast<const char *>(B);
  uint32_t okm = 0;
  auto fetch = [&](int k0) {
    okm = 0;
    const uint32_t bstep = BT ? uint32_t(k0) : uint32_t(k0) * uint32_t(g.ldb);
#pragma unroll
    for (int it = 0; it < PN; ++it) {
      const bool oka = ((rowok >> it) & 1u) && akk[it] + k0 < g.k;
      const bool okb = ((rowok >> (PN + it)) & 1u) && bkk[it] + k0 < g.k;
      ra[it] = double(*reinterpret_cast<const TA *>(
          Ab + (oka ? (aoff[it] + uint32_t(k0)) * uint32_t(sizeof(TA)) : 0u)));
      rb[it] = *reinterpret_cast<const double *>(Bb + (okb ? (boff[it] + bstep) * 8u : 0u));
      okm |= (oka ? 1u << it : 0u) | (okb ? 1u << (PN + it) : 0u);
    }
  };
  auto stash = [&](int buf) {
#pragma unroll
    for (int it = 0; it < PN; ++it) {
      const int e = tid + kThreads * it;
      const double va = ((okm >> it) & 1u) ? ra[it] : 0.0;
      const double vb = ((okm >> (PN + it)) & 1u) ? rb[it] : 0.0;
      sA[buf][e / kBK][e % kBK] = va;
      if (BT) sB[buf][e % kBK][e / kBK] = vb;
      else sB[buf][e / kTM][e % kTM] = vb;
    }
  };
  const int nch = (g.k + kBK - 1) / kBK;
  fetch(0);
  stash(0);
  if (nch > 1) fetch(kBK);
  __syncthreads();
  for (int c = 0; c < nch; ++c) {
    const int cur = c & 1;
    // operand fragments of the next 4-row step are read from LDS while the
    // current step's MFMAs run
    double af[2][2], bf[2][2];
    auto ld = [&](int ks, int q) {
      const int kr = ks * 4 + (lane >> 4);
#pragma unroll
      for (int i = 0; i < 2; ++i) af[q][i] = sA[cur][wm * 32 + i * 16 + (lane & 15)][kr];
#pragma unroll
      for (int j = 0; j < 2; ++j) bf[q][j] = sB[cur][kr][wn * 32 + j * 16 + (lane & 15)];
    };
    ld(0, 0);
#pragma unroll
    for (int ks = 0; ks < kBK / 4; ++ks) {
      const int q = ks & 1;
      if (ks + 1 < kBK / 4) ld(ks + 1, q ^ 1);
#pragma unroll
      for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j) acc[i][j] = mfma64(af[q][i], bf[q][j], acc[i][j]);
    }
    if (c + 1 < nch) stash(cur ^ 1);
    if (c + 2 < nch) fetch((c + 2) * kBK);
    __syncthreads();
  }
  // result layout of v_mfma_f64_16x16x4f64: row 4*r + lane/16, column lane%16
  if constexpr (EPI == 0) {
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
      for (int j = 0; j < 2; ++j)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const int gi = i0 + wm * 32 + i * 16 + 4 * r + (lane >> 4);
          const int gj = j0 + wn * 32 + j * 16 + (lane & 15);
          if (gi < g.m && gj < g.n) g.O[b * g.sO + int64_t(gi) * g.ldo + gj] = g.alpha * acc[i][j][r];
        }
  } else {
    // Every density value this lane needs is loaded before the first store:
    // with the loads and stores interleaved, each store would wait for its
    // load's round trip (G and P may alias as far as the compiler knows).
    const double *__restrict__ Pl = g.Pl;
    double *__restrict__ G = g.G + b * g.ldg;
    const double vb = g.gv * g.V[b];
    double pv[2][2][4];
    uint32_t pi[2][2][4];
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
      for (int j = 0; j < 2; ++j)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const uint32_t gi = uint32_t(i0 + wm * 32 + i * 16 + 4 * r + (lane >> 4));
          const uint32_t gj = uint32_t(j0 + wn * 32 + j * 16 + (lane & 15));
          const bool ok = gi < uint32_t(g.m) && gi >= gj;
          pi[i][j][r] = ok ? gi * (gi + 1u) / 2u + gj : ~0u;
          pv[i][j][r] = Pl[ok ? pi[i][j][r] : 0u];
        }
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
      for (int j = 0; j < 2; ++j)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const uint32_t p = pi[i][j][r];
          if (p == ~0u) continue;
          const uint32_t gi = uint32_t(i0 + wm * 32 + i * 16 + 4 * r + (lane >> 4));
          const uint32_t gj = uint32_t(j0 + wn * 32 + j * 16 + (lane & 15));
          const double s = (gi == gj) ? 1.0 : 2.0;
          G[p] = s * (vb * pv[i][j][r] + g.alpha * acc[i][j][r]);
        }
  }
}

// Dense symmetric n x n (row stride ld) from plain LT storage.
__global__ void k_unpack_lt(const double *__restrict__ lt, int n, double *__restrict__ out,
                            int64_t ld) {
  const int a = blockIdx.x;
  for (int b = threadIdx.x; b < n; b += blockDim.x) {
    const int hi = a > b ? a : b, lo = a > b ? b : a;
    out[int64_t(a) * ld + b] = lt[tri0(hi) + lo];
  }
}

// LT of scale * C C^T from the orbitals, C[a][k] = corb[k + a*o]; fold != 0
// doubles the off-diagonal (folded density), fold == 0 keeps plain storage.  One
// wave per 32 x 32 tile of the lower triangle, operands from memory: lane 16 g + m
// takes orbitals 16 c + 4 g + s of row m in the four steps s of chunk c (a thread
// per element read C with a stride of nocc: 53 us at n=536 nocc=98, now 8).
// grid = tiles, block 64.
__global__ __launch_bounds__(64) void k_density_lt(const double *__restrict__ corb, int o, int n, double scale,
                                                  int fold, double *__restrict__ p) {
  const int t = blockIdx.x;
  int ta = int((sqrt(8.0 * t + 1.0) - 1.0) * 0.5);
  while (ta * (ta + 1) / 2 > t) --ta;
  while ((ta + 1) * (ta + 2) / 2 <= t) ++ta;
  const int tb = t - ta * (ta + 1) / 2;
  const int lane = threadIdx.x, m = lane & 15, g = lane >> 4;
  const double *__restrict__ ra[2], *__restrict__ rb[2];
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    ra[h] = corb + int64_t(min(32 * ta + 16 * h + m, n - 1)) * o;
    rb[h] = corb + int64_t(min(32 * tb + 16 * h + m, n - 1)) * o;
  }
  v4d acc[2][2];
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j) acc[i][j] = v4d{0.0, 0.0, 0.0, 0.0};
  for (int k0 = 0; k0 < o; k0 += 16) {
    double a[4][2], b[4][2];
#pragma unroll
    for (int s = 0; s < 4; ++s) {
      const int k = k0 + 4 * g + s, kc = min(k, o - 1);
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        a[s][h] = k < o ? ra[h][kc] : 0.0;
        b[s][h] = k < o ? rb[h][kc] : 0.0;
      }
    }
#pragma unroll
    for (int s = 0; s < 4; ++s)
#pragma unroll
      for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j) acc[i][j] = mfma64(a[s][i], b[s][j], acc[i][j]);
  }
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int x = 32 * ta + 16 * i + 4 * r + g, y = 32 * tb + 16 * j + m;
        if (x < n && y <= x) p[tri0(x) + y] = (fold && x != y ? 2.0 : 1.0) * scale * acc[i][j][r];
      }
}

void density_launch(Context *c, const double *corb, int o, double scale, int fold, double *p) {
  const int64_t t = ceil_div(c->n, 32);
  hipLaunchKernelGGL(k_density_lt, dim3(unsigned(t * (t + 1) / 2)), dim3(64), 0, c->stream, corb, o, c->n, scale,
                     fold, p);
}

template <bool BT, int EPI, typename TA = double>
int gemm(Context *c, const GemmBatch &g0, int batch) {
  GemmBatch g = g0;
  // operands are addressed with 32-bit byte offsets inside one product
  constexpr int64_t kMaxElems = int64_t(1) << 28;
  if (int64_t(g.m) * g.lda >= kMaxElems || int64_t(BT ? g.n : g.k) * g.ldb >= kMaxElems)
    return set_error(c, MJK_ERR_ARG, "gemm: operand of more than 2^28 elements");
  const int ti = (g.m + kTM - 1) / kTM, tj = (g.n + kTM - 1) / kTM;
  g.tiles = EPI == 1 ? ti * (ti + 1) / 2 : ti * tj;  // EPI == 1: square lower-triangle output
  g.items = int64_t(g.tiles) * batch;
  hipLaunchKernelGGL((k_gemm<BT, EPI, TA>), dim3(unsigned(round_up(g.items, 8))), dim3(kThreads), 0,
                     c->stream, g);
  return MJK_OK;
}

// dL[J] = s * (alpha V_J P + beta W[J] C^T) for the jn vectors whose W = C Z
// sits at W (n_pad x ldc per vector): lower triangle, packed, row stride ldd.
int grad_from_w(Context *c, int nocc, const double *W, int ldc, const double *v, const double *P,
                 double alpha, double beta, double *dl, int64_t ldd, int64_t jn) {
  GemmBatch g{};
  g.A = W; g.sA = int64_t(c->n_pad) * ldc; g.lda = ldc;
  g.B = static_cast<const double *>(c->w->cbank.ptr); g.sB = 0; g.ldb = ldc;  // NT: B[j][k] = C[b][k]
  g.m = c->n; g.n = c->n; g.k = nocc; g.alpha = beta;
  g.G = dl; g.ldg = ldd; g.V = v; g.Pl = P; g.gv = alpha;
  return gemm<true, 1>(c, g, int(jn));
}

// ---- fused vector gradient ------------------------------------------------
// G[J] (packed lower triangle, row stride ldg) = s_ab (gv V_J P_ab +
// beta (C Z^J C^T)_ab) for the vectors J whose Z^J (nocc x nocc) has element
// (k, l) at z + J sz + k ldz + l.
struct GradRows {
  const void *ct;    // transposed orbital bank C^T[k][a], FP64 or FP32: 16 OC16 rows of n_pad,
                     // zero for k >= nocc or a >= n
  int n_pad;
  const double *z;
  int64_t sz;
  int ldz;
  int o;             // nocc
  const double *v;   // V[J]
  const double *p;   // P, plain LT (null: 2 C C^T)
  double gv, beta;
  double *g;
  int64_t ldg;
  int32_t rowbytes;  // bytes of one packed triangle n (n + 1) / 2 (< 2^31)
  int n, T;          // basis functions, strips of 32 rows
  int64_t jn;        // vectors
  int64_t items;     // strips x groups of four vectors
};
// Byte offset of a masked element in the packed triangle: past every row, so
// the buffer load returns 0 and the store is dropped by the range check of the
// buffer resource (stride 0, rowbytes records).
constexpr uint32_t kMasked = 0x80000000u;
constexpr int kRsrcWord3 = 0x00020000;  // buffer resource word 3 of this architecture family
typedef int v2u __attribute__((ext_vector_type(2)));  // operand types of the buffer builtins
typedef int v4u __attribute__((ext_vector_type(4)));
typedef float v2f __attribute__((ext_vector_type(2)));

// Arithmetic of k_grad_rows: FP64 MFMA, or FP32 MFMA (the split-precision
// backward's tail vectors: contractions of at most 128 terms, FP64 output).
// Operand layouts are those of v_mfma_f64_16x16x4f64 / v_mfma_f32_16x16x4f32
// (A[l%16][l/16], B[l/16][l%16]); result row of register r: 4r + l/16 (FP64),
// 4(l/16) + r (FP32), column l%16.
struct GR64 {
  typedef double T;
  typedef v2d T2;
  typedef v4d Acc;
  __device__ static Acc mma(T a, T b, Acc c) { return mfma64(a, b, c); }
  static constexpr int kStep = 4;  // row(g, r) - row(g, r - 1)
  __device__ static int row(int g, int r) { return 4 * r + g; }
};
struct GR32 {
  typedef float T;
  typedef v2f T2;
  typedef v4f Acc;
  __device__ static Acc mma(T a, T b, Acc c) { return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0); }
  static constexpr int kStep = 1;
  __device__ static int row(int g, int r) { return 4 * g + r; }
};

// Work item = (four vectors J, one per wave; strip of 32 rows a).  Phase 1 forms
// W^T = Z^T C^T of the strip (OC x 32, OC = 16 OC16 >= nocc): the transposed
// product, because its result layout (column a on the lane, row l in the
// register) is the A operand layout of phase 2, so W never leaves the
// accumulators.  Phase 2 walks the column tiles of 32 up to the diagonal: A = W
// from those registers, B = the tile's 32 columns of C^T, which the four waves
// share in LDS (double-buffered, one barrier per tile).  Loads and stores retire
// in one order, so a fragment loaded after a tile's stores is not there before
// their acknowledgement: the next tile's columns are loaded to registers before
// this tile's stores and no wait stands behind a store.  Lane l = 16 g + m takes
// columns 2 m, 2 m + 1 at once (row and column tile (i, h): AO 32 t + 2 m + h).  The
// tile is stored packed, two neighbours as 16 bytes, through a range-checked
// buffer resource that drops elements past n; only the diagonal tile masks
// element by element.  Contraction steps past nocc are left out.  The longest
// strip of a group of vectors runs first; its strips run on one XCD (they share
// the Z^J).
// Bound by the matrix cores from about 90 orbitals (n=536 nchol=2510 nocc=98
// 2.62 -> 1.98 ms, 56 TFLOP/s executed; n=600 nchol=2800 nocc=120 4.17 -> 3.11 ms),
// below that and in FP32 by the scattered stores (2.0-2.6 TB/s of output; n=600
// nchol=3000 nocc=75 2.83 -> 2.13 ms FP64, 2.07 -> 1.68 ms FP32; without them 0.4 ms
// less; aligned or non-temporal stores do not help).  Before, one workgroup per
// (J, 64 rows) kept W in LDS and read C AO-major: one L1 request per lane (74% of
// the L1's cycles), and padding to 64 rows and 16 contraction indices.
// HP: the density P is given.  Otherwise P = 2 C C^T, and gv V_J P + beta C Z C^T
// = C (beta Z + 2 gv V_J 1) C^T takes the first term into phase 1 (FP64 only: the
// V P term of an FP32 product stays in FP64, from P).
template <int OC16, class R, bool HP>
__global__ __launch_bounds__(kThreads, 2) void k_grad_rows(GradRows g) {
  typedef typename R::T T;
  typedef typename R::T2 T2;
  typedef typename R::Acc Acc;
  constexpr int OC = 16 * OC16;
  constexpr int V = 16 / int(sizeof(T));                 // elements of a 16-byte piece
  constexpr int NP = OC * 32 / V;                        // pieces of a column tile
  constexpr int PN = (NP + kThreads - 1) / kThreads;     // and per thread (the last one not for all)
  typedef T VT __attribute__((ext_vector_type(V)));
  __shared__ __attribute__((aligned(16))) T sB[2][OC * 32];
  const int64_t nblk = gridDim.x;  // multiple of 8
  const int64_t item = (int64_t(blockIdx.x) & 7) * (nblk >> 3) + (int64_t(blockIdx.x) >> 3);
  if (item >= g.items) return;
  const int64_t jr = item / g.T;
  const int I = g.T - 1 - int(item - jr * g.T);
  const int tid = threadIdx.x, lane = tid & 63, m = lane & 15, gq = lane >> 4;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int o = g.o, ldz = g.ldz, ldt = g.n_pad;
  const T *__restrict__ ct = static_cast<const T *>(g.ct);
  // a vector past the last repeats it, its stores dropped (a resource of no records)
  const int64_t J = min(4 * jr + w, g.jn - 1);
  const double *__restrict__ zj = g.z + J * g.sz;
  const double vj = g.gv * g.v[J];
  const __amdgpu_buffer_rsrc_t rg =
      __builtin_amdgcn_make_buffer_rsrc(g.g + J * g.ldg, 0, 4 * jr + w < g.jn ? g.rowbytes : 0, kRsrcWord3);
  const __amdgpu_buffer_rsrc_t rp =
      __builtin_amdgcn_make_buffer_rsrc(const_cast<double *>(g.p), 0, g.rowbytes, kRsrcWord3);

  // column tile j of C^T: global -> registers -> LDS rows of 32
  VT rs[PN];
  auto fetch = [&](int j) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < PN; ++i) {
      const int e = min(tid + kThreads * i, NP - 1);
      rs[i] = *reinterpret_cast<const VT *>(ct + uint32_t(e / (32 / V)) * uint32_t(ldt) + uint32_t(32 * j + V * (e % (32 / V))));
    }
  };
  auto stash = [&](int buf) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < PN; ++i)
      if (kThreads * (i + 1) <= NP || tid + kThreads * i < NP)
        *reinterpret_cast<VT *>(&sB[buf][V * (tid + kThreads * i)]) = rs[i];
  };
  fetch(0);

  // ---- phase 1: acc1[t][i] = rows l = 16 t .., columns a = 32 I + 2 m + i of W^T
  Acc acc1[OC16][2];
#pragma unroll
  for (int t = 0; t < OC16; ++t)
#pragma unroll
    for (int i = 0; i < 2; ++i) acc1[t][i] = Acc{0, 0, 0, 0};
  {
    const int ns = (o + 3) / 4;  // steps of four contraction indices
    T zr[2][OC16];
    T2 cr[2];
    const T *__restrict__ ca = ct + gq * int64_t(ldt) + 32 * I + 2 * m;
    uint32_t zo[OC16];  // column l of this lane, clamped
#pragma unroll
    for (int t = 0; t < OC16; ++t) zo[t] = uint32_t(min(16 * t + m, o - 1));
    auto load = [&](int s, int st) __attribute__((always_inline)) {
      s = min(s, ns - 1);
      const uint32_t zrow = uint32_t(min(4 * s + gq, o - 1)) * uint32_t(ldz);
      cr[st] = *reinterpret_cast<const T2 *>(ca + 4 * s * int64_t(ldt));
#pragma unroll
      for (int t = 0; t < OC16; ++t) zr[st][t] = T(zj[zrow + zo[t]]);
    };
    auto mul = [&](int s, int st) __attribute__((always_inline)) {
      const int k = 4 * s + gq;
#pragma unroll
      for (int t = 0; t < OC16; ++t) {
        T z = zr[st][t];
        if constexpr (!HP) z = T(g.beta) * z + (k == 16 * t + m ? T(2.0 * vj) : T(0));
        const T a = k < o && 16 * t + m < o ? z : T(0);
        acc1[t][0] = R::mma(a, cr[st][0], acc1[t][0]);
        acc1[t][1] = R::mma(a, cr[st][1], acc1[t][1]);
      }
    };
    load(0, 0);
    load(1, 1);
    // two steps per trip (one past the last multiplies by zeros: a conditional
    // step would give the accumulators a second set of registers)
#pragma unroll 1
    for (int s = 0; s < ns; s += 2) {
      mul(s, 0);
      __builtin_amdgcn_sched_barrier(0);
      load(s + 2, 0);
      __builtin_amdgcn_sched_barrier(0);
      mul(s + 1, 1);
      __builtin_amdgcn_sched_barrier(0);
      load(s + 3, 1);
      __builtin_amdgcn_sched_barrier(0);
    }
  }

  // ---- phase 2
  // steps of a tile's last chunk that hold an index below nocc: step s has the
  // indices row(g, s), 4 s + g (FP64) or 4 g + s (FP32)
  const int left = o - 16 * (OC16 - 1), tail = R::kStep == 4 ? (left + 3) / 4 : min(left, 4);
  uint32_t ro[2][4];  // byte offset of this lane's first element in each of its rows
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const uint32_t a = uint32_t(32 * I + 2 * R::row(gq, r) + i);
      ro[i][r] = a < uint32_t(g.n) ? (a * (a + 1u) / 2u + uint32_t(2 * m)) * 8u : kMasked;
    }
  Acc acc2[2][2];
  // The contraction index of (step s, lane group) is the one phase 1 left in
  // register s: row(gq, s) of the chunk.
  auto chunks = [&](int buf) __attribute__((always_inline)) {
    constexpr int D = OC16 < 8 || sizeof(T) == 4 ? 4 : 2;  // steps of fragments in flight (registers)
    T2 bq[D];
    auto load_b = [&](int u, T2 &dst) __attribute__((always_inline)) {
      dst = *reinterpret_cast<const T2 *>(&sB[buf][(16 * (u / 4) + R::row(gq, u % 4)) * 32 + 2 * m]);
    };
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
      for (int h = 0; h < 2; ++h) acc2[i][h] = Acc{0, 0, 0, 0};
#pragma unroll
    for (int u = 0; u < D; ++u) load_b(u, bq[u]);
#pragma unroll
    for (int u = 0; u < 4 * OC16; ++u) {
      if (u < 4 * (OC16 - 1) || u - 4 * (OC16 - 1) < tail) {
#pragma unroll
        for (int i = 0; i < 2; ++i)
#pragma unroll
          for (int h = 0; h < 2; ++h) acc2[i][h] = R::mma(acc1[u / 4][i][u % 4], bq[u % D][h], acc2[i][h]);
      }
      __builtin_amdgcn_sched_barrier(0);
      if (u + D < 4 * OC16) load_b(u + D, bq[u % D]);
      __builtin_amdgcn_sched_barrier(0);
    }
  };
  // element before the factor 2 off the diagonal
  auto value = [&](int i, int h, int r, double p) __attribute__((always_inline)) {
    const double x = double(acc2[i][h][r]);
    if constexpr (HP) return vj * p + g.beta * x;
    else return x;
  };
  stash(0);
  __syncthreads();
#pragma unroll 1
  for (int j = 0; j < I; ++j) {  // tiles wholly below the diagonal
    fetch(j + 1);
    v4u pv[2][4];
    constexpr bool kLate = OC16 >= 7 && sizeof(T) == 8;  // no registers for the densities beside the products
    auto load_p = [&]() __attribute__((always_inline)) {
#pragma unroll
      for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int r = 0; r < 4; ++r)
          pv[i][r] = __builtin_amdgcn_raw_buffer_load_b128(rp, int(ro[i][r] + 256u * uint32_t(j)), 0, 0);
    };
    if constexpr (HP && !kLate) load_p();
    __builtin_amdgcn_sched_barrier(0);
    chunks(j & 1);
    __builtin_amdgcn_sched_barrier(0);
    stash((j + 1) & 1);
    __builtin_amdgcn_sched_barrier(0);
    if constexpr (HP && kLate) load_p();
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        v2d p = {0.0, 0.0};
        if constexpr (HP) p = __builtin_bit_cast(v2d, pv[i][r]);
        v2d x;
#pragma unroll
        for (int h = 0; h < 2; ++h) x[h] = 2.0 * value(i, h, r, p[h]);
        __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(v4u, x), rg, int(ro[i][r] + 256u * uint32_t(j)), 0, 0);
      }
    __syncthreads();
  }
  // the diagonal tile
  auto po = [&](int i, int h, int r) __attribute__((always_inline)) {
    return int(2 * R::row(gq, r) + i >= 2 * m + h ? ro[i][r] + 256u * uint32_t(I) + 8u * h : kMasked);
  };
  chunks(I & 1);
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const double f = 2 * R::row(gq, r) + i == 2 * m + h ? 1.0 : 2.0;
        double p = 0.0;
        if constexpr (HP) p = __builtin_bit_cast(double, __builtin_amdgcn_raw_buffer_load_b64(rp, po(i, h, r), 0, 0));
        const double x = f * value(i, h, r, p);
        __builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(v2u, x), rg, po(i, h, r), 0, 0);
      }
}

// ct[k * n_pad + a] = T(cb[a * ldc + k]) for k < rows, 32 x 32 blocks through LDS.
// grid = (n_pad / 32, ceil(rows / 32)), block 256.
template <typename T>
__global__ __launch_bounds__(kThreads) void k_bank_t(const double *__restrict__ cb, int ldc, int n_pad, int rows,
                                                    T *__restrict__ ct) {
  __shared__ double t[32][33];
  const int a0 = blockIdx.x * 32, k0 = blockIdx.y * 32, x = threadIdx.x & 31, y = threadIdx.x >> 5;
#pragma unroll
  for (int i = y; i < 32; i += 8)
    t[i][x] = k0 + x < ldc ? cb[int64_t(a0 + i) * ldc + k0 + x] : 0.0;
  __syncthreads();
#pragma unroll
  for (int i = y; i < 32; i += 8)
    if (k0 + i < rows) ct[int64_t(k0 + i) * n_pad + a0 + x] = T(t[x][i]);
}

template <int OC16>
void launch_grad_rows(Context *c, const GradRows &g, bool f32) {
  const dim3 grid(unsigned(round_up(g.items, 8)));
  if (f32) hipLaunchKernelGGL((k_grad_rows<OC16, GR32, true>), grid, dim3(kThreads), 0, c->stream, g);
  else if (g.p) hipLaunchKernelGGL((k_grad_rows<OC16, GR64, true>), grid, dim3(kThreads), 0, c->stream, g);
  else hipLaunchKernelGGL((k_grad_rows<OC16, GR64, false>), grid, dim3(kThreads), 0, c->stream, g);
}

// Whether the fused k_grad_rows takes this shape: nocc <= 128, 32-bit bank
// offsets, and a packed dL row under 2^31 bytes (the range of its buffer
// resources).  Other shapes form W = C Z first.
bool grad_rows_fits(const Context *c, int nocc, int ldc) {
  const int64_t rowbytes = int64_t(c->n) * (c->n + 1) / 2 * int64_t(sizeof(double));
  return (nocc + 15) / 16 <= 8 && int64_t(c->n_pad) * ldc < (int64_t(1) << 28) && rowbytes < (int64_t(1) << 31);
}

// The transposed bank of k_grad_rows in FP64 or FP32 (workspaces gbt / gb32) from
// the packed FP64 bank.
int bank_t(Context *c, int nocc, int ldc, bool f32) {
  const int rows = 16 * ((nocc + 15) / 16);
  DevBuf &buf = f32 ? c->w->gb32 : c->w->gbt;
  const int rc = ensure(c, buf, (f32 ? sizeof(float) : sizeof(double)) * size_t(rows) * c->n_pad);
  if (rc) return rc;
  const double *cb = static_cast<const double *>(c->w->cbank.ptr);
  const dim3 grid(unsigned(c->n_pad / 32), unsigned(ceil_div(rows, 32)));
  if (f32)
    hipLaunchKernelGGL(k_bank_t<float>, grid, dim3(kThreads), 0, c->stream, cb, ldc, c->n_pad, rows,
                       static_cast<float *>(buf.ptr));
  else
    hipLaunchKernelGGL(k_bank_t<double>, grid, dim3(kThreads), 0, c->stream, cb, ldc, c->n_pad, rows,
                       static_cast<double *>(buf.ptr));
  return hip_check(c, hipGetLastError(), "bank transpose launch");
}

// dL of the jn vectors from Z in one fused launch, with FP64 or FP32 products
// (bank_t() of that precision first); returns MJK_ERR_ARG when grad_rows_fits
// rejects the shape (the caller then forms W = C Z first).
int grad_rows(Context *c, int nocc, int ldc, const double *z, int64_t sz, int ldz, const double *v,
              const double *P, double alpha, double beta, double *dl, int64_t ldd, int64_t jn, bool f32) {
  const int oc16 = (nocc + 15) / 16;
  if (!grad_rows_fits(c, nocc, ldc)) return MJK_ERR_ARG;
  if (jn < 1) return MJK_OK;
  GradRows g{};
  g.rowbytes = int32_t(int64_t(c->n) * (c->n + 1) / 2 * int64_t(sizeof(double)));
  g.ct = f32 ? c->w->gb32.ptr : c->w->gbt.ptr;
  g.n_pad = c->n_pad;
  g.z = z;
  g.sz = sz;
  g.ldz = ldz;
  g.o = nocc;
  g.v = v;
  g.p = P;
  g.gv = alpha;
  g.beta = beta;
  g.g = dl;
  g.ldg = ldd;
  g.n = c->n;
  g.T = int(ceil_div(c->n, 32));
  g.jn = jn;
  g.items = int64_t(g.T) * ceil_div(jn, 4);
  switch (oc16) {
    case 1: launch_grad_rows<1>(c, g, f32); break;
    case 2: launch_grad_rows<2>(c, g, f32); break;
    case 3: launch_grad_rows<3>(c, g, f32); break;
    case 4: launch_grad_rows<4>(c, g, f32); break;
    case 5: launch_grad_rows<5>(c, g, f32); break;
    case 6: launch_grad_rows<6>(c, g, f32); break;
    case 7: launch_grad_rows<7>(c, g, f32); break;
    default: launch_grad_rows<8>(c, g, f32); break;
  }
  return MJK_OK;
}

// P = 2 C C^T in plain LT storage (the misc workspace) unless the caller gave it.
int density_or(Context *c, int nocc, const double *corb, const double *p_lt, const double **P) {
  *P = p_lt;
  if (p_lt) return MJK_OK;
  int rc;
  if ((rc = ensure(c, c->w->misc, sizeof(double) * size_t(c->np)))) return rc;
  double *pw = static_cast<double *>(c->w->misc.ptr);
  density_launch(c, corb, nocc, 2.0, 0, pw);
  *P = pw;
  return MJK_OK;
}

// ---- Z^J = X^J C, lower blocks only ------------------------------------------
// Z^J = C^T L^J C is symmetric, so only its 16 x 16 blocks (i, j), j <= i are
// multiplied (OC16 = ceil(nocc/16) block rows, so at most 15 padding rows
// instead of a 64-wide tile's 63) and each off-diagonal block is also written
// transposed.  One workgroup per vector.  The block rows are dealt to the four
// waves at compile time (largest first, each to the wave with the fewest
// blocks), so every fragment index is static.  Per 16-row contraction chunk
// the bank rows C[a0 .. a0+15][0 .. 16 OC16) go through LDS (double-buffered,
// one barrier per chunk); a wave's X fragments are one 32-byte load per block
// row, lane group g taking the contraction indices 4g .. 4g+3 in the four
// MFMA steps (the B reads from LDS use the same order).
struct ZPlan {
  int nrows[4];
  int rows[4][16];
  int nblk[4];
};

constexpr ZPlan zplan(int oc16) {
  ZPlan p{};
  for (int i = oc16 - 1; i >= 0; --i) {  // row i holds i + 1 lower blocks
    int best = 0;
    for (int w = 1; w < 4; ++w)
      if (p.nblk[w] < p.nblk[best]) best = w;
    p.rows[best][p.nrows[best]++] = i;
    p.nblk[best] += i + 1;
  }
  return p;
}

template <int OC16, typename TX>
__global__ __launch_bounds__(kThreads) void k_zsym(const TX *__restrict__ X, int64_t sx, int ldx,
                                                  const double *__restrict__ cb, int ldc, int n,
                                                  int o, double *__restrict__ z, int64_t sz,
                                                  int ldz) {
  constexpr int OC = 16 * OC16;
  constexpr ZPlan P = zplan(OC16);
  constexpr int CL = (16 * OC) / kThreads > 0 ? (16 * OC) / kThreads : 1;  // bank doubles per thread
  __shared__ double sC[2][16 * OC];
  const int64_t J = blockIdx.x;
  const TX *__restrict__ xj = X + J * sx;
  const int tid = threadIdx.x, lane = tid & 63, gq = lane >> 4, w = tid >> 6;
  const int nch = (n + 15) / 16;
  double rc[CL];
  auto fetch = [&](int a0) {
#pragma unroll
    for (int q = 0; q < CL; ++q) {
      const int e = tid + kThreads * q;  // 16 * OC is a multiple of 256 or below it
      rc[q] = e < 16 * OC ? cb[(a0 + e / OC) * int64_t(ldc) + e % OC] : 0.0;
    }
  };
  auto stash = [&](int buf) {
#pragma unroll
    for (int q = 0; q < CL; ++q) {
      const int e = tid + kThreads * q;
      if (e < 16 * OC) sC[buf][e] = rc[q];
    }
  };
  auto wave = [&](auto wc) {
    constexpr int W = decltype(wc)::value;
    constexpr int NR = P.nrows[W];
    v4d acc[NR > 0 ? NR : 1][OC16];
#pragma unroll
    for (int r = 0; r < NR; ++r)
#pragma unroll
      for (int j = 0; j < OC16; ++j) acc[r][j] = v4d{0.0, 0.0, 0.0, 0.0};
    typedef TX TX4 __attribute__((ext_vector_type(4)));
    TX4 xs[2][NR > 0 ? NR : 1];  // [stage]: X fragments of chunk c in stage c & 1
    auto loadx = [&](int a0, TX4 (&dst)[NR > 0 ? NR : 1]) __attribute__((always_inline)) {
#pragma unroll
      for (int r = 0; r < NR; ++r)
        dst[r] = *reinterpret_cast<const TX4 *>(xj + int64_t(16 * P.rows[W][r] + (lane & 15)) * ldx + a0 +
                                                4 * gq);
    };
    // Every chunk issues the same loads (the ones past the last chunk clamped
    // to it, never used) and the X stages are compile-time (the loop runs two
    // chunks per trip), so no register copy of a load in flight and no
    // conditional load leaves the compiler a wait for the whole memory queue.
    auto chunk = [&](int c, auto stage) __attribute__((always_inline)) {
      constexpr int S = decltype(stage)::value;  // = c & 1: X stage and LDS buffer
      loadx(16 * (c + 1 < nch ? c + 1 : nch - 1), xs[S ^ 1]);
#pragma unroll
      for (int ks = 0; ks < 4; ++ks) {
        const double *__restrict__ brow = sC[S] + (4 * gq + ks) * OC + (lane & 15);
#pragma unroll
        for (int r = 0; r < NR; ++r) {
          const double a = double(xs[S][r][ks]);
#pragma unroll
          for (int j = 0; j < OC16; ++j)
            if (j <= P.rows[W][r]) acc[r][j] = mfma64(a, brow[16 * j], acc[r][j]);
        }
      }
      stash(S ^ 1);
      fetch(16 * (c + 2 < nch ? c + 2 : nch - 1));
      __syncthreads();
    };
    fetch(0);
    stash(0);
    loadx(0, xs[0]);
    fetch(16 * (nch > 1 ? 1 : 0));
    __syncthreads();
    int c = 0;
    for (; c + 1 < nch; c += 2) {
      chunk(c, std::integral_constant<int, 0>{});
      chunk(c + 1, std::integral_constant<int, 1>{});
    }
    if (c < nch) chunk(c, std::integral_constant<int, 0>{});
    double *__restrict__ zj = z + J * sz;
#pragma unroll
    for (int r = 0; r < NR; ++r) {
      const int i = P.rows[W][r];
#pragma unroll
      for (int j = 0; j < OC16; ++j) {
        if (j > i) continue;
        const int l = 16 * j + (lane & 15);
#pragma unroll
        for (int rr = 0; rr < 4; ++rr) {
          const int k = 16 * i + 4 * rr + gq;
          if (k < o && l < o) {
            zj[int64_t(k) * ldz + l] = acc[r][j][rr];
            if (j < i) zj[int64_t(l) * ldz + k] = acc[r][j][rr];
          }
        }
      }
    }
  };
  // every wave runs the chunk loop (its barriers) even when it owns no rows
  switch (w) {
    case 0: wave(std::integral_constant<int, 0>{}); break;
    case 1: wave(std::integral_constant<int, 1>{}); break;
    case 2: wave(std::integral_constant<int, 2>{}); break;
    default: wave(std::integral_constant<int, 3>{}); break;
  }
}

template <int OC16, typename TX>
void launch_zsym(Context *c, const TX *X, int64_t sx, const double *cb, int ldc, int nocc, double *z,
                 int64_t sz, int ldz, int64_t jn) {
  hipLaunchKernelGGL((k_zsym<OC16, TX>), dim3(unsigned(jn)), dim3(kThreads), 0, c->stream, X, sx,
                     c->n_pad, cb, ldc, c->n, nocc, z, sz, ldz);
}

// Z^J = X^J C for jn vectors (X rows of n_pad, sx apart per vector; bank cb of
// row stride ldc), Z^J at z + J sz with row stride ldz; nocc <= 128.
template <typename TX>
int zsym(Context *c, const TX *X, int64_t sx, const double *cb, int ldc, int nocc, double *z,
         int64_t sz, int ldz, int64_t jn) {
  if (nocc < 1 || nocc > 128 || jn < 1) return MJK_ERR_ARG;
  if (ldc < 16 * ((nocc + 15) / 16)) return set_error(c, MJK_ERR_ARG, "zsym: bank narrower than the blocks");
  switch ((nocc + 15) / 16) {
    case 1: launch_zsym<1>(c, X, sx, cb, ldc, nocc, z, sz, ldz, jn); break;
    case 2: launch_zsym<2>(c, X, sx, cb, ldc, nocc, z, sz, ldz, jn); break;
    case 3: launch_zsym<3>(c, X, sx, cb, ldc, nocc, z, sz, ldz, jn); break;
    case 4: launch_zsym<4>(c, X, sx, cb, ldc, nocc, z, sz, ldz, jn); break;
    case 5: launch_zsym<5>(c, X, sx, cb, ldc, nocc, z, sz, ldz, jn); break;
    case 6: launch_zsym<6>(c, X, sx, cb, ldc, nocc, z, sz, ldz, jn); break;
    case 7: launch_zsym<7>(c, X, sx, cb, ldc, nocc, z, sz, ldz, jn); break;
    default: launch_zsym<8>(c, X, sx, cb, ldc, nocc, z, sz, ldz, jn); break;
  }
  return hip_check(c, hipGetLastError(), "zsym launch");
}

}  // namespace

// O[i][j] = sum_k A[i][k] B[j][k], one launch per block of rows of A and of B
// that the 32-bit offsets of the kernel reach.
int gemm_nt(Context *c, const double *A, int64_t lda, const double *B, int64_t ldb, double *O, int64_t ldo,
            int64_t m, int n, int k) {
  constexpr int64_t kMost = (int64_t(1) << 28) - 1;
  const int64_t mi = std::max<int64_t>(1, kMost / lda), mj = std::max<int64_t>(1, kMost / ldb);
  for (int64_t i = 0; i < m; i += mi)
    for (int64_t j = 0; j < n; j += mj) {
      GemmBatch g{};
      g.A = A + i * lda; g.lda = lda;
      g.B = B + j * ldb; g.ldb = ldb;
      g.O = O + i * ldo + j; g.ldo = ldo;
      g.m = int(std::min(mi, m - i)); g.n = int(std::min<int64_t>(mj, n - j)); g.k = k; g.alpha = 1.0;
      const int rc = gemm<true, 0>(c, g, 1);
      if (rc) return rc;
    }
  return hip_check(c, hipGetLastError(), "gemm launch");
}

int z_from_x(Context *c, const void *X, bool x_f32, int ldc, int nocc, int64_t jn, double *z) {
  const double *cb = static_cast<const double *>(c->w->cbank.ptr);
  const int64_t sx = int64_t(ldc) * c->n_pad, sz = int64_t(nocc) * nocc;
  if (nocc <= 128)
    return x_f32 ? zsym(c, static_cast<const float *>(X), sx, cb, ldc, nocc, z, sz, nocc, jn)
                 : zsym(c, static_cast<const double *>(X), sx, cb, ldc, nocc, z, sz, nocc, jn);
  GemmBatch g{};
  if (x_f32) g.A32 = static_cast<const float *>(X);
  else g.A = static_cast<const double *>(X);
  g.sA = int64_t(ldc) * c->n_pad; g.lda = c->n_pad;                          // X[J][k][a]
  g.B = static_cast<const double *>(c->w->cbank.ptr); g.sB = 0; g.ldb = ldc;  // C[a][l] (NN)
  g.O = z; g.sO = int64_t(nocc) * nocc; g.ldo = nocc;                         // Z[J][k][l]
  g.m = nocc; g.n = nocc; g.k = c->n; g.alpha = 1.0;
  if (x_f32) return gemm<false, 0, float>(c, g, int(jn));
  return gemm<false, 0>(c, g, int(jn));
}

}  // namespace mjk

using namespace mjk;

extern "C" int mjk_density(mjk_context *c, int32_t nocc, const double *corb, double scale,
                           double *dlt) {
  if (!c) return MJK_ERR_ARG;
  if (nocc < 0 || (nocc > 0 && !corb) || !dlt) return set_error(c, MJK_ERR_ARG, "density: bad arguments");
  if (nocc == 0)
    return fill_zero(c, dlt, sizeof(double) * size_t(c->np));
  phase_begin(c);
  density_launch(c, corb, nocc, scale, 1, dlt);
  phase_end(c, MJK_PHASE_PACK);
  return hip_check(c, hipGetLastError(), "density launch");
}

extern "C" int mjk_grad_orbitals(mjk_context *c, int32_t nocc, const double *corb,
                                 const double *flt, double scale, double *dc) {
  if (!c) return MJK_ERR_ARG;
  if (nocc < 1 || !corb || !flt || !dc) return set_error(c, MJK_ERR_ARG, "grad_orbitals: bad arguments");
  const int n = c->n;
  int rc;
  if ((rc = ensure(c, c->w->misc, sizeof(double) * size_t(n) * n))) return rc;
  double *fd = static_cast<double *>(c->w->misc.ptr);
  phase_begin(c);
  hipLaunchKernelGGL(k_unpack_lt, dim3(unsigned(n)), dim3(256), 0, c->stream, flt, n, fd, int64_t(n));
  GemmBatch g{};
  g.A = fd; g.sA = 0; g.lda = n;           // F[a][b]
  g.B = corb; g.sB = 0; g.ldb = nocc;      // C[b][k] (NN)
  g.O = dc; g.sO = 0; g.ldo = nocc;        // dC[a][k]
  g.m = n; g.n = nocc; g.k = n; g.alpha = scale;
  if ((rc = gemm<false, 0>(c, g, 1))) return rc;
  phase_end(c, MJK_PHASE_ASSEMBLY);
  return hip_check(c, hipGetLastError(), "grad_orbitals launch");
}

extern "C" int mjk_grad_vectors(mjk_context *c, int32_t nocc, const double *corb,
                                const double *p_lt, const double *v, double alpha, double beta,
                                double *dl, int64_t ldd) {
  if (!c) return MJK_ERR_ARG;
  if (nocc < 1 || nocc > 256 || !corb || !v || !dl || ldd < c->np)
    return set_error(c, MJK_ERR_ARG, "grad_vectors: bad arguments");
  if (c->nloaded != c->nchol)
    return set_error(c, MJK_ERR_SHORT_READ, "grad_vectors: not all Cholesky vectors were uploaded");
  const int n = c->n, n_pad = c->n_pad;
  const int64_t M = c->nchol;
  int rc;
  // bank with the orbitals (FP64), X chunk, Z and W per vector
  std::vector<int> off, opad;
  int ot = 0, tot = 0;
  const double *sets[1] = {corb};
  if ((rc = pack_bank(c, 1, &nocc, sets, off, opad, &ot, &tot))) return rc;
  const int ldc = 16 * ot;
  const double *cb = static_cast<const double *>(c->w->cbank.ptr);
  // per vector: X (ldc x n_pad) + Z (ldc x ldc) + W (n_pad x ldc)
  const int64_t per_vec = int64_t(ldc) * n_pad * 2 + int64_t(ldc) * ldc;
  int64_t jc = std::max<int64_t>(1, std::min<int64_t>(M, c->x_budget / (8 * per_vec)));
  const int64_t nchunk = ceil_div(M, jc);
  jc = ceil_div(M, nchunk);
  if ((rc = ensure(c, c->w->x, sizeof(double) * size_t(jc * per_vec)))) return rc;
  double *X = static_cast<double *>(c->w->x.ptr);
  double *Z = X + jc * ldc * int64_t(n_pad);
  double *W = Z + jc * ldc * int64_t(ldc);
  const double *P = p_lt;  // caller's plain LT; without one the fused kernel needs none, the two-GEMM form 2 C C^T
  if (grad_rows_fits(c, nocc, ldc)) {
    if ((rc = bank_t(c, nocc, ldc, false))) return rc;
  } else if ((rc = density_or(c, nocc, corb, p_lt, &P))) {
    return rc;
  }
  for (int64_t ch = 0; ch < nchunk; ++ch) {
    const int64_t j0 = ch * jc, jn = std::min(jc, M - j0);
    phase_begin(c);
    ht_launch(c, tot, cb, j0, jn, X);  // X[J][k][a] = (C^T L^J)[k][a]
    phase_end(c, MJK_PHASE_HALF_TRANSFORM);
    phase_begin(c);
    GemmBatch g{};
    // Z[J] = X[J] C   (o x o), the same kernel as the forward's saved Z
    if (nocc <= 128) {
      if ((rc = zsym(c, static_cast<const double *>(X), int64_t(ldc) * n_pad, cb, ldc, nocc, Z,
                     int64_t(ldc) * ldc, ldc, jn)))
        return rc;
    } else {
      g.A = X; g.sA = int64_t(ldc) * n_pad; g.lda = n_pad;
      g.B = cb; g.sB = 0; g.ldb = ldc;
      g.O = Z; g.sO = int64_t(ldc) * ldc; g.ldo = ldc;
      g.m = nocc; g.n = nocc; g.k = n; g.alpha = 1.0;
      if ((rc = gemm<false, 0>(c, g, int(jn)))) return rc;
    }
    // dL[J] = s * (alpha V_J P + beta C Z[J] C^T), lower triangle, packed
    if (grad_rows(c, nocc, ldc, Z, int64_t(ldc) * ldc, ldc, v + j0, P, alpha, beta, dl + j0 * ldd,
                  ldd, jn, false) != MJK_OK) {  // nocc > 128: W = C Z first
      g = GemmBatch{};
      g.A = cb; g.sA = 0; g.lda = ldc;
      g.B = Z; g.sB = int64_t(ldc) * ldc; g.ldb = ldc;
      g.O = W; g.sO = int64_t(n_pad) * ldc; g.ldo = ldc;
      g.m = n; g.n = nocc; g.k = nocc; g.alpha = 1.0;
      if ((rc = gemm<false, 0>(c, g, int(jn)))) return rc;
      if ((rc = grad_from_w(c, nocc, W, ldc, v + j0, P, alpha, beta, dl + j0 * ldd, ldd, jn))) return rc;
    }
    phase_end(c, MJK_PHASE_BACKWARD);
  }
  return hip_check(c, hipGetLastError(), "grad_vectors launch");
}

namespace {
// dE/dL from a given Z; vectors [j_fp32, M) take FP32 products (nocc <= 128).
int grad_vectors_z_impl(Context *c, int32_t nocc, const double *corb, const double *p_lt,
                        const double *v, const double *z, double alpha, double beta, double *dl,
                        int64_t ldd, int64_t j_fp32, const char *who) {
  if (!c) return MJK_ERR_ARG;
  if (nocc < 1 || nocc > 256 || !corb || !v || !z || !dl || ldd < c->np)
    return set_error(c, MJK_ERR_ARG, std::string(who) + ": bad arguments");
  const int n_pad = c->n_pad;
  const int64_t M = c->nchol;
  if (j_fp32 < 0 || j_fp32 > M) return set_error(c, MJK_ERR_ARG, std::string(who) + ": split outside [0, nchol]");
  int rc;
  std::vector<int> off, opad;
  int ot = 0, tot = 0;
  const double *sets[1] = {corb};
  if ((rc = pack_bank(c, 1, &nocc, sets, off, opad, &ot, &tot))) return rc;
  const int ldc = 16 * ot;
  const double *cb = static_cast<const double *>(c->w->cbank.ptr);
  if (grad_rows_fits(c, nocc, ldc)) {  // one fused launch per precision: W = C Z stays on chip
    const double *P = p_lt;
    if (j_fp32 < M && (rc = density_or(c, nocc, corb, p_lt, &P))) return rc;
    if (j_fp32 > 0 && (rc = bank_t(c, nocc, ldc, false))) return rc;
    if (j_fp32 < M && (rc = bank_t(c, nocc, ldc, true))) return rc;
    const int64_t sz = int64_t(nocc) * nocc;
    phase_begin(c);
    if ((rc = grad_rows(c, nocc, ldc, z, sz, nocc, v, p_lt, alpha, beta, dl, ldd, j_fp32, false)) ||
        (rc = grad_rows(c, nocc, ldc, z + j_fp32 * sz, sz, nocc, v + j_fp32, P, alpha, beta,
                        dl + j_fp32 * ldd, ldd, M - j_fp32, true)))
      return set_error(c, rc, std::string(who) + ": fused gradient launch");
    phase_end(c, MJK_PHASE_BACKWARD);
    return hip_check(c, hipGetLastError(), "grad_vectors_z launch");
  }
  // per vector: W = C Z (n_pad x ldc)
  const int64_t per_vec = int64_t(n_pad) * ldc;
  int64_t jc = std::max<int64_t>(1, std::min<int64_t>(M, c->x_budget / (8 * per_vec)));
  const int64_t nchunk = ceil_div(M, jc);
  jc = ceil_div(M, nchunk);
  if ((rc = ensure(c, c->w->x, sizeof(double) * size_t(jc * per_vec)))) return rc;
  double *W = static_cast<double *>(c->w->x.ptr);
  const double *P = nullptr;
  if ((rc = density_or(c, nocc, corb, p_lt, &P))) return rc;
  for (int64_t ch = 0; ch < nchunk; ++ch) {
    const int64_t j0 = ch * jc, jn = std::min(jc, M - j0);
    phase_begin(c);
    GemmBatch g{};
    // W[J] = C Z[J]   (n x o), Z dense nocc x nocc per vector
    g.A = cb; g.sA = 0; g.lda = ldc;
    g.B = z + j0 * int64_t(nocc) * nocc; g.sB = int64_t(nocc) * nocc; g.ldb = nocc;
    g.O = W; g.sO = per_vec; g.ldo = ldc;
    g.m = c->n; g.n = nocc; g.k = nocc; g.alpha = 1.0;
    if ((rc = gemm<false, 0>(c, g, int(jn)))) return rc;
    if ((rc = grad_from_w(c, nocc, W, ldc, v + j0, P, alpha, beta, dl + j0 * ldd, ldd, jn))) return rc;
    phase_end(c, MJK_PHASE_BACKWARD);
  }
  return hip_check(c, hipGetLastError(), "grad_vectors_z launch");
}
}  // namespace

extern "C" int mjk_grad_vectors_z(mjk_context *c, int32_t nocc, const double *corb,
                                  const double *p_lt, const double *v, const double *z,
                                  double alpha, double beta, double *dl, int64_t ldd) {
  if (!c) return MJK_ERR_ARG;
  return grad_vectors_z_impl(c, nocc, corb, p_lt, v, z, alpha, beta, dl, ldd, c->nchol, "grad_vectors_z");
}

extern "C" int mjk_grad_vectors_z_mixed(mjk_context *c, int32_t nocc, const double *corb,
                                        const double *p_lt, const double *v, const double *z,
                                        double alpha, double beta, double *dl, int64_t ldd,
                                        int64_t j_fp32) {
  if (!c) return MJK_ERR_ARG;
  return grad_vectors_z_impl(c, nocc, corb, p_lt, v, z, alpha, beta, dl, ldd, j_fp32, "grad_vectors_z_mixed");
}
