// (pw|xy) integrals of the CASSCF Fock build.
//
// Reference: src/fock_util/cho_fmcscf.F90:403-487 and
// src/fock_util/cho_eval_waxy.F90:12-150 (nSym = 1):
//   L(v,b,J)  = sum_a C(v,a) L_ab,J              (CHO_VTRA iSwap = 0)
//   Lxy(J)    = sum_b L(x,b,J) C(y,b), x <= y    (DGEMM_Tri 'N','T')
//   Scr(w,a,xy) += sum_J L(w,a,J) Lxy(J)          (DGEMM over the batch)
//   W(p,w,xy) = sum_a CMO(a,nfro+p) Scr(w,a,xy)   (after the last batch)
// The first step is the exchange half-transform Y with the active orbitals as
// the only bank set, the second the Z = X C product of the exchange (all (x, y),
// symmetric), the third k_scr below and the last one GEMM.
#include "mjk_internal.h"

namespace mjk {
namespace {

constexpr int kThreads = 256;
constexpr int kTile = 64;
constexpr int kSlot = kTile * kTile;
constexpr int kD = 4;  // contraction steps in flight per wave

__device__ inline v4d mfma64(double a, double b, v4d c) {
  return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
}

// Partial Scr(xy, w, a) = sum_J Z[J][x][y] Y[J][w][a] over one slice of the
// chunk's vectors: workgroup = (64 pairs xy, orbital w, 64 AOs a, slice), its four
// waves taking the slice's steps of four vectors in turn, each accumulating the
// whole tile, summed through LDS once at the end.  Both operands go from memory
// into the MFMA registers: lane 16 g + m loads row J + g, columns 32 i + 2 m + c
// of Y (16 bytes) and pair 16 t + m of Z.  Bound by latency at the sizes in use
// (n=301 nchol=1505 10 active: 0.85 ms as per-thread FMA loops over all vectors,
// now 0.03 ms).  part[(slice * tiles + tile) * 4096 + 256 (4 t + 2 i + c) + 64 r + lane].
// One slice only: scr set, (+)= in place.
// grid = (tiles, slices), tile = (xt * na + w) * nat + at.
__global__ __launch_bounds__(kThreads, 2) void k_scr(const double *__restrict__ Y, int ldc, int n_pad, int na,
                                                  int nat, int64_t jn, const double *__restrict__ Z, int nxy,
                                                  double *__restrict__ part, bool add, double *__restrict__ scr) {
  __shared__ double red[4][4][4][64];
  const int tile = blockIdx.x, at = tile % nat, w = (tile / nat) % na, xt = tile / (nat * na);
  const int tid = threadIdx.x, lane = tid & 63, wv = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int m = lane & 15, g = lane >> 4;
  const int64_t jper = (jn + gridDim.y - 1) / gridDim.y, ja = blockIdx.y * jper, jz = min(jn, ja + jper);
  const int nst = jz > ja ? int((jz - ja + 3) / 4) : 0;
  const int ntt = min(4, (nxy - kTile * xt + 15) / 16);  // 16-pair tiles with pairs in them
  int zo[4];  // Z offset of this lane's pairs, clamped
#pragma unroll
  for (int t = 0; t < 4; ++t) {
    const int xy = min(kTile * xt + 16 * t + m, nxy - 1);
    int y = int((sqrt(8.0 * xy + 1.0) - 1.0) * 0.5);
    while (y * (y + 1) / 2 > xy) --y;
    while ((y + 1) * (y + 2) / 2 <= xy) ++y;
    zo[t] = (xy - y * (y + 1) / 2) * na + y;
  }
  v4d acc[4][4];
#pragma unroll
  for (int t = 0; t < 4; ++t)
#pragma unroll
    for (int j = 0; j < 4; ++j) acc[t][j] = v4d{0.0, 0.0, 0.0, 0.0};
  const int64_t ys = int64_t(ldc) * n_pad, zs = int64_t(na) * na;
  const double *__restrict__ y0 = Y + int64_t(w) * n_pad + kTile * at + 2 * m;
  const int ns = nst > wv ? (nst - wv + 3) / 4 : 0;
  if (ns > 0) {
    double za[kD][4];
    v2d yb[kD][2];
    auto load = [&](int i, int st) __attribute__((always_inline)) {
      const int64_t J = min(ja + 4 * (wv + 4 * int64_t(min(i, ns - 1))) + g, jz - 1);
      const double *__restrict__ yr = y0 + J * ys, *__restrict__ zr = Z + J * zs;
#pragma unroll
      for (int t = 0; t < 4; ++t) za[st][t] = zr[zo[t]];
#pragma unroll
      for (int h = 0; h < 2; ++h) yb[st][h] = *reinterpret_cast<const v2d *>(yr + 32 * h);
    };
    auto mul = [&](int i, int st) __attribute__((always_inline)) {
      const bool in = ja + 4 * (wv + 4 * int64_t(i)) + g < jz;  // rows past the slice count as zero
#pragma unroll
      for (int t = 0; t < 4; ++t) {
        if (t >= ntt) break;
        const double a = in ? za[st][t] : 0.0;
#pragma unroll
        for (int j = 0; j < 4; ++j) acc[t][j] = mfma64(a, in ? yb[st][j >> 1][j & 1] : 0.0, acc[t][j]);
      }
    };
#pragma unroll
    for (int st = 0; st < kD; ++st) load(st, st);
    for (int i = 0; i < ns; i += kD) {
#pragma unroll
      for (int st = 0; st < kD; ++st) {
        if (i + st < ns) mul(i + st, st);
        load(i + st + kD, st);
      }
    }
  }
  double *__restrict__ out = part + (int64_t(blockIdx.y) * gridDim.x + tile) * kSlot + lane;
#pragma unroll
  for (int t = 0; t < 4; ++t) {
    if (t) __syncthreads();
#pragma unroll
    for (int j = 0; j < 4; ++j)
#pragma unroll
      for (int r = 0; r < 4; ++r) red[wv][j][r][lane] = acc[t][j][r];
    __syncthreads();
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const double v = ((red[0][wv][r][lane] + red[1][wv][r][lane]) + red[2][wv][r][lane]) + red[3][wv][r][lane];
      if (scr) {
        const int xy = kTile * xt + 16 * t + 4 * r + g;
        if (xy < nxy) {
          double *__restrict__ o =
              scr + (int64_t(xy) * na + w) * n_pad + kTile * at + 32 * (wv >> 1) + 2 * m + (wv & 1);
          *o = add ? *o + v : v;
        }
      } else {
        out[256 * (4 * t + wv) + 64 * r] = v;
      }
    }
  }
}

// scr[(xy * na + w) * n_pad + a] (+)= the slices of one chunk in order.
// grid = tiles, block 256.
__global__ __launch_bounds__(kThreads) void k_scr_sum(const double *__restrict__ part, int slices, int n_pad, int na,
                                                      int nat, int nxy, bool add, double *__restrict__ scr) {
  const int tile = blockIdx.x, at = tile % nat, w = (tile / nat) % na, xt = tile / (nat * na);
  const int64_t stride = int64_t(gridDim.x) * kSlot;
  for (int e = threadIdx.x; e < kSlot; e += kThreads) {
    const int q = e >> 8, r = (e >> 6) & 3, lane = e & 63, t = q >> 2, j = q & 3;
    const int xy = kTile * xt + 16 * t + 4 * r + (lane >> 4);
    const int a = kTile * at + 32 * (j >> 1) + 2 * (lane & 15) + (j & 1);
    if (xy >= nxy) continue;
    double *__restrict__ o = scr + (int64_t(xy) * na + w) * n_pad + a;
    const double *__restrict__ src = part + int64_t(tile) * kSlot + e;
    double s = add ? *o : 0.0;
    int k = 0;
    for (; k + 8 <= slices; k += 8) {
      double v[8];
#pragma unroll
      for (int u = 0; u < 8; ++u) v[u] = src[(k + u) * stride];
#pragma unroll
      for (int u = 0; u < 8; ++u) s += v[u];
    }
    for (; k < slices; ++k) s += src[k * stride];
    *o = s;
  }
}

}  // namespace
}  // namespace mjk

using namespace mjk;

extern "C" int mjk_puvx(mjk_context *c, int32_t naorb, const double *porb3, const double *cmo,
                        int32_t nfro, int32_t norb, double *w) {
  if (!c) return MJK_ERR_ARG;
  if (naorb < 1 || naorb > 256 || !porb3 || !cmo || !w || nfro < 0 || norb < 0 ||
      nfro + norb > c->n)
    return set_error(c, MJK_ERR_ARG, "puvx: bad arguments");
  if (c->nloaded != c->nchol)
    return set_error(c, MJK_ERR_SHORT_READ, "puvx: not all Cholesky vectors were uploaded");
  const int n = c->n, n_pad = c->n_pad;
  const int nxy = naorb * (naorb + 1) / 2;
  const int64_t M = c->nchol;
  int rc;
  std::vector<int> off, opad;
  int ot = 0, tot = 0;
  const double *sets[1] = {porb3};
  if ((rc = pack_bank(c, 1, &naorb, sets, off, opad, &ot, &tot))) return rc;
  const int ldc = 16 * ot;
  const double *cb = static_cast<const double *>(c->w->cbank.ptr);
  const int64_t yvec = sizeof(double) * int64_t(ldc) * n_pad;
  int64_t jc = std::max<int64_t>(1, std::min<int64_t>(M, c->x_budget / yvec));
  const int64_t nchunk = ceil_div(M, jc);
  jc = ceil_div(M, nchunk);
  if ((rc = ensure(c, c->w->x, size_t(yvec * jc)))) return rc;
  double *Y = static_cast<double *>(c->w->x.ptr);
  // Scr and, per chunk, Z = Y C (naorb x naorb per vector) and the slices' partial
  // tiles: about two workgroups per CU, slices of at least 16 steps of four vectors
  const size_t scr_n = size_t(nxy) * naorb * n_pad, z_n = size_t(jc) * naorb * naorb;
  const int nat = int(ceil_div(n, kTile));
  const int64_t tiles = ceil_div(nxy, kTile) * naorb * nat;
  const int slices = int(std::max<int64_t>(1, std::min<int64_t>(2 * int64_t(c->ncu) / tiles, jc / 64)));
  if (tiles > (int64_t(1) << 30)) return set_error(c, MJK_ERR_ARG, "puvx: too many active orbitals");
  const size_t part_n = slices > 1 ? size_t(tiles) * slices * kSlot : 0;
  if ((rc = ensure(c, c->w->k, sizeof(double) * (scr_n + z_n + part_n)))) return rc;
  double *scr = static_cast<double *>(c->w->k.ptr);
  double *z = scr + scr_n, *part = z + z_n;
  for (int64_t ch = 0; ch < nchunk; ++ch) {
    const int64_t j0 = ch * jc, jn = std::min(jc, M - j0);
    phase_begin(c);
    ht_launch(c, tot, cb, j0, jn, Y);
    phase_end(c, MJK_PHASE_HALF_TRANSFORM);
    phase_begin(c);
    if ((rc = z_from_x(c, Y, false, ldc, naorb, jn, z))) return rc;
    hipLaunchKernelGGL(k_scr, dim3(unsigned(tiles), unsigned(slices)), dim3(kThreads), 0, c->stream, Y, ldc, n_pad,
                       naorb, nat, jn, z, nxy, part, ch > 0, slices > 1 ? nullptr : scr);
    if (slices > 1)
      hipLaunchKernelGGL(k_scr_sum, dim3(unsigned(tiles)), dim3(kThreads), 0, c->stream, part, slices, n_pad, naorb,
                         nat, nxy, ch > 0, scr);
    phase_end(c, MJK_PHASE_EXCHANGE);
  }
  // W(p, w, xy): rows (xy, w) of Scr times CMO
  phase_begin(c);
  if (norb > 0 && (rc = gemm_nt(c, scr, n_pad, cmo + int64_t(n) * nfro, n, w, norb, int64_t(nxy) * naorb, norb, n)))
    return rc;
  phase_end(c, MJK_PHASE_ASSEMBLY);
  return hip_check(c, hipGetLastError(), "puvx launch");
}
