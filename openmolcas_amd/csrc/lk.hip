// Reference-form LK screening of the exchange: the per-orbital shell lists,
// vector-pair and shell-pair cuts of CHO_LK_SCF (src/fock_util/
// cho_lk_scf.F90:143-171,547-627,659-830) and CHO_LK_CASSCF (src/fock_util/
// cho_lk_casscf.F90:164-200,604-930), on the device.
//
// The reference decides, per batch of at most 25 vectors of one reduced set
// and per orbital k, which shells a are listed (Y = sqrt|D| |C_k|, its
// largest element per shell MLk, a cut on MLk), which shell pairs (a, b) enter
// the half-transform X_k = L C_k (sqrt|SumAClk(b,k) SvShp(ab)| >= thrv), and
// which K blocks (a >= b) receive X_k,a X_k,b^T (MLk(a) MLk(b) >= tau,
// sqrt|Faa(a) Faa(b)| >= tau/MaxRed, Keep flags).  The same decisions are
// made here.  Between two evaluations of the shell lists (DoScreen) the batches
// do not depend on each other, so a group of batches goes through each kernel
// together; the decisions of one orbital become one bit of a 64-bit word, a word
// per (shell, shell) and 64 orbitals, which a wave forms with one ballot:
//   - the half-transform takes one shell a at a time, because for a fixed a the
//     mask depends on (orbital, b) only and can be applied to the orbital
//     operand: X_k(J, a) = sum_b [m C](k, b) L_J(a, b) is an MFMA product with
//     columns (J, a in the shell); steps of four b no orbital needs are left out;
//   - the K kernel forms S_k = sum_J X_k X_k^T of one orbital on a 32 x 32 tile
//     by MFMA and adds it under the mask of (orbital, shell a, shell b),
//     skipping orbitals whose mask is empty on the tile;
//   - decision quantities (diagonal, SvShp, SumAClk, Y, Faa) are evaluated
//     without FMA contraction, in the reference's summation order where it
//     has one, so the cuts fall where the reference's fall.
// Measured on a chain of 48 atoms (n=240, nchol=1200 in 48 batches, 48 orbitals),
// whole call: 33.2 -> 0.96 ms.  One batch at a time, each kernel had 10-144
// workgroups of serial work (K 0.35 ms per batch, half-transform 0.14, lists
// 0.06, norms 0.05); now per call 0.04, 0.18 (bound by its gathered loads of L,
// one cache line per lane), 0.13 (masks, bound by their scalar loads), 0.11
// (reads L once), K-block masks 0.09.  The MFMA sums run in the order of the
// scalar loops they replace: the result is bit for bit the same.
// The selection sort of the reference (:602-627) keeps the shells whose MLk
// passes the cut, in decreasing MLk order, stopping at the first failure;
// because the values along the sorted list do not increase and rounding is
// monotone, that set is exactly {s : MLk(s) max MLk >= tau} (SCF) or
// {s : MLk(s) >= sqrt(tau)} (CASSCF), which is what the list kernel forms.
#include <cmath>
#include <limits>
#include <utility>

#include "mjk_internal.h"

namespace mjk {
namespace {

constexpr int kLkBatch = 25;  // Cho_LK_MaxVecPerBatch (src/fock_util/cho_lk_maxvecperbatch.F90:30)
constexpr int kLkThreads = 256;
constexpr int kHtCols = 48;   // columns (J, a) of one half-transform wave
constexpr int kHtPanel = 1024;  // contraction indices b listed at a time

__device__ __forceinline__ int64_t shp_idx(int a, int b) {
  return a >= b ? int64_t(a) * (a + 1) / 2 + b : int64_t(b) * (b + 1) / 2 + a;
}

// One or two densities: orbital counts, first global orbital index, device
// orbital matrices (orbital-major), thresholds.  Mask words: density d owns the
// words q0[d] .. q0[d+1]-1, word q the orbitals 64 (q - q0[d]) .. of it.
struct LkDens {
  int nd;
  int nocc[2];
  int k0[2];           // global orbital offset of density d
  int q0[3];
  const double *c[2];  // C_d(b, k) at k + nocc[d]*b
  double tau[2], xtau[2];
  double thrv2[2];     // least x with sqrt(x) >= thrv
  double tk2[2];       // least x with sqrt(x) >= tau / MaxRed
  int ktot;            // sum of nocc
  int nq;              // words
};

// The batches of one group.
struct LkGroup {
  int nb;
  int64_t j0[kLkGroup];
  int jnum[kLkGroup];
  const uint8_t *present[kLkGroup];  // shell-pair occupancy of the batch's reduced set
};

__device__ __forceinline__ void dk_of(const LkDens &D, int g, int *d, int *k) {
  *d = (D.nd > 1 && g >= D.k0[1]) ? 1 : 0;
  *k = g - D.k0[*d];
}
__device__ __forceinline__ int d_of_word(const LkDens &D, int q) { return D.nd > 1 && q >= D.q0[1] ? 1 : 0; }
// Row length and position of orbital k of density d in the arrays that hold one
// value per (shell, orbital), orbital fastest, words aligned.
__device__ __forceinline__ int kpos(const LkDens &D, int d, int k) { return 64 * D.q0[d] + k; }

#pragma clang fp contract(off)

// Estimate: diag(p) = sum_J L_J(p)^2 of the batch (cho_lk_scf.F90:461-479).
__global__ void k_lk_est_diag(const double *__restrict__ L, int64_t ldl, int64_t j0, int jnum,
                              int64_t np, double *__restrict__ diag) {
  for (int64_t p = int64_t(blockIdx.x) * blockDim.x + threadIdx.x; p < np;
       p += int64_t(gridDim.x) * blockDim.x) {
    double s = 0.0;
    for (int j = 0; j < jnum; ++j) {
      const double v = L[(j0 + j) * ldl + p];
      s = s + v * v;
    }
    diag[p] = s;
  }
}

// Update: diag(p) = diag(p) - L_J(p)^2, vector by vector (:834-880).
__global__ void k_lk_update_diag(const double *__restrict__ L, int64_t ldl, int64_t j0, int jnum,
                                 int64_t np, double *__restrict__ diag) {
  for (int64_t p = int64_t(blockIdx.x) * blockDim.x + threadIdx.x; p < np;
       p += int64_t(gridDim.x) * blockDim.x) {
    double dv = diag[p];
    for (int j = 0; j < jnum; ++j) {
      const double v = L[(j0 + j) * ldl + p];
      dv = dv - v * v;
    }
    diag[p] = dv;
  }
}

// SvShp(ab) = max_J sum_{p in shell pair ab} L_J(p)^2 (CHO_GetShFull,
// src/fock_util/cho_getshfull.F90:48-96).  Small shells (kSmallShell functions
// at most): one lane per shell pair, a wave the pairs of one shell a with 64
// shells b, whose packed elements are neighbours in the rows of a.  grid =
// (shells a, ceil(nshell / 256), batches).
constexpr int kSmallShell = 8;
__global__ __launch_bounds__(kLkThreads) void k_lk_svshp(const double *__restrict__ L, int64_t ldl,
                                                         const LkGroup G, int nshell,
                                                         const int32_t *__restrict__ koff,
                                                         const int32_t *__restrict__ nbsh,
                                                         double *__restrict__ svall) {
  constexpr int U = 5;  // vectors in flight
  const int sa = blockIdx.x, sb = blockIdx.y * kLkThreads + threadIdx.x, bt = blockIdx.z;
  if (sb > sa) return;
  const int na = nbsh[sa], nb = nbsh[sb], a0 = koff[sa], b0 = koff[sb];
  const double *__restrict__ base = L + G.j0[bt] * ldl;
  const int jnum = G.jnum[bt];
  double best = 0.0;
  for (int j = 0; j < jnum; j += U) {
    double s[U] = {};
    for (int al = 0; al < na; ++al) {
      const int64_t row = int64_t(a0 + al) * (a0 + al + 1) / 2 + b0;
      const int nbe = sa == sb ? al + 1 : nb;
      for (int bl = 0; bl < nbe; ++bl) {
#pragma unroll
        for (int u = 0; u < U; ++u) {
          const double v = base[(j + u < jnum ? j + u : j) * ldl + row + bl];
          s[u] = s[u] + v * v;
        }
      }
    }
#pragma unroll
    for (int u = 0; u < U; ++u) best = s[u] > best ? s[u] : best;  // max(SvShp(:,1), SvShp(:,2))
  }
  svall[bt * (int64_t(nshell) * (nshell + 1) / 2) + shp_idx(sa, sb)] = best;
}

// The same for shells of any size: one wave per shell pair.  grid = (pairs / 4,
// batches).
__global__ __launch_bounds__(kLkThreads) void k_lk_svshp_wave(const double *__restrict__ L, int64_t ldl,
                                                              const LkGroup G, int nshell,
                                                              const int32_t *__restrict__ koff,
                                                              const int32_t *__restrict__ nbsh,
                                                              double *__restrict__ svall) {
  const int lane = threadIdx.x & 63, bt = blockIdx.y;
  const int64_t nshp = int64_t(nshell) * (nshell + 1) / 2;
  const int64_t p = int64_t(blockIdx.x) * (kLkThreads / 64) + (threadIdx.x >> 6);
  if (p >= nshp) return;
  int sa = int((sqrt(8.0 * double(p) + 1.0) - 1.0) * 0.5);
  while (int64_t(sa) * (sa + 1) / 2 > p) --sa;
  while (int64_t(sa + 1) * (sa + 2) / 2 <= p) ++sa;
  const int sb = int(p - int64_t(sa) * (sa + 1) / 2);
  const int na = nbsh[sa], nb = nbsh[sb], a0 = koff[sa], b0 = koff[sb];
  double best = 0.0;
  for (int j = 0; j < G.jnum[bt]; ++j) {
    const double *__restrict__ row = L + (G.j0[bt] + j) * ldl;
    double s = 0.0;
    for (int al = 0; al < na; ++al) {
      const int64_t a = a0 + al;
      const int nbe = sa == sb ? al + 1 : nb;
      for (int bl = lane; bl < nbe; bl += 64) {
        const double v = row[a * (a + 1) / 2 + b0 + bl];
        s = s + v * v;
      }
    }
    for (int off = 32; off > 0; off >>= 1) s = s + __shfl_xor(s, off, 64);
    best = s > best ? s : best;
  }
  if (lane == 0) svall[bt * nshp + p] = best;
}

// DH(a,b) = DH(b,a) = sqrt|D(ab)| (swap_tosqrt, src/fock_util/swap_tosqrt.F90:57-72).
__global__ void k_lk_diah(const double *__restrict__ diag, int n, double *__restrict__ dh) {
  const int a = blockIdx.x;
  for (int b = threadIdx.x; b <= a; b += blockDim.x) {
    const double v = sqrt(fabs(diag[int64_t(a) * (a + 1) / 2 + b]));
    dh[int64_t(a) * n + b] = v;
    dh[int64_t(b) * n + a] = v;
  }
}

// SumAClk(s,k) = sum_{i in s} C(i,k)^2 (cho_lk_scf.F90:235-253), at
// sumac[s * 64 nq + kpos].
__global__ void k_lk_sumac(LkDens D, int nshell, const int32_t *__restrict__ koff,
                           const int32_t *__restrict__ nbsh, double *__restrict__ sumac) {
  int d, k;
  dk_of(D, blockIdx.x, &d, &k);
  const double *c = D.c[d];
  const int no = D.nocc[d];
  for (int s = threadIdx.x; s < nshell; s += blockDim.x) {
    double t = 0.0;
    for (int i = 0; i < nbsh[s]; ++i) {
      const double v = c[k + int64_t(no) * (koff[s] + i)];
      t = t + v * v;
    }
    sumac[int64_t(s) * 64 * D.nq + kpos(D, d, k)] = t;
  }
}

// Per orbital (one workgroup each): Y = DH |C_k| (DGEMV 'N', :584-590), MLk per
// shell, the listed shells (:602-627).
__global__ __launch_bounds__(kLkThreads) void k_lk_screen(
    LkDens D, int n, int nshell, int cas_cut, const int32_t *__restrict__ koff,
    const int32_t *__restrict__ nbsh, const double *__restrict__ dh, double *__restrict__ ylk,
    double *__restrict__ mlk, uint8_t *__restrict__ listed, unsigned long long *__restrict__ stats) {
  constexpr int U = 16;  // rows of DH in flight
  __shared__ double red[kLkThreads / 64];
  __shared__ unsigned long long cnt;
  const int g = blockIdx.x;
  int d, k;
  dk_of(D, g, &d, &k);
  const int64_t ld = 64 * int64_t(D.nq);
  const int kp = kpos(D, d, k);
  if (threadIdx.x == 0) cnt = 0;
  const double *c = D.c[d];
  const int no = D.nocc[d];
  double *y = ylk + int64_t(g) * n;
  for (int l = threadIdx.x; l < n; l += blockDim.x) {
    double s = 0.0;
    int m = 0;
    for (; m + U <= n; m += U) {
      double v[U];
#pragma unroll
      for (int u = 0; u < U; ++u) v[u] = dh[int64_t(m + u) * n + l];
#pragma unroll
      for (int u = 0; u < U; ++u) s = s + v[u] * fabs(c[k + int64_t(no) * (m + u)]);
    }
    for (; m < n; ++m) s = s + dh[int64_t(m) * n + l] * fabs(c[k + int64_t(no) * m]);
    y[l] = s;
  }
  __syncthreads();
  double mx = 0.0;
  for (int s = threadIdx.x; s < nshell; s += blockDim.x) {
    double ym = 0.0;
    for (int i = 0; i < nbsh[s]; ++i) ym = fmax(ym, y[koff[s] + i]);
    mlk[s * ld + kp] = ym;
    mx = fmax(mx, ym);
  }
  for (int off = 32; off > 0; off >>= 1) mx = fmax(mx, __shfl_xor(mx, off, 64));
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = mx;
  __syncthreads();
  mx = fmax(fmax(red[0], red[1]), fmax(red[2], red[3]));
  unsigned long long nl = 0;
  for (int s = threadIdx.x; s < nshell; s += blockDim.x) {
    const double m = mlk[s * ld + kp];
    const bool ok = cas_cut ? (m >= D.xtau[d]) : (m * mx >= D.tau[d]);
    listed[s * ld + kp] = ok ? 1 : 0;
    nl += ok;
  }
  if (nl) atomicAdd(&cnt, nl);
  __syncthreads();
  if (threadIdx.x == 0 && cnt) atomicAdd(&stats[0], cnt);
}

// The half-transform's masks: bit k of word mw[((bt nq + q) nshell + sa) nshell
// + sb] = orbital k lists shell a and takes the pair (:659-702); kw[(bt nq + q)
// nshell + sa] = Keep(a).  Rows of shells with no kept orbital are not written.
// One lane per orbital.  grid = (shells a, batches * words).
__global__ __launch_bounds__(kLkThreads) void k_lk_mask(
    LkDens D, const LkGroup G, int nshell, const int32_t *__restrict__ nbsh,
    const uint8_t *__restrict__ listed, const double *__restrict__ sumac, const double *__restrict__ svall,
    unsigned long long *__restrict__ mw, unsigned long long *__restrict__ kw,
    unsigned long long *__restrict__ stats) {
  constexpr int U = 4;  // shells b in flight per wave
  __shared__ unsigned long long keep[kLkThreads / 64], cnt[kLkThreads / 64];
  const int sa = blockIdx.x, bt = blockIdx.y / D.nq, q = blockIdx.y % D.nq;
  const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int d = d_of_word(D, q), k = 64 * (q - D.q0[d]) + lane;
  const int64_t ld = 64 * int64_t(D.nq), col = 64 * int64_t(q) + lane;
  const double *__restrict__ sv = svall + bt * (int64_t(nshell) * (nshell + 1) / 2);
  const uint8_t *__restrict__ present = G.present[bt];
  const double thr = D.thrv2[d];
  const bool l = k < D.nocc[d] && listed[sa * ld + col] != 0;
  unsigned long long kept = 0, n = 0;
  if (__ballot(l) != 0 && nbsh[sa] > 0) {
    unsigned long long *__restrict__ row = mw + ((int64_t(bt) * D.nq + q) * nshell + sa) * nshell;
    for (int s0 = w * U; s0 < nshell; s0 += (kLkThreads / 64) * U) {
      double x[U];
      bool ok[U];
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const int sb = s0 + u < nshell ? s0 + u : nshell - 1;
        const int64_t p = shp_idx(sa, sb);
        ok[u] = l && present[p] != 0 && nbsh[sb] > 0;
        x[u] = sumac[sb * ld + col] * sv[p];
      }
#pragma unroll
      for (int u = 0; u < U; ++u) {
        if (s0 + u >= nshell) break;
        const unsigned long long b = __ballot(ok[u] && fabs(x[u]) >= thr);
        kept |= b;
        n += __popcll(b);
        if (lane == 0) row[s0 + u] = b;
      }
    }
  }
  if (lane == 0) {
    keep[w] = kept;
    cnt[w] = n;
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    kw[(int64_t(bt) * D.nq + q) * nshell + sa] = (keep[0] | keep[1]) | (keep[2] | keep[3]);
    const unsigned long long t = (cnt[0] + cnt[1]) + (cnt[2] + cnt[3]);
    if (t) atomicAdd(&stats[1], t);
  }
}

// Faa(a) = max_{i in a} |sum_J X(i,J)^2| (:713-743) at faa[(bt nshell + s) 64 nq
// + kpos], for the kept shells of each orbital.  grid = (orbitals, batches).
__global__ __launch_bounds__(kLkThreads) void k_lk_faa(
    LkDens D, const LkGroup G, int n_pad, int nshell, const int32_t *__restrict__ koff,
    const int32_t *__restrict__ nbsh, const double *__restrict__ X, const unsigned long long *__restrict__ kw,
    double *__restrict__ faa) {
  const int g = blockIdx.x, bt = blockIdx.y, jnum = G.jnum[bt];
  int d, k;
  dk_of(D, g, &d, &k);
  const int q = D.q0[d] + k / 64;
  const int64_t ld = 64 * int64_t(D.nq);
  const double *__restrict__ x = X + (int64_t(bt) * D.ktot + g) * kLkBatch * n_pad;
  for (int s = threadIdx.x; s < nshell; s += blockDim.x) {
    double t = 0.0;
    if ((kw[(int64_t(bt) * D.nq + q) * nshell + s] >> (k & 63)) & 1ull)
      for (int i = 0; i < nbsh[s]; ++i) {
        double f = 0.0;
        double v[kLkBatch];
#pragma unroll
        for (int j = 0; j < kLkBatch; ++j) v[j] = x[int64_t(j < jnum ? j : 0) * n_pad + koff[s] + i];
#pragma unroll
        for (int j = 0; j < kLkBatch; ++j) f = j < jnum ? f + v[j] * v[j] : f;
        t = fmax(t, fabs(f));
      }
    faa[(int64_t(bt) * nshell + s) * ld + kpos(D, d, k)] = t;
  }
}

// The K blocks each orbital keeps (:749-830): word pw[(bt nq + q) nshp + pair].
// grid = (shells a, batches * words).
__global__ __launch_bounds__(kLkThreads) void k_lk_pairs(
    LkDens D, int nshell, const unsigned long long *__restrict__ kw, const double *__restrict__ mlk,
    const double *__restrict__ faa, unsigned long long *__restrict__ pw, unsigned long long *__restrict__ stats) {
  constexpr int U = 4;
  __shared__ unsigned long long cnt[kLkThreads / 64];
  const int sa = blockIdx.x, bt = blockIdx.y / D.nq, q = blockIdx.y % D.nq;
  const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int d = d_of_word(D, q);
  const int64_t ld = 64 * int64_t(D.nq), col = 64 * int64_t(q) + lane;
  const int64_t nshp = int64_t(nshell) * (nshell + 1) / 2;
  const unsigned long long *__restrict__ kb = kw + (int64_t(bt) * D.nq + q) * nshell;
  const double *__restrict__ fb = faa + int64_t(bt) * nshell * ld;
  unsigned long long *__restrict__ row = pw + (int64_t(bt) * D.nq + q) * nshp + int64_t(sa) * (sa + 1) / 2;
  const unsigned long long ka = kb[sa];
  const double tau = D.tau[d], tk = D.tk2[d];
  unsigned long long n = 0;
  if (ka == 0) {
    for (int sb = threadIdx.x; sb <= sa; sb += kLkThreads) row[sb] = 0;
  } else {
    const bool la = (ka >> lane) & 1ull;
    const double ma = la ? mlk[sa * ld + col] : 0.0, fa = la ? fb[sa * ld + col] : 0.0;
    for (int s0 = w * U; s0 <= sa; s0 += (kLkThreads / 64) * U) {
      unsigned long long k2[U];
      double m[U], f[U];
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const int sb = s0 + u <= sa ? s0 + u : sa;
        k2[u] = kb[sb];
        m[u] = mlk[sb * ld + col];
        f[u] = fb[sb * ld + col];
      }
#pragma unroll
      for (int u = 0; u < U; ++u) {
        if (s0 + u > sa) break;
        const bool ok = la && ((k2[u] >> lane) & 1ull) && !(ma * m[u] < tau) && fabs(fa * f[u]) >= tk;
        const unsigned long long b = __ballot(ok);
        n += __popcll(b);
        if (lane == 0) row[s0 + u] = b;
      }
    }
  }
  if (lane == 0) cnt[w] = n;
  __syncthreads();
  if (threadIdx.x == 0) {
    const unsigned long long t = (cnt[0] + cnt[1]) + (cnt[2] + cnt[3]);
    if (t) atomicAdd(&stats[2], t);
  }
}

#pragma clang fp contract(fast)

__device__ inline v4d mfma64(double a, double b, v4d c) {
  return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
}

// Masked half-transform: X(bt, g, J, a) for one shell a, 64 orbitals (word q) and
// kHtCols columns (J, a in the shell, a fastest).  One wave; per step of four b
// it takes four A fragments (16 orbitals each, masked bit by bit) and three B
// fragments (packed elements gathered, one column per lane).  The steps whose
// mask words are all zero are left out.  X of orbitals that do not keep the
// shell is not meaningful and never read through its mask.
// grid = (shells a, column groups, batches * words).
__global__ __launch_bounds__(64) void k_lk_ht(
    LkDens D, const LkGroup G, const double *__restrict__ L, int64_t ldl, int n, int n_pad, int nshell,
    const int32_t *__restrict__ shell, const int32_t *__restrict__ koff, const int32_t *__restrict__ nbsh,
    const unsigned long long *__restrict__ mw, const unsigned long long *__restrict__ kw, double *__restrict__ X) {
  __shared__ unsigned long long sw[kHtPanel];
  __shared__ uint16_t steps[kHtPanel / 4];
  const int sa = blockIdx.x, bt = blockIdx.z / D.nq, q = blockIdx.z % D.nq;
  if (kw[(int64_t(bt) * D.nq + q) * nshell + sa] == 0) return;
  const int na = nbsh[sa], nc = na * G.jnum[bt], col0 = blockIdx.y * kHtCols;
  if (col0 >= nc) return;
  const int lane = threadIdx.x, m = lane & 15, g = lane >> 4;
  const int d = d_of_word(D, q), kb = 64 * (q - D.q0[d]), no = D.nocc[d];
  const int nkt = min(4, (no - kb + 15) / 16), nct = min(3, (nc - col0 + 15) / 16);
  const double *__restrict__ c = D.c[d];
  const unsigned long long *__restrict__ row = mw + ((int64_t(bt) * D.nq + q) * nshell + sa) * nshell;
  // this lane's columns: vector row pointer and AO
  const double *__restrict__ lp[3];
  int64_t xo[3];
  int ca[3];
#pragma unroll
  for (int j = 0; j < 3; ++j) {
    const int col = min(col0 + 16 * j + m, nc - 1);
    const int jl = col / na;
    ca[j] = koff[sa] + (col - jl * na);
    lp[j] = L + (G.j0[bt] + jl) * ldl;
    xo[j] = int64_t(jl) * n_pad + ca[j];
  }
  int kc[4];  // this lane's orbitals, clamped (their mask bits are zero past nocc)
#pragma unroll
  for (int i = 0; i < 4; ++i) kc[i] = min(kb + 16 * i + m, no - 1);
  v4d acc[4][3];
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int j = 0; j < 3; ++j) acc[i][j] = v4d{0.0, 0.0, 0.0, 0.0};
  for (int p0 = 0; p0 < n; p0 += kHtPanel) {
    const int pn = min(kHtPanel, n - p0);
    __syncthreads();
    for (int e = lane; e < kHtPanel; e += 64) sw[e] = e < pn ? row[shell[p0 + e]] : 0ull;
    __syncthreads();
    int nact = 0;
    for (int t0 = 0; 4 * t0 < pn; t0 += 64) {
      const int t = t0 + lane;
      const bool on = 4 * t < pn && ((sw[4 * t] | sw[4 * t + 1]) | (sw[4 * t + 2] | sw[4 * t + 3])) != 0;
      const unsigned long long b = __ballot(on);
      if (on) steps[nact + __popcll(b & ((1ull << lane) - 1ull))] = uint16_t(t);
      nact += __popcll(b);
    }
    __syncthreads();
    double ar[2][4], br[2][3];
    unsigned long long wr[2];
    auto load = [&](int i, int st) __attribute__((always_inline)) {
      const int e = 4 * steps[i] + g, b = min(p0 + e, n - 1);
      wr[st] = sw[e];
#pragma unroll
      for (int t = 0; t < 4; ++t) ar[st][t] = c[kc[t] + int64_t(no) * b];
#pragma unroll
      for (int j = 0; j < 3; ++j) {
        const int hi = max(ca[j], b), lo = min(ca[j], b);
        br[st][j] = lp[j][int64_t(hi) * (hi + 1) / 2 + lo];
      }
    };
    auto mul = [&](int st) __attribute__((always_inline)) {
#pragma unroll
      for (int t = 0; t < 4; ++t) {
        if (t >= nkt) break;
        const double a = (wr[st] >> (16 * t + m)) & 1ull ? ar[st][t] : 0.0;
        acc[t][0] = mfma64(a, br[st][0], acc[t][0]);
        if (nct > 1) acc[t][1] = mfma64(a, br[st][1], acc[t][1]);
        if (nct > 2) acc[t][2] = mfma64(a, br[st][2], acc[t][2]);
      }
    };
    if (nact > 0) {
      load(0, 0);
      for (int i = 0; i < nact; i += 2) {
        load(min(i + 1, nact - 1), 1);
        mul(0);
        if (i + 1 >= nact) break;
        load(min(i + 2, nact - 1), 0);
        mul(1);
      }
    }
  }
  double *__restrict__ xg = X + (int64_t(bt) * D.ktot + D.k0[d]) * kLkBatch * n_pad;
#pragma unroll
  for (int j = 0; j < 3; ++j) {
    if (col0 + 16 * j + m >= nc) continue;
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int k = kb + 16 * i + 4 * r + g;
        if (k < no) xg[int64_t(k) * kLkBatch * n_pad + xo[j]] = acc[i][j][r];
      }
  }
}

// K of one batch on the 32 x 32 tile t of the lower triangle, density d: the sum
// over the orbitals whose pair mask is set of S_k = sum_J X_k X_k^T, formed by
// MFMA per orbital and added under the mask.  One wave; a step's operands are
// reloaded with the next kept orbital's as soon as they are multiplied.  kpart[((bt nd + d) ntile
// + t) 1024 + (2 it + jt) 256 + 64 r + lane].  grid = (tiles, nd, batches).
__global__ __launch_bounds__(64) void k_lk_k(LkDens D, const LkGroup G, const double *__restrict__ X, int n,
                                             int n_pad, int nshell, const int32_t *__restrict__ shell,
                                             const unsigned long long *__restrict__ pw, double *__restrict__ kpart) {
  constexpr int KS = (kLkBatch + 3) / 4;
  const int t = blockIdx.x, d = blockIdx.y, bt = blockIdx.z, jnum = G.jnum[bt];
  int ta = int((sqrt(8.0 * t + 1.0) - 1.0) * 0.5);
  while (ta * (ta + 1) / 2 > t) --ta;
  while ((ta + 1) * (ta + 2) / 2 <= t) ++ta;
  const int tb = t - ta * (ta + 1) / 2;
  const int lane = threadIdx.x, m = lane & 15, g = lane >> 4;
  const int64_t nshp = int64_t(nshell) * (nshell + 1) / 2;
  v4d acc[2][2];
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j) acc[i][j] = v4d{0.0, 0.0, 0.0, 0.0};
  uint32_t pr[2][2][4];  // shell pair of each element, ~0: not in the lower triangle
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int a = 32 * ta + 16 * i + 4 * r + g, b = 32 * tb + 16 * j + m;
        pr[i][j][r] = a < n && b <= a ? uint32_t(shp_idx(shell[a], shell[b])) : ~0u;
      }
  const bool upper = ta != tb;  // tile (0, 1) of a diagonal tile lies above the diagonal
  uint32_t jo[KS];
#pragma unroll
  for (int s = 0; s < KS; ++s) jo[s] = uint32_t(min(4 * s + g, jnum - 1)) * uint32_t(n_pad) + uint32_t(m);
  for (int q = D.q0[d]; q < D.q0[d + 1]; ++q) {
    const unsigned long long *__restrict__ pq = pw + (int64_t(bt) * D.nq + q) * nshp;
    unsigned long long mk[2][2][4], any = 0;
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
      for (int j = 0; j < 2; ++j)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          mk[i][j][r] = pr[i][j][r] != ~0u ? pq[pr[i][j][r]] : 0ull;
          any |= mk[i][j][r];
        }
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) any |= __shfl_xor(any, o);
    any = (uint64_t(__builtin_amdgcn_readfirstlane(int(any >> 32))) << 32) |
          uint32_t(__builtin_amdgcn_readfirstlane(int(any)));
    if (any == 0) continue;
    const double *__restrict__ xq =
        X + (int64_t(bt) * D.ktot + D.k0[d] + 64 * (q - D.q0[d])) * kLkBatch * int64_t(n_pad);
    double ra[KS][2], rb[KS][2];
    auto load = [&](const double *__restrict__ x, int s) __attribute__((always_inline)) {
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        ra[s][h] = x[jo[s] + 32 * ta + 16 * h];
        rb[s][h] = x[jo[s] + 32 * tb + 16 * h];
      }
    };
    int k = __builtin_ctzll(any);
#pragma unroll
    for (int s = 0; s < KS; ++s) load(xq + int64_t(k) * kLkBatch * n_pad, s);
    for (;;) {
      any &= any - 1;
      const int kn = any ? __builtin_ctzll(any) : k;  // next kept orbital, or this one again
      const double *__restrict__ xn = xq + int64_t(kn) * kLkBatch * n_pad;
      v4d sm[2][2];
#pragma unroll
      for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j) sm[i][j] = v4d{0.0, 0.0, 0.0, 0.0};
#pragma unroll
      for (int s = 0; s < KS; ++s) {
        const bool in = 4 * s + g < jnum;
        double a[2], b[2];
#pragma unroll
        for (int h = 0; h < 2; ++h) {
          a[h] = in ? ra[s][h] : 0.0;
          b[h] = in ? rb[s][h] : 0.0;
        }
        sm[0][0] = mfma64(a[0], b[0], sm[0][0]);
        if (upper) sm[0][1] = mfma64(a[0], b[1], sm[0][1]);
        sm[1][0] = mfma64(a[1], b[0], sm[1][0]);
        sm[1][1] = mfma64(a[1], b[1], sm[1][1]);
        load(xn, s);
      }
#pragma unroll
      for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j)
#pragma unroll
          for (int r = 0; r < 4; ++r) acc[i][j][r] += (mk[i][j][r] >> k) & 1ull ? sm[i][j][r] : 0.0;
      if (any == 0) break;
      k = kn;
    }
  }
  double *__restrict__ out = kpart + ((int64_t(bt) * D.nd + d) * gridDim.x + t) * 1024 + lane;
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int r = 0; r < 4; ++r) out[(2 * i + j) * 256 + 64 * r] = acc[i][j][r];
}

// klt(d) += the group's batches in order.  grid = (tiles, nd), block 256.
__global__ __launch_bounds__(kLkThreads) void k_lk_reduce(const double *__restrict__ kpart, int nb, int nd, int n,
                                                          double *__restrict__ klt, int64_t ldk) {
  const int t = blockIdx.x, d = blockIdx.y;
  int ta = int((sqrt(8.0 * t + 1.0) - 1.0) * 0.5);
  while (ta * (ta + 1) / 2 > t) --ta;
  while ((ta + 1) * (ta + 2) / 2 <= t) ++ta;
  const int tb = t - ta * (ta + 1) / 2;
  const double *__restrict__ src = kpart + (int64_t(d) * gridDim.x + t) * 1024;
  const int64_t stride = int64_t(nd) * gridDim.x * 1024;
  for (int e = threadIdx.x; e < 1024; e += kLkThreads) {
    const int tile = e >> 8, r = (e >> 6) & 3, lane = e & 63;
    const int a = 32 * ta + 16 * (tile >> 1) + 4 * r + (lane >> 4), b = 32 * tb + 16 * (tile & 1) + (lane & 15);
    if (a >= n || b > a) continue;
    const int64_t p = d * ldk + int64_t(a) * (a + 1) / 2 + b;
    double s = klt[p];
    int k = 0;
    for (; k + 8 <= nb; k += 8) {
      double v[8];
#pragma unroll
      for (int u = 0; u < 8; ++u) v[u] = src[(k + u) * stride + e];
#pragma unroll
      for (int u = 0; u < 8; ++u) s += v[u];
    }
    for (; k < nb; ++k) s += src[k * stride + e];
    klt[p] = s;
  }
}

// Least double x >= 0 with sqrt(x) >= t (the rounded square root, as the device
// evaluates it, is monotone): sqrt|x| >= t can then be tested without a root.
double least_square(double t) {
  if (!(t > 0.0)) return 0.0;
  double x = t * t;
  if (std::isinf(x)) x = std::numeric_limits<double>::max();
  while (std::sqrt(x) >= t) {
    const double y = std::nextafter(x, 0.0);
    if (!(std::sqrt(y) >= t) || y == x) break;
    x = y;
  }
  while (std::sqrt(x) < t && !std::isinf(x)) x = std::nextafter(x, std::numeric_limits<double>::infinity());
  return x;
}

// Shell-pair occupancy of a reduced set (nnBstRSh > 0 of the reference).
int lk_present(Context *c, int rs, const uint8_t **out) {
  LKState &K = c->lk;
  const int ns = K.nshell;
  const int64_t nshp = int64_t(ns) * (ns + 1) / 2;
  std::vector<int32_t> shell(size_t(c->n));
  for (int s = 0, a = 0; s < ns; ++s)
    for (int i = 0; i < K.nbassh[size_t(s)]; ++i) shell[size_t(a++)] = s;
  auto lt_pair = [](int64_t idx, int64_t *a, int64_t *b) {
    int64_t r = int64_t((std::sqrt(8.0 * double(idx) + 1.0) - 1.0) * 0.5);
    while (r * (r + 1) / 2 > idx) --r;
    while ((r + 1) * (r + 2) / 2 <= idx) ++r;
    *a = r;
    *b = idx - r * (r + 1) / 2;
  };
  DevBuf *buf;
  int64_t *ver;
  std::vector<uint8_t> h(size_t(nshp), 0);
  if (rs < 0) {  // every pair: the store written in place
    buf = &K.present_all;
    ver = &K.present_all_version;
    if (*ver != K.version) std::fill(h.begin(), h.end(), 1);
  } else {
    if (K.present.size() < c->rsets.size()) {
      K.present.resize(c->rsets.size());
      K.present_version.resize(c->rsets.size(), -1);
    }
    buf = &K.present[size_t(rs)];
    ver = &K.present_version[size_t(rs)];
    if (*ver != K.version) {
      const ReducedSet &R = c->rsets[size_t(rs)];
      for (int64_t r = 0; r < R.nrs; ++r) {
        int64_t a, b;
        lt_pair(R.identity ? r : int64_t(R.h_map[size_t(r)]), &a, &b);
        const int s1 = shell[size_t(a)], s2 = shell[size_t(b)];
        h[size_t(s1 >= s2 ? int64_t(s1) * (s1 + 1) / 2 + s2 : int64_t(s2) * (s2 + 1) / 2 + s1)] = 1;
      }
    }
  }
  if (*ver != K.version) {
    int rc;
    if ((rc = ensure(c, *buf, size_t(nshp)))) return rc;
    if ((rc = hip_check(c, hipMemcpy(buf->ptr, h.data(), size_t(nshp), hipMemcpyHostToDevice),
                        "LK shell-pair occupancy")))
      return rc;
    *ver = K.version;
  }
  *out = static_cast<const uint8_t *>(buf->ptr);
  return MJK_OK;
}

}  // namespace

int lk_exchange(Context *c, int32_t nd, const int32_t *nocc, const double *const *corb,
                const double *tau, const double *thrv, bool cas_cut, double *klt, int64_t ldk) {
  LKState &K = c->lk;
  if (K.nshell < 1) return set_error(c, MJK_ERR_STATE, "LK screening: no shells (mjk_set_shells)");
  if (!K.diag_set)
    return set_error(c, MJK_ERR_STATE, "LK screening: no integral diagonal (mjk_set_lk_diag)");
  if (nd < 1 || nd > 2) return set_error(c, MJK_ERR_ARG, "LK screening: one or two densities");
  if (c->nloaded != c->nchol)
    return set_error(c, MJK_ERR_SHORT_READ, "LK screening: not all Cholesky vectors were uploaded");
  const int n = c->n, n_pad = c->n_pad, ns = K.nshell;
  const int64_t np = c->np, nshp = int64_t(ns) * (ns + 1) / 2;
  // vectors grouped by reduced set, in increasing order (InfVec(J,2) of the reference)
  struct Run { int rs; int64_t j0, jn; };
  std::vector<Run> runs;
  for (int64_t j = 0; j < c->nchol; ++j) {
    const int rs = c->vset[size_t(j)] > 0 ? c->vset[size_t(j)] - 1 : -1;
    if (runs.empty() || runs.back().rs != rs) runs.push_back({rs, j, 0});
    runs.back().jn += 1;
  }
  for (size_t i = 1; i < runs.size(); ++i)
    if (runs[i].rs < 0 || runs[i - 1].rs < 0 || runs[i].rs <= runs[i - 1].rs)
      return set_error(c, MJK_ERR_STATE,
                       "LK screening: vectors must come reduced set by reduced set, in order");
  const double maxred = double(K.maxred > 0 ? K.maxred : int(std::max<size_t>(c->rsets.size(), 1)));
  LkDens D{};
  D.nd = nd;
  int ktot = 0;
  for (int d = 0; d < nd; ++d) {
    D.nocc[d] = std::max(0, nocc[d]);
    D.k0[d] = ktot;
    D.q0[d + 1] = D.q0[d] + int(ceil_div(D.nocc[d], 64));
    D.c[d] = corb[d];
    D.tau[d] = tau[d];
    D.xtau[d] = std::sqrt(tau[d]);  // xtau = sqrt(tau), cho_lk_casscf.F90:193-194
    D.thrv2[d] = least_square(thrv[d]);
    D.tk2[d] = least_square(tau[d] / maxred);
    ktot += D.nocc[d];
  }
  D.ktot = ktot;
  D.nq = D.q0[nd];
  int rc;
  for (int d = 0; d < nd; ++d)
    if ((rc = fill_zero(c, klt + d * ldk, sizeof(double) * size_t(np)))) return rc;
  K.last_stats[0] = K.last_stats[1] = K.last_stats[2] = 0;
  K.last_batches = 0;
  if (ktot == 0 || runs.empty()) return MJK_OK;
  // the batches, and before which of them the shell lists are evaluated: the first
  // one, and every nScreen reduced sets, counting each of JRED1..JRED2 with or
  // without vectors (:336-337,374,831,891-898)
  struct Batch { int64_t j0; int jnum; const uint8_t *present; bool screen; };
  std::vector<Batch> batches;
  int kscreen = 1, max_rows = 0;
  bool doscreen = true;
  size_t ri = 0;
  for (int jred = runs.front().rs; jred <= runs.back().rs; ++jred) {
    if (ri < runs.size() && runs[ri].rs == jred) {
      const Run &R = runs[ri++];
      const uint8_t *present = nullptr;
      if ((rc = lk_present(c, R.rs, &present))) return rc;
      const int64_t nvec = std::min<int64_t>(kLkBatch, R.jn);
      for (int64_t b = 0; b < R.jn; b += nvec) {
        batches.push_back({R.j0 + b, int(std::min<int64_t>(nvec, R.jn - b)), present, doscreen});
        max_rows = std::max(max_rows, batches.back().jnum);
        doscreen = false;
      }
    }
    doscreen = kscreen == c->lk_nscreen;
    if (!doscreen) ++kscreen;
    else kscreen = 1;
  }
  K.last_batches = int64_t(batches.size());
  // Batches that go through the kernels together: as many as 1 GiB of per-batch
  // buffers holds (X, masks, partial K), or the X budget if that is less, up to
  // kLkGroup; half as many, and again, where the device has no room for them.
  const int nt = int(ceil_div(n, 32)), ntile = nt * (nt + 1) / 2;
  const int64_t ld = 64 * int64_t(D.nq);
  const size_t bx = sizeof(double) * size_t(ktot) * kLkBatch * n_pad, bm = 8 * size_t(D.nq) * ns * ns,
               bp = 8 * size_t(D.nq) * nshp, bk = sizeof(double) * 1024 * size_t(nd) * ntile,
               bs = sizeof(double) * size_t(nshp), bf = sizeof(double) * size_t(ns) * ld,
               bw = 8 * size_t(D.nq) * ns;
  const size_t room = size_t(std::min<int64_t>(int64_t(1) << 30, c->x_budget));
  int ng = int(std::max<size_t>(  // (batch, word) is one grid dimension
      1, std::min<size_t>({size_t(K.group_most), batches.size(), room / (bx + bm + bp + bk + bs + bf + bw),
                           size_t(65535 / D.nq)})));
  const size_t flag_bytes = size_t(ld) * ns;
  if ((rc = ensure(c, K.diag, sizeof(double) * size_t(np))) ||
      (rc = ensure(c, K.dh, sizeof(double) * size_t(n) * n)) ||
      (rc = ensure(c, K.ylk, sizeof(double) * size_t(ktot) * n)) ||
      (rc = ensure(c, K.sumac, sizeof(double) * size_t(ld) * ns)) ||
      (rc = ensure(c, K.mlk, sizeof(double) * size_t(ld) * ns)) || (rc = ensure(c, K.listed, flag_bytes)) ||
      (rc = ensure(c, K.stats, 3 * sizeof(unsigned long long))))
    return rc;
  const std::pair<DevBuf *, size_t> per_batch[] = {{&K.svshp, bs}, {&K.faa, bf},  {&K.keep, bw}, {&K.mask, bm},
                                                   {&K.pairs, bp}, {&K.kacc, bk}, {&K.x, bx}};
  for (;; ng = K.group_most = ng / 2) {
    for (const auto &b : per_batch)
      if ((rc = ensure(c, *b.first, b.second * ng))) break;
    if (!rc) break;
    if (rc != MJK_ERR_NOMEM || ng == 1) {
      K.group_most = kLkGroup;
      return rc;
    }
    int rs;
    if ((rs = hip_check(c, hipStreamSynchronize(c->stream), "LK buffers"))) return rs;
    for (const auto &b : per_batch) {  // room for the smaller ones
      if (b.first->ptr) (void)hipFree(b.first->ptr);
      *b.first = DevBuf{};
    }
  }
  double *diag = static_cast<double *>(K.diag.ptr);
  double *sv = static_cast<double *>(K.svshp.ptr), *sumac = static_cast<double *>(K.sumac.ptr);
  double *mlk = static_cast<double *>(K.mlk.ptr), *faa = static_cast<double *>(K.faa.ptr);
  double *X = static_cast<double *>(K.x.ptr), *kpart = static_cast<double *>(K.kacc.ptr);
  uint8_t *listed = static_cast<uint8_t *>(K.listed.ptr);
  typedef unsigned long long word;
  word *keep = static_cast<word *>(K.keep.ptr), *mask = static_cast<word *>(K.mask.ptr);
  word *pairs = static_cast<word *>(K.pairs.ptr), *stats = static_cast<word *>(K.stats.ptr);
  // mlk, sumac and listed have entries past each density's orbitals: zero, and no
  // mask bit is set for them
  if ((rc = hip_check(c, hipMemcpyAsync(diag, K.diag0.ptr, sizeof(double) * size_t(np),
                                        hipMemcpyDeviceToDevice, c->stream), "LK diagonal")) ||
      (rc = fill_zero(c, stats, 3 * sizeof(word))) || (rc = fill_zero(c, listed, flag_bytes)) ||
      (rc = fill_zero(c, mlk, sizeof(double) * size_t(ld) * ns)) ||
      (rc = fill_zero(c, sumac, sizeof(double) * size_t(ld) * ns)) || (rc = fill_zero(c, faa, bf * ng)))
    return rc;
  const int32_t *shell = static_cast<const int32_t *>(K.shell.ptr);
  const int32_t *koff = static_cast<const int32_t *>(K.koff.ptr);
  const int32_t *nbsh = static_cast<const int32_t *>(K.nbsh.ptr);
  hipLaunchKernelGGL(k_lk_sumac, dim3(unsigned(ktot)), dim3(kLkThreads), 0, c->stream, D, ns, koff,
                     nbsh, sumac);
  const unsigned gnp = unsigned(std::min<int64_t>(ceil_div(np, kLkThreads), 4096));
  int max_shell = 1;
  for (int32_t v : K.nbassh) max_shell = std::max(max_shell, int(v));
  const unsigned cols = unsigned(ceil_div(int64_t(max_rows) * max_shell, kHtCols));
  const bool update = K.update && c->lk_nscreen > 0;
  for (size_t b0 = 0; b0 < batches.size();) {
    LkGroup G{};
    size_t b1 = b0;
    int64_t jn = 0;
    for (; b1 < batches.size() && int(b1 - b0) < ng && (b1 == b0 || !batches[b1].screen); ++b1) {
      G.j0[b1 - b0] = batches[b1].j0;
      G.jnum[b1 - b0] = batches[b1].jnum;
      G.present[b1 - b0] = batches[b1].present;
      jn += batches[b1].jnum;
    }
    G.nb = int(b1 - b0);
    const unsigned nb = unsigned(G.nb), nbq = unsigned(G.nb * D.nq);
    if (max_shell <= kSmallShell)
      hipLaunchKernelGGL(k_lk_svshp, dim3(unsigned(ns), unsigned(ceil_div(ns, kLkThreads)), nb), dim3(kLkThreads), 0,
                         c->stream, c->L, c->ldl, G, ns, koff, nbsh, sv);
    else
      hipLaunchKernelGGL(k_lk_svshp_wave, dim3(unsigned(ceil_div(nshp, kLkThreads / 64)), nb), dim3(kLkThreads), 0,
                         c->stream, c->L, c->ldl, G, ns, koff, nbsh, sv);
    if (batches[b0].screen) {
      // Estimate: the diagonal of the batch the lists are evaluated before
      if (K.estimate)
        hipLaunchKernelGGL(k_lk_est_diag, dim3(gnp), dim3(kLkThreads), 0, c->stream, c->L, c->ldl,
                           G.j0[0], G.jnum[0], np, diag);
      hipLaunchKernelGGL(k_lk_diah, dim3(unsigned(n)), dim3(kLkThreads), 0, c->stream, diag, n,
                         static_cast<double *>(K.dh.ptr));
      hipLaunchKernelGGL(k_lk_screen, dim3(unsigned(ktot)), dim3(kLkThreads), 0, c->stream, D, n, ns,
                         int(cas_cut), koff, nbsh, static_cast<const double *>(K.dh.ptr),
                         static_cast<double *>(K.ylk.ptr), mlk, listed, stats);
    }
    hipLaunchKernelGGL(k_lk_mask, dim3(unsigned(ns), nbq), dim3(kLkThreads), 0, c->stream, D, G, ns, nbsh, listed,
                       sumac, sv, mask, keep, stats);
    hipLaunchKernelGGL(k_lk_ht, dim3(unsigned(ns), cols, nbq), dim3(64), 0, c->stream, D, G, c->L, c->ldl, n, n_pad,
                       ns, shell, koff, nbsh, mask, keep, X);
    hipLaunchKernelGGL(k_lk_faa, dim3(unsigned(ktot), nb), dim3(kLkThreads), 0, c->stream, D, G, n_pad, ns, koff,
                       nbsh, X, keep, faa);
    hipLaunchKernelGGL(k_lk_pairs, dim3(unsigned(ns), nbq), dim3(kLkThreads), 0, c->stream, D, ns, keep, mlk, faa,
                       pairs, stats);
    hipLaunchKernelGGL(k_lk_k, dim3(unsigned(ntile), unsigned(nd), nb), dim3(64), 0, c->stream, D, G, X, n, n_pad,
                       ns, shell, pairs, kpart);
    hipLaunchKernelGGL(k_lk_reduce, dim3(unsigned(ntile), unsigned(nd)), dim3(kLkThreads), 0, c->stream, kpart,
                       G.nb, nd, n, klt, ldk);
    // Update: only a later evaluation of the lists reads the diagonal, and with
    // Estimate it is formed anew there
    bool later = false;
    for (size_t b = b1; b < batches.size(); ++b) later |= batches[b].screen;
    if (update && later && !K.estimate)
      hipLaunchKernelGGL(k_lk_update_diag, dim3(gnp), dim3(kLkThreads), 0, c->stream, c->L, c->ldl, G.j0[0],
                         int(jn), np, diag);
    if ((rc = hip_check(c, hipGetLastError(), "LK group launch"))) return rc;
    b0 = b1;
  }
  unsigned long long h[3];
  if ((rc = hip_check(c, hipMemcpyAsync(h, stats, sizeof(h), hipMemcpyDeviceToHost, c->stream),
                      "LK counters")) ||
      (rc = hip_check(c, hipStreamSynchronize(c->stream), "LK sync")))
    return rc;
  for (int i = 0; i < 3; ++i) K.last_stats[i] = (long long)h[i];
  return MJK_OK;
}

}  // namespace mjk
