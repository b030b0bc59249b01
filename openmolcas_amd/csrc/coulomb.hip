// Coulomb (J) build from HBM-resident packed Cholesky vectors.
//
// Reference: the DGEMV pair of src/fock_util/cho_fscf.F90:208,215 (also
// cho_lk_scf.F90:442-449, cho_fmcscf.F90:261-285):
//   V_J  = sum_p L^J_p D_p          (D folded: off-diagonal doubled)
//   J_p  = sum_J L^J_p V_J
// Bound by HBM.  One or two densities of ordinary sizes read L once for both
// (k_coulomb_one); otherwise each pass streams L once.  L is stored vector-major
// (row J holds the packed LT of L^J, stride ldl, a multiple of 512 doubles),
// so whole 4 KiB row segments are read per workgroup iteration.
#include <mutex>
#include <string>

#include "mjk_internal.h"

namespace mjk {
namespace {

constexpr int kThreads = 256;
constexpr int kSeg = 2 * kThreads;  // doubles per row segment per iteration

template <int N>
__device__ inline void block_sum(double (&v)[N], double *lds /* [N][4] */) {
  const int lane = threadIdx.x & (kWave - 1);
  const int wave = threadIdx.x / kWave;
#pragma unroll
  for (int i = 0; i < N; ++i) {
    double x = v[i];
#pragma unroll
    for (int off = kWave / 2; off > 0; off >>= 1) x += __shfl_down(x, off, kWave);
    if (lane == 0) lds[i * 4 + wave] = x;
  }
  __syncthreads();
  if (threadIdx.x < N) {
    const double *p = lds + threadIdx.x * 4;
    v[0] = (p[0] + p[1]) + (p[2] + p[3]);
  }
}

// Pass 1.  grid = (ceil(M/JB), nsplit).  Workgroup (jb, s) accumulates
// V(J, d) for JB vectors over the pair range of split s into
// vpart[(s*M + J)*nd + d].
template <int JB, int ND>
__global__ __launch_bounds__(kThreads) void k_coulomb_v(
    const double *__restrict__ L, int64_t ldl, int64_t M, const double *__restrict__ D,
    int nd, int64_t pchunk, double *__restrict__ vpart) {
  __shared__ double lds[JB * ND * 4];
  const int64_t j0 = int64_t(blockIdx.x) * JB;
  const int64_t p0 = int64_t(blockIdx.y) * pchunk;
  const int64_t p1 = min(p0 + pchunk, ldl);
  double acc[JB * ND];
#pragma unroll
  for (int i = 0; i < JB * ND; ++i) acc[i] = 0.0;
  for (int64_t p = p0 + 2 * threadIdx.x; p < p1; p += kSeg) {
    v2d dv[ND];
#pragma unroll
    for (int d = 0; d < ND; ++d)
      dv[d] = (d < nd) ? *reinterpret_cast<const v2d *>(D + d * ldl + p)
                       : v2d{0.0, 0.0};
    // rows past M read the last row (their sums are never written): the loads
    // stay unconditional, so all JB of them are in flight together
#pragma unroll
    for (int jb = 0; jb < JB; ++jb) {
      const int64_t j = j0 + jb < M ? j0 + jb : M - 1;
      const v2d l = __builtin_nontemporal_load(reinterpret_cast<const v2d *>(L + j * ldl + p));
#pragma unroll
      for (int d = 0; d < ND; ++d) acc[jb * ND + d] += l.x * dv[d].x + l.y * dv[d].y;
    }
  }
  block_sum<JB * ND>(acc, lds);
  if (threadIdx.x < JB * ND) {
    const int jb = threadIdx.x / ND, d = threadIdx.x % ND;
    if (j0 + jb < M && d < nd) vpart[(int64_t(blockIdx.y) * M + j0 + jb) * nd + d] = acc[0];
  }
}

// V(J, d) = sum_s vpart[(s*M + J)*nd + d]  (fixed order: deterministic).
__global__ void k_reduce_v(const double *__restrict__ vpart, int64_t M, int nd, int nsplit,
                           double *__restrict__ v) {
  const int64_t i = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
  if (i >= M * nd) return;
  double s = 0.0;
  for (int k = 0; k < nsplit; ++k) s += vpart[int64_t(k) * M * nd + i];
  v[i] = s;
}

// Pass 2.  grid = (ceil(ldl/(W*kSeg)), nsplit).  Workgroup (c, s) owns pairs
// [c*W*kSeg, (c+1)*W*kSeg) (W row segments, so each vector row is read in
// W*4 KiB runs) and sums over the vectors of split s:
// jpart[(s*nd + d)*ldl + p] = sum_J L(J,p) V(J,d).  U rows in flight per thread.
template <int ND, int W, int U>
__global__ __launch_bounds__(kThreads) void k_coulomb_j(
    const double *__restrict__ L, int64_t ldl, int64_t M, const double *__restrict__ V,
    int nd, int64_t jchunk, double *__restrict__ jpart) {
  const int64_t pb = int64_t(blockIdx.x) * (W * kSeg) + 2 * threadIdx.x;
  const int64_t ja = int64_t(blockIdx.y) * jchunk;
  const int64_t jz = min(ja + jchunk, M);
  v2d acc[W][ND];
  bool ok[W];
#pragma unroll
  for (int w = 0; w < W; ++w) {
    ok[w] = pb + w * kSeg < ldl;
#pragma unroll
    for (int d = 0; d < ND; ++d) acc[w][d] = v2d{0.0, 0.0};
  }
  int64_t j = ja;
  for (; j + U <= jz; j += U) {
    v2d l[U][W];
#pragma unroll
    for (int u = 0; u < U; ++u)
#pragma unroll
      for (int w = 0; w < W; ++w)
        l[u][w] = ok[w] ? __builtin_nontemporal_load(
                              reinterpret_cast<const v2d *>(L + (j + u) * ldl + pb + w * kSeg))
                        : v2d{0.0, 0.0};
#pragma unroll
    for (int u = 0; u < U; ++u) {
#pragma unroll
      for (int d = 0; d < ND; ++d) {
        if (d < nd) {
          const double v = V[(j + u) * nd + d];
#pragma unroll
          for (int w = 0; w < W; ++w) {
            acc[w][d].x += l[u][w].x * v;
            acc[w][d].y += l[u][w].y * v;
          }
        }
      }
    }
  }
  for (; j < jz; ++j) {
#pragma unroll
    for (int w = 0; w < W; ++w) {
      if (!ok[w]) continue;
      const v2d l = __builtin_nontemporal_load(reinterpret_cast<const v2d *>(L + j * ldl + pb + w * kSeg));
#pragma unroll
      for (int d = 0; d < ND; ++d) {
        if (d < nd) {
          const double v = V[j * nd + d];
          acc[w][d].x += l.x * v;
          acc[w][d].y += l.y * v;
        }
      }
    }
  }
#pragma unroll
  for (int w = 0; w < W; ++w)
#pragma unroll
    for (int d = 0; d < ND; ++d)
      if (ok[w] && d < nd)
        *reinterpret_cast<v2d *>(jpart + (int64_t(blockIdx.y) * nd + d) * ldl + pb + w * kSeg) =
            acc[w][d];
}

// jlt(d*ldj + p) = sum_s jpart[(s*nd + d)*ldl + p], p < np.  Thread (q, pair)
// sums every fourth slice from the q-th, eight loads in flight, in a fixed order:
// one thread per pair took the slices one load after the other (137 of them at
// n=24: 33 us, now 4).  grid = (ceil(np / 64), nd), block 256.
__global__ __launch_bounds__(kThreads) void k_reduce_j(const double *__restrict__ jpart, int64_t ldl, int64_t np,
                                                      int nd, int nsplit, double *__restrict__ jlt, int64_t ldj) {
  __shared__ double red[3][64];
  const int cb = threadIdx.x & 63, q = threadIdx.x >> 6, d = blockIdx.y;
  const int64_t p = int64_t(blockIdx.x) * 64 + cb;
  const double *__restrict__ src = jpart + d * ldl + min(p, np - 1);
  const int64_t stride = nd * ldl;
  double s = 0.0;
  int k = q;
  for (; k + 28 < nsplit; k += 32) {
    double v[8];
#pragma unroll
    for (int u = 0; u < 8; ++u) v[u] = src[(k + 4 * u) * stride];
#pragma unroll
    for (int u = 0; u < 8; ++u) s += v[u];
  }
  for (; k < nsplit; k += 4) s += src[k * stride];
  if (q > 0) red[q - 1][cb] = s;
  __syncthreads();
  if (q == 0 && p < np) jlt[d * ldj + p] = ((s + red[0][cb]) + red[1][cb]) + red[2][cb];
}

// ---- one or two densities: both passes in one read of the vectors ----------
// A group of G workgroups holds one vector at a time in registers, each its slice
// of the pairs: a workgroup sums its part of V_J, publishes it, and adds V_J L^J to
// its J once the whole V_J is there.  Its ring of four vectors hides the exchange:
// while V_J is awaited the next is contracted and the one after is on its way.
// Bound by HBM (one read of L) once a group has its 48 KiB per step in flight.
// Measured against the two passes (two reads), us: n=701, 2804 vectors 1735 -> 946
// (5.8 TB/s), n=512 715 -> 385, n=301 164 -> 96, n=1200 8634 -> 4635; two densities
// n=701 1761 -> 1134, n=301 172 -> 106.  Rows and ring (rows x vectors of lag):
// one density, n=512: 8x0 457, 6x1 385, 6x2 387, 5x2 411, 4x3 451 us; two, n=512:
// 6x0 468, 5x1 440, 4x2 488 us.
constexpr int kOneWaves = 8, kOneRow = 2 * kWave * kOneWaves;  // streaming waves; doubles per workgroup row
constexpr int kOneRing = 4;                                    // vectors per workgroup: on its way, contracted, awaited
constexpr int64_t kOneEmpty = 0x7ff4a5c300f1d2e7;              // "not there yet" (a NaN) in the exchange array

template <int C>
__device__ inline double dpp_add(double x) {
  const int2 v = __builtin_bit_cast(int2, x);
  const int2 y = {__builtin_amdgcn_update_dpp(0, v.x, C, 0xf, 0xf, false),
                  __builtin_amdgcn_update_dpp(0, v.y, C, 0xf, 0xf, false)};
  return x + __builtin_bit_cast(double, y);
}

__device__ inline double lane_value(double x, int lane) {
  const int2 v = __builtin_bit_cast(int2, x);
  return __builtin_bit_cast(double, int2{__builtin_amdgcn_readlane(v.x, lane), __builtin_amdgcn_readlane(v.y, lane)});
}

// Sum over the wave, the same in every lane.
__device__ inline double wave_sum(double x) {
  x = dpp_add<0xB1>(x);   // lane ^ 1
  x = dpp_add<0x4E>(x);   // lane ^ 2
  x = dpp_add<0x141>(x);  // the other quad of eight lanes
  x = dpp_add<0x140>(x);  // the other eight of sixteen
  return (lane_value(x, 0) + lane_value(x, 16)) + (lane_value(x, 32) + lane_value(x, 48));
}

// LDS written before is seen after; loads from memory stay in flight across it.
__device__ inline void lds_barrier() {
  asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
}

// Part of V of one vector that a wave sums: each lane's pairs in rising order, then
// the wave.
template <int ROWS>
__device__ inline double one_dot(const v2d (&x)[ROWS], const v2d *sD, int t) {
  double a = 0.0;
#pragma unroll
  for (int i = 0; i < ROWS; ++i) {
    const v2d d = sD[i * (kOneWaves * kWave) + t];
    a = __builtin_fma(x[i].x, d.x, a);
    a = __builtin_fma(x[i].y, d.y, a);
    if (i & 1) asm volatile("" : "+v"(a) : : "memory");  // two rows of D in registers, not all
  }
  return wave_sum(a);
}

// What rows past the end of a slice, and steps past the last vector, read.
__device__ const v2d one_zeros[kWave] = {};

__device__ inline double sum_waves(const double *s) {
  return ((s[0] + s[1]) + (s[2] + s[3])) + ((s[4] + s[5]) + (s[6] + s[7]));
}

// Rows of a slice of len doubles that belong to wave w.
__device__ inline int one_rows(int64_t len, int w) {
  const int64_t left = len - 2 * kWave * w;
  return left <= 0 ? 0 : int((left + kOneRow - 1) / kOneRow);
}

// How the members of a group meet, one per group, zero at the start.
struct OneGate {
  int arrived;  // members that have started; kOneApart set: the group works apart
  int parts, done, sums;  // apart: runs of parts begun, ended; slices begun for J
};
constexpr int kOneApart = 1 << 30;
// Apart, a slice's parts go in up to 16 runs of vectors, at least 16 vectors each:
// whoever finds no more of them waits for the last ones.
constexpr int kOneRuns = 16, kOneRunLeast = 16;

// Whether all G members of a group run at the same time, the same answer for each: a
// member waits for the others for `looks` looks (about 1 us each).
__device__ inline bool one_together(OneGate *g, int G, int looks) {
  int v = __hip_atomic_fetch_add(&g->arrived, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) + 1;
  for (int left = looks;; --left) {
    if (v & kOneApart) return false;
    if (v == G) return true;
    if (left <= 0 && __hip_atomic_compare_exchange_strong(&g->arrived, &v, v | kOneApart, __ATOMIC_RELAXED,
                                                          __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT))
      return false;
    __builtin_amdgcn_s_sleep(1);
    v = __hip_atomic_load(&g->arrived, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  }
}

__device__ inline int one_take(int *n) {
  return __hip_atomic_fetch_add(n, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// grid = ngrp * G; workgroup b belongs to group b / G (workgroups start in this order:
// with part of the GPU free the first groups are whole).  Group g takes vectors g,
// g + ngrp, ...  Slice m is pairs [m * slice, (m+1) * slice), slice a multiple of 128
// and at most ROWS rows of 1024.  D: padded densities (stride ldl).
// part[(J * G + m) * ND + d]: the exchange, all kOneEmpty at the start (unused for
// G = 1; G * ND <= 256).
//
// Waiting for another member is safe only while it runs, and other streams may hold
// part of the GPU.  A group whose members have not all started after `looks` looks
// works apart: whoever of it runs takes runs of vectors of a slice and sums its parts of
// their V (nothing is waited for), then, all parts being there, takes slices for J.  That
// is two reads of the vectors, with any number of members, and the same bits.
// Contexts at once on streams of their own, J alone, us, two-pass kernels -> this one, on
// two and on four streams: n=301, 1200 vectors 286 -> 172, 584 -> 379; n=512, 1000 668 ->
// 445, 1329 -> 1305; n=701, 700 876 -> 591, 1721 -> 1712; n=900, 700 1424 -> 1254, 2771 ->
// 2931; n=1100, 600 1821 -> 1164, 3536 -> 3633.  J and K on four: n=301 2186 -> 1629,
// n=701 9552 -> 7925.  (Apart, whole slices at a time in the loop that reads once, with two vectors
// on their way: n=900 on four streams 3574, n=1100 4413.)  With 4096 looks 4 x J at
// n=900 took 23000; 16 or 8 looks: up to +29% at n=301, none gained.
//
// STEP kParts, then kSums in a second launch: every member does that for its own slice
// and waits for nobody, whatever other calls write to the exchange and the gates.
//
// waits: looks (about 1 us each) at what a running member owes, after which V is NaN and
// nothing more is waited for.  A member answers within milliseconds; only a call that
// writes to this one's workspace meanwhile (contexts that share one, or one context,
// on two streams at once) can keep it away for ever.
enum OneStep { kTogether, kParts, kSums };

// The vectors that a workgroup works on: T of its group's from the one with index J0 on.
struct OneRun {
  int64_t J0, p0, len;  // first pair and pairs of the slice
  int ngrp, T;
};

using OneRow = const __attribute__((address_space(1))) v2d *;

// Rows of this wave of vector s of a run; zeros past its end.
template <int ROWS>
__device__ __forceinline__ void one_fetch(const double *__restrict__ L, int64_t ldl, const OneRun &r, int s, int nv, int w,
                                          int lane, v2d (&x)[ROWS]) {
  const uint64_t row = reinterpret_cast<uint64_t>(L + (r.J0 + int64_t(s) * r.ngrp) * ldl + r.p0 + 2 * kWave * w);
  int have = s < r.T ? nv : 0;
  asm("" : "+s"(have));  // one number to compare each row with, not two conditions
#pragma unroll
  for (int i = 0; i < ROWS; ++i)
    x[i] = __builtin_nontemporal_load(
        reinterpret_cast<OneRow>(i < have ? row + i * (kOneRow * sizeof(double)) : reinterpret_cast<uint64_t>(one_zeros)) + lane);
}

// This wave's rows of D to LDS.
template <int ND, int ROWS>
__device__ __forceinline__ void one_dens(const double *__restrict__ D, int64_t ldl, const OneRun &r, int nv, int w, int lane,
                                         v2d (*sD)[ROWS * kOneWaves * kWave]) {
#pragma unroll
  for (int d = 0; d < ND; ++d)
#pragma unroll
    for (int i = 0; i < ROWS; ++i)
      sD[d][(i * kOneWaves + w) * kWave + lane] =
          reinterpret_cast<OneRow>(i < nv ? reinterpret_cast<uint64_t>(D + d * ldl + r.p0 + i * kOneRow + 2 * kWave * w)
                                          : reinterpret_cast<uint64_t>(one_zeros))[lane];
}

template <int ND, int ROWS>
__device__ __forceinline__ void one_add(const v2d (&x)[ROWS], const double *sV, v2d (&acc)[ND][ROWS]) {
#pragma unroll
  for (int d = 0; d < ND; ++d) {
    const double v = sV[d];
#pragma unroll
    for (int i = 0; i < ROWS; ++i) {
      acc[d][i].x = __builtin_fma(x[i].x, v, acc[d][i].x);
      acc[d][i].y = __builtin_fma(x[i].y, v, acc[d][i].y);
      asm volatile("" : "+v"(acc[d][i]));  // summed here, not where it is next read
    }
  }
}

template <int ND, int ROWS>
__device__ __forceinline__ void one_store(const v2d (&acc)[ND][ROWS], int64_t ldl, int grp, const OneRun &r, int nv, int w,
                                          int lane, double *__restrict__ jpart) {
#pragma unroll
  for (int d = 0; d < ND; ++d)
#pragma unroll
    for (int i = 0; i < ROWS; ++i)
      if (i < nv)
        *reinterpret_cast<v2d *>(jpart + (int64_t(grp) * ND + d) * ldl + r.p0 + i * kOneRow + 2 * (kWave * w + lane)) = acc[d][i];
}

// A member's part of V_J(d) to the exchange.
__device__ __forceinline__ void one_publish(const double *sP, double *part) {
  double mine = sum_waves(sP);
  if (__builtin_bit_cast(int64_t, mine) == kOneEmpty) mine = __builtin_nan("");
  __hip_atomic_store(part, mine, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// Parts of V_J of all members (cnt = G ND <= 256 of them), looked for up to `waits` more
// times; waits becomes 0 when they do not come, and V_J is NaN.
__device__ __forceinline__ double one_collect(const double *row, int cnt, int lane, int &waits) {
  double x[4];
  for (int left = waits;; --left) {
    bool ok = true;
    auto look = [&](int k) {
      return __hip_atomic_load(row + min(lane + 64 * k, cnt - 1), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    };
    x[0] = look(0);
    x[1] = x[2] = x[3] = 0.0;
    if (cnt > 128) {
      x[1] = look(1), x[2] = look(2), x[3] = look(3);
    } else if (cnt > 64) {
      x[1] = look(1);
    }
#pragma unroll
    for (int k = 0; k < 4; ++k) ok = ok && __builtin_bit_cast(int64_t, x[k]) != kOneEmpty;
    if (__all(ok)) break;
    if (left <= 0) {
      waits = 0;
      break;
    }
    __builtin_amdgcn_s_sleep(1);
  }
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    asm("" : "+v"(x[k]));  // one select each: merged, they lie on the way from the last part to V (n=701 986, now 984 us)
    x[k] = lane + 64 * k < cnt ? x[k] : 0.0;
  }
  return (x[0] + x[1]) + (x[2] + x[3]);
}

// V_J from the collected parts: entry 2 m + d, even lanes density 0, odd lanes density 1.
template <int ND>
__device__ __forceinline__ void one_total(double y, int lane, double (&v)[ND]) {
  if constexpr (ND == 1) {
    v[0] = wave_sum(y);
  } else {
    v[0] = wave_sum(lane & 1 ? 0.0 : y);
    v[1] = wave_sum(lane & 1 ? y : 0.0);
  }
}

// One slice with nothing to wait for: its parts of V of a run of vectors, or its J with
// all parts there.  Three vectors on their way while one is worked on and one barrier for
// four of them, which the one-read loop has no registers and no time for.
template <int ND, int ROWS, bool SUMS>
__device__ __forceinline__ void one_slice(const double *__restrict__ L, int64_t ldl, const double *__restrict__ D, int grp,
                                          int G, int mem, const OneRun &r, int &waits, double *part,
                                          double *__restrict__ V, double *__restrict__ jpart, int w, int lane,
                                          v2d (*sD)[ROWS * kOneWaves * kWave], double (*sP)[4][ND][kOneWaves],
                                          double (*sV)[4][ND]) {
  const int trips = (r.T + 3) / 4;
  if (w == kOneWaves) {
    if constexpr (SUMS) {
      auto values = [&](int q) {  // V of trip q
        for (int u = 0; u < 4; ++u) {
          const int s = 4 * q + u;
          double v[ND] = {};
          if (s < r.T) {
            const int64_t J = r.J0 + int64_t(s) * r.ngrp;
            one_total<ND>(one_collect(part + J * G * ND, G * ND, lane, waits), lane, v);
            if (mem == 0 && lane == 0) {
#pragma unroll
              for (int d = 0; d < ND; ++d) V[J * ND + d] = v[d];
            }
          }
          if (lane == 0) {
#pragma unroll
            for (int d = 0; d < ND; ++d) sV[q & 1][u][d] = v[d];
          }
        }
      };
      values(0);
      lds_barrier();
      for (int q = 0; q < trips; ++q) {
        values(q + 1);
        lds_barrier();
      }
    } else {
      lds_barrier();
      for (int q = 0; q < trips; ++q) {
        lds_barrier();
        const int u = lane / ND, d = lane % ND, s = 4 * q + u;
        if (lane < 4 * ND && s < r.T)
          one_publish(sP[q & 1][u][d], part + ((r.J0 + int64_t(s) * r.ngrp) * G + mem) * ND + d);
      }
    }
    return;
  }
  const int nv = __builtin_amdgcn_readfirstlane(one_rows(r.len, w));
  v2d buf[4][ROWS], acc[ND][ROWS];
#pragma unroll
  for (int u = 0; u < 3; ++u) one_fetch<ROWS>(L, ldl, r, u, nv, w, lane, buf[u]);
  if constexpr (SUMS) {
#pragma unroll
    for (int d = 0; d < ND; ++d)
#pragma unroll
      for (int i = 0; i < ROWS; ++i) acc[d][i] = v2d{0.0, 0.0};
  } else {
    one_dens<ND, ROWS>(D, ldl, r, nv, w, lane, sD);
  }
  lds_barrier();
  for (int q = 0; q < trips; ++q) {
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      __builtin_amdgcn_sched_barrier(0);  // the buffer has been used before it is loaded again
      one_fetch<ROWS>(L, ldl, r, 4 * q + u + 3, nv, w, lane, buf[(u + 3) % 4]);
      __builtin_amdgcn_sched_barrier(0);
      if constexpr (SUMS) {
        one_add<ND, ROWS>(buf[u], sV[q & 1][u], acc);
      } else {
#pragma unroll
        for (int d = 0; d < ND; ++d) sP[q & 1][u][d][w] = one_dot<ROWS>(buf[u], sD[d], kWave * w + lane);
      }
    }
    lds_barrier();
  }
  if constexpr (SUMS) one_store<ND, ROWS>(acc, ldl, grp, r, nv, w, lane, jpart);
}

template <int ND, int ROWS, OneStep STEP>
__global__ __launch_bounds__((kOneWaves + 1) * kWave) void k_coulomb_one(
    const double *__restrict__ L, int64_t ldl, int64_t M, const double *__restrict__ D, int ngrp, int G, int64_t slice,
    int looks, int waits, OneGate *gate, double *part, double *__restrict__ V, double *__restrict__ jpart) {
  constexpr int R = kOneRing, LAG = R - 3;
  __shared__ __attribute__((aligned(16))) v2d sD[ND][ROWS * kOneWaves * kWave];
  __shared__ double sP[2][4][ND][kOneWaves];
  __shared__ double sV[2][4][ND];
  __shared__ int sTask;  // together: whether; apart: what to do next, < 0: nothing
  const int lane = threadIdx.x & (kWave - 1), w = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
  const int grp = blockIdx.x / G, mem = blockIdx.x % G;
  const int T = int((M - grp + ngrp - 1) / ngrp);  // vectors of the group
  auto run = [&](int m, int s0, int cnt) {
    OneRun r;
    r.J0 = grp + int64_t(s0) * ngrp;
    r.p0 = min(m * slice, ldl);
    r.len = min(slice, ldl - r.p0);
    r.ngrp = ngrp;
    r.T = cnt;
    return r;
  };
  const OneRun r = run(mem, 0, T);
  if constexpr (STEP != kTogether) {
    int none = 0;
    one_slice<ND, ROWS, STEP == kSums>(L, ldl, D, grp, G, mem, r, none, part, V, jpart, w, lane, sD, sP, sV);
    return;
  }

  const int steps = (T + LAG + R - 1) / R * R;
  if (w == kOneWaves) {  // ---- together: the wave that exchanges V
    const bool one = G == 1 || __builtin_amdgcn_readfirstlane(lane == 0 ? one_together(gate + grp, G, looks) : 0);
    if (lane == 0) sTask = one ? 0 : -1;
    lds_barrier();  // D is there
    lds_barrier();  // parts of the first vector
    if (one) {
      for (int s = 0; s < steps; ++s) {
        double v[ND] = {};
        if (G > 1 && s < T && lane < ND)
          one_publish(sP[0][s % R][lane], part + ((grp + int64_t(s) * ngrp) * G + mem) * ND + lane);
        const int64_t J = grp + int64_t(s - LAG) * ngrp;
        const bool have = s >= LAG && s - LAG < T;
        if (have && G == 1) {
#pragma unroll
          for (int d = 0; d < ND; ++d) v[d] = sum_waves(sP[0][(s - LAG) % R][d]);
        }
        if (have && G > 1)  // the others run: their parts come
          one_total<ND>(one_collect(part + J * G * ND, G * ND, lane, waits), lane, v);
        if (lane == 0) {
#pragma unroll
          for (int d = 0; d < ND; ++d) sV[0][s & 1][d] = v[d];
          if (mem == 0 && have) {
#pragma unroll
            for (int d = 0; d < ND; ++d) V[J * ND + d] = v[d];
          }
        }
        lds_barrier();
      }
    }
  } else {  // ---- together: the streaming waves
    const int nv = __builtin_amdgcn_readfirstlane(one_rows(r.len, w));
    v2d buf[R][ROWS], acc[ND][ROWS];
#pragma unroll
    for (int u = 0; u < R; ++u) one_fetch<ROWS>(L, ldl, r, u < 2 ? u : T, nv, w, lane, buf[u]);
    one_dens<ND, ROWS>(D, ldl, r, nv, w, lane, sD);
#pragma unroll
    for (int d = 0; d < ND; ++d)
#pragma unroll
      for (int i = 0; i < ROWS; ++i) acc[d][i] = v2d{0.0, 0.0};
    lds_barrier();
    auto parts = [&](int s, const v2d(&x)[ROWS]) {
#pragma unroll
      for (int d = 0; d < ND; ++d) sP[0][s % R][d][w] = one_dot<ROWS>(x, sD[d], kWave * w + lane);  // the same in every lane
    };
    parts(0, buf[0]);
    lds_barrier();
    // step s: vector s + 2 on its way, parts of s + 1, V of s - LAG
    auto step = [&](int s, v2d(&cur)[ROWS], v2d(&nxt)[ROWS], v2d(&far)[ROWS]) {
      __builtin_amdgcn_sched_barrier(0);  // `far` has been used before it is loaded again
      one_fetch<ROWS>(L, ldl, r, s + 2, nv, w, lane, far);
      __builtin_amdgcn_sched_barrier(0);
      parts(s + 1, nxt);
      lds_barrier();
      one_add<ND, ROWS>(cur, sV[0][s & 1], acc);
    };
    if (__builtin_amdgcn_readfirstlane(sTask) >= 0) {
      for (int s = 0; s < steps; s += R) {  // steps of zeros at both ends
#pragma unroll
        for (int u = 0; u < R; ++u) step(s + u, buf[(u + 3) % R], buf[(u + 1) % R], buf[(u + 2) % R]);
      }
      one_store<ND, ROWS>(acc, ldl, grp, r, nv, w, lane, jpart);
    }
  }
  if (__builtin_amdgcn_readfirstlane(sTask) >= 0) return;

  // ---- apart: a run of a slice's parts, or a slice for J, as they come
  const int runs = max(1, min(kOneRuns, T / kOneRunLeast)), per = (T + runs - 1) / runs;
  for (int mode = kTogether;;) {
    lds_barrier();  // everybody has read sTask
    if (w == kOneWaves && lane == 0) {
      OneGate *g = gate + grp;
      int next = 0, m = mode;
      if (m == kParts) one_take(&g->done);
      if (m != kSums) {
        m = kParts;
        next = one_take(&g->parts);
        if (next >= G * runs) {
          // runs not done are being worked on, and nothing is waited for there
          for (int left = waits; left > 0; --left) {
            if (__hip_atomic_load(&g->done, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) >= G * runs) break;
            __builtin_amdgcn_s_sleep(8);
          }
          m = kSums;
        }
      }
      if (m == kSums) next = one_take(&g->sums);
      sTask = m == kParts || next < G ? next * 4 + m : -1;
    }
    lds_barrier();
    const int task = __builtin_amdgcn_readfirstlane(sTask);
    if (task < 0) return;
    mode = task & 3;
    const int k = task >> 2;
    int ln = lane;
    asm volatile("" : "+v"(ln));  // nothing of the slices is prepared before the loop
    if (mode == kParts)
      one_slice<ND, ROWS, false>(L, ldl, D, grp, G, k / runs, run(k / runs, k % runs * per, max(0, min(per, T - k % runs * per))),
                                 waits, part, V, jpart, w, ln, sD, sP, sV);
    else
      one_slice<ND, ROWS, true>(L, ldl, D, grp, G, k, run(k, 0, T), waits, part, V, jpart, w, ln, sD, sP, sV);
  }
}

// Copies nd densities of stride ldd into the zero-padded staging buffer of
// stride ldl; on the way nempty elements of `part` become kOneEmpty and nzero
// after them 0.
__global__ void k_pack_dens(const double *__restrict__ dlt, int64_t ldd, int64_t np,
                            int64_t ldl, double *__restrict__ out, int64_t *__restrict__ part, int64_t nempty,
                            int64_t nzero) {
  const int64_t p = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
  const int d = blockIdx.y;
  const int64_t threads = int64_t(gridDim.x) * blockDim.x;
  for (int64_t i = p + d * threads; i < nempty + nzero; i += threads * gridDim.y) part[i] = i < nempty ? kOneEmpty : 0;
  if (p >= ldl) return;
  out[d * ldl + p] = (p < np) ? dlt[d * ldd + p] : 0.0;
}

// ---- many densities (3..16): both passes on FP64 MFMA ---------------------
// With nd densities each vector element is used nd times; the per-vector
// kernels above would re-read every density for every vector.  Both passes
// below read each L element once per pass and each density (or V) element
// once per 64 vectors: still HBM-bound, at the single-density byte count.
// MFMA v_mfma_f64_16x16x4f64: lane l supplies A[l%16][l/16] and B[l/16][l%16];
// result register r holds row 4r + l/16, column l%16.
__device__ inline v4d mfma64(double a, double b, v4d c) {
  return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
}

// Pass 1 as V = L D^T.  grid = (ceil(M/VM), nsplit); workgroup (x, s) stages
// VM vectors x VK pairs of L (rows read in VK*8-byte runs with 16-byte loads)
// and the same VK pairs of the densities in LDS, the next chunk being fetched
// to registers meanwhile.  Row tile rt = w / WPT of 16 vectors is contracted
// by WPT waves, each taking every WPT-th group of k-steps; their partial
// tiles are summed through LDS.  vpart[(s*M + J)*nd + d].
template <int VM, int VK>
__global__ __launch_bounds__(kThreads) void k_coulomb_v_tile(
    const double *__restrict__ L, int64_t ldl, int64_t M, const double *__restrict__ D, int nd,
    int64_t pchunk, double *__restrict__ vpart) {
  constexpr int RT = VM / 16, WPT = 4 / RT, KS = VK / 4 / WPT;
  constexpr int NL = VM * VK / 2 / kThreads, NDD = 16 * VK / 2 / kThreads;
  static_assert(NL >= 1 && NDD >= 1 && KS >= 1, "tile shape");
  __shared__ double sL[VM][VK + 1];
  __shared__ double sD[16][VK + 1];
  const int64_t J0 = int64_t(blockIdx.x) * VM;
  const int64_t p0 = int64_t(blockIdx.y) * pchunk;
  const int64_t p1 = min(p0 + pchunk, ldl);
  const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
  const int rt = w / WPT, wk = w % WPT;
  v4d acc = {0.0, 0.0, 0.0, 0.0};
  v2d rl[NL], rd[NDD];
  // Out-of-range rows (vectors >= M, densities >= nd) load row 0 and are
  // zeroed when stashed, so the chunk's loads stay in flight across the
  // multiply of the previous chunk.
  auto fetch = [&](int64_t pc) {
#pragma unroll
    for (int i = 0; i < NL; ++i) {
      const int e = tid + kThreads * i, r = e / (VK / 2), k2 = e % (VK / 2);
      rl[i] = __builtin_nontemporal_load(
          reinterpret_cast<const v2d *>(L + (J0 + r < M ? J0 + r : 0) * ldl + pc + 2 * k2));
    }
#pragma unroll
    for (int i = 0; i < NDD; ++i) {
      const int e = tid + kThreads * i, d = e / (VK / 2), k2 = e % (VK / 2);
      rd[i] = *reinterpret_cast<const v2d *>(D + (d < nd ? d : 0) * ldl + pc + 2 * k2);
    }
  };
  if (p0 < p1) fetch(p0);
  for (int64_t pc = p0; pc < p1; pc += VK) {
    if (pc != p0) __syncthreads();
#pragma unroll
    for (int i = 0; i < NL; ++i) {
      const int e = tid + kThreads * i, r = e / (VK / 2), k2 = e % (VK / 2);
      const bool ok = J0 + r < M;
      sL[r][2 * k2] = ok ? rl[i].x : 0.0;
      sL[r][2 * k2 + 1] = ok ? rl[i].y : 0.0;
    }
#pragma unroll
    for (int i = 0; i < NDD; ++i) {
      const int e = tid + kThreads * i, d = e / (VK / 2), k2 = e % (VK / 2);
      sD[d][2 * k2] = d < nd ? rd[i].x : 0.0;
      sD[d][2 * k2 + 1] = d < nd ? rd[i].y : 0.0;
    }
    __syncthreads();
    if (pc + VK < p1) fetch(pc + VK);
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) {
      const int k = (ks * WPT + wk) * 4 + (lane >> 4);
      acc = mfma64(sL[16 * rt + (lane & 15)][k], sD[lane & 15][k], acc);
    }
  }
  if constexpr (WPT > 1) {
    __syncthreads();
    double *red = &sL[0][0];  // WPT-1 partial tiles per row tile: 4 x 64 doubles each
    if (wk > 0) {
#pragma unroll
      for (int r = 0; r < 4; ++r) red[((rt * (WPT - 1) + wk - 1) * 4 + r) * 64 + lane] = acc[r];
    }
    __syncthreads();
    if (wk > 0) return;
#pragma unroll
    for (int q = 0; q < WPT - 1; ++q)
#pragma unroll
      for (int r = 0; r < 4; ++r) acc[r] += red[((rt * (WPT - 1) + q) * 4 + r) * 64 + lane];
  }
  const int d = lane & 15;
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    const int64_t J = J0 + 16 * rt + 4 * r + (lane >> 4);
    if (J < M && d < nd) vpart[(int64_t(blockIdx.y) * M + J) * nd + d] = acc[r];
  }
}

// Pass 2 as J^T = V^T L, L streamed from HBM straight into registers.
// grid = (ldl/512, nsplit).  Wave w of workgroup (x, s) owns the 128 pairs
// from 512x + 128w; per step of 4 vectors J..J+3, lane l (n = l%16, g = l/16)
// loads L[J + g][base + 32i + 2n .. + 1] for i < 4 (16 lanes cover 256
// contiguous bytes of a row), and MFMA (i, c) produces output columns
// base + 32i + 2n + c.  A operand: V[J + l/16][l%16].  Groups of U steps are
// fetched one group ahead.  jpart[(s*nd + d)*ldl + p].
template <int U>
__global__ __launch_bounds__(kThreads) void k_coulomb_j_stream(
    const double *__restrict__ L, int64_t ldl, int64_t M, const double *__restrict__ V, int nd,
    int64_t jchunk, double *__restrict__ jpart) {
  const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
  const int n16 = lane & 15, g = lane >> 4;
  const int64_t pw = int64_t(blockIdx.x) * 512 + 128 * w + 2 * n16;
  const int64_t ja = int64_t(blockIdx.y) * jchunk;
  const int64_t jz = min(ja + jchunk, M);
  const int ngrp = int(jz > ja ? (jz - ja + 4 * U - 1) / (4 * U) : 0);
  v4d acc[8];
#pragma unroll
  for (int t = 0; t < 8; ++t) acc[t] = v4d{0.0, 0.0, 0.0, 0.0};
  v2d la[U][4], lb[U][4];
  double va[U], vb[U];
  auto fetch = [&](int q, v2d(&x)[U][4], double(&v)[U]) {
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int64_t J = ja + int64_t(q) * 4 * U + 4 * u + g;
      const bool ok = J < jz;
      const double *__restrict__ row = L + (ok ? J : ja) * ldl + pw;
#pragma unroll
      for (int i = 0; i < 4; ++i)
        x[u][i] = ok ? __builtin_nontemporal_load(reinterpret_cast<const v2d *>(row + 32 * i))
                     : v2d{0.0, 0.0};
      v[u] = (ok && n16 < nd) ? V[J * nd + n16] : 0.0;
    }
  };
  auto body = [&](int q, v2d(&cur)[U][4], double(&vc)[U], v2d(&nxt)[U][4], double(&vn)[U]) {
    if (q + 1 < ngrp) fetch(q + 1, nxt, vn);
#pragma unroll
    for (int u = 0; u < U; ++u)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        acc[2 * i] = mfma64(vc[u], cur[u][i].x, acc[2 * i]);
        acc[2 * i + 1] = mfma64(vc[u], cur[u][i].y, acc[2 * i + 1]);
      }
  };
  if (ngrp > 0) {
    fetch(0, la, va);
    for (int q = 0; q < ngrp; q += 2) {
      body(q, la, va, lb, vb);
      if (q + 1 < ngrp) body(q + 1, lb, vb, la, va);
    }
  }
  // acc[t][rr]: density 4rr + g, pair pw + t
#pragma unroll
  for (int rr = 0; rr < 4; ++rr) {
    const int m = 4 * rr + g;
    if (m < nd) {
      double *__restrict__ out = jpart + (int64_t(blockIdx.y) * nd + m) * ldl + pw;
#pragma unroll
      for (int i = 0; i < 4; ++i)
        *reinterpret_cast<v2d *>(out + 32 * i) = v2d{acc[2 * i][rr], acc[2 * i + 1][rr]};
    }
  }
}

template <int JB, int ND>
void launch_v(Context *c, const double *D, int nd, double *vpart, int nsplit, int64_t pchunk) {
  dim3 grid(unsigned(ceil_div(c->nchol, JB)), unsigned(nsplit));
  hipLaunchKernelGGL((k_coulomb_v<JB, ND>), grid, dim3(kThreads), 0, c->stream, c->L, c->ldl,
                     c->nchol, D, nd, pchunk, vpart);
}

// Row segments per workgroup of the J pass for one or two densities (8 KiB runs per
// vector row, measured faster than one).
constexpr int kJWidth = 2;

template <int ND>
void launch_j(Context *c, const double *V, int nd, double *jpart, int nsplit, int64_t jchunk) {
  constexpr int W = kJWidth, U = 4;
  dim3 grid(unsigned(ceil_div(c->ldl / kSeg, W)), unsigned(nsplit));
  hipLaunchKernelGGL((k_coulomb_j<ND, W, U>), grid, dim3(kThreads), 0, c->stream, c->L, c->ldl,
                     c->nchol, V, nd, jchunk, jpart);
}

// w[J] = ||L^J||_F^2 of the full symmetric matrix = 2 sum_p L_p^2 - sum_a L_aa^2.
// grid = M, one workgroup per vector.
__global__ __launch_bounds__(kThreads) void k_vector_norms(const double *__restrict__ L,
                                                           int64_t ldl, int64_t np, int n,
                                                           double *__restrict__ w) {
  __shared__ double lds[4];
  const double *__restrict__ row = L + int64_t(blockIdx.x) * ldl;
  double s[1] = {0.0};
  for (int64_t p = threadIdx.x; p < np; p += kThreads) s[0] += 2.0 * row[p] * row[p];
  for (int a = threadIdx.x; a < n; a += kThreads) {
    const double x = row[int64_t(a) * (a + 1) / 2 + a];
    s[0] -= x * x;
  }
  block_sum<1>(s, lds);
  if (threadIdx.x == 0) w[blockIdx.x] = s[0];
}

}  // namespace

int vector_norms(Context *c, double *w) {
  if (!w) return set_error(c, MJK_ERR_ARG, "vector_norms: null pointer");
  if (c->nloaded != c->nchol)
    return set_error(c, MJK_ERR_SHORT_READ, "vector_norms: not all Cholesky vectors were uploaded");
  hipLaunchKernelGGL(k_vector_norms, dim3(unsigned(c->nchol)), dim3(kThreads), 0, c->stream, c->L,
                     c->ldl, c->np, c->n, w);
  return hip_check(c, hipGetLastError(), "vector_norms launch");
}

namespace {

constexpr size_t kScratchBytes = size_t(64) << 20;  // the fixed buffer of coulomb_noalloc, below

// Work split and scratch of one Coulomb build (both passes).
struct CoulombPlan {
  bool tile = false;                   // nd >= 3: the MFMA passes
  int group = 0, ngrp = 0;             // one pass: workgroups per group, groups (0: two passes)
  int64_t slice = 0, nparts = 0;       // one pass: pairs per workgroup; parts of V to exchange
  int nsplit1 = 0, nsplit2 = 0;
  int64_t nblk = 0, pchunk = 0, jchunk = 0;
  size_t bytes_d = 0, bytes_vpart = 0, bytes_v = 0, bytes_jpart = 0;
};

constexpr int kTileVM = 64, kTileVK = 64, kTileU = 4;  // MFMA passes (nd >= 3)

inline size_t piece(size_t bytes) { return size_t(round_up(int64_t(bytes), 256)); }

// Pass 2 split of the streaming J pass: about 1024 workgroups of two segments, at
// least eight vectors each (a slice of one vector costs more to write and reduce than
// to read).
void plan_j_stream(const Context *c, int nd, CoulombPlan *p) {
  const int64_t M = c->nchol, nseg = c->ldl / kSeg;
  const int64_t nxj = ceil_div(nseg, kJWidth);
  int nsplit2 = int(std::min<int64_t>(std::max<int64_t>(ceil_div(2048 / kJWidth, nxj), 1), M));
  p->jchunk = std::max<int64_t>(ceil_div(M, nsplit2), 8);
  p->nsplit2 = int(ceil_div(M, p->jchunk));
  p->bytes_jpart = sizeof(double) * size_t(p->nsplit2) * nd * c->ldl;
}

// Rows of 1024 pairs per workgroup of the one-pass kernel (register budget: four
// vectors and the J of each density, three waves per SIMD).
constexpr int one_rows_max(int nd) { return nd == 1 ? 6 : 5; }
constexpr int kOneGrid = 256;  // workgroups at most: one per CU, as many as there are

// The one-pass kernel takes one or two densities from 8192 pairs on (n = 131, 524
// vectors: 34 us, 38 in two passes; n = 110: 36 against 31, the members' meeting is not
// hidden) up to 786432, so that there are two groups (n = 1200: 4970 against 8630 us;
// n = 1300, 200 vectors, one group: 403 against 474 alone but 1006 against 889 on two
// streams).  Groups: as many as fit, with at least eight vectors each, below which
// their J costs more to write and reduce than the wait for V (n = 130: 33.8 us with
// two each, 29.8 with eight), but up to 32 when vectors are few (n = 500, 16 vectors:
// 36 us in two groups, 28 in eight).  Its scratch stays within the fixed buffer of
// coulomb_noalloc (tens of thousands of vectors reach it), so that entry takes what
// the two passes take.
bool plan_one(const Context *c, int nd, CoulombPlan *p) {
  const int64_t M = c->nchol, ldl = c->ldl;
  if (nd > 2 || ldl < 8192) return false;
  const int64_t gmin = ceil_div(ldl, kOneRow * one_rows_max(nd));
  const int64_t grid = std::min(kOneGrid, c->ncu);
  if (gmin > grid / 2 || gmin * nd > 256) return false;
  const int64_t want = std::max<int64_t>({M / 8, std::min<int64_t>(M / 2, 32), 1});
  const int64_t ngrp = std::min<int64_t>(grid / gmin, want);
  const int64_t slice = round_up(ceil_div(ldl, std::min<int64_t>(grid / ngrp, 256 / nd)), 2 * kWave);
  const int64_t group = ceil_div(ldl, slice);
  if ((M * (group + 1) + (ngrp + 1) * ldl) * nd * sizeof(double) > kScratchBytes - 65536) return false;
  p->ngrp = int(ngrp);
  p->slice = slice;
  p->group = int(group);
  p->nsplit2 = p->ngrp;
  p->nparts = p->group > 1 ? M * p->group * nd : 0;
  p->bytes_vpart = sizeof(double) * size_t(p->nparts) + sizeof(OneGate) * size_t(p->ngrp);
  p->bytes_jpart = sizeof(double) * size_t(p->ngrp) * nd * ldl;
  return true;
}

CoulombPlan plan_coulomb(const Context *c, int nd) {
  CoulombPlan p;
  const int64_t M = c->nchol, ldl = c->ldl;
  p.bytes_d = sizeof(double) * size_t(nd) * ldl;
  p.bytes_v = sizeof(double) * size_t(M) * nd;
  if (plan_one(c, nd, &p)) return p;
  if (nd >= 3) {
    p.tile = true;
    p.nblk = ceil_div(M, kTileVM);
    const int64_t nk = ldl / kTileVK;
    int nsplit1 = int(std::min<int64_t>(std::max<int64_t>(ceil_div(2048, p.nblk), 1), nk));
    p.pchunk = ceil_div(nk, nsplit1) * kTileVK;  // whole chunks: ldl % VK == 0
    p.nsplit1 = int(ceil_div(ldl, p.pchunk));
    const int64_t npc = ldl / 512;
    int nsplit2 = int(std::min<int64_t>(std::max<int64_t>(ceil_div(2048, npc), 1),
                                        ceil_div(M, 4 * kTileU)));
    p.jchunk = round_up(ceil_div(M, nsplit2), 4 * kTileU);
    p.nsplit2 = int(ceil_div(M, p.jchunk));
    p.bytes_jpart = sizeof(double) * size_t(p.nsplit2) * nd * ldl;
  } else {
    const int jb = 8;
    p.nblk = ceil_div(M, jb);
    const int64_t nseg = ldl / kSeg;
    int nsplit1 = int(std::min<int64_t>(std::max<int64_t>(ceil_div(2048, p.nblk), 1), nseg));
    p.pchunk = ceil_div(nseg, nsplit1) * kSeg;
    p.nsplit1 = int(ceil_div(ldl, p.pchunk));
    plan_j_stream(c, nd, &p);
  }
  p.bytes_vpart = sizeof(double) * size_t(p.nsplit1) * M * nd;
  return p;
}

// Where the passes put their scratch: the context's grow-only workspaces, or
// (arena set) consecutive 256-byte pieces of a fixed device buffer that is
// neither allocated nor freed here.
struct Scratch {
  double *arena = nullptr;
  size_t cap = 0, used = 0;  // bytes
};

int take(Context *c, Scratch &s, DevBuf &ws, size_t bytes, double **out) {
  if (!s.arena) {
    const int rc = ensure(c, ws, bytes);
    if (rc) return rc;
    *out = static_cast<double *>(ws.ptr);
    return MJK_OK;
  }
  if (s.used + piece(bytes) > s.cap)
    return set_error(c, MJK_ERR_ARG, "coulomb: scratch exceeds the fixed buffer");
  *out = s.arena + s.used / sizeof(double);
  s.used += piece(bytes);
  return MJK_OK;
}

// Pass 2 for one or two densities: J = L V, then the fixed-order reduction of the vector slices into jlt.
int j_pass(Context *c, Scratch &s, const CoulombPlan &p, int nd, const double *V, double *jlt,
           int64_t ldj) {
  int rc;
  double *jpart;
  if ((rc = take(c, s, c->w->jpart, p.bytes_jpart, &jpart))) return rc;
  phase_begin(c);
  if (nd == 1) launch_j<1>(c, V, nd, jpart, p.nsplit2, p.jchunk);
  else launch_j<2>(c, V, nd, jpart, p.nsplit2, p.jchunk);
  phase_end(c, MJK_PHASE_COULOMB_J);
  phase_begin(c);
  hipLaunchKernelGGL(k_reduce_j, dim3(unsigned(ceil_div(c->np, 64)), unsigned(nd)), dim3(256), 0,
                     c->stream, jpart, c->ldl, c->np, nd, p.nsplit2, jlt, ldj);
  phase_end(c, MJK_PHASE_REDUCE);
  return hip_check(c, hipGetLastError(), "coulomb launch");
}

int coulomb_run(Context *c, Scratch &s, int32_t nd, const double *dlt, int64_t ldd, double *jlt,
                int64_t ldj, double *v_out) {
  if (nd < 1 || nd > 16) return set_error(c, MJK_ERR_ARG, "coulomb: nd must be in [1,16]");
  if (ldd < c->np || ldj < c->np) return set_error(c, MJK_ERR_ARG, "coulomb: ld < nbas(nbas+1)/2");
  if (c->nloaded != c->nchol)
    return set_error(c, MJK_ERR_SHORT_READ, "coulomb: not all Cholesky vectors were uploaded");
  const int64_t M = c->nchol, ldl = c->ldl;
  const CoulombPlan p = plan_coulomb(c, nd);
  int rc;
  double *Dp, *vpart, *V;
  // staging copy of the densities (zero padded to ldl)
  if ((rc = take(c, s, c->w->d, p.bytes_d, &Dp)) || (rc = take(c, s, c->w->vpart, p.bytes_vpart, &vpart)))
    return rc;
  if (v_out) V = v_out;
  else if ((rc = take(c, s, c->w->v, p.bytes_v, &V))) return rc;
  phase_begin(c);
  hipLaunchKernelGGL(k_pack_dens, dim3(unsigned(ceil_div(ldl, 256)), unsigned(nd)), dim3(256), 0,
                     c->stream, dlt, ldd, c->np, ldl, Dp, reinterpret_cast<int64_t *>(vpart),
                     p.nparts, p.group > 1 ? int64_t(sizeof(OneGate) / 8) * p.ngrp : 0);
  phase_end(c, MJK_PHASE_PACK);

  if (p.group) {
    double *jpart;
    if ((rc = take(c, s, c->w->jpart, p.bytes_jpart, &jpart))) return rc;
    const dim3 grid(unsigned(p.ngrp * p.group)), block((kOneWaves + 1) * kWave);
    OneGate *gate = reinterpret_cast<OneGate *>(vpart + p.nparts);
    auto one = [&](auto kernel, int phase) {
      phase_begin(c);
      hipLaunchKernelGGL(kernel, grid, block, 0, c->stream, c->L, ldl, M, Dp, p.ngrp, p.group, p.slice, c->coulomb_looks,
                         c->coulomb_waits, gate, vpart, V, jpart);
      phase_end(c, phase);
    };
    constexpr int R1 = one_rows_max(1), R2 = one_rows_max(2);
    // The fixed buffer may be written by an overlapping call, so nothing is waited for
    // in it: two reads of the vectors, the same bits.
    if (s.arena && p.group > 1) {
      one(nd == 1 ? k_coulomb_one<1, R1, kParts> : k_coulomb_one<2, R2, kParts>, MJK_PHASE_COULOMB_V);
      one(nd == 1 ? k_coulomb_one<1, R1, kSums> : k_coulomb_one<2, R2, kSums>, MJK_PHASE_COULOMB_J);
    } else {
      one(nd == 1 ? k_coulomb_one<1, R1, kTogether> : k_coulomb_one<2, R2, kTogether>, MJK_PHASE_COULOMB_J);
    }
    phase_begin(c);
    hipLaunchKernelGGL(k_reduce_j, dim3(unsigned(ceil_div(c->np, 64)), unsigned(nd)), dim3(256), 0, c->stream, jpart,
                       ldl, c->np, nd, p.ngrp, jlt, ldj);
    phase_end(c, MJK_PHASE_REDUCE);
    return hip_check(c, hipGetLastError(), "coulomb launch");
  }

  if (p.tile) {
    // ---- pass 1: V = L D^T, split over pairs to fill the device
    phase_begin(c);
    hipLaunchKernelGGL((k_coulomb_v_tile<kTileVM, kTileVK>), dim3(unsigned(p.nblk), unsigned(p.nsplit1)),
                       dim3(kThreads), 0, c->stream, c->L, ldl, M, Dp, nd, p.pchunk, vpart);
    phase_end(c, MJK_PHASE_COULOMB_V);
    phase_begin(c);
    hipLaunchKernelGGL(k_reduce_v, dim3(unsigned(ceil_div(M * nd, 256))), dim3(256), 0, c->stream,
                       vpart, M, nd, p.nsplit1, V);
    phase_end(c, MJK_PHASE_REDUCE);
    // ---- pass 2: J = L^T V, split over vectors
    double *jpart;
    if ((rc = take(c, s, c->w->jpart, p.bytes_jpart, &jpart))) return rc;
    phase_begin(c);
    hipLaunchKernelGGL(k_coulomb_j_stream<kTileU>, dim3(unsigned(ldl / 512), unsigned(p.nsplit2)),
                       dim3(kThreads), 0, c->stream, c->L, ldl, M, V, nd, p.jchunk, jpart);
    phase_end(c, MJK_PHASE_COULOMB_J);
    phase_begin(c);
    hipLaunchKernelGGL(k_reduce_j, dim3(unsigned(ceil_div(c->np, 64)), unsigned(nd)), dim3(256), 0,
                       c->stream, jpart, ldl, c->np, nd, p.nsplit2, jlt, ldj);
    phase_end(c, MJK_PHASE_REDUCE);
    return hip_check(c, hipGetLastError(), "coulomb launch");
  }

  // ---- pass 1: V = L^T D
  phase_begin(c);
  if (nd == 1) launch_v<8, 1>(c, Dp, nd, vpart, p.nsplit1, p.pchunk);
  else launch_v<8, 2>(c, Dp, nd, vpart, p.nsplit1, p.pchunk);
  phase_end(c, MJK_PHASE_COULOMB_V);
  phase_begin(c);
  hipLaunchKernelGGL(k_reduce_v, dim3(unsigned(ceil_div(M * nd, 256))), dim3(256), 0, c->stream,
                     vpart, M, nd, p.nsplit1, V);
  phase_end(c, MJK_PHASE_REDUCE);
  return j_pass(c, s, p, nd, V, jlt, ldj);
}

// ---- the allocation-free Coulomb build ----------------------------------
// Its scratch is one fixed device array per GPU, allocated with the code
// object and held until the process ends.  Host code uses the address that
// hipGetSymbolAddress returns for the current device, never the array's name
// (that is a host-side stand-in, not a device address).
constexpr int kMaxDevices = 64;
__device__ __align__(256) double scratch[kScratchBytes / sizeof(double)];

}  // namespace

// Device address of this GPU's scratch array, looked up once per device (with
// that device current) and cached.
static int scratch_device_ptr(Context *c, double **out) {
  static double *ptr[kMaxDevices] = {};
  static std::mutex mu;
  if (c->device < 0 || c->device >= kMaxDevices)
    return set_error(c, MJK_ERR_ARG, "coulomb_noalloc: device index out of range");
  std::lock_guard<std::mutex> lock(mu);
  if (!ptr[c->device]) {
    int cur = -1;
    int rc;
    if ((rc = hip_check(c, hipGetDevice(&cur), "hipGetDevice"))) return rc;
    if (cur != c->device)
      return set_error(c, MJK_ERR_STATE, "coulomb_noalloc: the context's device is not current");
    void *p = nullptr;
    if ((rc = hip_check(c, hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)), "hipGetSymbolAddress(scratch)")))
      return rc;
    ptr[c->device] = static_cast<double *>(p);
  }
  *out = ptr[c->device];
  return MJK_OK;
}

int coulomb(Context *c, int32_t nd, const double *dlt, int64_t ldd, double *jlt, int64_t ldj,
            double *v_out) {
  Scratch s;  // the context's workspaces
  return coulomb_run(c, s, nd, dlt, ldd, jlt, ldj, v_out);
}

int coulomb_noalloc(Context *c, int32_t nd, const double *dlt, int64_t ldd, double *jlt, int64_t ldj,
                    double *v_out) {
  if (nd < 1 || nd > 16) return set_error(c, MJK_ERR_ARG, "coulomb: nd must be in [1,16]");
  const CoulombPlan p = plan_coulomb(c, nd);
  const size_t need = piece(p.bytes_d) + piece(p.bytes_vpart) + piece(p.bytes_jpart) +
                      (v_out ? 0 : piece(p.bytes_v));
  if (need > kScratchBytes)
    return set_error(c, MJK_ERR_ARG,
                     "coulomb_noalloc: this build needs " + std::to_string(need >> 20) +
                         " MiB of scratch, more than the fixed " +
                         std::to_string(kScratchBytes >> 20) + " MiB");
  Scratch s;
  int rc;
  if ((rc = scratch_device_ptr(c, &s.arena))) return rc;
  s.cap = kScratchBytes;
  return coulomb_run(c, s, nd, dlt, ldd, jlt, ldj, v_out);
}

namespace {
int coulomb_exchange_run(Context *c, const double *dlt, int64_t ldd, double *jlt, int64_t ldj,
                         int32_t nk, const int32_t *nocc, const double *const *corb, double *klt,
                         int64_t ldk, double *v_out) {
  if (ldd < c->np || ldj < c->np) return set_error(c, MJK_ERR_ARG, "coulomb: ld < nbas(nbas+1)/2");
  if (c->nloaded != c->nchol)
    return set_error(c, MJK_ERR_SHORT_READ, "coulomb: not all Cholesky vectors were uploaded");
  if (nk < 1 || !nocc) return set_error(c, MJK_ERR_ARG, "exchange: nk < 1");
  int64_t tot = 0;
  for (int d = 0; d < nk; ++d) tot += std::max(nocc[d], 0);
  int rc;
  if (tot == 0) {  // no half-transform to carry the V pass
    if ((rc = coulomb(c, 1, dlt, ldd, jlt, ldj, v_out))) return rc;
    return exchange(c, nk, nocc, corb, klt, ldk, MJK_PREC_FP64);
  }
  const int64_t M = c->nchol;
  const int ntmax = int(ceil_div(c->n, 16));  // at most one wave per 16 columns
  if ((rc = ensure(c, c->w->vpart, sizeof(double) * size_t(ntmax) * M)) ||
      (rc = ensure(c, c->w->v, sizeof(double) * M)))
    return rc;
  double *vpart = static_cast<double *>(c->w->vpart.ptr);
  double *V = v_out ? v_out : static_cast<double *>(c->w->v.ptr);
  // the fused pass must not outlive this call on any return path
  struct FuseReset {
    Context *c;
    ~FuseReset() { c->fv = FuseV{}; }
  } fuse_reset{c};
  // the half-transform reads the caller's density at packed indices < nbas(nbas+1)/2
  // only (masked elements read index 0), so no padded copy is needed
  c->fv.p = dlt;
  c->fv.vpart = vpart;
  c->fv.m = M;
  c->fv.ntile = 0;
  if ((rc = exchange(c, nk, nocc, corb, klt, ldk, MJK_PREC_FP64))) return rc;
  const int ntile = c->fv.ntile;
  c->fv = FuseV{};
  if (ntile < 1 || ntile > ntmax)
    return set_error(c, MJK_ERR_ARG, "coulomb_exchange: the half-transform did not run");
  phase_begin(c);
  hipLaunchKernelGGL(k_reduce_v, dim3(unsigned(ceil_div(M, 256))), dim3(256), 0, c->stream, vpart,
                     M, 1, ntile, V);
  phase_end(c, MJK_PHASE_REDUCE);
  CoulombPlan p;
  plan_j_stream(c, 1, &p);
  Scratch s;  // the context's workspaces
  return j_pass(c, s, p, 1, V, jlt, ldj);
}

}  // namespace

int coulomb_exchange(Context *c, const double *dlt, int64_t ldd, double *jlt, int64_t ldj,
                     int32_t nk, const int32_t *nocc, const double *const *corb, double *klt,
                     int64_t ldk, double *v_out) {
  return coulomb_exchange_run(c, dlt, ldd, jlt, ldj, nk, nocc, corb, klt, ldk, v_out);
}

}  // namespace mjk
