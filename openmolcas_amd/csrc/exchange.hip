// Exchange (K) build: half-transform X^J = C^T L^J and K = sum_J X^J^T X^J.
//
// Reference: Cho_X_getVtra -> CHO_VTRA iSwap=2 (src/cholesky_util/cho_vtra.F90:
// 318-363), a scatter-AXPY over reduced-set pairs, followed by DGEMM_Tri
// (src/linalg_util/dgemm_tri.F90:122-147), a lower-triangle SYRK over the merged
// (k,J) index executed as per-column DGEMV (src/fock_util/cho_fscf.F90:276).
//
// MI355X design:
//  * All orbital sets of one call are concatenated into one "orbital bank"
//    Cb[b][k] (AO row b, orbital column k; every set starts at a multiple of 4
//    columns, padded with zeros), so ONE pass over L serves every density.
//  * Half-transform X[J][k][a] (a fastest): FP64 k_ht64, L from memory into MFMA
//    registers; FP32 k_ht, a workgroup per (vector J, AO tile) that unpacks the
//    packed-triangle block L^J[b0:b0+BK, tile] into a square LDS tile (mirroring
//    across the diagonal; the reference's 1/2 on diagonal pairs added twice is
//    the same as taking the diagonal once).  Workgroups of one vector are placed
//    on one XCD so that the two reads of every packed element (as row and as
//    transposed column) share that XCD's L2.
//  * SYRK: a workgroup owns one tile (A >= B) of K and a slice of the
//    vectors; it contracts over (J, k in the density's bank columns) with
//    MFMA (FP64: k_syrk64, operands straight from memory into registers) and
//    writes an FP64 partial tile.  A final
//    deterministic reduction sums the slices into LT storage.
#include <type_traits>

#include "mjk_internal.h"

namespace mjk {
namespace {

constexpr int kThreads = 256;

// 16x16x4 products: lane l holds A[l%16][l/16] and B[l/16][l%16].  Register r of the
// result is row 4 r + l/16 in FP64, row32(l, r) in FP32, column l%16.
__device__ inline v4d mma64(double a, double b, v4d c) { return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0); }
__device__ inline v4f mma32(float a, float b, v4f c) { return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0); }
__device__ inline int row32(int lane, int r) { return 4 * (lane >> 4) + r; }

// FP32 SYRK partial sums are folded into FP64 registers every kFlushRows
// contraction rows, so no FP32 sum runs over more than kFlushRows products.
constexpr int kFlushRows = 512;

// Densities of one SYRK launch: workgroup b belongs to the set d with
// item0[d] <= b < item0[d+1]; inside it, tile = local % ntiles and slice
// s = local / ntiles.  Set d contracts over bank columns off..off+opad-1 and
// writes partial tiles at kpart + kbase[d].
constexpr int kMaxSets = 16;
struct SyrkSets {
  int n;
  int off[kMaxSets];
  int opad[kMaxSets];
  int nsplit[kMaxSets];
  int item0[kMaxSets + 1];
  int64_t kbase[kMaxSets];
};

// The same for the FP64 SYRK (k_syrk64): 64x64 tiles only, the off-diagonal and
// the diagonal tiles sliced separately (nsf / nsd slices), because a diagonal
// tile costs 10 MFMAs per step where an off-diagonal one costs 16.  Set d owns
// the blocks item0[d] .. item0[d+1]-1 (multiples of 8: block b runs on XCD
// b % 8) and the partial tiles at kf[d] (off-diagonal) and kd[d] (diagonal).
constexpr int kT64 = 64;
constexpr int kSlot64 = kT64 * kT64;
struct Syrk64Sets {
  int n;
  int off[kMaxSets];
  int opad[kMaxSets];
  int nsf[kMaxSets], nsd[kMaxSets];
  int item0[kMaxSets + 1];
  int64_t kf[kMaxSets], kd[kMaxSets];
};

// K tiles and vector slices that screening decides on (k_keep), `strips` 64-AO strips
// to a side, ntiles in the lower triangle: set d owns the flags item0[d] + tile *
// nref[d] + slice.
struct ScreenSets {
  int n, strips, ntiles;
  int nref[kMaxSets];
  int item0[kMaxSets + 1];
};

__device__ inline int find_set(const SyrkSets &sets, int b) {
  int d = 0;
  while (d + 1 < sets.n && b >= sets.item0[d + 1]) ++d;
  return d;
}

__device__ inline int64_t tri0(int64_t a) { return a * (a + 1) / 2; }
// Offset of packed row a within one vector in 32-bit arithmetic: contexts hold
// at most 46340 basis functions, so a(a+1) and the triangle fit in 32 bits.
__device__ inline uint32_t tri0u(uint32_t a) { return a * (a + 1u) / 2u; }

// Maps blockIdx.x so that consecutive logical blocks land on the same XCD
// (hardware dispatches block i to XCD i % 8).  Returns -1 for padding blocks.
__device__ inline int64_t xcd_logical(int64_t nblocks) {
  const int64_t g = gridDim.x;  // multiple of 8
  const int64_t b = blockIdx.x;
  const int64_t l = (b & 7) * (g >> 3) + (b >> 3);
  return l < nblocks ? l : -1;
}

// ---- orbital bank --------------------------------------------------------
// Orbital sets of one call: set d fills the bank columns off[d] .. of nocc[d]
// orbitals, element (k, a) at c[d][k + a * nocc[d]].
struct OrbSets {
  int n;
  const double *c[kMaxSets];
  int nocc[kMaxSets];
  int off[kMaxSets];
};

__device__ __forceinline__ double bank_value(const OrbSets &sets, int a, int col, int n) {
  int d = 0;
  while (d + 1 < sets.n && col >= sets.off[d + 1]) ++d;
  const int k = col - sets.off[d];
  return a < n && k < sets.nocc[d] ? sets.c[d][k + int64_t(a) * sets.nocc[d]] : 0.0;
}

// Cb[a*ldc + col], every element of the n_pad x ldc bank in one launch (a zero
// fill and a launch per set before).
template <typename T>
__global__ void k_pack_orb(const OrbSets sets, int n, int n_pad, int ldc, T *__restrict__ cb) {
  const int64_t i = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
  if (i >= int64_t(n_pad) * ldc) return;
  cb[i] = T(bank_value(sets, int(i / ldc), int(i % ldc), n));
}

// FP32 shadow of the resident vectors for the mixed-precision exchange.
__global__ void k_to_f32(const double *__restrict__ src, float *__restrict__ dst, int64_t cnt) {
  for (int64_t i = int64_t(blockIdx.x) * blockDim.x + threadIdx.x; i < cnt;
       i += int64_t(gridDim.x) * blockDim.x)
    dst[i] = float(src[i]);
}

// ---- FP32 half-transform -------------------------------------------------
// grid.x = round_up(ceil(jc/NJ) * ntile_a, 8), block = 256.  Workgroup (jr,
// a-tile of TA columns) computes, for the NJ vectors J = NJ*jr + q < jc,
// X[(J*LDC + k)*n_pad + a] = sum_b Cb[b*LDC + k] L^J_ab for all LDC = 16*OT
// bank columns k.  Wave w owns AO columns a0 + w*TA/4 .. a0 + (w+1)*TA/4 - 1
// (TA/64 MFMA column tiles) and all OT row tiles; each orbital fragment read
// from LDS feeds the MFMAs of all NJ vectors.  The next b-chunk is fetched
// into registers while the current one is multiplied out of LDS.
template <int OT, int TA, int BK, int NJ>
__global__ __launch_bounds__(kThreads) void k_ht(
    const float *__restrict__ L, int64_t ldl, int n, int n_pad,
    const float *__restrict__ Cb, int64_t j0, int64_t jc, int ntile_a, int64_t nblocks,
    float *__restrict__ X, const Screen sc) {
  typedef float T;
  typedef v4f Acc;
  constexpr int LDC = 16 * OT;
  // Wave layout.  Narrow banks: wave w owns AO columns w*TA/4 .. (w+1)*TA/4-1
  // and all OT row tiles.  Wide banks (one vector, even OT >= 6, TA = 64): 2 x 2
  // waves, wave w owns row tiles (w>>1)*OT/2 .. and AO columns (w&1)*TA/2 ..,
  // so a step reads OT/2 + 2 fragments for OT MFMAs instead of OT + 1.
  constexpr int SPLIT = (NJ == 1 && OT % 2 == 0 && OT >= 6 && TA == 64) ? 2 : 1;
  constexpr int OTW = OT / SPLIT;         // row tiles per wave
  constexpr int NB = TA * SPLIT / 64;     // 16-column MFMA tiles per wave
  constexpr int SLD = TA + 1;            // LDS row stride of the L tile
  constexpr int CN = BK * LDC / kThreads;
  constexpr int LN = BK * TA / kThreads;
  static_assert(BK * LDC % kThreads == 0 && BK * TA % kThreads == 0, "tile shape");
  __shared__ __attribute__((aligned(16))) T sC[2][BK * LDC];
  __shared__ T sL[2][NJ][BK * SLD];
  const int64_t lb = xcd_logical(nblocks);
  if (lb < 0) return;
  const int64_t jr = lb / ntile_a;
  const int a0 = int(lb % ntile_a) * TA;
  const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
  const int t0 = SPLIT == 2 ? (w >> 1) * OTW : 0;
  const int c0 = SPLIT == 2 ? (w & 1) * (TA / 2) : w * (TA / 4);
  // vectors of this workgroup: present (J < jc) and not screened out
  bool live[NJ];
  const T *__restrict__ Lq[NJ];
#pragma unroll
  for (int q = 0; q < NJ; ++q) {
    const int64_t J = NJ * jr + q;
    live[q] = J < jc;
    Lq[q] = L + (j0 + (live[q] ? J : NJ * jr)) * ldl;
  }
  if (sc.lnorm) {  // screened: ||X tile||_F <= ||L^J[:, tile]||_F max_d ||C_d||_F
    bool any = false;
#pragma unroll
    for (int q = 0; q < NJ; ++q) {
      if (!live[q]) continue;
      const int64_t J = NJ * jr + q;
      double s2 = 0.0;
      for (int st = a0 / 64; st < (a0 + TA) / 64; ++st) {
        const double v = sc.lnorm[(j0 + J) * sc.nstrip + st];
        s2 += v * v;
      }
      if (sqrt(s2) * sc.cmax[0] < sc.thr_x) {
        T *__restrict__ xj = X + J * LDC * int64_t(n_pad);
        for (int e = tid; e < LDC * TA; e += kThreads) xj[int64_t(e / TA) * n_pad + a0 + e % TA] = T(0);
        if (tid == 0) atomicAdd(sc.cnt + 1, 1ull);
        live[q] = false;
      }
      any = any || live[q];
    }
    if (!any) return;
  }

  Acc acc[NJ][OTW][NB];
#pragma unroll
  for (int q = 0; q < NJ; ++q)
#pragma unroll
    for (int t = 0; t < OTW; ++t)
#pragma unroll
      for (int j = 0; j < NB; ++j) acc[q][t][j] = Acc{0, 0, 0, 0};

  if (a0 < n) {
    // orbital bank rows are contiguous: 16-byte pieces where the tile divides
    constexpr int VW = (CN * int(sizeof(T))) % 16 == 0 ? 16 / int(sizeof(T)) : 1;
    typedef T VT __attribute__((ext_vector_type(VW)));
    constexpr int CV = CN / VW;
    VT rc[CV];
    T rl[NJ][LN];
    // bit i: element i lies inside the matrix.  The mask is applied when the
    // chunk is stashed, so the loads stay in flight across the multiply of
    // the current chunk (a select right after the load would wait for it).
    uint32_t lok = 0;
    static_assert(LN <= 32, "element mask");
    // Element i of a thread: "row-major" chunks (b > a and diagonal blocks)
    // walk e -> (bb = e / TA, aa = e % TA); "column" chunks (b < a, where the
    // packed row a holds b contiguous) walk e -> (bb = e % BK, aa = e / BK).
    // Chunks wholly inside the matrix and wholly below (column chunks) or above
    // the diagonal block (uniform per workgroup) step each thread's packed
    // offsets instead of forming tri0 per element: a thread's elements lie DA
    // columns (column chunks) or DB rows apart, and tri0(x + d) - tri0(x) =
    // d x + d (d + 1) / 2.  Diagonal and edge chunks take the general path.
    constexpr int DA = kThreads / BK, DB = kThreads / TA;
    static_assert(kThreads % BK == 0 && kThreads % TA == 0, "element walk");
    // The chunk kinds differ only in the packed index of each element: the
    // branches form the indices, and one load sequence after them fills rl.
    // Loads issued inside the branches left their registers to be
    // merged by copies at the join, and a copy of a register whose load is in
    // flight waits for the whole memory queue: the chunk after next was then
    // waited for right after its loads were issued.
    auto fetch = [&](int b0) {
      const bool colmajor = b0 + BK <= a0;
      const bool inside = b0 + BK <= n && a0 + TA <= n;
      const T *__restrict__ cs = Cb + int64_t(b0) * LDC;
#pragma unroll
      for (int i = 0; i < CV; ++i)
        rc[i] = *reinterpret_cast<const VT *>(cs + (tid + kThreads * i) * VW);
      uint32_t idx[LN];
      if (inside && colmajor) {  // packed row a = a0 + tid/BK + DA i holds b0 + tid%BK
        uint32_t a = uint32_t(a0 + tid / BK);
        uint32_t x = tri0u(a) + uint32_t(b0 + tid % BK);
#pragma unroll
        for (int i = 0; i < LN; ++i) {
          idx[i] = x;
          x += uint32_t(DA) * a + uint32_t(DA * (DA + 1) / 2);
          a += uint32_t(DA);
        }
        lok = LN == 32 ? ~0u : (1u << LN) - 1u;
      } else if (inside && b0 >= a0 + TA) {  // packed row b = b0 + tid/TA + DB i at column a0 + tid%TA
        uint32_t b = uint32_t(b0 + tid / TA);
        uint32_t x = tri0u(b) + uint32_t(a0 + tid % TA);
#pragma unroll
        for (int i = 0; i < LN; ++i) {
          idx[i] = x;
          x += uint32_t(DB) * b + uint32_t(DB * (DB + 1) / 2);
          b += uint32_t(DB);
        }
        lok = LN == 32 ? ~0u : (1u << LN) - 1u;
      } else {
#pragma unroll
        for (int i = 0; i < LN; ++i) {
          const int e = tid + kThreads * i;
          const int bb = colmajor ? e % BK : e / TA, aa = colmajor ? e / BK : e % TA;
          const int b = b0 + bb, a = a0 + aa;
          const bool ok = (b < n) && (a < n);
          const int hi = b >= a ? b : a, lo = b >= a ? a : b;
          idx[i] = ok ? tri0u(uint32_t(hi)) + uint32_t(lo) : 0u;  // branch-free masked load
          lok = ok ? (lok | (1u << i)) : (lok & ~(1u << i));
        }
      }
#pragma unroll
      for (int i = 0; i < LN; ++i)
#pragma unroll
        for (int q = 0; q < NJ; ++q) rl[q][i] = Lq[q][idx[i]];
    };
    auto stash = [&](int b0, int buf) {
      const bool colmajor = b0 + BK <= a0;
#pragma unroll
      for (int i = 0; i < CV; ++i)
        *reinterpret_cast<VT *>(&sC[buf][(tid + kThreads * i) * VW]) = rc[i];
#pragma unroll
      for (int i = 0; i < LN; ++i) {
        const int e = tid + kThreads * i;
        const int bb = colmajor ? e % BK : e / TA, aa = colmajor ? e / BK : e % TA;
#pragma unroll
        for (int q = 0; q < NJ; ++q)
          sL[buf][q][bb * SLD + aa] = ((lok >> i) & 1u) ? rl[q][i] : T(0);
      }
    };
    // Double-buffered LDS: chunk c is multiplied out of buffer c&1 while
    // chunk c+1 is stored into the other buffer and chunk c+2 is fetched to
    // registers; one barrier per chunk.  The operand fragments of the next
    // 4-row step are read while the current step's MFMAs run.
    const int nch = (n + BK - 1) / BK;
    fetch(0);
    stash(0, 0);
    if (nch > 1) fetch(BK);
    __syncthreads();
    for (int c = 0; c < nch; ++c) {
      const int cur = c & 1;
      const T *__restrict__ sc = sC[cur];
      T af[2][OTW], bf[2][NJ][NB];
      auto ld = [&](int ks, int qq) {
        const int kr = ks * 4 + (lane >> 4);
#pragma unroll
        for (int q = 0; q < NJ; ++q)
#pragma unroll
          for (int j = 0; j < NB; ++j)
            bf[qq][q][j] = sL[cur][q][kr * SLD + c0 + j * 16 + (lane & 15)];
#pragma unroll
        for (int t = 0; t < OTW; ++t) af[qq][t] = sc[kr * LDC + 16 * (t0 + t) + (lane & 15)];
      };
      ld(0, 0);
#pragma unroll
      for (int ks = 0; ks < BK / 4; ++ks) {
        const int qq = ks & 1;
        if (ks + 1 < BK / 4) ld(ks + 1, qq ^ 1);
#pragma unroll
        for (int q = 0; q < NJ; ++q)
#pragma unroll
          for (int t = 0; t < OTW; ++t)
#pragma unroll
            for (int j = 0; j < NB; ++j) acc[q][t][j] = mma32(af[qq][t], bf[qq][q][j], acc[q][t][j]);
      }
      if (c + 1 < nch) stash((c + 1) * BK, cur ^ 1);
      if (c + 2 < nch) fetch((c + 2) * BK);
      __syncthreads();
    }
  }
#pragma unroll
  for (int q = 0; q < NJ; ++q) {
    if (!live[q]) continue;
    T *__restrict__ xj = X + (NJ * jr + q) * LDC * int64_t(n_pad);
#pragma unroll
    for (int j = 0; j < NB; ++j) {
      const int a = a0 + c0 + j * 16 + (lane & 15);
#pragma unroll
      for (int t = 0; t < OTW; ++t)
#pragma unroll
        for (int r = 0; r < 4; ++r)
          xj[int64_t(16 * (t0 + t) + row32(lane, r)) * n_pad + a] = acc[q][t][j][r];
    }
  }
}

// ---- FP64 half-transform ------------------------------------------------------
// Wave item = (vector J, up to NB blocks of 16 AO columns a); the wave forms all
// OT 16-row orbital tiles of its columns and walks b in 16-row chunks.  No other
// wave needs its elements of L^J for this product, so L goes from memory into
// the wave's registers with no staging shared between waves; only the bank
// chunk, which the workgroup's four waves share, is staged in LDS (one barrier
// per chunk).  Every load instruction covers 128-byte runs of packed rows:
//  * below the diagonal block (b >= a) packed row b holds a contiguous and lane
//    l = 16 g + m loads L(b, a) at b = 16 c + 4 g + s, a = a0 + 16 j + m: these
//    are the MFMA operands of the four steps s (the bank rows in the same
//    order), and step s of chunk c + 1 is loaded into the registers of step s
//    of chunk c as soon as that is multiplied;
//  * above it (b < a) packed row a holds b contiguous: lane l loads
//    b = 16 c + m of row a = a0 + 16 j + 4 q + g (q = 0..3) and each 16 x 16
//    block is turned through a wave-private LDS tile (loads that follow the
//    operand layout there touch one cache line per lane, four times over:
//    the L1 request rate bound the kernel);
//  * the diagonal chunks gather element by element.
// Orbital tile pair (i, h) holds the bank columns 32 i + 2 m + h, so one 16-byte
// LDS read gives two A fragments.  Indices past n are clamped to n - 1 (always
// inside the packed row) and the values zeroed where that can happen.
// FV: sum_{b >= a} L_ba D_ba of the wave's columns into *vout.
// Bound by the matrix cores (busy 74-85% of the cycles) at the clock they leave
// (2.1-2.3 GHz); where few orbitals share an element, by the L traffic too (each
// packed element is read twice, 3.7 TB/s at n=512 nocc=64).  With the V work:
// n=1200 nchol=6000 nocc=150 55.3 -> 43.3 ms (65 TFLOP/s executed), n=536
// nchol=2510 nocc=98 3.7 -> 2.8 ms, n=512 nchol=2048 nocc=64 1.40 -> 1.34 ms,
// n=187 nchol=905 nocc=23 0.116 -> 0.077 ms, against staging square tiles of L
// in LDS (its transposing stores, their waits and 5 VALU operations per MFMA
// stood between the MFMAs).
// TQ: columns past the OT full tiles go in quarters of four, v_mfma_f64_4x4x4 (four
// 4x4 blocks, one per four AO columns): it takes the same B operand and runs at the
// same rate (76 TFLOP/s measured), so the bank is padded to 4 columns, not 16.  Lane
// group g holds row g of a quarter; quarters 0 and 1 take alternate columns of eight
// (one 16-byte read).  Without the V work, against full tiles only: n=1200 nocc=150
// 43.3 -> 40.1 ms, n=536 nocc=98 2.81 -> 2.63, n=400 nocc=50 0.78 -> 0.70, n=301
// nocc=40 0.28 -> 0.25, n=187 nocc=23 0.061 -> 0.053 ms.
constexpr int kHtB = 16;       // contraction rows per chunk
constexpr int kHtS = 17;       // row stride of a turned block
constexpr int ht64_ldc(int ot, int tq) { return 16 * (ot + (tq > 0)); }  // bank columns

template <int OT, int TQ, int NBV, bool FV>
__device__ __forceinline__ void ht64_wave(const double *__restrict__ Lj, int n, int nch, int n_pad,
                                          const double *__restrict__ Cb, int a0, double *__restrict__ xj,
                                          const double *__restrict__ dens, double *__restrict__ vout,
                                          double (*__restrict__ sC)[kHtB * ht64_ldc(OT, TQ)], double *__restrict__ sT) {
  constexpr int LDC = ht64_ldc(OT, TQ);
  constexpr int HP = OT / 2;                 // pairs of orbital tiles; an odd last tile stands alone
  constexpr int NB1 = NBV > 0 ? NBV : 1;
  constexpr int CN = kHtB * LDC / 2 / kThreads;  // 16-byte pieces of a bank chunk per thread ...
  constexpr int CR = kHtB * LDC / 2 % kThreads;  // ... and those of a last, partial round
  const int tid = threadIdx.x, lane = tid & 63, m = lane & 15, g = lane >> 4;
  v4d acc[OT > 0 ? OT : 1][NB1];
  double accq[TQ > 0 ? TQ : 1][NB1];
#pragma unroll
  for (int j = 0; j < NBV; ++j) {
#pragma unroll
    for (int t = 0; t < OT; ++t) acc[t][j] = v4d{0.0, 0.0, 0.0, 0.0};
#pragma unroll
    for (int q = 0; q < TQ; ++q) accq[q][j] = 0.0;
  }
  double vp = 0.0;
  // bank chunk: global -> registers -> LDS, the layout unchanged
  v2d rc[CN + (CR ? 1 : 0)];
  auto fetch_c = [&](int c) __attribute__((always_inline)) {
    const double *__restrict__ src = Cb + int64_t(c) * kHtB * LDC;
#pragma unroll
    for (int i = 0; i < CN; ++i) rc[i] = *reinterpret_cast<const v2d *>(src + 2 * (tid + kThreads * i));
    if constexpr (CR > 0)
      rc[CN] = *reinterpret_cast<const v2d *>(src + 2 * (tid < CR ? tid + kThreads * CN : 0));
  };
  auto stash_c = [&](int buf) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < CN; ++i) *reinterpret_cast<v2d *>(&sC[buf][2 * (tid + kThreads * i)]) = rc[i];
    if constexpr (CR > 0)
      if (tid < CR) *reinterpret_cast<v2d *>(&sC[buf][2 * (tid + kThreads * CN)]) = rc[CN];
  };
  const int ncol = a0 / kHtB;  // chunks wholly above the diagonal block
  double rl[4][NB1];
  double rd[2][NB1];  // FV: density values of two steps in flight
  // General loads, for the chunks outside the two long runs below.  The lane's
  // parts of the packed indices are hidden from the loop-invariant code motion,
  // which would keep an index per load in registers.
  auto load_low = [&](int c, int s) __attribute__((always_inline)) {  // c >= ncol
    const int b0 = c * kHtB;
    int mm = m, gg = g;
    asm volatile("" : "+v"(mm), "+v"(gg));
    const uint32_t b = uint32_t(min(b0 + 4 * gg + s, n - 1));
    const uint32_t tb = tri0u(b);
    uint32_t x[NB1];
#pragma unroll
    for (int j = 0; j < NBV; ++j) {
      const uint32_t a = uint32_t(min(a0 + 16 * j + mm, n - 1));
      x[j] = b >= a ? tb + a : tri0u(a) + b;
    }
#pragma unroll
    for (int j = 0; j < NBV; ++j) rl[s][j] = Lj[x[j]];
  };
  auto load_col = [&](int c, int s) __attribute__((always_inline)) {  // c < ncol
    int mm = m, gg = g;
    asm volatile("" : "+v"(mm), "+v"(gg));
#pragma unroll
    for (int j = 0; j < NBV; ++j)
      rl[s][j] = Lj[tri0u(uint32_t(min(a0 + 16 * j + 4 * s + gg, n - 1))) + uint32_t(c * kHtB + mm)];
  };
  // density of the step's elements with b >= a (the others: one cached address)
  auto load_d = [&](int c, int s) __attribute__((always_inline)) {
    if constexpr (FV) {
      int mm = m, gg = g;
      asm volatile("" : "+v"(mm), "+v"(gg));
      const int b = min(c * kHtB + 4 * gg + s, n - 1);
      const uint32_t tb = tri0u(uint32_t(b)) + uint32_t(a0 + mm);
#pragma unroll
      for (int j = 0; j < NBV; ++j) rd[s & 1][j] = dens[a0 + 16 * j + mm <= b ? tb + 16u * j : 0u];
    }
  };
  // A fragments of one step, each pair replaced by the next step's once used
  v2d cf[HP > 0 ? HP : 1];
  double co = 0.0;
  auto load_cp = [&](int buf, int s, int i) __attribute__((always_inline)) {
    cf[i] = *reinterpret_cast<const v2d *>(&sC[buf][(4 * g + s) * LDC + 32 * i + 2 * m]);
  };
  auto load_co = [&](int buf, int s) __attribute__((always_inline)) {
    if constexpr (OT % 2 == 1) co = sC[buf][(4 * g + s) * LDC + 16 * (OT - 1) + m];
  };
  v2d cq = {0.0, 0.0};  // quarter tiles 0 and 1 take alternate columns
  double ct = 0.0;
  auto load_cq = [&](int buf, int s) __attribute__((always_inline)) {
    const double *__restrict__ row = &sC[buf][(4 * g + s) * LDC + 16 * OT];
    if constexpr (TQ == 1) cq[0] = row[m & 3];
    if constexpr (TQ >= 2) cq = *reinterpret_cast<const v2d *>(row + 2 * (m & 3));
    if constexpr (TQ == 3) ct = row[8 + (m & 3)];
  };
  auto step = [&](int buf, int s, const double(&x)[NB1]) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < HP; ++i) {
#pragma unroll
      for (int h = 0; h < 2; ++h)
#pragma unroll
        for (int j = 0; j < NBV; ++j) acc[2 * i + h][j] = mma64(cf[i][h], x[j], acc[2 * i + h][j]);
      if (s < 3) load_cp(buf, s + 1, i);
    }
    if constexpr (OT % 2 == 1) {
#pragma unroll
      for (int j = 0; j < NBV; ++j) acc[OT - 1][j] = mma64(co, x[j], acc[OT - 1][j]);
      if (s < 3) load_co(buf, s + 1);
    }
    if constexpr (TQ > 0) {
#pragma unroll
      for (int q = 0; q < TQ; ++q)
#pragma unroll
        for (int j = 0; j < NBV; ++j)
          accq[q][j] = __builtin_amdgcn_mfma_f64_4x4x4f64(q < 2 ? cq[q] : ct, x[j], accq[q][j], 0, 0, 0);
      if (s < 3) load_cq(buf, s + 1);
    }
  };
  auto first_c = [&](int buf) __attribute__((always_inline)) {
    if constexpr (NBV > 0) {
#pragma unroll
      for (int i = 0; i < HP; ++i) load_cp(buf, 0, i);
      load_co(buf, 0);
      load_cq(buf, 0);
    }
  };

  auto next_c = [&](int c) __attribute__((always_inline)) {  // end of chunk c
    stash_c((c & 1) ^ 1);
    fetch_c(min(c + 2, nch - 1));
    __syncthreads();
  };
  fetch_c(0);
  stash_c(0);
  fetch_c(min(1, nch - 1));
#pragma unroll
  for (int s = 0; s < 4; ++s) {
    if (ncol > 0) load_col(0, s);
    else load_low(0, s);
  }
  __syncthreads();
  int c = 0;
  // ---- chunks above the diagonal block (b < a): blocks turned through LDS;
  // the next chunk is loaded as soon as this one is in LDS
  auto upper = [&](int c, auto load) __attribute__((always_inline)) {
    const int cur = c & 1;
    first_c(cur);
    if constexpr (NBV > 0) {
#pragma unroll
      for (int s = 0; s < 4; ++s)
#pragma unroll
        for (int j = 0; j < NBV; ++j) sT[(16 * j + 4 * s + g) * kHtS + m] = rl[s][j];
      __builtin_amdgcn_sched_barrier(0);
      load();
      __builtin_amdgcn_sched_barrier(0);
      __builtin_amdgcn_wave_barrier();
      double xs[2][NB1];
      auto turn = [&](int s) __attribute__((always_inline)) {
#pragma unroll
        for (int j = 0; j < NBV; ++j) xs[s & 1][j] = sT[(16 * j + m) * kHtS + 4 * g + s];
      };
      turn(0);
#pragma unroll
      for (int s = 0; s < 4; ++s) {
        if (s < 3) turn(s + 1);
        step(cur, s, xs[s & 1]);
        __builtin_amdgcn_sched_barrier(0);
      }
      __builtin_amdgcn_wave_barrier();
    }
    next_c(c);
  };
  // byte offsets of the long runs are 32-bit: below 2^29 packed elements
  const bool small = uint32_t(n) < 32768u;
  if (small) {
    // chunk c + 1 of every row is 128 bytes after chunk c: one offset per load,
    // kept, and a uniform pointer that moves
    uint32_t off[4][NB1];
#pragma unroll
    for (int s = 0; s < 4; ++s)
#pragma unroll
      for (int j = 0; j < NBV; ++j) off[s][j] = 8u * (tri0u(uint32_t(min(a0 + 16 * j + 4 * s + g, n - 1))) + uint32_t(m));
    const char *__restrict__ p = reinterpret_cast<const char *>(Lj);
#pragma unroll 1
    for (; c + 1 < ncol; ++c) {
      p += 8 * kHtB;
      upper(c, [&]() __attribute__((always_inline)) {
#pragma unroll
        for (int s = 0; s < 4; ++s)
#pragma unroll
          for (int j = 0; j < NBV; ++j) rl[s][j] = *reinterpret_cast<const double *>(p + off[s][j]);
      });
    }
  }
#pragma unroll 1
  for (; c + 1 < ncol; ++c)
    upper(c, [&]() __attribute__((always_inline)) {
#pragma unroll
      for (int s = 0; s < 4; ++s) load_col(c + 1, s);
    });
  if (c < ncol) {
    upper(c, [&]() __attribute__((always_inline)) {
#pragma unroll
      for (int s = 0; s < 4; ++s) load_low(c + 1, s);
    });
    ++c;
  }
  // ---- diagonal block and below
  auto lower = [&](int c) __attribute__((always_inline)) {
    const int cur = c & 1, cn = min(c + 1, nch - 1);
    first_c(cur);
#pragma unroll
    for (int s = 0; s < 4; ++s) {
      if constexpr (NBV > 0) {
        // masks by selects into temporaries: a branch that rewrote the loaded
        // registers made the compiler copy them while their loads were in flight
        const int b = c * kHtB + 4 * g + s;
        double x[NB1];
#pragma unroll
        for (int j = 0; j < NBV; ++j) x[j] = b < n ? rl[s][j] : 0.0;
        if constexpr (FV) {
#pragma unroll
          for (int j = 0; j < NBV; ++j) vp += x[j] * (b >= a0 + 16 * j + m ? rd[s & 1][j] : 0.0);
          asm volatile("" : "+v"(vp));  // summed here: sunk to the end of the chunk, the operands would stay live
          __builtin_amdgcn_sched_barrier(0);
          load_d(s < 2 ? c : cn, (s + 2) & 3);
        }
        step(cur, s, x);
        __builtin_amdgcn_sched_barrier(0);
        load_low(cn, s);
        __builtin_amdgcn_sched_barrier(0);
      }
    }
    next_c(c);
  };
  load_d(c, 0);
  load_d(c, 1);
  const int cd = min(ncol + NBV, nch);            // past the diagonal chunks
  const int cr = n % kHtB == 0 ? nch - 1 : nch - 2;  // the next chunk has all its rows inside up to here
#pragma unroll 1
  for (; c < cd; ++c) lower(c);
  if (NBV > 0 && small && c < cr) {
    // chunks below the diagonal block whose next chunk needs no clamp: the
    // offset of row 16 c + 4 g + s of the next chunk steps by its row distance
    const char *__restrict__ lp = reinterpret_cast<const char *>(Lj);
    const char *__restrict__ dp = reinterpret_cast<const char *>(dens);
    uint32_t off[4], inc[4];  // this chunk's rows; bytes to the next chunk's: 8 (16 b + 136)
#pragma unroll
    for (int s = 0; s < 4; ++s) {
      const uint32_t b = uint32_t(c * kHtB + 4 * g + s);
      off[s] = 8u * (tri0u(b) + uint32_t(a0 + m));
      inc[s] = 8u * (16u * b + 136u);
    }
#pragma unroll 1
    for (; c < cr; ++c) {
      const int cur = c & 1;
      first_c(cur);
#pragma unroll
      for (int s = 0; s < 4; ++s) {
        double x[NB1];
#pragma unroll
        for (int j = 0; j < NBV; ++j) x[j] = rl[s][j];
        if constexpr (FV) {
#pragma unroll
          for (int j = 0; j < NBV; ++j) vp += x[j] * rd[s & 1][j];
          asm volatile("" : "+v"(vp));
          __builtin_amdgcn_sched_barrier(0);
#pragma unroll
          for (int j = 0; j < NBV; ++j)
            rd[s & 1][j] = *reinterpret_cast<const double *>(dp + off[(s + 2) & 3] + 128 * j);
        }
        step(cur, s, x);
        __builtin_amdgcn_sched_barrier(0);
        off[s] += inc[s];
        inc[s] += 8u * 256u;
#pragma unroll
        for (int j = 0; j < NBV; ++j) rl[s][j] = *reinterpret_cast<const double *>(lp + off[s] + 128 * j);
        __builtin_amdgcn_sched_barrier(0);
      }
      next_c(c);
    }
  }
#pragma unroll 1
  for (; c < nch; ++c) lower(c);
  if constexpr (FV) {
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) vp += __shfl_xor(vp, o);
    if (NBV > 0 && lane == 0) *vout = vp;
  }
#pragma unroll
  for (int j = 0; j < NBV; ++j) {
    const int a = a0 + 16 * j + m;
#pragma unroll
    for (int t = 0; t < OT; ++t)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int row = 4 * r + g;
        const int k = t < 2 * HP ? 32 * (t >> 1) + 2 * row + (t & 1) : 16 * t + row;
        xj[int64_t(k) * n_pad + a] = a < n ? acc[t][j][r] : 0.0;  // clamped columns
      }
#pragma unroll
    for (int q = 0; q < TQ; ++q) {
      const int k = 16 * OT + (TQ == 1 ? g : q < 2 ? 2 * g + q : 8 + g);
      xj[int64_t(k) * n_pad + a] = a < n ? accq[q][j] : 0.0;
    }
  }
}

// grid.x = round_up(ceil(jc * W / 4), 8): four wave items per workgroup, item =
// J * W + t over the W = ceil(nblk / nb) waves of a vector (nblk = ceil(n / 16)
// column blocks, nb <= NB of them per wave).
template <int OT, int TQ, int NB, bool FV>
__global__ __launch_bounds__(kThreads, 2) void k_ht64(const double *__restrict__ L, int64_t ldl, int n, int n_pad,
                                                   const double *__restrict__ Cb, int64_t j0, int64_t jc, int W,
                                                   int nb, int64_t nblocks, double *__restrict__ X,
                                                   const Screen sc, const FuseV fv) {
  static_assert(NB <= 4, "tail widths");
  constexpr int LDC = ht64_ldc(OT, TQ);
  __shared__ __attribute__((aligned(16))) double sC[2][kHtB * LDC];
  __shared__ __attribute__((aligned(16))) double sT[4][NB * 16 * kHtS];
  const int64_t lb = xcd_logical(nblocks);
  if (lb < 0) return;
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int64_t item = 4 * lb + w;
  const bool live = item < jc * W;
  const int64_t J = live ? item / W : jc - 1;
  const int t = live ? int(item - J * W) : 0;
  const int nblk = (n + 15) / 16, nch = nblk;
  const int a0 = 16 * nb * t;
  int nbv = live ? min(nb, nblk - nb * t) : 0;
  const double *__restrict__ Lj = L + (j0 + J) * ldl;
  double *__restrict__ xj = X + J * LDC * int64_t(n_pad);
  if (sc.lnorm && live) {  // screened: ||X tile||_F <= ||L^J[:, tile]||_F max_d ||C_d||_F; the wave lies in one tile
    const int st0 = a0 / (64 * sc.xw) * sc.xw;
    double s2 = 0.0;
    for (int st = st0; st < st0 + sc.xw; ++st) {
      const double v = sc.lnorm[(j0 + J) * sc.nstrip + st];
      s2 += v * v;
    }
    if (sqrt(s2) * sc.cmax[0] < sc.thr_x) {
      for (int e = threadIdx.x & 63; e < LDC * 16 * nbv; e += 64)
        xj[int64_t(e / (16 * nbv)) * n_pad + a0 + e % (16 * nbv)] = 0.0;
      if ((threadIdx.x & 63) == 0 && a0 == 64 * st0) atomicAdd(sc.cnt + 1, 1ull);
      nbv = 0;
    }
  }
  double *vout = FV ? fv.vpart + int64_t(t) * fv.m + j0 + J : nullptr;
  // a wave without columns still stages its share of the bank and joins the barriers
  switch (nbv) {
    case 0: ht64_wave<OT, TQ, 0, FV>(Lj, n, nch, n_pad, Cb, a0, xj, fv.p, vout, sC, sT[w]); break;
    case 1: ht64_wave<OT, TQ, 1, FV>(Lj, n, nch, n_pad, Cb, a0, xj, fv.p, vout, sC, sT[w]); break;
    case 2: if constexpr (NB >= 2) ht64_wave<OT, TQ, 2, FV>(Lj, n, nch, n_pad, Cb, a0, xj, fv.p, vout, sC, sT[w]); break;
    case 3: if constexpr (NB >= 3) ht64_wave<OT, TQ, 3, FV>(Lj, n, nch, n_pad, Cb, a0, xj, fv.p, vout, sC, sT[w]); break;
    default: if constexpr (NB >= 4) ht64_wave<OT, TQ, 4, FV>(Lj, n, nch, n_pad, Cb, a0, xj, fv.p, vout, sC, sT[w]); break;
  }
}

// ---- SYRK ------------------------------------------------------------------
// grid.x = ntiles * nsplit.  Tile t = A(A+1)/2 + B (A >= B) of TMxTM, split s
// covers chunk vectors [s*jper, min(jc,(s+1)*jper)).  The contraction runs
// over f = (J, k), k in [off, off+opad) of the bank columns.
// kpart[(s*ntiles + t)*TM*TM + al*TM + bl] (+)= sum_f X[f][A*TM+al] X[f][B*TM+bl]
// On diagonal tiles (A == B) only one operand is staged and the MFMA tiles
// strictly above the diagonal are skipped (those entries are never read).
template <int TM, int BKF>
__global__ __launch_bounds__(kThreads) __attribute__((amdgpu_waves_per_eu(2))) void k_syrk(
    const float *__restrict__ X, int n_pad, int ldc, int64_t jc, int ntiles,
    const SyrkSets sets, double *__restrict__ kpart_all, int chunk, const Screen sc) {
  typedef float T;
  typedef v4f Acc;
  constexpr int WT = TM / 2;
  constexpr int MT = WT / 16;
  constexpr int VW = 16 / int(sizeof(T));  // elements per 16-byte load
  typedef T VT __attribute__((ext_vector_type(VW)));
  constexpr int PN = BKF * TM / kThreads / VW;
  static_assert(PN >= 1 && BKF * TM % (kThreads * VW) == 0, "tile shape");
  __shared__ __attribute__((aligned(16))) T sA[2][BKF * TM];
  __shared__ __attribute__((aligned(16))) T sB[2][BKF * TM];
  const int set = find_set(sets, blockIdx.x);
  const int local = blockIdx.x - sets.item0[set];
  const int tile = local % ntiles;
  const int s = local / ntiles;
  const int off = sets.off[set], opad = sets.opad[set];
  const int64_t jper = (jc + sets.nsplit[set] - 1) / sets.nsplit[set];
  double *__restrict__ kpart = kpart_all + sets.kbase[set];
  int A = int((sqrt(8.0 * tile + 1.0) - 1.0) * 0.5);
  while (A * (A + 1) / 2 > tile) --A;
  while ((A + 1) * (A + 2) / 2 <= tile) ++A;
  const int B = tile - A * (A + 1) / 2;
  const bool diag = (A == B);
  const int64_t ja = int64_t(s) * jper;
  const int64_t jz = min(jc, ja + jper);
  const int nf = int((jz > ja ? jz - ja : 0) * opad);  // < 2^31, checked on the host
  const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
  const int wm = w >> 1, wn = w & 1;
  const bool idle = diag && wm < wn;  // wave tile entirely above the diagonal
  // slot (chunk, slice): every chunk of vectors writes its own partial tiles
  double *__restrict__ kp =
      kpart + ((int64_t(chunk) * sets.nsplit[set] + s) * ntiles + tile) * TM * TM;
  if (sc.xn2 && nf > 0) {  // screened: |K_ab| of this slice <= sum_J ||X^J_A||_F ||X^J_B||_F
    double bound = 0.0;
    for (int64_t J = ja; J < jz; ++J) {
      const double *__restrict__ r = sc.xn2 + (int64_t(set) * jc + J) * sc.nstrip;
      double sa2 = 0.0, sb2 = 0.0;
#pragma unroll
      for (int st = 0; st < TM / 64; ++st) {
        sa2 += r[A * (TM / 64) + st];
        sb2 += r[B * (TM / 64) + st];
      }
      bound += sqrt(sa2 * sb2);
    }
    if (bound < sc.tau) {
      for (int e = tid; e < TM * TM; e += kThreads) kp[e] = 0.0;
      if (tid == 0) atomicAdd(sc.cnt, 1ull);
      return;
    }
  }

  Acc acc[MT][MT];
  double accd[MT][MT][4];
#pragma unroll
  for (int i = 0; i < MT; ++i)
#pragma unroll
    for (int j = 0; j < MT; ++j) acc[i][j] = Acc{0, 0, 0, 0};
#pragma unroll
  for (int i = 0; i < MT; ++i)
#pragma unroll
    for (int j = 0; j < MT; ++j)
#pragma unroll
      for (int r = 0; r < 4; ++r) accd[i][j][r] = 0.0;
  auto flush = [&]() {
#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
      for (int j = 0; j < MT; ++j) {
#pragma unroll
        for (int r = 0; r < 4; ++r) accd[i][j][r] += double(acc[i][j][r]);
        acc[i][j] = Acc{0, 0, 0, 0};
      }
  };

  VT ra[PN], rb[PN];
  uint32_t rok = 0;  // bit i: piece i lies inside the slice (applied at stash time)
  static_assert(PN <= 32, "piece mask");
  // Piece i of a thread (VW consecutive columns from cc) is row
  // f0 + ff0 + STEP*i; the row's (vector, bank column) pair is stepped
  // incrementally (one division per chunk).
  constexpr int STEP = kThreads * VW / TM;
  const int cc = (tid % (TM / VW)) * VW, ff0 = tid / (TM / VW);
  const int64_t row0 = (ja * ldc + off) * int64_t(n_pad);
  auto fetch = [&](int f0) {
    int f = f0 + ff0;
    int J = f / opad, kk = f - J * opad;
#pragma unroll
    for (int i = 0; i < PN; ++i) {
      const bool ok = f < nf;
      const int64_t ro = ok ? ((ja + J) * ldc + off + kk) * int64_t(n_pad) : row0;  // masked load
      ra[i] = *reinterpret_cast<const VT *>(X + ro + A * TM + cc);
      rb[i] = *reinterpret_cast<const VT *>(X + ro + B * TM + cc);
      rok = ok ? (rok | (1u << i)) : (rok & ~(1u << i));
      f += STEP;
      kk += STEP;
      while (kk >= opad) {  // opad >= 4: at most STEP / 4 wraps
        kk -= opad;
        ++J;
      }
    }
  };
  // FP32: a fragment read pass (32 lanes of 4 bytes, 32 banks) covers rows kr,
  // kr + 1 of TM floats, a multiple of 32 apart; column c of row f sits at
  // c ^ 16 (f & 1) so the two rows fall in different bank halves (the 16-byte
  // stores keep their four columns together)
  auto spos = [](int f, int c) { return f * TM + (c ^ ((f & 1) << 4)); };
  auto stash = [&](int buf) {
#pragma unroll
    for (int i = 0; i < PN; ++i)
      *reinterpret_cast<VT *>(&sA[buf][spos(ff0 + STEP * i, cc)]) = ((rok >> i) & 1u) ? ra[i] : VT(0);
    if (!diag) {
#pragma unroll
      for (int i = 0; i < PN; ++i)
        *reinterpret_cast<VT *>(&sB[buf][spos(ff0 + STEP * i, cc)]) = ((rok >> i) & 1u) ? rb[i] : VT(0);
    }
  };
  // Double-buffered LDS: chunk c is multiplied out of buffer c&1 while chunk
  // c+1 is stored into the other buffer and chunk c+2 is fetched to
  // registers; one barrier per chunk.  Operand fragments of the next
  // 4-row step are read from LDS while the current step's MFMAs run.
  const int nch = (nf + BKF - 1) / BKF;
  if (nch > 0) {
    fetch(0);
    stash(0);
  }
  if (nch > 1) fetch(BKF);
  __syncthreads();
  for (int c = 0; c < nch; ++c) {
    const int cur = c & 1;
    if (!idle) {
      const T *__restrict__ sa = sA[cur];
      const T *__restrict__ sb = diag ? sA[cur] : sB[cur];
      T af[2][MT], bf[2][MT];
      auto ld = [&](int ks, int q) {
        const int kr = ks * 4 + (lane >> 4);
#pragma unroll
        for (int i = 0; i < MT; ++i) af[q][i] = sa[spos(kr, wm * WT + i * 16 + (lane & 15))];
#pragma unroll
        for (int j = 0; j < MT; ++j) bf[q][j] = sb[spos(kr, wn * WT + j * 16 + (lane & 15))];
      };
      // LO: a wave on the diagonal of a diagonal tile, MFMA tiles i >= j only
      // (a compile-time pattern, so the MFMAs issue back to back)
      auto steps = [&](auto lower_only) {
        constexpr bool LO = decltype(lower_only)::value;
        ld(0, 0);
#pragma unroll
        for (int ks = 0; ks < BKF / 4; ++ks) {
          const int q = ks & 1;
          if (ks + 1 < BKF / 4) ld(ks + 1, q ^ 1);
#pragma unroll
          for (int i = 0; i < MT; ++i)
#pragma unroll
            for (int j = 0; j < MT; ++j)
              if (!LO || i >= j) acc[i][j] = mma32(af[q][i], bf[q][j], acc[i][j]);
        }
      };
      if (!diag || wm > wn) steps(std::false_type{});
      else steps(std::true_type{});
    }
    if (((c + 1) * BKF) % kFlushRows == 0) flush();
    if (c + 1 < nch) stash(cur ^ 1);
    if (c + 2 < nch) fetch((c + 2) * BKF);
    __syncthreads();
  }
  flush();
#pragma unroll
  for (int i = 0; i < MT; ++i)
#pragma unroll
    for (int j = 0; j < MT; ++j)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int al = wm * WT + i * 16 + row32(lane, r);
        const int bl = wn * WT + j * 16 + (lane & 15);
        kp[al * TM + bl] = accd[i][j][r];
      }
}

// ---- FP64 SYRK -------------------------------------------------------------
// Workgroup = (one 64x64 tile A >= B of K, one slice of the chunk's vectors);
// its four waves share the tile and take the slice's 4-row contraction steps
// in turn (wave w: steps w, w+4, ...), each accumulating the whole tile, and
// are summed through LDS once at the end.  A step is four rows of X (one
// vector, four bank columns: opad is a multiple of 4); lane l = 16 g + m loads
// columns 32 i + 2 m, 2 m + 1 (i = 0, 1) of row g of both tile sides, 16 bytes
// each, and these ARE the MFMA operands: tile (i, c) holds the columns
// 32 i + 2 m + c.  So no LDS, no barrier and no address arithmetic sits
// between the loads and the MFMAs: per step 4 loads and 16 MFMAs of 64 cycles,
// kSyrkD steps of loads in flight per wave, two waves per SIMD.
// Bound by the matrix cores and the clock they leave: at n=1200 nchol=6000
// nocc=150 they are busy 88% of the cycles and the clock settles near 2.1 GHz
// (63 TFLOP/s executed; the card's own large FP64 product reaches 70).  The
// LDS-staged 128x128 tile it replaces ran the same shape in 27.3 ms (now 21.8)
// and n=536 nchol=2510 nocc=98 in 2.18 ms (now 1.26): whole 128-wide diagonal
// and edge tiles, whose idle waves held their workgroup's slots, cost a third.
// SH: the tile row holds rows in its first 32 columns only (ragged n); DG:
// diagonal tile, its 10 lower MFMA tiles ((i, 0) x (i, 1) is the transpose of
// (i, 1) x (i, 0) and is read from there).
constexpr int kSyrkD = 4;

// Slot layout of a partial tile: MFMA tile q = 4 (2 i + c) + 2 i' + c', result
// register r, lane: position 256 q + 64 r + lane.
__device__ __forceinline__ int slot64_pos(int al, int bl) {
  const int m = (al >> 1) & 15;  // row index inside MFMA tile (i, c)
  const int q = 4 * (2 * (al >> 5) + (al & 1)) + 2 * (bl >> 5) + (bl & 1);
  return 256 * q + 64 * (m >> 2) + 16 * (m & 3) + ((bl >> 1) & 15);
}

// SCR: of the vectors ja .. jz-1 only those whose slice of jref vectors is kept
// (keep[J / jref]), run by run; with all kept it is the same one run.
template <bool SH, bool DG, bool SCR>
__device__ __forceinline__ void syrk64_tile(const double *__restrict__ X, int n_pad, int ldc, int off,
                                            int q4, int64_t ja, int64_t jz, int A, int B, double *__restrict__ kp,
                                            double (*__restrict__ red)[4][4][64], const uint8_t *__restrict__ keep,
                                            int64_t jref) {
  constexpr int HA = SH ? 1 : 2, HB = (SH && DG) ? 1 : 2;  // 32-column halves of the two sides
  const int tid = threadIdx.x, lane = tid & 63, w = __builtin_amdgcn_readfirstlane(tid >> 6);
  v4d acc[2 * HA][2 * HB];
#pragma unroll
  for (int i = 0; i < 2 * HA; ++i)
#pragma unroll
    for (int j = 0; j < 2 * HB; ++j) acc[i][j] = v4d{0.0, 0.0, 0.0, 0.0};
  auto used = [](int i, int j) { return !DG || (i >> 1) > (j >> 1) || ((i >> 1) == (j >> 1) && i >= j); };
  auto run = [&](int64_t ja, int nst) __attribute__((always_inline)) {
    // steps of this wave and the row pointer of its next load (uniform)
    const int ns = nst > w ? (nst - w + 3) / 4 : 0;
    if (ns <= 0) return;
    int kk = w % q4, left = ns;
    const int64_t row4 = 4 * int64_t(n_pad);
    const double *p = X + ((ja + w / q4) * ldc + off) * int64_t(n_pad) + kk * row4;
    const int64_t wrap = (int64_t(ldc) - 4 * q4) * n_pad;  // from one vector's bank columns to the next's
    const uint32_t la = uint32_t((lane >> 4) * n_pad + A * kT64 + 2 * (lane & 15)) * 8u;
    const uint32_t lb = uint32_t((lane >> 4) * n_pad + B * kT64 + 2 * (lane & 15)) * 8u;
    v2d ra[kSyrkD][HA], rb[kSyrkD][DG ? 1 : 2];
    // every call issues the same loads; past the last step the pointer stays
    auto load = [&](v2d(&a)[HA], v2d(&b)[DG ? 1 : 2]) __attribute__((always_inline)) {
      const char *c = reinterpret_cast<const char *>(p);
#pragma unroll
      for (int i = 0; i < HA; ++i) a[i] = *reinterpret_cast<const v2d *>(c + la + 256 * i);
      if constexpr (!DG) {
#pragma unroll
        for (int i = 0; i < 2; ++i) b[i] = *reinterpret_cast<const v2d *>(c + lb + 256 * i);
      }
      if (--left > 0) {
        p += 4 * row4;
        kk += 4;
        while (kk >= q4) {
          kk -= q4;
          p += wrap;
        }
      }
    };
    auto mul = [&](const v2d(&a)[HA], const v2d(&b)[DG ? 1 : 2]) __attribute__((always_inline)) {
#pragma unroll
      for (int i = 0; i < 2 * HA; ++i)
#pragma unroll
        for (int j = 0; j < 2 * HB; ++j)
          if (used(i, j)) {
            double bv;
            if constexpr (DG) bv = a[j >> 1][j & 1];
            else bv = b[j >> 1][j & 1];
            acc[i][j] = mma64(a[i >> 1][i & 1], bv, acc[i][j]);
          }
    };
#pragma unroll
    for (int s = 0; s < kSyrkD; ++s) load(ra[s], rb[s]);
    int t = 0;
    for (; t + kSyrkD <= ns; t += kSyrkD) {
#pragma unroll
      for (int s = 0; s < kSyrkD; ++s) {
        mul(ra[s], rb[s]);
        __builtin_amdgcn_sched_barrier(0);
        load(ra[s], rb[s]);
        __builtin_amdgcn_sched_barrier(0);
      }
    }
#pragma unroll
    for (int s = 0; s < kSyrkD - 1; ++s)
      if (t + s < ns) mul(ra[s], rb[s]);
  };
  if constexpr (SCR) {
    for (int64_t j = ja; j < jz;) {
      int64_t e = (j / jref + 1) * jref;
      if (keep[j / jref]) {
        while (e < jz && keep[e / jref]) e += jref;
        e = min(e, jz);
        run(j, int(e - j) * q4);
      }
      j = e;
    }
  } else {
    run(ja, int(jz > ja ? jz - ja : 0) * q4);  // < 2^29, checked on the host
  }
  // sum of the four waves in wave order: MFMA tiles four at a time through
  // LDS, wave w finishing the w-th of them
  constexpr int NT = 4 * HA * HB;
#pragma unroll
  for (int q0 = 0; q0 < NT; q0 += 4) {
    if (q0) __syncthreads();
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const int i = (q0 + u) / (2 * HB), j = (q0 + u) % (2 * HB);
      if (used(i, j)) {
#pragma unroll
        for (int r = 0; r < 4; ++r) red[w][u][r][lane] = acc[i][j][r];
      }
    }
    __syncthreads();
    const int i = (q0 + w) / (2 * HB), j = (q0 + w) % (2 * HB);
    if (used(i, j)) {
      double *__restrict__ out = kp + 256 * (4 * i + j) + lane;
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        double v = red[0][w][r][lane];
#pragma unroll
        for (int u = 1; u < 4; ++u) v += red[u][w][r][lane];
        out[64 * r] = v;
      }
    }
  }
}

template <bool SCR>
__global__ __launch_bounds__(kThreads, 2) void k_syrk64(const double *__restrict__ X, int n, int n_pad,
                                                     int ldc, int64_t jc, int T, const Syrk64Sets sets,
                                                     double *__restrict__ kpart, int chunk, const ScreenSets ref,
                                                     const uint8_t *__restrict__ keep) {
  __shared__ double red[4][4][4][64];
  int set = 0;
  while (set + 1 < sets.n && int(blockIdx.x) >= sets.item0[set + 1]) ++set;
  const int local = blockIdx.x - sets.item0[set], x = local & 7, li = local >> 3;
  const int nf = T * (T - 1) / 2;
  const int nsf = sets.nsf[set], nsd = sets.nsd[set];
  // XCD x takes the x-th eighth of the diagonal items (first: their slices are
  // the longer ones) and of the off-diagonal ones, both slice by slice, so the
  // tiles that read the same rows of X run on one XCD
  const int nd8 = (nsd * T + 7) / 8, nf8 = (nsf * nf + 7) / 8;
  const bool diag = li < nd8;
  const int l = diag ? x * nd8 + li : x * nf8 + (li - nd8);
  if (l >= (diag ? nsd * T : nsf * nf)) return;
  int A, B, s, ns;
  double *kp;
  if (diag) {
    s = l / T;
    A = B = l - s * T;
    ns = nsd;
    kp = kpart + sets.kd[set] + (int64_t(chunk) * nsd * T + l) * kSlot64;
  } else {
    s = l / nf;
    const int t = l - s * nf;
    ns = nsf;
    A = int((sqrt(8.0 * t + 1.0) + 1.0) * 0.5);
    while (A * (A - 1) / 2 > t) --A;
    while (A * (A + 1) / 2 <= t) ++A;
    B = t - A * (A - 1) / 2;
    kp = kpart + sets.kf[set] + (int64_t(chunk) * nsf * nf + l) * kSlot64;
  }
  const int64_t jper = (jc + ns - 1) / ns;
  const int64_t ja = s * jper, jz = min(jc, ja + jper);
  const int q4 = sets.opad[set] / 4;
  int64_t jref = 1;
  if constexpr (SCR) {
    const int ta = A / ref.strips, tb = B / ref.strips, nref = ref.nref[set];
    jref = (jc + nref - 1) / nref;
    keep += ref.item0[set] + (int64_t(ta) * (ta + 1) / 2 + tb) * nref;
    bool any = false;
    for (int64_t r = ja / jref; r * jref < jz; ++r) any |= keep[r] != 0;
    if (!any) {
      for (int e = threadIdx.x; e < kSlot64; e += kThreads) kp[e] = 0.0;
      return;
    }
  }
  const bool half = n - A * kT64 <= 32;
  const int off = sets.off[set];
  if (diag) {
    if (half) syrk64_tile<true, true, SCR>(X, n_pad, ldc, off, q4, ja, jz, A, B, kp, red, keep, jref);
    else syrk64_tile<false, true, SCR>(X, n_pad, ldc, off, q4, ja, jz, A, B, kp, red, keep, jref);
  } else {
    if (half) syrk64_tile<true, false, SCR>(X, n_pad, ldc, off, q4, ja, jz, A, B, kp, red, keep, jref);
    else syrk64_tile<false, false, SCR>(X, n_pad, ldc, off, q4, ja, jz, A, B, kp, red, keep, jref);
  }
}

// ---- screening norms -------------------------------------------------------
// keep[item] of the chunk's jn vectors for k_syrk64: a slice's part of a K tile is left
// out when |K_ab| <= sum_J ||X^J_A||_F ||X^J_B||_F < tau there.  One wave per (set,
// tile, slice), four per workgroup.
__global__ __launch_bounds__(kThreads) void k_keep(const double *__restrict__ xn2, int nstrip, int64_t jn,
                                                  const ScreenSets ref, double tau, uint8_t *__restrict__ keep,
                                                  unsigned long long *__restrict__ cnt) {
  const int item = blockIdx.x * (kThreads / 64) + (threadIdx.x >> 6), lane = threadIdx.x & 63;
  if (item >= ref.item0[ref.n]) return;
  int set = 0;
  while (set + 1 < ref.n && item >= ref.item0[set + 1]) ++set;
  const int nref = ref.nref[set], t = (item - ref.item0[set]) / nref, s = (item - ref.item0[set]) % nref;
  int A = int((sqrt(8.0 * t + 1.0) - 1.0) * 0.5);
  while (A * (A + 1) / 2 > t) --A;
  while ((A + 1) * (A + 2) / 2 <= t) ++A;
  const int B = t - A * (A + 1) / 2;
  const int64_t jref = (jn + nref - 1) / nref, ja = s * jref, jz = min(jn, ja + jref);
  double bound = 0.0;
  for (int64_t J = ja + lane; J < jz; J += 64) {
    const double *__restrict__ r = xn2 + (int64_t(set) * jn + J) * nstrip;
    double a2 = 0.0, b2 = 0.0;
    for (int st = 0; st < ref.strips; ++st) {
      a2 += r[A * ref.strips + st];
      b2 += r[B * ref.strips + st];
    }
    bound += sqrt(a2 * b2);
  }
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) bound += __shfl_xor(bound, o);
  if (lane > 0) return;
  const bool skip = jz > ja && bound < tau;
  keep[item] = !skip;
  if (skip) atomicAdd(cnt, 1ull);
}

__device__ inline double block_sum256(double x, double *red) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) x += __shfl_down(x, off, 64);
  if (lane == 0) red[wave] = x;
  __syncthreads();
  const double t = (red[0] + red[1]) + (red[2] + red[3]);
  __syncthreads();  // red is reused by the next call
  return t;
}

// out[J*nstrip + st] = ||L^J[:, 64*st .. 64*st+63]||_F of the symmetric matrix.
// grid = (M, nstrip), 256 threads.
__global__ __launch_bounds__(kThreads) void k_strip_norms(const double *__restrict__ L,
                                                          int64_t ldl, int n, int nstrip,
                                                          double *__restrict__ out) {
  __shared__ double red[4];
  const int64_t J = blockIdx.x;
  const int st = blockIdx.y;
  const double *__restrict__ Lj = L + J * ldl;
  double s = 0.0;
  for (int e = threadIdx.x; e < 64 * n; e += kThreads) {
    const int a = st * 64 + (e & 63), b = e >> 6;
    if (a < n) {
      const int hi = a > b ? a : b, lo = a > b ? b : a;
      const double v = Lj[tri0(hi) + lo];
      s += v * v;
    }
  }
  s = block_sum256(s, red);
  if (threadIdx.x == 0) out[J * nstrip + st] = sqrt(s);
}

// xn2[(d*jn + J)*nstrip + st] = sum over the rows of set d and the 64 AOs of
// strip st of X[J]^2.  grid = (jn, nstrip, nk), 256 threads.
template <typename T>
__global__ __launch_bounds__(kThreads) void k_xnorms(const T *__restrict__ X, int ldc, int n, int n_pad,
                                                     const SyrkSets sets, int nstrip,
                                                     double *__restrict__ xn2) {
  __shared__ double red[4];
  const int64_t J = blockIdx.x;
  const int st = blockIdx.y, d = blockIdx.z;
  const int off = sets.off[d], opad = sets.opad[d];
  double s = 0.0;
  for (int e = threadIdx.x; e < opad * 64; e += kThreads) {
    if (st * 64 + (e & 63) >= n) continue;  // columns past n need not be written
    const double v = double(X[(J * ldc + off + (e >> 6)) * int64_t(n_pad) + st * 64 + (e & 63)]);
    s += v * v;
  }
  s = block_sum256(s, red);
  if (threadIdx.x == 0) xn2[(int64_t(d) * gridDim.x + J) * nstrip + st] = s;
}

// out[d] = ||C_d||_F from the bank (rows a < n, columns off_d .. off_d+opad_d-1),
// out[nk] = max_d out[d].  One workgroup.
template <typename T>
__global__ __launch_bounds__(kThreads) void k_cnorm(const T *__restrict__ Cb, int ldc, int n,
                                                    const SyrkSets sets, double *__restrict__ out) {
  __shared__ double red[4];
  double mx = 0.0;
  for (int d = 0; d < sets.n; ++d) {
    const int off = sets.off[d], opad = sets.opad[d];
    double s = 0.0;
    for (int e = threadIdx.x; e < n * opad; e += kThreads) {
      const double v = double(Cb[int64_t(e / opad) * ldc + off + e % opad]);
      s += v * v;
    }
    s = block_sum256(s, red);
    mx = fmax(mx, sqrt(s));
    if (threadIdx.x == 0) out[d] = sqrt(s);
  }
  if (threadIdx.x == 0) out[sets.n] = mx;
}

// ---- split-BF16, three products ---------------------------------------------
// x = hi + lo with hi = bf16(x), lo = bf16(x - hi); a product is taken as
// lo*hi + hi*lo + hi*hi (lo*lo dropped) with v_mfma_f32_16x16x32_bf16 and FP32
// accumulation.  That MFMA takes 8 consecutive contraction indices per lane
// (lane l: row/column l%16, indices 8*(l/16)..8*(l/16)+7), so both operands are
// staged contraction-contiguous in LDS: rows of kB3S bf16 (32 used, padded to
// keep 16-byte alignment).  Result layout: row 4*(l/16) + r, column l%16.
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));

constexpr int kB3K = 32;          // contraction indices per MFMA
constexpr int kB3S = kB3K + 8;    // LDS row stride in bf16 elements

// LDS position of contraction index k (0..31) of row r in a split-BF16 tile:
// the 16-byte granule k / 8 is XOR-ed with bits 3-4 of the row.  A fragment
// read pass (8 lanes of 16 bytes, 32 banks of 4 bytes) covers 8 consecutive
// rows of one granule and stays conflict-free (rows 80 bytes apart); stores
// whose lanes walk rows 4 or 8 apart (SYRK staging, the half-transform's row
// chunks) no longer pile onto two bank groups.
__device__ __forceinline__ int b3pos(int r, int k) {
  return r * kB3S + ((((k >> 3) ^ (r >> 3)) & 3) << 3) + (k & 7);
}

__device__ inline void split_bf16(float x, __bf16 &hi, __bf16 &lo) {
  hi = __bf16(x);
  lo = __bf16(x - float(hi));
}

__device__ inline v4f mma_b3(bf16x8 ah, bf16x8 al, bf16x8 bh, bf16x8 bl, v4f acc) {
  acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(al, bh, acc, 0, 0, 0);
  acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ah, bl, acc, 0, 0, 0);
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(ah, bh, acc, 0, 0, 0);
}

// Transposed split bank: ch/cl[col*n_pad + a] = hi/lo of the bank element.
__global__ void k_pack_orb_b3(const OrbSets sets, int n, int n_pad, int ldc, __bf16 *__restrict__ ch,
                              __bf16 *__restrict__ cl) {
  const int64_t i = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
  if (i >= int64_t(n_pad) * ldc) return;
  __bf16 h, l;
  split_bf16(float(bank_value(sets, int(i % n_pad), int(i / n_pad), n)), h, l);
  ch[i] = h;
  cl[i] = l;
}

// Half-transform, same work decomposition as k_ht: X[(jr*LDC + k)*n_pad + a].
template <int OT, int TA>
__global__ __launch_bounds__(kThreads) void k_ht_b3(
    const float *__restrict__ L, int64_t ldl, int n, int n_pad, const __bf16 *__restrict__ CbH,
    const __bf16 *__restrict__ CbL, int64_t j0, int ntile_a, int64_t nblocks,
    float *__restrict__ X) {
  constexpr int LDC = 16 * OT;
  constexpr int NB = TA / 64;
  constexpr int LN = kB3K * TA / kThreads;
  constexpr int CCH = LDC * kB3K / 8;  // 16-byte pieces of one bank array per chunk
  constexpr int CN = (CCH + kThreads - 1) / kThreads;
  static_assert(kB3K * TA % kThreads == 0, "tile shape");
  __shared__ __attribute__((aligned(16))) __bf16 sCh[LDC * kB3S];
  __shared__ __attribute__((aligned(16))) __bf16 sCl[LDC * kB3S];
  __shared__ __attribute__((aligned(16))) __bf16 sLh[TA * kB3S];
  __shared__ __attribute__((aligned(16))) __bf16 sLl[TA * kB3S];
  const int64_t lb = xcd_logical(nblocks);
  if (lb < 0) return;
  const int64_t jr = lb / ntile_a;
  const int a0 = int(lb % ntile_a) * TA;
  const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
  const float *__restrict__ Lj = L + (j0 + jr) * ldl;

  v4f acc[OT][NB];
#pragma unroll
  for (int t = 0; t < OT; ++t)
#pragma unroll
    for (int j = 0; j < NB; ++j) acc[t][j] = v4f{0, 0, 0, 0};

  if (a0 < n) {
    // L staging: thread t owns LG groups of four consecutive contraction
    // indices b (one AO column a each) and writes each group as one 8-byte LDS
    // store per hi/lo array.  Row chunks (packed row b holds a contiguous) put
    // a on consecutive lanes; column chunks (packed row a holds b contiguous)
    // put the eight groups of one column on consecutive lanes.
    typedef __bf16 bf16x4 __attribute__((ext_vector_type(4)));
    constexpr int LG = LN / 4;
    static_assert(LN % 4 == 0, "staging shape");
    float rl[LG][4];
    int lo[LG];
    typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));  // 16 bytes, promotable to registers
    u32x4 rch[CN], rcl[CN];
    auto fetch = [&](int b0) {
#pragma unroll
      for (int i = 0; i < CN; ++i) {
        const int p = tid + kThreads * i;
        if (p < CCH) {
          const int64_t src = int64_t(p / 4) * n_pad + b0 + (p % 4) * 8;
          rch[i] = *reinterpret_cast<const u32x4 *>(CbH + src);
          rcl[i] = *reinterpret_cast<const u32x4 *>(CbL + src);
        }
      }
      // chunks wholly inside the matrix step each thread's packed offsets
      // (tri0(x + d) - tri0(x) = d x + d (d + 1) / 2) instead of forming tri0
      // per element; diagonal and edge chunks take the general path
      const bool inside = b0 + kB3K <= n && a0 + TA <= n;
      constexpr int GA = kThreads / (kB3K / 4);  // column step between a thread's groups
      constexpr int GB = 4 * (kThreads / TA);     // row step between a thread's groups
      if (inside && b0 + kB3K <= a0) {  // packed row a holds b0 + 4q .. contiguous
        uint32_t a = uint32_t(a0 + tid / (kB3K / 4));
        uint32_t off = tri0u(a) + uint32_t(b0 + 4 * (tid % (kB3K / 4)));
#pragma unroll
        for (int i = 0; i < LG; ++i) {
#pragma unroll
          for (int k = 0; k < 4; ++k) rl[i][k] = Lj[off + uint32_t(k)];
          lo[i] = b3pos(tid / (kB3K / 4) + GA * i, 4 * (tid % (kB3K / 4)));
          off += uint32_t(GA) * a + uint32_t(GA * (GA + 1) / 2);
          a += uint32_t(GA);
        }
      } else if (inside && b0 >= a0 + TA) {  // packed rows b, b+1, b+2, b+3 at column a
        const uint32_t a = uint32_t(a0 + tid % TA);
        uint32_t b = uint32_t(b0 + 4 * (tid / TA));
#pragma unroll
        for (int i = 0; i < LG; ++i) {
          uint32_t idx = tri0u(b) + a;
#pragma unroll
          for (int k = 0; k < 4; ++k) {
            rl[i][k] = Lj[idx];
            idx += b + uint32_t(k) + 1u;
          }
          lo[i] = b3pos(tid % TA, 4 * (tid / TA + (GB / 4) * i));
          b += uint32_t(GB);
        }
      } else if (b0 + kB3K <= a0) {  // every b < a
#pragma unroll
        for (int i = 0; i < LG; ++i) {
          const int g = tid + kThreads * i, q = g % (kB3K / 4), aa = g / (kB3K / 4), a = a0 + aa;
          const float *__restrict__ row = Lj + (tri0u(uint32_t(a)) + uint32_t(b0 + 4 * q));
#pragma unroll
          for (int k = 0; k < 4; ++k) rl[i][k] = (a < n) ? row[k] : 0.f;
          lo[i] = b3pos(aa, 4 * q);
        }
      } else {
#pragma unroll
        for (int i = 0; i < LG; ++i) {
          const int g = tid + kThreads * i, aa = g % TA, q = g / TA, a = a0 + aa;
#pragma unroll
          for (int k = 0; k < 4; ++k) {
            const int b = b0 + 4 * q + k;
            float v = 0.f;
            if (b < n && a < n)
              v = (b >= a) ? Lj[tri0u(uint32_t(b)) + uint32_t(a)] : Lj[tri0u(uint32_t(a)) + uint32_t(b)];
            rl[i][k] = v;
          }
          lo[i] = b3pos(aa, 4 * q);
        }
      }
    };
    fetch(0);
    for (int b0 = 0; b0 < n; b0 += kB3K) {
      if (b0) __syncthreads();
#pragma unroll
      for (int i = 0; i < CN; ++i) {
        const int p = tid + kThreads * i;
        if (p < CCH) {
          const int dst = (p / 4) * kB3S + (p % 4) * 8;
          *reinterpret_cast<u32x4 *>(sCh + dst) = rch[i];
          *reinterpret_cast<u32x4 *>(sCl + dst) = rcl[i];
        }
      }
#pragma unroll
      for (int i = 0; i < LG; ++i) {
        bf16x4 h, l;
#pragma unroll
        for (int k = 0; k < 4; ++k) {
          __bf16 hh, ll;
          split_bf16(rl[i][k], hh, ll);
          h[k] = hh;
          l[k] = ll;
        }
        *reinterpret_cast<bf16x4 *>(sLh + lo[i]) = h;
        *reinterpret_cast<bf16x4 *>(sLl + lo[i]) = l;
      }
      __syncthreads();
      if (b0 + kB3K < n) fetch(b0 + kB3K);
      const int ko = 8 * (lane >> 4);
      bf16x8 bh[NB], bl[NB];
#pragma unroll
      for (int j = 0; j < NB; ++j) {
        const int r = w * (TA / 4) + 16 * j + (lane & 15);
        bh[j] = *reinterpret_cast<const bf16x8 *>(sLh + b3pos(r, ko));
        bl[j] = *reinterpret_cast<const bf16x8 *>(sLl + b3pos(r, ko));
      }
#pragma unroll
      for (int t = 0; t < OT; ++t) {
        const int r = 16 * t + (lane & 15);
        const bf16x8 ah = *reinterpret_cast<const bf16x8 *>(sCh + r * kB3S + ko);
        const bf16x8 al = *reinterpret_cast<const bf16x8 *>(sCl + r * kB3S + ko);
#pragma unroll
        for (int j = 0; j < NB; ++j) acc[t][j] = mma_b3(ah, al, bh[j], bl[j], acc[t][j]);
      }
    }
  }
  float *__restrict__ xj = X + jr * LDC * int64_t(n_pad);
#pragma unroll
  for (int j = 0; j < NB; ++j) {
    const int a = a0 + w * (TA / 4) + j * 16 + (lane & 15);
#pragma unroll
    for (int t = 0; t < OT; ++t)
#pragma unroll
      for (int r = 0; r < 4; ++r) xj[int64_t(16 * t + 4 * (lane >> 4) + r) * n_pad + a] = acc[t][j][r];
  }
}

// SYRK on FP32 X with split-BF16 products; same tiles, slices and FP64 flush
// as k_syrk.
template <int TM>
__global__ __launch_bounds__(kThreads) void k_syrk_b3(
    const float *__restrict__ X, int n_pad, int ldc, int64_t jc, int ntiles, const SyrkSets sets,
    double *__restrict__ kpart_all, int chunk) {
  constexpr int WT = TM / 2;
  constexpr int MT = WT / 16;
  __shared__ __attribute__((aligned(16))) __bf16 sAh[TM * kB3S];
  __shared__ __attribute__((aligned(16))) __bf16 sAl[TM * kB3S];
  __shared__ __attribute__((aligned(16))) __bf16 sBh[TM * kB3S];
  __shared__ __attribute__((aligned(16))) __bf16 sBl[TM * kB3S];
  const int set = find_set(sets, blockIdx.x);
  const int local = blockIdx.x - sets.item0[set];
  const int tile = local % ntiles;
  const int s = local / ntiles;
  const int off = sets.off[set], opad = sets.opad[set];
  const int64_t jper = (jc + sets.nsplit[set] - 1) / sets.nsplit[set];
  double *__restrict__ kpart = kpart_all + sets.kbase[set];
  int A = int((sqrt(8.0 * tile + 1.0) - 1.0) * 0.5);
  while (A * (A + 1) / 2 > tile) --A;
  while ((A + 1) * (A + 2) / 2 <= tile) ++A;
  const int B = tile - A * (A + 1) / 2;
  const bool diag = (A == B);
  const int64_t ja = int64_t(s) * jper;
  const int64_t jz = min(jc, ja + jper);
  const int nf = int((jz > ja ? jz - ja : 0) * opad);
  const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
  const int wm = w >> 1, wn = w & 1;
  const bool idle = diag && wm < wn;

  v4f acc[MT][MT];
  double accd[MT][MT][4];
#pragma unroll
  for (int i = 0; i < MT; ++i)
#pragma unroll
    for (int j = 0; j < MT; ++j) {
      acc[i][j] = v4f{0, 0, 0, 0};
#pragma unroll
      for (int r = 0; r < 4; ++r) accd[i][j][r] = 0.0;
    }
  // Thread t stages columns 4cq..4cq+3 of rows RQ*fq .. RQ*fq+RQ-1 of each
  // chunk (cq = t % (TM/4), fq = t / (TM/4)): RQ 16-byte row loads per operand
  // and, per column, one LDS write of RQ consecutive contraction indices for
  // each of hi and lo.  The RQ rows share one vector J (chunk starts, RQ*fq
  // and opad are multiples of RQ, which divides 4).
  constexpr int RQ = kB3K * TM / (4 * kThreads);
  static_assert(RQ == 2 || RQ == 4, "staging shape");
  typedef float f4 __attribute__((ext_vector_type(4)));
  typedef __bf16 bfq __attribute__((ext_vector_type(RQ)));
  const int cq = tid % (TM / 4), fq = tid / (TM / 4);
  f4 ra[RQ], rb[RQ];
  auto fetch = [&](int f0) {
    const int f = f0 + RQ * fq;
    const int J = f / opad, kk = f - J * opad;
    const bool ok = f < nf;  // nf is a multiple of 4: the group is all in or all out
    const int64_t ro = ok ? ((ja + J) * ldc + off + kk) * int64_t(n_pad) : 0;
#pragma unroll
    for (int k = 0; k < RQ; ++k) {
      f4 va = f4(0.f), vb = f4(0.f);
      if (ok) {
        va = *reinterpret_cast<const f4 *>(X + ro + k * int64_t(n_pad) + A * TM + 4 * cq);
        if (!diag) vb = *reinterpret_cast<const f4 *>(X + ro + k * int64_t(n_pad) + B * TM + 4 * cq);
      }
      ra[k] = va;
      rb[k] = vb;
    }
  };
  auto stash_one = [&](const f4 (&r)[RQ], __bf16 *sh, __bf16 *sl) {
#pragma unroll
    for (int c = 0; c < 4; ++c) {
      bfq h, l;
#pragma unroll
      for (int k = 0; k < RQ; ++k) {
        __bf16 hh, ll;
        split_bf16(r[k][c], hh, ll);
        h[k] = hh;
        l[k] = ll;
      }
      *reinterpret_cast<bfq *>(sh + b3pos(4 * cq + c, RQ * fq)) = h;
      *reinterpret_cast<bfq *>(sl + b3pos(4 * cq + c, RQ * fq)) = l;
    }
  };
  if (nf > 0) fetch(0);
  for (int f0 = 0; f0 < nf; f0 += kB3K) {
    if (f0) __syncthreads();
    stash_one(ra, sAh, sAl);
    if (!diag) stash_one(rb, sBh, sBl);
    __syncthreads();
    if (f0 + kB3K < nf) fetch(f0 + kB3K);
    if (!idle) {
      const __bf16 *sbh = diag ? sAh : sBh;
      const __bf16 *sbl = diag ? sAl : sBl;
      const int ko = 8 * (lane >> 4);
      bf16x8 ah[MT], al[MT], bh[MT], bl[MT];
#pragma unroll
      for (int i = 0; i < MT; ++i) {
        const int r = wm * WT + 16 * i + (lane & 15);
        ah[i] = *reinterpret_cast<const bf16x8 *>(sAh + b3pos(r, ko));
        al[i] = *reinterpret_cast<const bf16x8 *>(sAl + b3pos(r, ko));
      }
#pragma unroll
      for (int j = 0; j < MT; ++j) {
        const int r = wn * WT + 16 * j + (lane & 15);
        bh[j] = *reinterpret_cast<const bf16x8 *>(sbh + b3pos(r, ko));
        bl[j] = *reinterpret_cast<const bf16x8 *>(sbl + b3pos(r, ko));
      }
      if (!diag || wm > wn) {
#pragma unroll
        for (int i = 0; i < MT; ++i)
#pragma unroll
          for (int j = 0; j < MT; ++j) acc[i][j] = mma_b3(ah[i], al[i], bh[j], bl[j], acc[i][j]);
      } else {  // diagonal wave of a diagonal tile: MFMA tiles i >= j
#pragma unroll
        for (int i = 0; i < MT; ++i)
#pragma unroll
          for (int j = 0; j <= i; ++j) acc[i][j] = mma_b3(ah[i], al[i], bh[j], bl[j], acc[i][j]);
      }
    }
    if ((f0 + kB3K) % kFlushRows == 0) {
#pragma unroll
      for (int i = 0; i < MT; ++i)
#pragma unroll
        for (int j = 0; j < MT; ++j) {
#pragma unroll
          for (int r = 0; r < 4; ++r) accd[i][j][r] += double(acc[i][j][r]);
          acc[i][j] = v4f{0, 0, 0, 0};
        }
    }
  }
  // slot (chunk, slice): every chunk of vectors writes its own partial tiles
  double *__restrict__ kp =
      kpart + ((int64_t(chunk) * sets.nsplit[set] + s) * ntiles + tile) * TM * TM;
#pragma unroll
  for (int i = 0; i < MT; ++i)
#pragma unroll
    for (int j = 0; j < MT; ++j)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int al_ = wm * WT + i * 16 + 4 * (lane >> 4) + r;
        const int bl_ = wn * WT + j * 16 + (lane & 15);
        kp[al_ * TM + bl_] = accd[i][j][r] + double(acc[i][j][r]);
      }
}

// Sum of every fourth value, from the q-th, of cnt values `stride` apart, eight
// loads in flight, in a fixed order.
__device__ __forceinline__ double strided_sum(const double *__restrict__ src, int64_t stride, int cnt, int q) {
  double s = 0.0;
  int k = q;
  for (; k + 28 < cnt; k += 32) {
    double v[8];
#pragma unroll
    for (int u = 0; u < 8; ++u) v[u] = src[(k + 4 * u) * stride];
#pragma unroll
    for (int u = 0; u < 8; ++u) s += v[u];
  }
  for (; k < cnt; k += 4) s += src[k * stride];
  return s;
}

// klt[d*ldk + a*(a+1)/2 + b] = sum over the partial tiles of (a, b): the FP64
// chunks' (k_syrk64, nchunk64 of them, slots of sets64) and the reduced-
// precision chunks' (nchunk of them, slots of sets, row-major TM x TM tiles).
// grid = (n rows a, column blocks of 64, nsets), block 256: thread (q, column)
// sums every fourth slot, so that a small K, which has few rows to run side by
// side, is not one long chain of loads per element.
__global__ __launch_bounds__(kThreads) void k_reduce_k(const double *__restrict__ kpart64, const Syrk64Sets sets64,
                                                      int nchunk64, const double *__restrict__ kpart_all, int tm,
                                                      const SyrkSets sets, int nchunk, int n,
                                                      double *__restrict__ klt, int64_t ldk) {
  __shared__ double red[3][64];
  const int a = blockIdx.x, d = blockIdx.z;
  const int cb = threadIdx.x & 63, q = threadIdx.x >> 6;
  const int b = blockIdx.y * 64 + cb;
  if (int(blockIdx.y) * 64 > a) return;
  double s = 0.0;
  if (b <= a) {
    if (nchunk64 > 0) {
      const int T = (n + kT64 - 1) / kT64;
      const int A = a / kT64, B = b / kT64;
      int al = a % kT64, bl = b % kT64;
      const double *src;
      int64_t stride;
      int cnt;
      if (A == B) {
        if ((al >> 5) == (bl >> 5) && !(al & 1) && (bl & 1)) {  // stored as its transpose
          const int t = al;
          al = bl;
          bl = t;
        }
        cnt = sets64.nsd[d] * nchunk64;
        stride = int64_t(T) * kSlot64;
        src = kpart64 + sets64.kd[d] + int64_t(A) * kSlot64;
      } else {
        const int nf = T * (T - 1) / 2;
        cnt = sets64.nsf[d] * nchunk64;
        stride = int64_t(nf) * kSlot64;
        src = kpart64 + sets64.kf[d] + (int64_t(A) * (A - 1) / 2 + B) * kSlot64;
      }
      s = strided_sum(src + slot64_pos(al, bl), stride, cnt, q);
    }
    if (nchunk > 0) {
      const int ntile1 = (n + tm - 1) / tm, ntiles = ntile1 * (ntile1 + 1) / 2;
      const int A = a / tm, B = b / tm;
      const double *src = kpart_all + sets.kbase[d] + (int64_t(A) * (A + 1) / 2 + B) * tm * tm +
                          int64_t(a % tm) * tm + b % tm;
      s += strided_sum(src, int64_t(ntiles) * tm * tm, sets.nsplit[d] * nchunk, q);
    }
  }
  if (q > 0) red[q - 1][cb] = s;
  __syncthreads();
  if (q == 0 && b <= a) klt[d * ldk + tri0(a) + b] = ((s + red[0][cb]) + red[1][cb]) + red[2][cb];
}

template <int OT, int TA, int BK>
void launch_ht(Context *c, const float *L, const float *cb, int64_t j0, int64_t jc, float *X) {
  // two vectors per workgroup while the accumulators stay small (half the
  // orbital-fragment LDS reads per MFMA) and at OT = 7
  constexpr int NJ = (OT * (TA / 64) <= 4 || (TA == 64 && OT == 7)) ? 2 : 1;
  const int ntile_a = c->n_pad / TA;
  const int64_t nblocks = ceil_div(jc, NJ) * ntile_a;
  const int64_t grid = round_up(nblocks, 8);
  hipLaunchKernelGGL((k_ht<OT, TA, BK, NJ>), dim3(unsigned(grid)), dim3(kThreads), 0,
                     c->stream, L, c->ldl, c->n, c->n_pad, cb, j0, jc, ntile_a, nblocks, X, c->scr);
  if (c->scr.lnorm) c->x_tiles += jc * ntile_a;
}

// Column blocks per wave.  Few enough for three waves per SIMD up to five orbital
// tiles (n=300 nocc=45: 0.32 ms with two blocks, 0.38 with four; n=512 nocc=64
// 1.34 / 1.37 ms), two from there to ten tiles (n=536 nocc=98 2.81 ms, with one
// block 2.91; n=1200 nocc=150 43.3 / 44.1 ms), one past that (registers).
constexpr int ht64_nb(int ot) { return ot == 1 ? 4 : ot == 2 ? 3 : ot <= 10 ? 2 : 1; }

template <int OT, int TQ>
void launch_ht64(Context *c, const double *cb, int64_t j0, int64_t jc, double *X) {
  constexpr int NB = ht64_nb(OT + (TQ > 0));
  const int64_t nblk = ceil_div(c->n, 16);
  // Column blocks per wave of a launch of few rounds of resident workgroups: the
  // count whose last round wastes least (a wave's time goes with its blocks, plus
  // about half a block for its share of the bank and the barriers).  n=187
  // nchol=905 nocc=23: three blocks 84 us (905 workgroups on 768 slots), two 77.
  constexpr int64_t kPerCu = OT + (TQ > 0) <= 5 ? 3 : 2;
  const int64_t slots = kPerCu * c->ncu;
  int nb = c->fv.p ? c->fv.nb : 0;  // V: as the first chunk of this exchange
  if (!nb) {
    nb = NB;
    double least = 1e300;
    for (int v = NB; v >= 1; --v) {
      if (v == 3 && c->scr.lnorm) continue;  // a screened wave lies in one tile of 64
      const int64_t wgs = ceil_div(jc * ceil_div(nblk, v), 4), rounds = ceil_div(wgs, slots);
      if (v == NB && rounds > 8) break;
      const double cost = double(rounds) * (v + 0.5);
      if (cost < least) {
        least = cost;
        nb = v;
      }
    }
  }
  const int W = int(ceil_div(nblk, nb));
  const int64_t nblocks = ceil_div(jc * W, 4);
  const dim3 grid(unsigned(round_up(nblocks, 8)));
  if (c->fv.p) {  // fused Coulomb pass (never together with screening)
    c->fv.ntile = W;
    c->fv.nb = nb;
    hipLaunchKernelGGL((k_ht64<OT, TQ, NB, true>), grid, dim3(kThreads), 0, c->stream, c->L, c->ldl, c->n, c->n_pad, cb,
                       j0, jc, W, nb, nblocks, X, Screen{}, c->fv);
    return;
  }
  hipLaunchKernelGGL((k_ht64<OT, TQ, NB, false>), grid, dim3(kThreads), 0, c->stream, c->L, c->ldl, c->n, c->n_pad, cb,
                     j0, jc, W, nb, nblocks, X, c->scr, FuseV{});
  if (c->scr.lnorm) c->x_tiles += jc * ceil_div(c->n, 64 * c->scr.xw);
}

// Three quarters only up to four full tiles: past that they save a quarter of one
// tile in six or more, less than the variants' place in the library is worth.
template <int OT>  // full tiles before the last
void launch_ht64_q(Context *c, int rest, const double *cb, int64_t j0, int64_t jn, double *X) {
  switch ((rest + 3) / 4) {
    case 1:
      return launch_ht64<OT, 1>(c, cb, j0, jn, X);
    case 2:
      return launch_ht64<OT, 2>(c, cb, j0, jn, X);
    case 3:
      if constexpr (OT < 5) return launch_ht64<OT, 3>(c, cb, j0, jn, X);
      break;
    default: break;
  }
  launch_ht64<OT + 1, 0>(c, cb, j0, jn, X);
}

// X^J = C^T L^J of the first tot bank columns (stride 16 ceil(tot / 16)).
void ht64_dispatch(Context *c, int tot, const double *cb, int64_t j0, int64_t jn, double *X) {
  switch ((tot - 1) / 16) {
    case 0: launch_ht64_q<0>(c, tot % 16, cb, j0, jn, X); break;
    case 1: launch_ht64_q<1>(c, tot % 16, cb, j0, jn, X); break;
    case 2: launch_ht64_q<2>(c, tot % 16, cb, j0, jn, X); break;
    case 3: launch_ht64_q<3>(c, tot % 16, cb, j0, jn, X); break;
    case 4: launch_ht64_q<4>(c, tot % 16, cb, j0, jn, X); break;
    case 5: launch_ht64_q<5>(c, tot % 16, cb, j0, jn, X); break;
    case 6: launch_ht64_q<6>(c, tot % 16, cb, j0, jn, X); break;
    case 7: launch_ht64_q<7>(c, tot % 16, cb, j0, jn, X); break;
    case 8: launch_ht64_q<8>(c, tot % 16, cb, j0, jn, X); break;
    case 9: launch_ht64_q<9>(c, tot % 16, cb, j0, jn, X); break;
    case 10: launch_ht64_q<10>(c, tot % 16, cb, j0, jn, X); break;
    case 11: launch_ht64_q<11>(c, tot % 16, cb, j0, jn, X); break;
    case 12: launch_ht64_q<12>(c, tot % 16, cb, j0, jn, X); break;
    case 13: launch_ht64_q<13>(c, tot % 16, cb, j0, jn, X); break;
    case 14: launch_ht64_q<14>(c, tot % 16, cb, j0, jn, X); break;
    default: launch_ht64_q<15>(c, tot % 16, cb, j0, jn, X); break;
  }
}

// FP32 AO tile width: 128 while the accumulators fit (ot <= 6), else 64; the
// context's ht_ta overrides (autotuner).
inline int ht_tile(const Context *c, int ot) { return c->ht_ta ? c->ht_ta : ot <= 6 ? 128 : 64; }

template <int OT>
void launch_ht_w(Context *c, bool wide, const float *L, const float *cb, int64_t j0, int64_t jn, float *X) {
  // 8-row chunks where the staging pieces divide, else 16 (odd OT)
  constexpr int BK = (8 * 16 * OT) % kThreads == 0 ? 8 : 16;
  if (wide) return launch_ht<OT, 128, BK>(c, L, cb, j0, jn, X);
  launch_ht<OT, 64, BK>(c, L, cb, j0, jn, X);
}

void ht32_dispatch(Context *c, int ot, const float *L, const float *cb, int64_t j0, int64_t jn, float *X) {
  // BK = 8 where the staging pieces divide (16 for one or three tiles)
  const bool wide = ht_tile(c, ot) == 128;
  switch (ot) {
    case 1: wide ? launch_ht<1, 128, 16>(c, L, cb, j0, jn, X) : launch_ht<1, 64, 16>(c, L, cb, j0, jn, X); break;
    case 2: wide ? launch_ht<2, 128, 16>(c, L, cb, j0, jn, X) : launch_ht<2, 64, 8>(c, L, cb, j0, jn, X); break;
    case 3: wide ? launch_ht<3, 128, 16>(c, L, cb, j0, jn, X) : launch_ht<3, 64, 16>(c, L, cb, j0, jn, X); break;
    case 4: wide ? launch_ht<4, 128, 16>(c, L, cb, j0, jn, X) : launch_ht<4, 64, 8>(c, L, cb, j0, jn, X); break;
    case 5: wide ? launch_ht<5, 128, 16>(c, L, cb, j0, jn, X) : launch_ht<5, 64, 16>(c, L, cb, j0, jn, X); break;
    case 6: wide ? launch_ht<6, 128, 16>(c, L, cb, j0, jn, X) : launch_ht<6, 64, 8>(c, L, cb, j0, jn, X); break;
    case 7: launch_ht_w<7>(c, wide, L, cb, j0, jn, X); break;
    case 8: launch_ht_w<8>(c, wide, L, cb, j0, jn, X); break;
    case 10: launch_ht_w<10>(c, wide, L, cb, j0, jn, X); break;
    case 12: launch_ht_w<12>(c, wide, L, cb, j0, jn, X); break;
    case 14: launch_ht_w<14>(c, wide, L, cb, j0, jn, X); break;
    default: launch_ht_w<16>(c, wide, L, cb, j0, jn, X); break;
  }
}

void syrk_launch64(Context *c, const double *X, int ldc, int64_t jn, const Syrk64Sets &sets, double *kpart,
                   int chunk, const ScreenSets &ref, uint8_t *keep) {
  const int T = int(ceil_div(c->n, kT64));
  const dim3 grid(unsigned(sets.item0[sets.n]));
  if (c->scr.xn2) {
    const int items = ref.item0[ref.n];
    hipLaunchKernelGGL(k_keep, dim3(unsigned(ceil_div(items, kThreads / 64))), dim3(kThreads), 0, c->stream,
                       c->scr.xn2, c->scr.nstrip, jn, ref, c->scr.tau, keep, c->scr.cnt);
    c->k_items += items;
    hipLaunchKernelGGL((k_syrk64<true>), grid, dim3(kThreads), 0, c->stream, X, c->n, c->n_pad, ldc, jn, T, sets, kpart,
                       chunk, ref, keep);
    return;
  }
  hipLaunchKernelGGL((k_syrk64<false>), grid, dim3(kThreads), 0, c->stream, X, c->n, c->n_pad, ldc, jn, T, sets, kpart,
                     chunk, ref, keep);
}

void syrk_launch32(Context *c, int tm, int items, const float *X, int ldc, int64_t jn, int ntiles,
                   const SyrkSets &sets, double *kpart, int chunk) {
  if (tm == 128)
    hipLaunchKernelGGL((k_syrk<128, 16>), dim3(unsigned(items)), dim3(kThreads), 0, c->stream, X,
                       c->n_pad, ldc, jn, ntiles, sets, kpart, chunk, c->scr);
  else
    hipLaunchKernelGGL((k_syrk<64, 32>), dim3(unsigned(items)), dim3(kThreads), 0, c->stream, X,
                       c->n_pad, ldc, jn, ntiles, sets, kpart, chunk, c->scr);
  if (c->scr.xn2) c->k_items += items;
}

template <int OT, int TA>
void launch_ht_b3(Context *c, const float *L, const __bf16 *ch, const __bf16 *cl, int64_t j0,
                  int64_t jc, float *X) {
  const int ntile_a = c->n_pad / TA;
  const int64_t nblocks = jc * ntile_a;
  hipLaunchKernelGGL((k_ht_b3<OT, TA>), dim3(unsigned(round_up(nblocks, 8))), dim3(kThreads), 0,
                     c->stream, L, c->ldl, c->n, c->n_pad, ch, cl, j0, ntile_a, nblocks, X);
}

void ht_dispatch_b3(Context *c, int ot, const float *L, const __bf16 *ch, const __bf16 *cl,
                    int64_t j0, int64_t jn, float *X) {
  // 128-wide AO tiles unless the context's ht_ta asks for 64: twice the MFMA
  // work per staged chunk (measured 36-38% faster at 10 and 14 bank tiles)
  const bool wide = c->ht_ta != 64;
  switch (ot) {
    case 1: wide ? launch_ht_b3<1, 128>(c, L, ch, cl, j0, jn, X) : launch_ht_b3<1, 64>(c, L, ch, cl, j0, jn, X); break;
    case 2: wide ? launch_ht_b3<2, 128>(c, L, ch, cl, j0, jn, X) : launch_ht_b3<2, 64>(c, L, ch, cl, j0, jn, X); break;
    case 3: wide ? launch_ht_b3<3, 128>(c, L, ch, cl, j0, jn, X) : launch_ht_b3<3, 64>(c, L, ch, cl, j0, jn, X); break;
    case 4: wide ? launch_ht_b3<4, 128>(c, L, ch, cl, j0, jn, X) : launch_ht_b3<4, 64>(c, L, ch, cl, j0, jn, X); break;
    case 5: wide ? launch_ht_b3<5, 128>(c, L, ch, cl, j0, jn, X) : launch_ht_b3<5, 64>(c, L, ch, cl, j0, jn, X); break;
    case 6: wide ? launch_ht_b3<6, 128>(c, L, ch, cl, j0, jn, X) : launch_ht_b3<6, 64>(c, L, ch, cl, j0, jn, X); break;
    case 7: wide ? launch_ht_b3<7, 128>(c, L, ch, cl, j0, jn, X) : launch_ht_b3<7, 64>(c, L, ch, cl, j0, jn, X); break;
    case 8: wide ? launch_ht_b3<8, 128>(c, L, ch, cl, j0, jn, X) : launch_ht_b3<8, 64>(c, L, ch, cl, j0, jn, X); break;
    case 10: wide ? launch_ht_b3<10, 128>(c, L, ch, cl, j0, jn, X) : launch_ht_b3<10, 64>(c, L, ch, cl, j0, jn, X); break;
    case 12: wide ? launch_ht_b3<12, 128>(c, L, ch, cl, j0, jn, X) : launch_ht_b3<12, 64>(c, L, ch, cl, j0, jn, X); break;
    case 14: wide ? launch_ht_b3<14, 128>(c, L, ch, cl, j0, jn, X) : launch_ht_b3<14, 64>(c, L, ch, cl, j0, jn, X); break;
    default: wide ? launch_ht_b3<16, 128>(c, L, ch, cl, j0, jn, X) : launch_ht_b3<16, 64>(c, L, ch, cl, j0, jn, X); break;
  }
}

void syrk_launch_b3(Context *c, int tm, int items, const float *X, int ldc, int64_t jn, int ntiles,
                    const SyrkSets &sets, double *kpart, int chunk) {
  if (tm == 128)
    hipLaunchKernelGGL((k_syrk_b3<128>), dim3(unsigned(items)), dim3(kThreads), 0, c->stream, X,
                       c->n_pad, ldc, jn, ntiles, sets, kpart, chunk);
  else
    hipLaunchKernelGGL((k_syrk_b3<64>), dim3(unsigned(items)), dim3(kThreads), 0, c->stream, X,
                       c->n_pad, ldc, jn, ntiles, sets, kpart, chunk);
}

OrbSets orb_sets(int32_t nk, const int32_t *nocc, const double *const *corb, const std::vector<int> &off) {
  OrbSets s{};
  s.n = nk;
  for (int d = 0; d < nk; ++d) {
    s.c[d] = corb[d];
    s.nocc[d] = nocc[d];
    s.off[d] = off[size_t(d)];
  }
  return s;
}

int pack_bank_b3(Context *c, int32_t nk, const int32_t *nocc, const double *const *corb,
                 const std::vector<int> &off, int ldc, DevBuf &buf) {
  const int64_t half = int64_t(ldc) * c->n_pad;
  int rc;
  if ((rc = ensure(c, buf, 2 * sizeof(__bf16) * size_t(half)))) return rc;
  __bf16 *ch = static_cast<__bf16 *>(buf.ptr);
  phase_begin(c);
  hipLaunchKernelGGL(k_pack_orb_b3, dim3(unsigned(ceil_div(half, 256))), dim3(256), 0, c->stream,
                     orb_sets(nk, nocc, corb, off), c->n, c->n_pad, ldc, ch, ch + half);
  phase_end(c, MJK_PHASE_PACK);
  return hip_check(c, hipGetLastError(), "bank launch");
}

// Layout of the bank for nk sets; returns MJK_OK and ot = 0 when empty.  The
// reduced-precision kernels exist for even widths above eight tiles only.
int bank_layout(Context *c, int32_t nk, const int32_t *nocc, std::vector<int> &off,
                std::vector<int> &opad, bool fp64_only, int *ot_out, int *tot_out) {
  off.assign(size_t(nk), 0);
  opad.assign(size_t(nk), 0);
  int tot = 0;
  for (int d = 0; d < nk; ++d) {
    if (nocc[d] < 0 || nocc[d] > 256)
      return set_error(c, MJK_ERR_ARG, "orbital set larger than 256 columns");
    off[size_t(d)] = tot;
    opad[size_t(d)] = int(round_up(nocc[d], 4));
    tot += opad[size_t(d)];
  }
  *tot_out = tot;
  *ot_out = 0;
  if (tot == 0) return MJK_OK;
  int ot = int(ceil_div(tot, 16));
  if (!fp64_only && ot > 8) ot = int(round_up(ot, 2));
  if (ot <= 16) {
    *ot_out = ot;
    return MJK_OK;
  }
  return set_error(c, MJK_ERR_ARG, "more than 256 orbital columns in one call");
}

template <typename T>
int pack_bank_t(Context *c, int32_t nk, const int32_t *nocc, const double *const *corb,
                const std::vector<int> &off, int ldc, DevBuf &buf) {
  const int64_t cnt = int64_t(c->n_pad) * ldc;
  int rc;
  if ((rc = ensure(c, buf, sizeof(T) * size_t(cnt)))) return rc;
  phase_begin(c);
  hipLaunchKernelGGL(k_pack_orb<T>, dim3(unsigned(ceil_div(cnt, 256))), dim3(256), 0, c->stream,
                     orb_sets(nk, nocc, corb, off), c->n, c->n_pad, ldc, static_cast<T *>(buf.ptr));
  phase_end(c, MJK_PHASE_PACK);
  return hip_check(c, hipGetLastError(), "bank launch");
}

// FP32 copy of L, made once after the vectors change.
int ensure_l32(Context *c) {
  if (c->l32_valid) return MJK_OK;
  const int64_t cnt = c->nchol * c->ldl;
  int rc;
  if ((rc = ensure(c, c->ws_l32, sizeof(float) * size_t(cnt)))) return rc;
  phase_begin(c);
  hipLaunchKernelGGL(k_to_f32, dim3(4096), dim3(256), 0, c->stream, c->L,
                     static_cast<float *>(c->ws_l32.ptr), cnt);
  phase_end(c, MJK_PHASE_PACK);
  c->l32_valid = true;
  return hip_check(c, hipGetLastError(), "L to FP32");
}

// Slices of the FP64 SYRK (k_syrk64) for chunks of jc vectors: fills sets and
// returns the doubles its partial tiles take over nchunk chunks.
// Workgroups per launch: whole rounds of two per CU, as many (up to 64) as leave
// each of a workgroup's four waves about 160 steps (a step is four rows, 16
// MFMAs); a diagonal tile (10 MFMAs per step) gets 10/16 of the slices.  The
// tiles of one slice drift apart as they run, and once they are further apart
// than the XCD's L2 holds, each fetches X from HBM by itself; short slices bound
// the drift until the partial tiles' traffic takes over.  Measured (workgroups
// per launch: 1024, 4096, 16384, 32768): n=512 nchol=2048 nocc=64 0.58, 0.61,
// 0.73, 0.95 ms; n=800 nchol=3600 nocc=150 6.5, 6.1, 5.7, 5.8 ms; n=1200
// nchol=6000 nocc=150 22.9, 21.4, 22.4, 21.5 ms.
// most: partial tiles (32 KiB) that a launch may take, but at least one round.
int64_t plan_syrk64(const Context *c, int32_t nk, const int32_t *nocc, const std::vector<int> &off,
                    const std::vector<int> &opad, int64_t jc, int64_t work, int64_t nchunk, int64_t most,
                    Syrk64Sets *out) {
  Syrk64Sets &s = *out;
  s.n = nk;
  const int64_t T = ceil_div(c->n, kT64), nf = T * (T - 1) / 2;
  const int64_t units = 16 * nf + 10 * T;  // MFMAs of one step over all tiles
  const int64_t slots = 2 * int64_t(c->ncu), steps = jc * work / 4;
  const int64_t rounds = std::min<int64_t>(64, std::max<int64_t>(1, steps * units / (16 * 4 * 160 * slots)));
  const int64_t target = c->split_target ? c->split_target : std::max(slots, std::min(slots * rounds, most));
  // Slices of every set for `aim` workgroups; the number there will be (each XCD's
  // eighth of a set's two item lists is rounded up).
  auto slices = [&](int64_t aim) {
    for (int d = 0; d < nk; ++d) {
      s.nsf[d] = s.nsd[d] = 0;
      if (nocc[d] > 0) {
        const int64_t own = aim * opad[size_t(d)];
        // at least 4 steps per wave, at most one slice per vector
        const int64_t fit = std::max<int64_t>(1, std::min<int64_t>(jc, jc * opad[size_t(d)] / 64));
        auto clip = [&](int64_t v) { return int(std::max<int64_t>(1, std::min<int64_t>(v, fit))); };
        s.nsf[d] = clip(own * 16 / (work * units));
        s.nsd[d] = clip(own * 10 / (work * units));
      }
      s.item0[d + 1] = s.item0[d] + int(8 * (ceil_div(s.nsd[d] * T, 8) + ceil_div(s.nsf[d] * nf, 8)));
    }
    return int64_t(s.item0[nk]);
  };
  // No more than the target: 520 workgroups on 512 slots took a second round
  // (two or three tiles across: n=187 nocc=23 30.5 -> 22.6 us, n=175 nocc=50 52 -> 37,
  // n=131 nocc=42 31 -> 26).
  for (int64_t aim = target; slices(aim) > target && aim > target / 2;) aim -= 8;
  int64_t kb = 0;
  for (int d = 0; d < nk; ++d) {
    s.off[d] = off[size_t(d)];
    s.opad[d] = std::max(opad[size_t(d)], 4);
    s.kf[d] = kb;
    kb += s.nsf[d] * nchunk * nf * kSlot64;
    s.kd[d] = kb;
    kb += s.nsd[d] * nchunk * T * kSlot64;
  }
  return kb;
}

// A run of vectors [j0, j1) computed in one precision.
struct Segment {
  int64_t j0, j1;
  int32_t prec;
};

int exchange_segments(Context *c, int32_t nk, const int32_t *nocc, const double *const *corb,
                      double *klt, int64_t ldk, const std::vector<Segment> &segs,
                      double tau = 0.0, double thr_x = 0.0) {
  const int n = c->n, n_pad = c->n_pad;
  int rc;
  if (nk > kMaxSets) return set_error(c, MJK_ERR_ARG, "exchange: more than 16 orbital sets");
  std::vector<int> off, opad;
  int ot = 0, tot = 0;
  bool use[3] = {false, false, false};
  for (const Segment &s : segs)
    if (s.j1 > s.j0) use[s.prec] = true;
  if ((rc = bank_layout(c, nk, nocc, off, opad, !use[MJK_PREC_FP32] && !use[MJK_PREC_BF16X3], &ot, &tot)))
    return rc;
  if (tot == 0) {  // no orbitals: K = 0
    for (int d = 0; d < nk; ++d)
      if ((rc = fill_zero(c, klt + d * ldk, sizeof(double) * c->np))) return rc;
    return MJK_OK;
  }
  const int ldc = 16 * ot;
  const bool zsave = c->zs.z != nullptr;
  if (zsave && (nk != 1 || nocc[0] != c->zs.nocc))
    return set_error(c, MJK_ERR_ARG, "exchange: Z output needs exactly one orbital set");
  if (zsave && (tau > 0.0 || thr_x > 0.0))
    return set_error(c, MJK_ERR_ARG, "exchange: Z output cannot be screened");
  // one bank per precision in use; the reduced-precision ones read the FP32
  // copy of L.  Z = X C always multiplies by the FP64 bank.
  if ((use[MJK_PREC_FP64] || zsave) &&
      (rc = pack_bank_t<double>(c, nk, nocc, corb, off, ldc, c->w->cbank)))
    return rc;
  if (use[MJK_PREC_FP32] && (rc = pack_bank_t<float>(c, nk, nocc, corb, off, ldc, c->w->cb32)))
    return rc;
  if (use[MJK_PREC_BF16X3] && (rc = pack_bank_b3(c, nk, nocc, corb, off, ldc, c->w->cb3)))
    return rc;
  if ((use[MJK_PREC_FP32] || use[MJK_PREC_BF16X3]) && (rc = ensure_l32(c))) return rc;
  const float *L32 = static_cast<const float *>(c->ws_l32.ptr);

  // ---- chunking over vectors (X budget, sized for the widest element in use)
  const int64_t elem = use[MJK_PREC_FP64] ? 8 : 4;
  const int64_t xvec_bytes = elem * ldc * n_pad;
  int64_t jc = std::max<int64_t>(1, std::min<int64_t>(c->nchol, c->x_budget / xvec_bytes));
  int64_t nchunk = 0, nchunk64 = 0;  // chunks in reduced precision, in FP64
  for (const Segment &s : segs)
    if (s.j1 > s.j0) (s.prec == MJK_PREC_FP64 ? nchunk64 : nchunk) += ceil_div(s.j1 - s.j0, jc);
  if (jc * ldc >= (int64_t(1) << 31))
    return set_error(c, MJK_ERR_ARG, "exchange: chunk contraction length exceeds 2^31");
  if ((rc = ensure(c, c->w->x, size_t(xvec_bytes) * jc))) return rc;

  // ---- SYRK tiling and slices (one launch per chunk covers every density)
  int64_t work = 0;  // contraction rows per vector over all densities
  for (int d = 0; d < nk; ++d)
    if (nocc[d] > 0) work += opad[size_t(d)];
  int tm = c->tile_syrk ? c->tile_syrk : (n_pad >= 512 && n_pad % 128 == 0 ? 128 : 64);
  if (n_pad % tm) tm = 64;
  const int ntile1 = int(ceil_div(n, tm));
  const int ntiles = ntile1 * (ntile1 + 1) / 2;
  SyrkSets sets{};
  sets.n = nk;
  int64_t kb = 0;
  sets.item0[0] = 0;
  // slices per density in proportion to its contraction length (opad rows per vector).
  // Workgroups per launch: at most the target, rounded down, so that a target of
  // whole resident rounds (k_syrk keeps two workgroups per CU) leaves no handful
  // of items to a round of its own.  Default: the most rounds (1, 2, 4 or 8) that
  // still give every item >= 2048 contraction rows; shorter items lose more to
  // their pipeline fill and store-out than finer balancing gains.
  const int64_t slots = 2 * int64_t(c->ncu);
  auto slices = [&](int d, int64_t tiles) {
    int rounds = 1;
    while (rounds < 8 && jc * work * tiles >= int64_t(2048) * slots * (2 * rounds)) rounds *= 2;
    const int target = c->split_target ? c->split_target : int(slots * rounds);
    const int64_t want = int64_t(target) * opad[size_t(d)] / (tiles * std::max<int64_t>(work, 1));
    return nocc[d] > 0 ? int(std::max<int64_t>(1, std::min<int64_t>(want, jc))) : 0;
  };
  // What a screened call leaves out at a given tau depends on the tiles and slices that
  // the bound is tested over.  They are the same in every precision, whatever the
  // kernels themselves use: TM x TM, slices counted over the tiles of n_pad.  The FP32
  // kernel, which tests its own slices, scales tau where it has more of them.
  ScreenSets ref{};
  ref.n = nk;
  ref.strips = tm / 64;
  ref.ntiles = ntiles;
  double tau32 = tau;
  const int pad1 = n_pad / tm;
  for (int d = 0; d < nk; ++d) {
    sets.nsplit[d] = slices(d, ntiles);
    sets.off[d] = off[size_t(d)];
    sets.opad[d] = std::max(opad[size_t(d)], 1);
    sets.kbase[d] = kb;
    kb += int64_t(sets.nsplit[d]) * nchunk * ntiles * tm * tm;
    sets.item0[d + 1] = sets.item0[d] + sets.nsplit[d] * ntiles;
    ref.nref[d] = slices(d, int64_t(pad1) * (pad1 + 1) / 2);
    ref.item0[d + 1] = ref.item0[d] + ref.nref[d] * ntiles;
    if (ref.nref[d] < sets.nsplit[d]) tau32 = std::min(tau32, tau * ref.nref[d] / sets.nsplit[d]);
  }
  const int items = sets.item0[nk];
  // Partial tiles of all FP64 chunks together: a sixteenth of the X budget (so that a
  // smaller budget, which means more chunks, takes less), and less again where the
  // device has no room for that.
  Syrk64Sets sets64{};
  int64_t kb64 = 0, &most = c->w->kpart_most;
  for (int64_t tried = -1;; tried = kb64) {
    const int64_t bytes = std::min(most, c->x_budget / 16);
    if (nchunk64)
      kb64 = plan_syrk64(c, nk, nocc, off, opad, jc, work, nchunk64,
                         bytes / (int64_t(sizeof(double)) * kSlot64 * nchunk64), &sets64);
    if (kb64 == tried) break;  // no smaller plan
    if ((rc = ensure(c, c->w->kpart, sizeof(double) * size_t(std::max<int64_t>(kb64 + kb, 1)))) != MJK_ERR_NOMEM) break;
    most = bytes / 2;
  }
  if (rc) {
    most = INT64_MAX;
    return rc;
  }
  double *kpart64 = static_cast<double *>(c->w->kpart.ptr), *kpart = kpart64 + kb64;

  // ---- screening set-up (norms of L strips, of the orbital sets, counters)
  const bool screen = tau > 0.0 || thr_x > 0.0;
  const int nstrip = n_pad / 64;
  uint8_t *keep = nullptr;
  c->k_items = c->x_tiles = 0;
  c->scr = Screen{};
  // the screening state must not outlive this call on any return path: other
  // users of the half-transform (puvx, backward) launch unscreened
  struct ScreenReset {
    Context *c;
    ~ScreenReset() { c->scr = Screen{}; }
  } screen_reset{c};
  if (screen) {
    if (use[MJK_PREC_BF16X3])
      return set_error(c, MJK_ERR_ARG, "exchange: screening is not available for split-BF16");
    if ((rc = ensure(c, c->scount, 2 * sizeof(unsigned long long))) ||
        (rc = fill_zero(c, c->scount.ptr, 2 * sizeof(unsigned long long))))
      return rc;
    c->scr.cnt = static_cast<unsigned long long *>(c->scount.ptr);
    c->scr.nstrip = nstrip;
    c->scr.xw = c->ht_ta == 128 && ot <= 6 ? 2 : 1;
    if (thr_x > 0.0) {
      if (!c->lnorm_valid) {
        if ((rc = ensure(c, c->lnorm, sizeof(double) * size_t(c->nchol) * nstrip))) return rc;
        hipLaunchKernelGGL(k_strip_norms, dim3(unsigned(c->nchol), unsigned(nstrip)), dim3(kThreads),
                           0, c->stream, c->L, c->ldl, n, nstrip,
                           static_cast<double *>(c->lnorm.ptr));
        c->lnorm_valid = true;
      }
      if ((rc = ensure(c, c->w->cnorm, sizeof(double) * (kMaxSets + 1)))) return rc;
      double *cn = static_cast<double *>(c->w->cnorm.ptr);
      if (use[MJK_PREC_FP64])
        hipLaunchKernelGGL(k_cnorm<double>, dim3(1), dim3(kThreads), 0, c->stream,
                           static_cast<const double *>(c->w->cbank.ptr), ldc, n, sets, cn);
      else
        hipLaunchKernelGGL(k_cnorm<float>, dim3(1), dim3(kThreads), 0, c->stream,
                           static_cast<const float *>(c->w->cb32.ptr), ldc, n, sets, cn);
      c->scr.lnorm = static_cast<const double *>(c->lnorm.ptr);
      c->scr.cmax = cn + nk;
      c->scr.thr_x = thr_x;
    }
    if (tau > 0.0) {
      const size_t norms = size_t(nk) * jc * nstrip;
      if ((rc = ensure(c, c->w->xn2, sizeof(double) * norms + size_t(ref.item0[nk])))) return rc;
      keep = static_cast<uint8_t *>(static_cast<void *>(static_cast<double *>(c->w->xn2.ptr) + norms));
      c->scr.tau = use[MJK_PREC_FP64] ? tau : tau32;
    }
  }

  int64_t slot = 0, slot64 = 0;  // running chunk indices
  for (const Segment &s : segs) {
    for (int64_t j0 = s.j0; j0 < s.j1; j0 += jc, ++(s.prec == MJK_PREC_FP64 ? slot64 : slot)) {
      const int64_t jn = std::min(jc, s.j1 - j0);
      phase_begin(c);
      switch (s.prec) {
        case MJK_PREC_FP64:
          // the reduced precisions may round the bank up by a tile: all of it then
          ht64_dispatch(c, ceil_div(tot, 16) == ot ? tot : ldc, static_cast<const double *>(c->w->cbank.ptr), j0, jn,
                        static_cast<double *>(c->w->x.ptr));
          break;
        case MJK_PREC_FP32:
          ht32_dispatch(c, ot, L32, static_cast<const float *>(c->w->cb32.ptr), j0, jn,
                           static_cast<float *>(c->w->x.ptr));
          break;
        default: {
          const __bf16 *cbh = static_cast<const __bf16 *>(c->w->cb3.ptr);
          ht_dispatch_b3(c, ot, L32, cbh, cbh + size_t(ldc) * n_pad, j0, jn,
                         static_cast<float *>(c->w->x.ptr));
        }
      }
      phase_end(c, MJK_PHASE_HALF_TRANSFORM);
      if (zsave) {
        phase_begin(c);
        if ((rc = z_from_x(c, c->w->x.ptr, s.prec != MJK_PREC_FP64, ldc, nocc[0], jn,
                           c->zs.z + j0 * int64_t(nocc[0]) * nocc[0])))
          return rc;
        phase_end(c, MJK_PHASE_ZSAVE);
      }
      if (screen && tau > 0.0) {
        double *xn2 = static_cast<double *>(c->w->xn2.ptr);
        if (s.prec == MJK_PREC_FP64)
          hipLaunchKernelGGL(k_xnorms<double>, dim3(unsigned(jn), unsigned(nstrip), unsigned(nk)),
                             dim3(kThreads), 0, c->stream, static_cast<const double *>(c->w->x.ptr),
                             ldc, n, n_pad, sets, nstrip, xn2);
        else
          hipLaunchKernelGGL(k_xnorms<float>, dim3(unsigned(jn), unsigned(nstrip), unsigned(nk)),
                             dim3(kThreads), 0, c->stream, static_cast<const float *>(c->w->x.ptr),
                             ldc, n, n_pad, sets, nstrip, xn2);
        c->scr.xn2 = xn2;
      }
      phase_begin(c);
      switch (s.prec) {
        case MJK_PREC_FP64:
          syrk_launch64(c, static_cast<const double *>(c->w->x.ptr), ldc, jn, sets64, kpart64, int(slot64), ref, keep);
          break;
        case MJK_PREC_FP32:
          syrk_launch32(c, tm, items, static_cast<const float *>(c->w->x.ptr), ldc, jn, ntiles,
                        sets, kpart, int(slot));
          break;
        default:
          syrk_launch_b3(c, tm, items, static_cast<const float *>(c->w->x.ptr), ldc, jn, ntiles,
                         sets, kpart, int(slot));
      }
      phase_end(c, MJK_PHASE_EXCHANGE);
    }
  }
  phase_begin(c);
  hipLaunchKernelGGL(k_reduce_k, dim3(unsigned(n), unsigned(ceil_div(n, 64)), unsigned(nk)), dim3(kThreads), 0,
                     c->stream, kpart64, sets64, int(nchunk64), kpart, tm, sets, int(nchunk), n, klt, ldk);
  phase_end(c, MJK_PHASE_REDUCE);
  return hip_check(c, hipGetLastError(), "exchange launch");
}

}  // namespace

int pack_bank(Context *c, int32_t nk, const int32_t *nocc, const double *const *corb,
              std::vector<int> &off, std::vector<int> &opad, int *ot, int *tot) {
  int rc = bank_layout(c, nk, nocc, off, opad, true, ot, tot);
  if (rc || *tot == 0) return rc;
  return pack_bank_t<double>(c, nk, nocc, corb, off, 16 * *ot, c->w->cbank);
}

void ht_launch(Context *c, int tot, const double *cb, int64_t j0, int64_t jn, double *X) {
  ht64_dispatch(c, tot, cb, j0, jn, X);
}

int exchange(Context *c, int32_t nk, const int32_t *nocc, const double *const *corb, double *klt,
             int64_t ldk, int32_t precision) {
  const int64_t M = c->nchol;
  if (precision == MJK_PREC_LADDER)  // split points of mjk_set_ladder; FP64 until set
    return exchange_mixed(c, nk, nocc, corb, klt, ldk, c->lad_fp32 < 0 ? M : c->lad_fp32,
                          c->lad_bf16 < 0 ? M : c->lad_bf16);
  if (precision < MJK_PREC_FP64 || precision > MJK_PREC_BF16X3)
    return set_error(c, MJK_ERR_ARG, "exchange: precision mode not available");
  return exchange_mixed(c, nk, nocc, corb, klt, ldk, precision == MJK_PREC_FP64 ? M : 0,
                        precision == MJK_PREC_BF16X3 ? 0 : M);
}

int exchange_screened(Context *c, int32_t nk, const int32_t *nocc, const double *const *corb,
                      double *klt, int64_t ldk, int32_t precision, double tau, double thr_x) {
  if (nk < 1) return set_error(c, MJK_ERR_ARG, "exchange: nk < 1");
  if (ldk < c->np) return set_error(c, MJK_ERR_ARG, "exchange: ldk < nbas(nbas+1)/2");
  if (c->nloaded != c->nchol)
    return set_error(c, MJK_ERR_SHORT_READ, "exchange: not all Cholesky vectors were uploaded");
  if (!(tau >= 0.0) || !(thr_x >= 0.0))
    return set_error(c, MJK_ERR_ARG, "exchange: screening thresholds must be >= 0");
  if (precision == MJK_PREC_LADDER) {
    if (tau > 0.0 || thr_x > 0.0)
      return set_error(c, MJK_ERR_ARG, "exchange: the precision ladder cannot be screened");
    return exchange(c, nk, nocc, corb, klt, ldk, precision);
  }
  if (precision < MJK_PREC_FP64 || precision > MJK_PREC_BF16X3)
    return set_error(c, MJK_ERR_ARG, "exchange: precision mode not available");
  std::vector<Segment> segs = {{0, c->nchol, precision}};
  return exchange_segments(c, nk, nocc, corb, klt, ldk, segs, tau, thr_x);
}

int exchange_mixed(Context *c, int32_t nk, const int32_t *nocc, const double *const *corb,
                   double *klt, int64_t ldk, int64_t j_fp32, int64_t j_bf16) {
  if (nk < 1) return set_error(c, MJK_ERR_ARG, "exchange: nk < 1");
  if (ldk < c->np) return set_error(c, MJK_ERR_ARG, "exchange: ldk < nbas(nbas+1)/2");
  if (c->nloaded != c->nchol)
    return set_error(c, MJK_ERR_SHORT_READ, "exchange: not all Cholesky vectors were uploaded");
  const int64_t M = c->nchol;
  if (j_fp32 < 0 || j_fp32 > j_bf16 || j_bf16 > M)
    return set_error(c, MJK_ERR_ARG, "exchange: need 0 <= j_fp32 <= j_bf16 <= nchol");
  std::vector<Segment> segs = {{0, j_fp32, MJK_PREC_FP64},
                               {j_fp32, j_bf16, MJK_PREC_FP32},
                               {j_bf16, M, MJK_PREC_BF16X3}};
  return exchange_segments(c, nk, nocc, corb, klt, ldk, segs);
}

}  // namespace mjk
