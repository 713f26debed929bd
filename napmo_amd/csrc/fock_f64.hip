// FP64 contraction F = Phi^T diag(s) Phi over the 16 x 16 blocks of the upper triangle
// (src/wavefunction/nwavefunction.cpp:77-107), for up to FOCK_MAX_NB block rows; 64 x 64 tiles
// for two operands and larger bases.
//
// The nb (nb + 1) / 2 upper blocks, in row order, are cut into equal strips; a workgroup takes
// one strip over one chunk of points, and its 4 or 8 waves hold consecutive runs of at most 16
// blocks in MFMA accumulators. So no block below the diagonal and no padding column is
// computed, and every wave has the same work (within one block): the 64 x 64 tiles did 15 x 16
// blocks for the 190 of 300 functions and 36 x 16 for the 465 of 480. Strips of up to 10 blocks
// (4 block rows) split the points of a stage over sets of waves and add the sets in LDS.
//
// Points run through LDS in stages, double buffered, with two more stages of loads in flight in
// registers: the strip's columns of Phi, and s Phi for its rows. An FP64 MFMA (64 cycles per
// 16 x 16 x 4 product) holds its SIMD's VALU, and every VALU instruction between two products
// costs 6 to 8 cycles of matrix time (measured), so the product loop holds no other arithmetic:
// fragment addresses stay in registers and s is multiplied in while staging. What is left above
// the MFMA time is that staging (LDS writes 15 %, loads 10 % at n = 300).
// Measured, 64 x 64 tiles -> this: n = 300, 472,000 points 1.02 -> 0.74 ms (62 TFLOP/s on the
// upper blocks); n = 480, 1,062,000 points 5.4 -> 4.1 ms (62); n = 130, 140,000 points 0.122 ->
// 0.086 ms; n = 10, 22,000 points 16.7 -> 6.2 us.
#include <algorithm>

#include "common.hpp"
#include "kernels.hpp"

namespace napmo {

typedef double d4 __attribute__((ext_vector_type(4)));
typedef double d2 __attribute__((ext_vector_type(2)));

void launch_fock_blocks(const FockShape &sh, const double *X, const double *s, double *partial, hipStream_t st);
void launch_fock_block_reduce(const FockShape &sh, const double *partial, int n, double *F, hipStream_t st);

// ------------------------------------------------------------------ 64 x 64 tiles
// Two operands (X^T diag(s) Y, all tiles), bases past FOCK_MAX_NB block rows, and the shape of
// the BF16 contractions.
// F[mu][nu] = sum_p X[p][mu] s[p] Y[p][nu]: A[m][k] = X[p0+k][mu0+m], B[k][n] =
// s[p0+k] Y[p0+k][nu0+n]. Split over points (chunks); one workgroup per (tile, chunk).
FockShape fock_shape(int ld, long Npad, bool symmetric, long wg_target) {
  FockShape sh;
  sh.ld = ld;
  sh.nt = ld / TILE;
  sh.ntiles = symmetric ? sh.nt * (sh.nt + 1) / 2 : sh.nt * sh.nt;
  sh.symmetric = symmetric;
  sh.Npad = Npad;
  // aim at ~2048 workgroups (or wg_target); chunks a multiple of 256 points (the mixed
  // kernel's FP32 accumulation block)
  long want = std::max(1L, (wg_target > 0 ? wg_target : 2048L) / sh.ntiles);
  long chunk = round_up(div_up(Npad, want), 256);
  sh.chunk = std::max<long>(chunk, 256);
  sh.nchunk = (int)div_up(Npad, sh.chunk);
  return sh;
}

__device__ inline void tile_coords(int t, int nt, bool symmetric, int &ti, int &tj) {
  if (!symmetric) {
    ti = t / nt, tj = t % nt;
    return;
  }
  int i = 0, rem = t;
  while (rem >= nt - i) rem -= nt - i, ++i;
  ti = i, tj = i + rem;
}

// Points run in stages of KS: the next stage's rows (4 consecutive doubles of one point
// per thread for each operand) are loaded into registers while the current stage's MFMAs
// run, then stored to the other LDS buffer (one barrier per stage). LDS rows hold 64
// functions plus 16 doubles of padding, so a 16 x 4 fragment read touches each bank once
// per half-wave.
constexpr int KS = 16;  // points staged in LDS per step
constexpr int FSTRIDE = TILE + 16;
constexpr size_t TILE_LDS = 4 * KS * FSTRIDE * sizeof(double);

__device__ __forceinline__ void fock_f64_body(const double *__restrict__ X,
                                              const double *__restrict__ Yv,
                                              const double *__restrict__ s, int ld, int nt,
                                              int symmetric, int ntiles, int nchunk, long Npad,
                                              long chunk, double *__restrict__ partial, int g,
                                              double *lds) {
  auto As = (double (*)[KS][FSTRIDE])lds;  // As[.][k][m] = X[p0 + k][mu0 + m]
  auto Bs = As + 2;                        // Bs[.][k][n] = s[p0 + k] Y[p0 + k][nu0 + n]
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  // XCD-aware order: workgroup g runs on XCD g % 8; all tiles of one chunk of points get
  // ids congruent mod 8 (g = 8 i + x: tile i % ntiles, chunk (i / ntiles) * 8 + x), so the
  // chunk's Phi rows are shared through one L2
  const int xcd = g & 7, gi = g >> 3;
  const int tile = gi % ntiles, chunk_id = (gi / ntiles) * 8 + xcd;
  if (chunk_id >= nchunk) return;
  int ti, tj;
  tile_coords(tile, nt, symmetric, ti, tj);
  const int mu0 = ti * TILE, nu0 = tj * TILE;
  const bool same = (X == Yv) && (ti == tj);
  const long pbeg = (long)chunk_id * chunk;
  const long pend = min(Npad, pbeg + chunk);
  const int wr = (wave >> 1) * 32, wc = (wave & 1) * 32;
  const int lr = tid >> 4, lc = (tid & 15) * 4;  // this thread's stage row and 4 columns
  d4 ra, rb;
  double rs = 0.0;
  auto load = [&](long k0) {
    const long p = k0 + lr;
    ra = *(const d4 *)&X[p * ld + mu0 + lc];
    if (!same) rb = *(const d4 *)&Yv[p * ld + nu0 + lc];
    rs = s[p];
  };
  auto store = [&](int buf) {
    const d4 b = same ? ra : rb;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      As[buf][lr][lc + e] = ra[e];
      Bs[buf][lr][lc + e] = rs * b[e];
    }
  };
  d4 acc[2][2];
  for (int a = 0; a < 2; ++a)
    for (int b = 0; b < 2; ++b) acc[a][b] = (d4){0, 0, 0, 0};
  if (pbeg < pend) {
    load(pbeg);
    store(0);
  }
  __syncthreads();
  int buf = 0;
  const int kr0 = lane >> 4, mi = lane & 15;
  for (long k0 = pbeg; k0 < pend; k0 += KS) {
    const bool more = k0 + KS < pend;
    if (more) load(k0 + KS);
#pragma unroll
    for (int ks = 0; ks < KS; ks += 4) {
      const int kr = ks + kr0;
      const double a0 = As[buf][kr][wr + mi], a1 = As[buf][kr][wr + 16 + mi];
      const double b0 = Bs[buf][kr][wc + mi], b1 = Bs[buf][kr][wc + 16 + mi];
      acc[0][0] = __builtin_amdgcn_mfma_f64_16x16x4f64(a0, b0, acc[0][0], 0, 0, 0);
      acc[0][1] = __builtin_amdgcn_mfma_f64_16x16x4f64(a0, b1, acc[0][1], 0, 0, 0);
      acc[1][0] = __builtin_amdgcn_mfma_f64_16x16x4f64(a1, b0, acc[1][0], 0, 0, 0);
      acc[1][1] = __builtin_amdgcn_mfma_f64_16x16x4f64(a1, b1, acc[1][1], 0, 0, 0);
    }
    if (more) store(buf ^ 1);
    __syncthreads();
    buf ^= 1;
  }
  double *out = partial + (long)chunk_id * ((long)ntiles * TILE * TILE + 32) +
                (long)tile * TILE * TILE;
  const int col16 = lane & 15, rg = lane >> 4;
  for (int a = 0; a < 2; ++a)
    for (int b = 0; b < 2; ++b)
      for (int r = 0; r < 4; ++r)
        out[(wr + a * 16 + rg + 4 * r) * TILE + wc + b * 16 + col16] = acc[a][b][r];
}

__global__ void __launch_bounds__(256) k_fock_f64(const double *__restrict__ X,
                                                  const double *__restrict__ Yv,
                                                  const double *__restrict__ s, int ld, int nt,
                                                  int symmetric, int ntiles, int nchunk, long Npad,
                                                  long chunk, double *__restrict__ partial) {
  extern __shared__ d4 fock_lds[];
  fock_f64_body(X, Yv, s, ld, nt, symmetric, ntiles, nchunk, Npad, chunk, partial, blockIdx.x,
                (double *)fock_lds);
}

void launch_fock_f64(const FockShape &sh, const double *X, const double *Y, const double *s,
                     double *partial, hipStream_t st) {
  if (sh.nb > 0) {
    NAPMO_REQUIRE(X == Y, "FP64 contraction: block shapes are symmetric");
    launch_fock_blocks(sh, X, s, partial, st);
    return;
  }
  const dim3 grid((unsigned)(sh.ntiles * round_up(sh.nchunk, 8)));
  k_fock_f64<<<grid, 256, TILE_LDS, st>>>(X, Y, s, sh.ld, sh.nt, sh.symmetric ? 1 : 0, sh.ntiles,
                                   sh.nchunk, sh.Npad, sh.chunk, partial);
  NAPMO_HIP(hipGetLastError());
}

// Sum the chunk partials of each computed tile element: 4 slices of chunks per element
// (slice k takes chunks k, k + 4, ...), combined in slice order (deterministic). Threads
// walk the tile-element space of the partials, so every load is coalesced; the mirror
// image of an off-diagonal upper tile is written by the same thread. Partials are FP64
// (per-tile kernels) or FP32 (the one-pass mixed kernel, whose accumulators are FP32).
template <class T>
__device__ __forceinline__ void fock_reduce_body(const T *__restrict__ partial, int nt, int ntiles,
                                                 int nchunk, int symmetric, int n,
                                                 int upper_mirror, double scale, int accumulate,
                                                 double *__restrict__ F, long g) {
  __shared__ double red[4][64];
  const int el = threadIdx.x & 63, slice = threadIdx.x >> 6;
  const long u = g * 64 + el;
  const long nel = (long)ntiles * TILE * TILE;
  double sum = 0.0;
  if (u < nel) {
    const long cstride = nel + 32;
    int c = slice;
    // 8 loads in flight, added in chunk order
    for (; c + 28 < nchunk; c += 32) {
      double v[8];
#pragma unroll
      for (int k = 0; k < 8; ++k) v[k] = (double)partial[(long)(c + 4 * k) * cstride + u];
#pragma unroll
      for (int k = 0; k < 8; ++k) sum += v[k];
    }
    for (; c < nchunk; c += 4) sum += (double)partial[(long)c * cstride + u];
  }
  red[slice][el] = sum;
  __syncthreads();
  if (slice != 0 || u >= nel) return;
  const double tot = ((red[0][el] + red[1][el]) + red[2][el] + red[3][el]) * scale;
  const int t = (int)(u / (TILE * TILE)), r = (int)(u % (TILE * TILE)) / TILE, cc = (int)(u % TILE);
  int ti, tj;
  if (symmetric) {
    // upper tiles in row order: (0,0), (0,1), ..., (0,nt-1), (1,1), ...
    int rem = t;
    ti = 0;
    while (rem >= nt - ti) rem -= nt - ti, ++ti;
    tj = ti + rem;
  } else {
    ti = t / nt, tj = t % nt;
  }
  const int i = ti * TILE + r, j = tj * TILE + cc;
  if (i >= n || j >= n) return;
  auto put = [&](int a, int b) {
    const long e = (long)a * n + b;
    F[e] = accumulate ? F[e] + tot : tot;
  };
  if (symmetric) {
    // the upper triangle is mirrored, so F is exactly symmetric (a diagonal tile's own
    // lower half, equal to rounding, is not used)
    if (i > j) return;
    put(i, j);
    if (i != j) put(j, i);
  } else if (upper_mirror) {
    if (i <= j) {
      put(i, j);
      if (i != j) put(j, i);
    }
  } else {
    put(i, j);
  }
}

template <class T>
__global__ void __launch_bounds__(256) k_fock_reduce(const T *__restrict__ partial, int nt,
                                                     int ntiles, int nchunk, int symmetric, int n,
                                                     int upper_mirror, double scale, int accumulate,
                                                     double *__restrict__ F) {
  fock_reduce_body<T>(partial, nt, ntiles, nchunk, symmetric, n, upper_mirror, scale, accumulate,
                      F, blockIdx.x);
}

void launch_fock_reduce(const FockShape &sh, const double *partial, int n, int upper_mirror,
                        double scale, int accumulate, double *F, hipStream_t st) {
  if (sh.nb > 0) {
    NAPMO_REQUIRE(scale == 1.0 && !accumulate, "FP64 contraction reduction: block shapes");
    launch_fock_block_reduce(sh, partial, n, F, st);
    return;
  }
  const long nel = (long)sh.ntiles * TILE * TILE;
  k_fock_reduce<double><<<div_up(nel, 64), 256, 0, st>>>(partial, sh.nt, sh.ntiles, sh.nchunk,
                                                         sh.symmetric ? 1 : 0, n, upper_mirror,
                                                         scale, accumulate, F);
  NAPMO_HIP(hipGetLastError());
}

void launch_fock_reduce_f32(const FockShape &sh, const float *partial, int n, double *F,
                            hipStream_t st) {
  const long nel = (long)sh.ntiles * TILE * TILE;
  k_fock_reduce<float><<<div_up(nel, 64), 256, 0, st>>>(partial, sh.nt, sh.ntiles, sh.nchunk,
                                                        sh.symmetric ? 1 : 0, n, 0, 1.0, 0, F);
  NAPMO_HIP(hipGetLastError());
}


// ---------------------------------------------------------------- upper 16 x 16 blocks
namespace {

constexpr int FOCK_BPW = 16;  // most blocks per wave: 128 accumulator registers, two waves per SIMD
constexpr int FOCK_CUS = 256;

// first linear index of block row i in the upper triangle of nb rows
__host__ __device__ inline int tri_first(int i, int nb) { return i * nb - i * (i - 1) / 2; }

__host__ __device__ inline int tri_row(int b, int nb) {
  int i = 0;
  while (i + 1 < nb && tri_first(i + 1, nb) <= b) ++i;
  return i;
}

// Shape classes by CW, the LDS row stride of the columns in blocks (odd, so that it is 16 mod
// 32 doubles): nb = 1, <= 3, 4, <= 8, <= 10, <= 20, <= FOCK_MAX_NB. Short strips use few waves per
// workgroup and several workgroups per CU; from 11 block rows on 8 waves share a stage, so its
// columns are staged for twice the blocks (4 waves -> 8 on one card: n = 300 0.86 -> 0.83 ms, n = 480 4.95 -> 4.06 ms).
__host__ __device__ constexpr int cw_of(int nb) {
  return nb == 1 ? 1 : (nb <= 3 ? 3 : (nb == 4 ? 5 : (nb <= 8 ? 9 : (nb <= 10 ? 21 : (nb <= 20 ? 25 : 41)))));
}
__host__ __device__ constexpr int maxnb_of(int cw) { return cw <= 3 ? cw : (cw == 21 ? 10 : (cw == 25 ? 20 : cw - 1)); }
// stride of the scaled rows: a strip of at most 16 nw_of(cw) blocks meets at most 11 or 16 block
// rows (12 or 16 with the last load's width)
__host__ __device__ constexpr int ra_of(int cw) { return cw == 21 ? 13 : (cw >= 25 ? 17 : cw); }
// points per stage
__host__ __device__ constexpr int kst_of(int cw) { return cw <= 3 ? 32 : (cw == 5 ? 16 : 8); }
// waves per workgroup
__host__ __device__ constexpr int nw_of(int cw) { return cw >= 25 ? 8 : 4; }
// workgroups per CU that LDS and the accumulators leave room for
__host__ __device__ constexpr int occ_of(int cw) { return cw >= 25 ? 1 : (cw == 21 ? 2 : 3); }
__host__ __device__ constexpr int lds_doubles(int cw) { return 2 * kst_of(cw) * 16 * (cw + ra_of(cw)); }

// columns that one 16-byte load per thread covers, and the most and fewest loads of a strip
__host__ __device__ constexpr int lcols_of(int cw) { return 128 * nw_of(cw) / kst_of(cw); }
__host__ __device__ constexpr int maxl_of(int cw) { return (16 * maxnb_of(cw) + lcols_of(cw) - 1) / lcols_of(cw); }

// BPW: blocks per wave; NSET: sets of waves that take different points of a stage; NCH: 16-byte
// loads per thread and stage (the strip's columns; a constant, so that no load is conditional
// and a wait for the older stage does not wait for the newer one)
template <int BPW, int CW, int NSET, int NCH>
__device__ __forceinline__ void fock_strip(const FockMember &f, int strip, int chunk_id, double *lds) {
  constexpr int KST = kst_of(CW), SB = 16 * CW, SA = 16 * ra_of(CW);
  constexpr int NW = nw_of(CW), TPR = 64 * NW / KST;  // threads per staged point
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int nb = f.nb, T = nb * (nb + 1) / 2;
  const int b0 = (int)((long)T * strip / f.nstrip), b1 = (int)((long)T * (strip + 1) / f.nstrip);
  constexpr int WS = NW / NSET;
  const int set = wave / WS, wis = wave - set * WS;
  const int w0 = b0 + (b1 - b0) * wis / WS, w1 = b0 + (b1 - b0) * (wis + 1) / WS;
  const int row0 = tri_row(b0, nb), ncol = 16 * (nb - row0);
  const int nrow = 16 * (tri_row(b1 - 1, nb) - row0 + 1);
  // lds: [2][KST][SB] Phi, then [2][KST][SA] s Phi of the strip's rows
  const int kr = lane >> 4, mi = lane & 15;
  // this wave's fragments, fixed addresses (buffer and k step are immediate offsets): a product
  // on the FP64 matrix cores holds the SIMD's VALU, so an address add in the loop is lost time
  int pa[BPW], pb[BPW];
  {
    int i = tri_row(w0, nb), j = i + (w0 - tri_first(i, nb));
    const int k = kr + 4 * set;
#pragma unroll
    for (int s = 0; s < BPW; ++s) {
      pa[s] = 2 * KST * SB + k * SA + mi + 16 * (i - row0), pb[s] = k * SB + mi + 16 * (j - row0);
      asm("" : "+v"(pa[s]), "+v"(pb[s]));  // kept, not added up again in the loop
      if (w0 + s + 1 < w1) {  // past the run: the last block again, not written
        if (++j == nb) ++i, j = i;
      }
    }
  }
  const long pbeg = (long)chunk_id * f.chunk, pend = min(f.Npad, pbeg + f.chunk);
  // thread t stages point t / TPR, columns 2 (t % TPR) + 2 TPR c; columns past the strip repeat
  // its last two (never used), so that no load or store is conditional
  const int srow = tid / TPR, scol = 2 * (tid % TPR);
  double *db = lds + srow * SB + scol, *da = lds + 2 * KST * SB + srow * SA + scol;
  unsigned off[NCH];
#pragma unroll
  for (int c = 0; c < NCH; ++c) off[c] = srow * f.ld + 16 * row0 + min(scol + 2 * TPR * c, ncol - 2);
  d2 r[2][NCH];
  double rs[2];
  // the stage from point p on (the last one again past the end), two stages ahead of its products:
  // one stage (about 1 us) does not cover the latency of a busy HBM
  auto load = [&](int q, long p) {
    p = min(p, pend - KST);
    const double *src = f.X + p * f.ld;
#pragma unroll
    for (int c = 0; c < NCH; ++c) r[q][c] = *(const d2 *)(src + off[c]);
    rs[q] = (f.s + p)[(unsigned)srow];
    __builtin_amdgcn_sched_barrier(0);
  };
  auto store = [&](int buf) {
#pragma unroll
    for (int c = 0; c < NCH; ++c) *(d2 *)(db + buf * KST * SB + 2 * TPR * c) = r[buf][c];
#pragma unroll
    for (int c = 0; c < NCH; ++c)
      if (2 * TPR * (c + 1) <= SA && 2 * TPR * c < nrow) *(d2 *)(da + buf * KST * SA + 2 * TPR * c) = rs[buf] * r[buf][c];
  };
  d4 acc[BPW];
#pragma unroll
  for (int s = 0; s < BPW; ++s) acc[s] = (d4){0, 0, 0, 0};
  // GB blocks of one k step at a time, the next group's fragments read while a group's products
  // run (left to itself the compiler reads each group's just before it, or all of them first)
  constexpr int GB = BPW < 4 ? BPW : 4, NG = (BPW + GB - 1) / GB, NK = KST / (4 * NSET);
  auto compute = [&](int buf) {
    double a[2][GB], b[2][GB];
    auto frag = [&](int u) {  // u = k step * NG + group
#pragma unroll
      for (int t = 0; t < GB; ++t) {
        const int s = (u % NG) * GB + t, ks = (u / NG) * 4 * NSET;
        if (s < BPW) {
          a[u & 1][t] = lds[pa[s] + (buf * KST + ks) * SA];
          b[u & 1][t] = lds[pb[s] + (buf * KST + ks) * SB];
        }
      }
    };
    frag(0);
#pragma unroll
    for (int u = 0; u < NG * NK; ++u) {
      if (u + 1 < NG * NK) frag(u + 1);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int t = 0; t < GB; ++t)
        if ((u % NG) * GB + t < BPW)
          acc[(u % NG) * GB + t] = __builtin_amdgcn_mfma_f64_16x16x4f64(a[u & 1][t], b[u & 1][t], acc[(u % NG) * GB + t], 0, 0, 0);
      __builtin_amdgcn_sched_barrier(0);
    }
  };
  load(0, pbeg);
  load(1, pbeg + KST);
  store(0);
  __syncthreads();
  // two stages per turn, one per buffer (chunks and Npad are whole pairs of stages)
#pragma unroll 1
  for (long p = pbeg; p < pend; p += 2 * KST) {
    load(0, p + 2 * KST);
    compute(0);
    store(1);
    __syncthreads();
    load(1, p + 3 * KST);
    compute(1);
    store(0);
    __syncthreads();
  }
  double *out = f.partial + (long)chunk_id * f.cstride;
  if constexpr (NSET == 1) {
#pragma unroll
    for (int s = 0; s < BPW; ++s)
      if (w0 + s < w1)
#pragma unroll
        for (int q = 0; q < 4; ++q) out[(long)(w0 + s) * 256 + (kr + 4 * q) * 16 + mi] = acc[s][q];
    return;
  }
  // sets of waves over different points: added in set order through LDS
  const int nblk = b1 - b0;
  double *red = lds;  // [NSET][nblk][256], at most 24 x 256
#pragma unroll
  for (int s = 0; s < BPW; ++s)
    if (w0 + s < w1)
#pragma unroll
      for (int q = 0; q < 4; ++q)
        red[(set * nblk + w0 + s - b0) * 256 + (kr + 4 * q) * 16 + mi] = acc[s][q];
  __syncthreads();
  for (int e = tid; e < nblk * 256; e += 64 * NW) {
    double sum = red[e];
    for (int k = 1; k < NSET; ++k) sum += red[k * nblk * 256 + e];
    out[(long)b0 * 256 + e] = sum;
  }
}

template <int BPW, int CW, int NSET, int NCH>
__device__ __forceinline__ void fock_strip_from(int nch, const FockMember &f, int strip, int chunk_id, double *lds) {
  if constexpr (NCH <= 1) {
    fock_strip<BPW, CW, NSET, 1>(f, strip, chunk_id, lds);
  } else if (nch >= NCH || NCH == 2) {
    fock_strip<BPW, CW, NSET, NCH>(f, strip, chunk_id, lds);
  } else {
    fock_strip_from<BPW, CW, NSET, NCH - 1>(nch, f, strip, chunk_id, lds);
  }
}

template <int BPW, int CW, int NSET>
__device__ __forceinline__ void fock_block_body(const FockMember &f, int g, double *lds) {
  // workgroup g runs on XCD g % 8: the strips of one chunk share that XCD's L2
  const int xcd = g & 7, gi = g >> 3;
  const int strip = gi % f.nstrip, chunk_id = (gi / f.nstrip) * 8 + xcd;
  if (chunk_id >= f.nchunk) return;
  const int T = f.nb * (f.nb + 1) / 2, row0 = tri_row((int)((long)T * strip / f.nstrip), f.nb);
  fock_strip_from<BPW, CW, NSET, maxl_of(CW)>((16 * (f.nb - row0) + lcols_of(CW) - 1) / lcols_of(CW), f, strip,
                                              chunk_id, lds);
}

size_t fock_block_lds(const FockShape &sh) {
  size_t d = lds_doubles(cw_of(sh.nb));
  if (sh.nset > 1) d = std::max(d, (size_t)sh.nset * (sh.nb * (sh.nb + 1) / 2) * 256);
  return d * sizeof(double);
}

template <int BPW, int CW, int NSET>
__global__ void __launch_bounds__(64 * nw_of(CW), 4 * occ_of(CW) * nw_of(CW) / 16) k_fock_blocks(FockMember f) {
  extern __shared__ d4 fock_lds[];
  fock_block_body<BPW, CW, NSET>(f, blockIdx.x, (double *)fock_lds);
}

// (blocks per wave, CW, sets) of nb = 1 | 2, 3 | 4 | 5, 6, 7, 8 | 9, 10; 11 .. 20 | 21 .. 40
#define NAPMO_FOCK_SHAPES4(M)                                                                   \
  M(1, 1, 4) M(3, 3, 4) M(6, 3, 4) M(5, 5, 2) M(4, 9, 1) M(6, 9, 1) M(7, 9, 1) M(9, 9, 1)       \
  M(12, 21, 1) M(14, 21, 1)
#define NAPMO_FOCK_SHAPES8(M) M(9, 25, 1) M(10, 25, 1) M(11, 25, 1) M(12, 25, 1) M(14, 25, 1) M(15, 25, 1) M(12, 41, 1) M(13, 41, 1) M(14, 41, 1) M(15, 41, 1) M(16, 41, 1)

// the block partials of every chunk, as k_fock_reduce does for 64 x 64 tiles: 4 slices of
// chunks per element, added in slice order; F mirrored from the upper triangle
__device__ __forceinline__ void fock_block_reduce_body(const double *__restrict__ partial, int nb,
                                                       int nchunk, long cstride, int n,
                                                       double *__restrict__ F, long g) {
  __shared__ double red[4][64];
  const int el = threadIdx.x & 63, slice = threadIdx.x >> 6;
  const long u = g * 64 + el;  // 256 elements per block: a workgroup stays inside one block
  double sum = 0.0;
  int c = slice;
  for (; c + 28 < nchunk; c += 32) {
    double v[8];
#pragma unroll
    for (int k = 0; k < 8; ++k) v[k] = partial[(long)(c + 4 * k) * cstride + u];
#pragma unroll
    for (int k = 0; k < 8; ++k) sum += v[k];
  }
  for (; c < nchunk; c += 4) sum += partial[(long)c * cstride + u];
  red[slice][el] = sum;
  __syncthreads();
  if (slice != 0) return;
  const double tot = (red[0][el] + red[1][el]) + red[2][el] + red[3][el];
  const int b = (int)(u / 256), bi = tri_row(b, nb), bj = bi + (b - tri_first(bi, nb));
  const int i = 16 * bi + (int)(u % 256) / 16, j = 16 * bj + (int)(u % 16);
  if (i > j || j >= n) return;
  F[(long)i * n + j] = tot;
  F[(long)j * n + i] = tot;
}

__global__ void __launch_bounds__(256) k_fock_block_reduce(const double *__restrict__ partial, int nb,
                                                           int nchunk, long cstride, int n,
                                                           double *__restrict__ F) {
  fock_block_reduce_body(partial, nb, nchunk, cstride, n, F, blockIdx.x);
}

FockMember member(const FockShape &sh, const double *X, const double *s, double *partial) {
  FockMember f = {};
  f.X = X, f.s = s, f.partial = partial, f.Npad = sh.Npad, f.chunk = sh.chunk, f.ld = sh.ld;
  f.nchunk = sh.nchunk, f.nb = sh.nb, f.bpw = sh.bpw, f.nstrip = sh.nstrip, f.nset = sh.nset;
  f.cstride = sh.cstride(), f.nt = sh.nt, f.ntiles = sh.ntiles;
  return f;
}

void set_lds(const void *kern) {
  NAPMO_HIP(hipFuncSetAttribute(kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)max_lds_per_block()));
}

}  // namespace

FockShape fock_block_shape(int n, int ld, long Npad, long wg_target) {
  FockShape sh = {};
  const int nb = (int)div_up(n, 16), T = nb * (nb + 1) / 2;
  sh.ld = ld, sh.symmetric = true, sh.Npad = Npad, sh.nb = nb;
  sh.nset = T <= 6 ? 4 : (T <= 12 ? 2 : 1);
  const int nw = nw_of(cw_of(nb));
  sh.nstrip = (int)div_up(T, FOCK_BPW * nw);
  sh.bpw = (int)div_up(div_up(T, sh.nstrip), nw / sh.nset);
  // one round of the workgroups that the device holds at once, every one the same work, since
  // every further round leaves more partials to add: contraction + reduction at n = 300, 472,000
  // points in one, two, four rounds 741 + 13, 748 + 21, 763 + 37 us; n = 480, 1,062,000 points
  // 4112 + 15, 4119 + 25, 4135 + 49; n = 130, 135,900 points in half a round, one, two 72 + 10,
  // 74 + 13, 82 + 20. At least 128 points each, so that short grids do not leave mostly partials.
  // Whole pairs of stages: 32 or 64 points.
  const long want = std::max(1L, (wg_target > 0 ? wg_target : (long)FOCK_CUS * occ_of(cw_of(nb))) / sh.nstrip);
  const long per = div_up(Npad, want);
  sh.chunk = std::max(128L, round_up(per, nb <= 3 || per > 1024 ? 64 : 32));
  sh.nchunk = (int)div_up(Npad, sh.chunk);
  return sh;
}

void launch_fock_blocks(const FockShape &sh, const double *X, const double *s, double *partial, hipStream_t st) {
  NAPMO_REQUIRE(sh.nb >= 1 && sh.nb <= FOCK_MAX_NB && 16 * sh.nb <= sh.ld && sh.ld % 2 == 0 &&
                    sh.Npad % 64 == 0 && sh.chunk % (2 * kst_of(cw_of(sh.nb))) == 0 && sh.bpw >= 1,
                "FP64 contraction: shape");
  const dim3 grid((unsigned)(sh.nstrip * round_up(sh.nchunk, 8)));
  const FockMember f = member(sh, X, s, partial);
  const size_t lds = fock_block_lds(sh);
  switch ((sh.bpw * 64 + cw_of(sh.nb)) * 8 + sh.nset) {
#define NAPMO_CASE(B, C, S)                                  \
  case (B * 64 + C) * 8 + S:                                       \
    set_lds((const void *)k_fock_blocks<B, C, S>);            \
    k_fock_blocks<B, C, S><<<grid, 64 * nw_of(C), lds, st>>>(f);        \
    break;
    NAPMO_FOCK_SHAPES4(NAPMO_CASE)
    NAPMO_FOCK_SHAPES8(NAPMO_CASE)
#undef NAPMO_CASE
    default: throw Error("FP64 contraction: no kernel for " + std::to_string(sh.bpw) + " blocks per wave");
  }
  NAPMO_HIP(hipGetLastError());
}

void launch_fock_block_reduce(const FockShape &sh, const double *partial, int n, double *F, hipStream_t st) {
  NAPMO_REQUIRE(n > 16 * (sh.nb - 1) && n <= 16 * sh.nb, "FP64 contraction reduction: shape");
  k_fock_block_reduce<<<4 * (sh.nb * (sh.nb + 1) / 2), 256, 0, st>>>(partial, sh.nb, sh.nchunk, sh.cstride(), n, F);
  NAPMO_HIP(hipGetLastError());
}

// ------------------------------------------------------------------ many plans in one launch
// (each workgroup finds its member and runs that member's own shape)
namespace {

__global__ void __launch_bounds__(256, 2) k_fock_f64_group(const FockMember *__restrict__ mem, int nmem) {
  extern __shared__ d4 fock_lds[];
  const long g = blockIdx.x;
  const FockMember f = mem[group_member(mem, nmem, g)];
  double *lds = (double *)fock_lds;
  switch ((f.bpw * 64 + cw_of(f.nb)) * 8 + f.nset) {
#define NAPMO_CASE(B, C, S) \
  case (B * 64 + C) * 8 + S: fock_block_body<B, C, S>(f, (int)(g - f.block0), lds); break;
    NAPMO_FOCK_SHAPES4(NAPMO_CASE)
    default:
      fock_f64_body(f.X, f.X, f.s, f.ld, f.nt, 1, f.ntiles, f.nchunk, f.Npad, f.chunk, f.partial,
                    (int)(g - f.block0), lds);
  }
}

// the members with eight waves per workgroup
__global__ void __launch_bounds__(512, 2) k_fock_f64_group8(const FockMember *__restrict__ mem, int nmem) {
  extern __shared__ d4 fock_lds[];
  const long g = blockIdx.x;
  const FockMember f = mem[group_member(mem, nmem, g)];
  double *lds = (double *)fock_lds;
  switch ((f.bpw * 64 + cw_of(f.nb)) * 8 + f.nset) {
    NAPMO_FOCK_SHAPES8(NAPMO_CASE)
#undef NAPMO_CASE
    default: break;
  }
}

__global__ void __launch_bounds__(256) k_fock_reduce_group(const FockReduceMember *__restrict__ mem,
                                                           int nmem) {
  const long g = blockIdx.x;
  const FockReduceMember &f = mem[group_member(mem, nmem, g)];
  if (f.nb > 0)
    fock_block_reduce_body(f.partial, f.nb, f.nchunk, f.cstride, f.n, f.F, g - f.block0);
  else
    fock_reduce_body<double>(f.partial, f.nt, f.ntiles, f.nchunk, 1, f.n, 0, 1.0, 0, f.F, g - f.block0);
}

}  // namespace

long fock_group_fill(FockMember &f, const FockShape &sh, const double *X, const double *s,
                     double *partial, long block0) {
  NAPMO_REQUIRE(sh.symmetric && block0 % 8 == 0, "grouped Fock: symmetric shapes, aligned blocks");
  f = member(sh, X, s, partial);
  f.block0 = block0;
  return (sh.nb > 0 ? sh.nstrip : (long)sh.ntiles) * round_up(sh.nchunk, 8);
}

int fock_group_waves(const FockShape &sh) { return sh.nb > 0 ? nw_of(cw_of(sh.nb)) : 4; }

size_t fock_group_lds(const FockShape &sh) { return sh.nb > 0 ? fock_block_lds(sh) : TILE_LDS; }

void launch_fock_group(const FockMember *d_mem, int nmem, long nblocks, int waves, size_t lds, hipStream_t st) {
  if (nmem <= 0 || nblocks <= 0) return;
  const dim3 grid((unsigned)nblocks);
  if (waves == 8) {
    set_lds((const void *)k_fock_f64_group8);
    k_fock_f64_group8<<<grid, 512, lds, st>>>(d_mem, nmem);
  } else {
    set_lds((const void *)k_fock_f64_group);
    k_fock_f64_group<<<grid, 256, lds, st>>>(d_mem, nmem);
  }
  NAPMO_HIP(hipGetLastError());
}

long fock_reduce_group_fill(FockReduceMember &f, const FockShape &sh, const double *partial, int n,
                            double *F, long block0) {
  NAPMO_REQUIRE(sh.symmetric, "grouped Fock reduction: symmetric shapes");
  f = {};
  f.partial = partial, f.F = F, f.block0 = block0, f.cstride = sh.cstride();
  f.nt = sh.nt, f.ntiles = sh.ntiles, f.nchunk = sh.nchunk, f.n = n, f.nb = sh.nb;
  return sh.nb > 0 ? 4L * (sh.nb * (sh.nb + 1) / 2) : div_up((long)sh.ntiles * TILE * TILE, 64);
}

void launch_fock_reduce_group(const FockReduceMember *d_mem, int nmem, long nblocks, hipStream_t st) {
  if (nmem <= 0 || nblocks <= 0) return;
  k_fock_reduce_group<<<dim3((unsigned)nblocks), 256, 0, st>>>(d_mem, nmem);
  NAPMO_HIP(hipGetLastError());
}

}  // namespace napmo
