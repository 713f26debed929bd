// gfx950 kernels of the nAPMO grid hot path: Becke partition, GTO collocation,
// Poisson projection / radial Green solve / synthesis, and the FP64 MFMA grid
// contractions rho = diag(Phi P Phi^T) and F = Phi^T diag(s) Phi.
#include <hip/hip_runtime.h>

#include <cmath>

#include "common.hpp"
#include "kernels.hpp"
#include "synth_launch.hpp"

namespace napmo {

typedef double d4 __attribute__((ext_vector_type(4)));

static constexpr double INV_SQRT_4_PI = 0.28209479177387814347;

// ================================================================ Becke partition
// One thread per point. Pair tables are wave-uniform loads (scalar cache).
__global__ void k_becke(const double *__restrict__ x, const double *__restrict__ y,
                        const double *__restrict__ z, long N, const int *__restrict__ owner, int M,
                        const double *__restrict__ center, const double *__restrict__ R,
                        const double *__restrict__ As, double *__restrict__ bw) {
  // Same operation order as the reference loop (no FMA contraction): the weights pass
  // through 1 - s with s near 1, where contraction changes the last bits visibly.
#pragma clang fp contract(off)
  long p = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (p >= N) return;
  const double px = x[p], py = y[p], pz = z[p];
  const int own = owner[p];
  double sum = 0.0, mine = 0.0;
  for (int i = 0; i < M; ++i) {
    double dx = px - center[3 * i], dy = py - center[3 * i + 1], dz = pz - center[3 * i + 2];
    const double ri = sqrt(dx * dx + dy * dy + dz * dz);
    double prod = 1.0;
    for (int j = 0; j < M; ++j) {
      if (j == i) continue;
      double ex = px - center[3 * j], ey = py - center[3 * j + 1], ez = pz - center[3 * j + 2];
      const double rj = sqrt(ex * ex + ey * ey + ez * ez);
      const double mu = (ri - rj) / R[i * M + j];
      double sv = mu + As[i * M + j] * (1.0 - mu * mu);
      sv = 0.5 * sv * (3 - sv * sv);
      sv = 0.5 * sv * (3 - sv * sv);
      sv = 0.5 * sv * (3 - sv * sv);
      prod *= 0.5 * (1.0 - sv);
    }
    if (i == own) mine = prod;
    sum += prod;
  }
  bw[p] = mine / sum;
}

void launch_becke(const double *x, const double *y, const double *z, long N, const int *owner,
                  int M, const double *center, const double *R, const double *As, double *bw,
                  hipStream_t s) {
  if (N <= 0) return;
  k_becke<<<div_up(N, 256), 256, 0, s>>>(x, y, z, N, owner, M, center, R, As, bw);
  NAPMO_HIP(hipGetLastError());
}

// ==================================================================== collocation
// Thread per (point, function): lanes run over functions so row writes coalesce.
__device__ inline double ipow(double v, int e) {
  double r = 1.0;
  for (int k = 0; k < e; ++k) r *= v;
  return r;
}

__global__ void k_collocate(const double *__restrict__ x, const double *__restrict__ y,
                            const double *__restrict__ z, long N, long Npad, int n, int ld,
                            const double *__restrict__ fo, const int *__restrict__ fl,
                            const int *__restrict__ ff, const int *__restrict__ fnp,
                            const double *__restrict__ fnorm, const double *__restrict__ pz,
                            const double *__restrict__ pc, double *__restrict__ out64,
                            float *__restrict__ out32) {
  const int mu = blockIdx.x * blockDim.x + threadIdx.x;
  const long p = (long)blockIdx.y * blockDim.y + threadIdx.y;
  if (mu >= ld || p >= Npad) return;
  double val = 0.0;
  if (mu < n && p < N) {
    const double dx = x[p] - fo[3 * mu], dy = y[p] - fo[3 * mu + 1], dz = z[p] - fo[3 * mu + 2];
    const double r2 = dx * dx + dy * dy + dz * dz;
    const double ang = ipow(dx, fl[3 * mu]) * ipow(dy, fl[3 * mu + 1]) * ipow(dz, fl[3 * mu + 2]);
    double acc = 0.0;
    const int f0 = ff[mu], np = fnp[mu];
    for (int k = 0; k < np; ++k) acc += pc[f0 + k] * ang * exp(-pz[f0 + k] * r2);
    val = acc * fnorm[mu];
  }
  const size_t o = (size_t)p * ld + mu;
  if (out64) out64[o] = val;
  if (out32) out32[o] = (float)val;
}

void launch_collocate(const double *x, const double *y, const double *z, long N, long Npad, int n,
                      int ld, const double *fo, const int *fl, const int *ff, const int *fnp,
                      const double *fnorm, const double *pz, const double *pc, double *out64,
                      float *out32, hipStream_t s) {
  dim3 block(64, 4);
  dim3 grid(div_up(ld, 64), div_up(Npad, 4));
  k_collocate<<<grid, block, 0, s>>>(x, y, z, N, Npad, n, ld, fo, fl, ff, fnp, fnorm, pz, pc, out64,
                                     out32);
  NAPMO_HIP(hipGetLastError());
}

// ========================================================= Poisson: projection
// rho_lm[A][i][lm] = sum_j f_Aij Yhat[j][lm] with f = dens * bw and the Lebedev table
// Yhat[j][lm] = aw_j S_lm(u_j) sqrt(4 pi (2l+1)) / sum aw: per atom a product of nset x nrad
// rows (density o, shell i) with Yhat, on FP64 MFMA. One workgroup forms 16 R rows x 16 C harmonics;
// its 8 waves share the angular points in groups of four (wave w the groups w, w + 8, ...), f is
// staged in LDS PJ points at a time (the next PJ read meanwhile), Yhat goes straight to the
// operand registers, and the waves' sums are added in order at the end. What bounds the product
// is reading Yhat from L2, once per 16 R rows (the rows of one density, 5 a workgroup, read
// 5.8 GB for 40 densities): 16 atoms x 50 x 590 points, lmax 12, 40 densities 0.63 -> 0.22
// ms, one density 24 -> 21 us; 8 atoms, 21 densities 74 -> 37 us. A row's sum does not depend on
// R and C, nor on the densities that share the launch.
constexpr int PJ = 128, PPITCH = PJ + 2, PWAVES = 8;

template <int R, int C>
__global__ void __launch_bounds__(64 * PWAVES, 4) k_project(AtomTables at, const double *__restrict__ dens,
                                                         const double *__restrict__ bw,
                                                         const double *__restrict__ yhat, int L,
                                                         double *__restrict__ rho_lm, int nset,
                                                         long dstride, long ostride) {
  constexpr int ROWS = 16 * R, NV = ROWS * PJ / (64 * PWAVES);
  constexpr int CP = C > 1 ? 2 : 1, NG = PJ / 4 / PWAVES;
  __shared__ double sh[ROWS * PPITCH > PWAVES * 256 * CP ? ROWS * PPITCH : PWAVES * 256 * CP];
  __shared__ long row_d[ROWS], row_p[ROWS], row_o[ROWS];
  const int A = blockIdx.z, tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int nr = at.nrad[A], na = at.nang[A];
  const int rows = nset * nr, q0 = blockIdx.x * ROWS, lm0 = blockIdx.y * 16 * C;
  if (q0 >= rows) return;
  if (tid < ROWS) {  // rows past the last repeat it and are not written
    const int q = min(q0 + tid, rows - 1), o = q / nr, i = q % nr;
    row_p[tid] = at.point_off[A] + (long)i * na;
    row_d[tid] = o * dstride + row_p[tid];
    row_o[tid] = o * ostride + (at.rad_off[A] + i) * (long)L;
  }
  __syncthreads();
  // harmonics above the centre's cut are zero (written, not summed)
  const int Lc = at.lcut ? (at.lcut[A] + 1) * (at.lcut[A] + 1) : L;
  const int kr = lane >> 4, mi = lane & 15;
  d4 acc[R][C];
#pragma unroll
  for (int r = 0; r < R; ++r)
#pragma unroll
    for (int c = 0; c < C; ++c) acc[r][c] = (d4){0, 0, 0, 0};
  if (lm0 < Lc) {
    const int sj = tid & (PJ - 1), sr = tid / PJ;
    double vd[NV], vb[NV];
    auto load = [&](int j0) {
      const int j = min(j0 + sj, na - 1);
#pragma unroll
      for (int t = 0; t < NV; ++t) {
        const int row = sr + t * (64 * PWAVES / PJ);
        vd[t] = dens[row_d[row] + j], vb[t] = bw[row_p[row] + j];
      }
    };
    const double *Y = yhat + at.yhat_off[A];
    int col[C];
#pragma unroll
    for (int c = 0; c < C; ++c) col[c] = min(lm0 + 16 * c + mi, L - 1);
    auto yload = [&](int j0, int u, double *y) {
      const int off = min(j0 + 4 * (wave + u * PWAVES) + kr, na - 1) * L;
#pragma unroll
      for (int c = 0; c < C; ++c) y[c] = Y[(unsigned)(off + col[c])];
    };
    auto multiply = [&](int u, const double *b) {
      double a[R];
#pragma unroll
      for (int r = 0; r < R; ++r) a[r] = sh[(16 * r + mi) * PPITCH + 4 * (wave + u * PWAVES) + kr];
#pragma unroll
      for (int r = 0; r < R; ++r)
#pragma unroll
        for (int c = 0; c < C; ++c)
          acc[r][c] = __builtin_amdgcn_mfma_f64_16x16x4f64(a[r], b[c], acc[r][c], 0, 0, 0);
    };
    double y[NG][C];
    load(0);
    if (C == 1)
#pragma unroll
      for (int u = 0; u < NG; ++u) yload(0, u, y[u]);
    for (int j0 = 0; j0 < na; j0 += PJ) {
#pragma unroll
      for (int t = 0; t < NV; ++t)
        sh[(sr + t * (64 * PWAVES / PJ)) * PPITCH + sj] = j0 + sj < na ? vd[t] * vb[t] : 0.0;
      __syncthreads();
      if (j0 + PJ < na) load(j0 + PJ);
      if (C == 1) {
        // few products: the wave's whole share of the next PJ points is in flight
        double b[NG][C];
#pragma unroll
        for (int u = 0; u < NG; ++u) b[u][0] = y[u][0];
#pragma unroll
        for (int u = 0; u < NG; ++u) yload(j0 + PJ, u, y[u]);
#pragma unroll
        for (int u = 0; u < NG; ++u) multiply(u, b[u]);
      } else {
        const int ng = ((min(PJ, na - j0) + 3) / 4 - wave + PWAVES - 1) / PWAVES;
        yload(j0, 0, y[0]);
        for (int u = 0; u < ng; ++u) {
          double b[C];
#pragma unroll
          for (int c = 0; c < C; ++c) b[c] = y[0][c];
          yload(j0, u + 1, y[0]);
          multiply(u, b);
        }
      }
      __syncthreads();
    }
  }
  // the waves' sums, 16 rows x 16 CP harmonics at a time (element e of a lane: row kr + 4 e)
#pragma unroll
  for (int h = 0; h < R * C / CP; ++h) {
    const int r = h / (C / CP), c0 = h % (C / CP) * CP;
#pragma unroll
    for (int c = 0; c < CP; ++c)
#pragma unroll
      for (int e = 0; e < 4; ++e)
        sh[(wave * 16 + kr + 4 * e) * 16 * CP + 16 * c + mi] = acc[r][c0 + c][e];
    __syncthreads();
    if (tid < 256 * CP) {
      double t = 0.0;
#pragma unroll
      for (int w = 0; w < PWAVES; ++w) t += sh[w * 256 * CP + tid];
      const int row = 16 * r + tid / (16 * CP), lm = lm0 + 16 * c0 + tid % (16 * CP);
      if (q0 + row < rows && lm < L) rho_lm[row_o[row] + lm] = lm < Lc ? t : 0.0;
    }
    __syncthreads();
  }
}

void launch_project(const AtomTables &at, const double *dens, const double *bw, const double *yhat,
                    int lmax, double *rho_lm, hipStream_t s, int nset, long dstride, long ostride) {
  const int L = (lmax + 1) * (lmax + 1);
  NAPMO_REQUIRE(nset >= 1 && (long)nset * at.M <= 65535, "projection: too many density sets");
  const long rows = (long)nset * at.max_nrad, cols = div_up(L, 64) * at.M;
  auto grid = [&](int r, int c) { return dim3((unsigned)div_up(rows, r), (unsigned)div_up(L, c), at.M); };
  // 32 rows x 64 harmonics read Yhat and f least, with at least two workgroups a CU (40 densities
  // on 16 atoms 0.22 ms; at 528 workgroups, 21 densities on 8 atoms, 16 rows take the same 37 us);
  // 16 rows down to one a CU (24 atoms, one density: 288 workgroups 26 us, 16 x 16 37 us); else
  // 16 x 16 (16 atoms: 192 workgroups of 16 x 64 21 us, 16 x 16 21 us; 3 atoms 10 -> 7.8 us)
  if (div_up(rows, 32) * cols >= 512)
    k_project<2, 4><<<grid(32, 64), 64 * PWAVES, 0, s>>>(at, dens, bw, yhat, L, rho_lm, nset, dstride, ostride);
  else if (div_up(rows, 16) * cols >= 256)
    k_project<1, 4><<<grid(16, 64), 64 * PWAVES, 0, s>>>(at, dens, bw, yhat, L, rho_lm, nset, dstride, ostride);
  else
    k_project<1, 1><<<grid(16, 16), 64 * PWAVES, 0, s>>>(at, dens, bw, yhat, L, rho_lm, nset, dstride, ostride);
  NAPMO_HIP(hipGetLastError());
}

// ====================================================== Poisson: radial solves
// U[A][i][lm] = sum_j G_{A,l}[i][j] rho_lm[A][j][lm] for y and dt; one workgroup per
// (atom, l, chunk of 256 outputs): the (nr x 2l+1) block of rho_lm is staged in LDS and
// each thread forms one output from a contiguous Green row. green block of an atom: for
// l = 0..lmax: Gy [nr x nr], then Gd [nr x nr].
constexpr int RMAX_STAGE = 4096;  // doubles of rho_lm staged per (atom, l)
constexpr int RADIAL_CHUNK = 256;

__global__ void __launch_bounds__(RADIAL_CHUNK) k_radial(AtomTables at, const double *__restrict__ rho_lm,
                                                const double *__restrict__ green, int L,
                                                double *__restrict__ Uy, double *__restrict__ Udt,
                                                int nchunk, long stride) {
  __shared__ double sr[RMAX_STAGE];
  const int A = blockIdx.x, l = blockIdx.y;
  if (at.lcut && l > at.lcut[A]) return;  // above the centre's cut: never read
  // blockIdx.z = set * nchunk + chunk: set k reads rho_lm + k stride, writes U + k stride
  const long set = blockIdx.z / nchunk;
  rho_lm += set * stride, Uy += set * stride, Udt += set * stride;
  const int nr = at.nrad[A], nm = 2 * l + 1;
  const int total = 2 * nr * nm;
  const int o0 = (blockIdx.z % nchunk) * RADIAL_CHUNK;
  if (o0 >= total) return;
  const double *G = green + at.green_off[A] + (long)l * 2 * nr * nr;
  const long roff = at.rad_off[A] * (long)L;
  const bool staged = nr * nm <= RMAX_STAGE;
  if (staged)
    for (int e = threadIdx.x; e < nr * nm; e += blockDim.x)
      sr[e] = rho_lm[roff + (long)(e / nm) * L + l * l + e % nm];
  __syncthreads();
  const int o = o0 + threadIdx.x;
  if (o >= total) return;
  const int m = o % nm, row = o / nm;  // row in [0, 2 nr): which * nr + i
  const int which = row / nr, i = row - which * nr;
  const double *g = G + (long)which * nr * nr + (long)i * nr;
  double acc = 0.0;
  if (staged) {
    for (int j = 0; j < nr; ++j) acc += g[j] * sr[j * nm + m];
  } else {
    const double *r = rho_lm + roff + l * l + m;
    for (int j = 0; j < nr; ++j) acc += g[j] * r[(long)j * L];
  }
  (which ? Udt : Uy)[roff + (long)i * L + l * l + m] = acc;
}

void launch_radial(const AtomTables &at, const double *rho_lm, const double *green, int lmax,
                   double *Uy, double *Udt, hipStream_t s, int nset, long stride) {
  const int L = (lmax + 1) * (lmax + 1);
  const int nchunk = (int)div_up(2L * at.max_nrad * (2 * lmax + 1), RADIAL_CHUNK);
  NAPMO_REQUIRE(nset >= 1 && (long)nset * nchunk <= 65535, "radial solves: too many sets");
  dim3 grid(at.M, lmax + 1, (unsigned)(nset * nchunk));
  k_radial<<<grid, RADIAL_CHUNK, 0, s>>>(at, rho_lm, green, L, Uy, Udt, nchunk, stride);
  NAPMO_HIP(hipGetLastError());
}

// ====================================================== Poisson: synthesis tables
// Synthesis order q: for m = 0..lmax, for l = m..lmax: C_lm (and S_lm when m > 0).
// Reference order index of (l, m, cs): l*l + (m ? 2m - 1 + cs : 0).
// Each coefficient carries sqrt(2l+1)/sqrt(4 pi) (evaluate.cpp:195-205) and the Racah
// factor sqrt(2 (l-m)!/(l+m)!) of moments.cpp:106-112, so that the kernel multiplies
// by (x + i y)^m times the PI_l^m(z) polynomial of the unit vector only.
__device__ inline void q_decode(int q, int lmax, int &l, int &m, int &cs) {
  int base = 0;
  for (m = 0; m <= lmax; ++m) {
    const int cnt = (lmax - m + 1) * (m ? 2 : 1);
    if (q < base + cnt) {
      const int r = q - base;
      if (m == 0) {
        l = r, cs = 0;
      } else {
        l = m + r / 2, cs = r % 2;
      }
      return;
    }
    base += cnt;
  }
  l = m = cs = 0;
}

__device__ inline double q_factor(int l, int m) {
  double f = sqrt(2.0 * l + 1.0) * INV_SQRT_4_PI;
  if (m > 0) {
    double r = M_SQRT2;
    for (int k = 1; k <= m; ++k) r /= sqrt((double)((l + k) * (l - k + 1)));
    f *= r;
  }
  return f;
}

void synth_order(int lmax, std::vector<int> &l, std::vector<int> &m, std::vector<int> &cs,
                 std::vector<double> &scale) {
  l.clear(), m.clear(), cs.clear(), scale.clear();
  for (int mm = 0; mm <= lmax; ++mm)
    for (int ll = mm; ll <= lmax; ++ll)
      for (int c = 0; c < (mm ? 2 : 1); ++c) {
        double f = std::sqrt(2.0 * ll + 1.0) * INV_SQRT_4_PI;
        if (mm > 0) {
          double r = M_SQRT2;
          for (int k = 1; k <= mm; ++k) r /= std::sqrt((double)((ll + k) * (ll - k + 1)));
          f *= r;
        }
        f *= pi_sigma(ll, mm);
        l.push_back(ll), m.push_back(mm), cs.push_back(c), scale.push_back(f);
      }
}

constexpr int SYNTH_TAB_J = 4;  // intervals per workgroup (the factors are formed once for them)

// Layout of the tables: coefficient c of (set, centre A, interval j, q) at
// T[set tset + (A (max_nrad - 1) + j) trow + q tq + c], amplitudes at
// amp[set aset + A arow + q aq]. Sets nvalid .. gridDim.z - 1 are written as zeros (the
// padding columns of the density-interleaved layout).
struct SynthTabLayout {
  long tset, trow, tq, aset, arow, aq;
  int nvalid;
};

__global__ void k_synth_tables(AtomTables at, const double *__restrict__ Uy,
                               const double *__restrict__ Udt, int lmax, int L,
                               int write_amps, double *__restrict__ T,
                               double *__restrict__ ampL, double *__restrict__ ampR,
                               long ustride, SynthTabLayout lay) {
  const int A = blockIdx.y, jb = blockIdx.x * SYNTH_TAB_J;
  // blockIdx.z = set: U + set ustride -> its tables
  const long set = blockIdx.z;
  const bool pad = set >= lay.nvalid;
  Uy += set * ustride, Udt += set * ustride, T += set * lay.tset;
  ampL += set * lay.aset, ampR += set * lay.aset;
  const int nr = at.nrad[A];
  if (jb >= nr - 1) return;
  const long roff = at.rad_off[A];
  // a centre with its own cut: its harmonics only, in its own synthesis order, in its own
  // rows (at.toff)
  const int la = at.lcut ? at.lcut[A] : lmax, La = (la + 1) * (la + 1);
  for (int q = threadIdx.x; q < La; q += blockDim.x) {
    int l, m, cs;
    q_decode(q, la, l, m, cs);
    const int ref = l * l + (m ? 2 * m - 1 + cs : 0);
    const double f = q_factor(l, m) * pi_sigma(l, m);
    for (int j = jb; j < min(jb + SYNTH_TAB_J, nr - 1); ++j) {
      double *t = at.toff ? T + at.toff[A] + ((long)j * La + q) * 4
                          : T + ((long)A * (at.max_nrad - 1) + j) * lay.trow + q * lay.tq;
      if (pad) {
        t[0] = t[1] = t[2] = t[3] = 0.0;
        if (j == 0 && write_amps) ampL[A * lay.arow + q * lay.aq] = ampR[A * lay.arow + q * lay.aq] = 0.0;
        continue;
      }
      const double y0 = Uy[(roff + j) * L + ref], y1 = Uy[(roff + j + 1) * L + ref];
      const double d0 = Udt[(roff + j) * L + ref], d1 = Udt[(roff + j + 1) * L + ref];
      const double zz = y1 - y0;
      t[0] = y0 * f;
      t[1] = d0 * f;
      t[2] = (3 * zz - 2 * d0 - d1) * f;
      t[3] = (-2 * zz + d0 + d1) * f;
      if (j == 0 && write_amps) {
        // PotentialExtrapolation::prepare (src/horton/extrapolation.cpp:156-159)
        const double r0 = at.r[roff], rn = at.r[roff + nr - 1];
        const double yn = Uy[(roff + nr - 1) * L + ref];
        ampL[A * lay.arow + q * lay.aq] = y0 / pow(r0, (double)l) * f;
        ampR[A * lay.arow + q * lay.aq] = yn * pow(rn, (double)(l + 1)) * f;
      }
    }
  }
}

long synth_table_size(const AtomTables &at, int lmax) {
  return (long)at.M * std::max(at.max_nrad - 1, 1) * (lmax + 1) * (lmax + 1) * 4;
}

void launch_synth_tables(const AtomTables &at, const double *Uy, const double *Udt, int lmax,
                         double *T, double *ampL, double *ampR, hipStream_t s, int write_amps,
                         int nset, long ustride) {
  const int L = (lmax + 1) * (lmax + 1);
  NAPMO_REQUIRE(nset >= 1 && nset <= 65535, "synthesis tables: too many sets");
  dim3 grid((unsigned)div_up(at.max_nrad - 1, SYNTH_TAB_J), at.M, nset);
  const SynthTabLayout lay{synth_table_size(at, lmax), (long)L * 4, 4, (long)at.M * L, L, 1, nset};
  k_synth_tables<<<grid, 256, 0, s>>>(at, Uy, Udt, lmax, L, write_amps, T, ampL, ampR, ustride, lay);
  NAPMO_HIP(hipGetLastError());
}

void launch_synth_tables_cols(const AtomTables &at, const double *Uy, const double *Udt, int lmax,
                              int nset, long ustride, int ndp, double *T, double *ampL,
                              double *ampR, hipStream_t s) {
  const int L = (lmax + 1) * (lmax + 1);
  NAPMO_REQUIRE(nset >= 1 && nset <= ndp && ndp % 16 == 0 && ndp <= 65535,
                "interleaved synthesis tables: 1 <= sets <= columns, columns a multiple of 16");
  dim3 grid((unsigned)div_up(at.max_nrad - 1, SYNTH_TAB_J), at.M, ndp);
  const SynthTabLayout lay{4, (long)L * ndp * 4, (long)ndp * 4, 1, (long)L * ndp, ndp, nset};
  k_synth_tables<<<grid, 256, 0, s>>>(at, Uy, Udt, lmax, L, 1, T, ampL, ampR, ustride, lay);
  NAPMO_HIP(hipGetLastError());
}

// ============================================== Poisson: the transposed operator
// z = V^T y for the discrete Becke-Poisson operator v = V rho (projection, radial Green
// solves, synthesis tables, synthesis over the (point, centre) pairs, sum over centres),
// each step transposed exactly, in the reverse order. Used for the derivative of
// E = 1/2 sum_p w bw rho v = 1/2 rho^T W V rho: dE/drho = 1/2 (W v + V^T (W rho)).

// synthesis^T: T[q][c] = sum over a bucket's pairs of y_p Y_q(p) u^c (spline rows) or
// y_p Y_q(p) d^l / d^-(l+1) (extrapolation amplitudes). Buckets hold from one pair to tens of
// thousands, so the work is cut along the slots and not along the buckets: workgroup g takes
// the slots g K .. g K + K - 1 and writes one row of partial sums per bucket that it meets, at
// row g + bucket (both grow along the slots, so the rows of one bucket are contiguous);
// k_synth_adjoint_sum adds them in that order. One workgroup per bucket, every thread
// redoing its own recurrence per pair, took 94 ms for 8 x 50 x 194 points at lmax 8 (a few
// long buckets in series); this form takes 0.10 ms there.
//
// A stage is 32 pairs. First the harmonics, pair by pair: 8 groups of 32 lanes share the m
// values, each running the forward recurrences in l, and write y Y_q to LDS as [q][pair]
// (row stride 33 doubles: neither the writes along pairs nor the reads along q conflict).
// Then the sums, q by q: lane = q, wave w adds its 8 pairs into 4 accumulators per q, u^c
// read as wave-uniform values. Bound by FP64 VALU: 4 FMA per (pair, q) and about one LDS
// read; the four waves are added in wave order at the end of a row, so a result does not
// depend on timing.
constexpr int ADJ_P = 32;      // pairs per stage
constexpr int ADJ_QB = 256;    // synthesis indices per workgroup (blockIdx.y), 64 NQ of them used

// first synthesis index of order m
__device__ inline int q_base(int m, int lmax) {
  return m == 0 ? 0 : (lmax + 1) + 2 * (m - 1) * (lmax + 1) - m * (m - 1);
}

__device__ inline double lane_value(double v, int lane) {
  union { double d; int i[2]; } a;
  a.d = v;
  a.i[0] = __builtin_amdgcn_readlane(a.i[0], lane);
  a.i[1] = __builtin_amdgcn_readlane(a.i[1], lane);
  return a.d;
}

template <int NQ>
__global__ void __launch_bounds__(256) k_synth_adjoint(AtomTables at, int lmax, int L,
                                                       const double *__restrict__ geo,
                                                       const int *__restrict__ list,
                                                       const int *__restrict__ wave_bucket, long nslots,
                                                       int kslots, const double *__restrict__ y,
                                                       double *__restrict__ part) {
  extern __shared__ double adj_lds[];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int q0 = blockIdx.y * ADJ_QB, nq = min(L - q0, 64 * NQ);
  double *beta = adj_lds;                             // [l (l + 1) / 2 + m]
  double *yt = adj_lds + (lmax + 1) * (lmax + 2) / 2;  // [nq][ADJ_P + 1]
  for (int e = tid; e < (lmax + 1) * (lmax + 2) / 2; e += 256) {
    int l = (int)((sqrt(8.0 * e + 1.0) - 1.0) * 0.5);
    while ((l + 1) * (l + 2) / 2 <= e) ++l;
    while (l * (l + 1) / 2 > e) --l;
    const int m = e - l * (l + 1) / 2;
    beta[e] = l >= m + 2 ? pi_beta(l, m) : 0.0;
  }
  __syncthreads();
  double acc[NQ][4];
#pragma unroll
  for (int g = 0; g < NQ; ++g)
#pragma unroll
    for (int c = 0; c < 4; ++c) acc[g][c] = 0.0;
  const long s0 = (long)blockIdx.x * kslots, s1 = min(nslots, s0 + kslots);
  const int pp = tid & (ADJ_P - 1), cls = tid / ADJ_P;  // pair of the stage, m group
  // pair data of the next stage, loaded one stage ahead
  const long nst = 2 * (s1 - s0);
  auto pair_at = [&](long st, int p) { return (s0 + (st >> 1)) * 64 + (st & 1) * ADJ_P + p; };
  auto geo_at = [&](long st, int p) { return (s0 + (st >> 1)) * 256 + (st & 1) * ADJ_P + p; };
  int pn = list[pair_at(0, pp)];
  double g0n = geo[geo_at(0, pp)], uxn = geo[geo_at(0, pp) + 64], uyn = geo[geo_at(0, pp) + 128],
         uzn = geo[geo_at(0, pp) + 192], upn = geo[geo_at(0, 8 * wave + (lane & 7))];
  double yn = pn >= 0 ? y[pn] : 0.0;
  for (long st = 0; st < nst; ++st) {
    const int gb = __builtin_amdgcn_readfirstlane(wave_bucket[s0 + (st >> 1)]);
    const int A = gb / (at.max_nrad + 1), loc = gb - A * (at.max_nrad + 1);
    const int nr = at.nrad[A];
    const int reg = loc == 0 ? 0 : (loc == nr ? 2 : 1);
    const double g0 = g0n, ux = uxn, uy = uyn, uz = uzn, yy = yn;
    const double u = reg == 1 ? upn : 0.0;
    if (st + 1 < nst) {
      const double *g = geo + geo_at(st + 1, pp);
      pn = list[pair_at(st + 1, pp)];
      g0n = g[0], uxn = g[64], uyn = g[128], uzn = g[192];
      upn = geo[geo_at(st + 1, 8 * wave + (lane & 7))];
    }
    const double base = reg == 0 ? g0 : (reg == 2 ? 1.0 / g0 : 1.0);
    double Am = yy, Bm = 0.0, pwm = reg == 2 ? base : 1.0;
    int mdone = 0;
    // m = cls, 15 - cls, 16 + cls, 31 - cls: about as many harmonics for every group
    for (int t = 0; t < 4; ++t) {
      const int m = (t & 1) ? 16 * (t >> 1) + 15 - cls : 16 * (t >> 1) + cls;
      if (m > lmax) continue;
      for (; mdone < m; ++mdone) {
        const double re = fma(ux, Am, -(uy * Bm));
        Bm = fma(ux, Bm, uy * Am);
        Am = re;
        pwm *= base;
      }
      const int step = m ? 2 : 1;
      int q = q_base(m, lmax) - q0;
      double pil = 1.0, pi1 = 1.0, pi2 = 0.0, pw = pwm;
      for (int l = m; l <= lmax; ++l) {
        if (l > m) {
          pil = l == m + 1 ? uz : fma(uz, pi1, -(beta[l * (l + 1) / 2 + m] * pi2));
          pi2 = pi1;
          pi1 = pil;
          pw *= base;
        }
        const double h = pil * pw;
        // a zero cotangent adds nothing, whatever its pair's geometry (padding slots)
        if (q >= 0 && q < nq) yt[q * (ADJ_P + 1) + pp] = yy != 0.0 ? Am * h : 0.0;
        if (m && q + 1 >= 0 && q + 1 < nq) yt[(q + 1) * (ADJ_P + 1) + pp] = yy != 0.0 ? Bm * h : 0.0;
        q += step;
      }
    }
    if (st + 1 < nst) yn = pn >= 0 ? y[pn] : 0.0;
    __syncthreads();
    const double u2 = u * u, u3 = u2 * u;
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const double v1 = lane_value(u, i), v2 = lane_value(u2, i), v3 = lane_value(u3, i);
#pragma unroll
      for (int g = 0; g < NQ; ++g) {
        const double h = yt[min(64 * g + lane, nq - 1) * (ADJ_P + 1) + 8 * wave + i];
        acc[g][0] += h;
        acc[g][1] = fma(h, v1, acc[g][1]);
        acc[g][2] = fma(h, v2, acc[g][2]);
        acc[g][3] = fma(h, v3, acc[g][3]);
      }
    }
    __syncthreads();
    if (st + 1 == nst || wave_bucket[s0 + ((st + 1) >> 1)] != gb) {
      // end of the bucket or of the slots: the four waves' sums, in wave order, in yt
#pragma unroll
      for (int g = 0; g < NQ; ++g)
        if (64 * g + lane < nq)
#pragma unroll
          for (int c = 0; c < 4; ++c) {
            yt[(wave * nq + 64 * g + lane) * 4 + c] = acc[g][c];
            acc[g][c] = 0.0;
          }
      __syncthreads();
      double *row = part + ((long)blockIdx.x + gb) * 4 * L + 4 * q0;
      for (int e = tid; e < 4 * nq; e += 256)
        row[e] = ((yt[e] + yt[4 * nq + e]) + yt[8 * nq + e]) + yt[12 * nq + e];
      __syncthreads();
    }
  }
}

// The partial rows of each bucket, in slot order, into the table and amplitude cotangents.
__global__ void __launch_bounds__(256) k_synth_adjoint_sum(AtomTables at, int L, int kslots,
                                                           const long *__restrict__ slot0,
                                                           const double *__restrict__ part,
                                                           double *__restrict__ Tt,
                                                           double *__restrict__ aLt,
                                                           double *__restrict__ aRt) {
  const int b = blockIdx.x, nb = at.max_nrad + 1;
  const int A = b / nb, loc = b % nb;
  const int nr = at.nrad[A];
  if (loc > nr) return;
  const int e = blockIdx.y * 256 + threadIdx.x;
  if (e >= 4 * L) return;
  const long s0 = slot0[b], s1 = slot0[b + 1];
  double sum = 0.0;
  if (s1 > s0) {
    long r = s0 / kslots + b;
    const long r1 = (s1 - 1) / kslots + b;
    for (; r + 7 <= r1; r += 8) {
      double v[8];
#pragma unroll
      for (int k = 0; k < 8; ++k) v[k] = part[(r + k) * 4 * L + e];
#pragma unroll
      for (int k = 0; k < 8; ++k) sum += v[k];
    }
    for (; r <= r1; ++r) sum += part[r * 4 * L + e];
  }
  if (loc == 0 || loc == nr) {
    if ((e & 3) == 0) (loc == 0 ? aLt : aRt)[(long)A * L + (e >> 2)] = sum;
  } else {
    Tt[(((long)A * (at.max_nrad - 1) + loc - 1) * L) * 4 + e] = sum;
  }
}

// Slots per workgroup: about 3,000 workgroups (12 waves per CU), from 2 to 64 slots each, so
// that short grids still fill the device and the partial rows stay few on long ones.
int synth_adjoint_slots(long nslots) { return (int)std::min(64L, std::max(2L, div_up(nslots, 3072))); }

long synth_adjoint_rows(const AtomTables &at, long nslots) {
  return div_up(nslots, synth_adjoint_slots(nslots)) + (long)at.M * (at.max_nrad + 1);
}

// synthesis tables^T: one workgroup per (radial node, centre), one thread per q; node i
// collects interval i (as its left end) and interval i - 1 (as its right end), and the
// extrapolation amplitudes at the first and last node.
__global__ void k_synth_tables_adjoint(AtomTables at, int lmax, int L, const double *__restrict__ Tt,
                                       const double *__restrict__ aLt, const double *__restrict__ aRt,
                                       double *__restrict__ Uyt, double *__restrict__ Udtt) {
  const int i = blockIdx.x, A = blockIdx.y;
  const int nr = at.nrad[A];
  if (i >= nr) return;
  const long roff = at.rad_off[A];
  for (int q = threadIdx.x; q < L; q += blockDim.x) {
    int l, m, cs;
    q_decode(q, lmax, l, m, cs);
    const int ref = l * l + (m ? 2 * m - 1 + cs : 0);
    const double f = q_factor(l, m) * pi_sigma(l, m);
    double gy = 0.0, gd = 0.0;
    if (i <= nr - 2) {
      const double *t = Tt + (((long)A * (at.max_nrad - 1) + i) * L + q) * 4;
      gy += f * (t[0] - 3 * t[2] + 2 * t[3]);
      gd += f * (t[1] - 2 * t[2] + t[3]);
    }
    if (i >= 1) {
      const double *t = Tt + (((long)A * (at.max_nrad - 1) + i - 1) * L + q) * 4;
      gy += f * (3 * t[2] - 2 * t[3]);
      gd += f * (t[3] - t[2]);
    }
    if (i == 0) gy += aLt[(long)A * L + q] * f / pow(at.r[roff], (double)l);
    if (i == nr - 1) gy += aRt[(long)A * L + q] * f * pow(at.r[roff + nr - 1], (double)(l + 1));
    Uyt[(roff + i) * L + ref] = gy;
    Udtt[(roff + i) * L + ref] = gd;
  }
}

// radial solves^T: rho_lm^T[A][j][lm] = sum_i Gy[i][j] Uy^T[A][i][lm] + Gd[i][j] Udt^T[A][i][lm].
__global__ void __launch_bounds__(256) k_radial_adjoint(AtomTables at, const double *__restrict__ green,
                                                        int L, const double *__restrict__ Uyt,
                                                        const double *__restrict__ Udtt,
                                                        double *__restrict__ rt) {
  const int A = blockIdx.z, lm = blockIdx.y;
  const int j = blockIdx.x * blockDim.x + threadIdx.x;
  const int nr = at.nrad[A];
  if (j >= nr) return;
  const int l = (int)sqrt((double)lm + 0.5);
  const double *G = green + at.green_off[A] + (long)l * 2 * nr * nr;
  const long roff = at.rad_off[A];
  double acc = 0.0;
  for (int i = 0; i < nr; ++i)
    acc += G[(long)i * nr + j] * Uyt[(roff + i) * L + lm] + G[(long)nr * nr + (long)i * nr + j] * Udtt[(roff + i) * L + lm];
  rt[(roff + j) * L + lm] = acc;
}

// projection^T: z_p = bw_p sum_lm Yhat[j][lm] rho_lm^T[A][i][lm] on atom A's own points
// (p = point_off[A] + i na + j).
__global__ void __launch_bounds__(256) k_project_adjoint(AtomTables at, const int *__restrict__ owner,
                                                         const double *__restrict__ bw,
                                                         const double *__restrict__ yhat, int L, long N,
                                                         const double *__restrict__ rt,
                                                         double *__restrict__ z) {
  const long p = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (p >= N) return;
  const int A = owner[p];
  const int na = at.nang[A];
  const long loc = p - at.point_off[A];
  const long i = loc / na, j = loc - i * na;
  const double *Y = yhat + at.yhat_off[A] + j * L;
  const double *r = rt + (at.rad_off[A] + i) * L;
  double acc = 0.0;
  for (int lm = 0; lm < L; ++lm) acc += Y[lm] * r[lm];
  z[p] = bw[p] * acc;
}

__global__ void k_half_sum(const double *__restrict__ a, const double *__restrict__ b, long N, long Npad,
                           double *__restrict__ out) {
  const long p = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (p < Npad) out[p] = p < N ? 0.5 * (a[p] + b[p]) : 0.0;
}

void launch_half_sum(const double *a, const double *b, long N, long Npad, double *out, hipStream_t st) {
  if (Npad <= 0) return;
  k_half_sum<<<div_up(Npad, 256), 256, 0, st>>>(a, b, N, Npad, out);
  NAPMO_HIP(hipGetLastError());
}

void launch_poisson_adjoint(const AtomTables &at, int lmax, const double *geo, const int *list,
                            const int *wave_bucket, long nslots, const long *slot0, const int *owner,
                            const double *bw, const double *yhat, const double *green, long N,
                            const double *y, double *part, double *Tt, double *aLt, double *aRt,
                            double *Uyt, double *Udtt, double *rt, double *z, hipStream_t s) {
  NAPMO_REQUIRE(lmax >= 0 && lmax <= MAX_LMAX, "lmax out of range for the transposed synthesis");
  const int L = (lmax + 1) * (lmax + 1);
  const int nb = at.M * (at.max_nrad + 1);
  const int ks = synth_adjoint_slots(nslots);
  if (nslots > 0) {
    const int nq = (int)div_up(std::min(L, ADJ_QB), 64);
    const dim3 grid((unsigned)div_up(nslots, ks), (unsigned)div_up(L, ADJ_QB));
    const size_t lds = sizeof(double) * ((lmax + 1) * (lmax + 2) / 2 + (size_t)std::min(L, ADJ_QB) * (ADJ_P + 1));
    auto kern = nq == 1 ? k_synth_adjoint<1> : nq == 2 ? k_synth_adjoint<2> : nq == 3 ? k_synth_adjoint<3> : k_synth_adjoint<4>;
    NAPMO_HIP(hipFuncSetAttribute((const void *)kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)max_lds_per_block()));
    kern<<<grid, 256, lds, s>>>(at, lmax, L, geo, list, wave_bucket, nslots, ks, y, part);
  }
  k_synth_adjoint_sum<<<dim3(nb, (unsigned)div_up(4 * L, 256)), 256, 0, s>>>(at, L, ks, slot0, part, Tt, aLt, aRt);
  k_synth_tables_adjoint<<<dim3(at.max_nrad, at.M), 256, 0, s>>>(at, lmax, L, Tt, aLt, aRt, Uyt, Udtt);
  k_radial_adjoint<<<dim3(div_up(at.max_nrad, 256), L, at.M), 256, 0, s>>>(at, green, L, Uyt, Udtt, rt);
  if (N > 0) k_project_adjoint<<<div_up(N, 256), 256, 0, s>>>(at, owner, bw, yhat, L, N, rt, z);
  NAPMO_HIP(hipGetLastError());
}

// ================================================================ Poisson: synthesis
// (kernel template in synth_kernel.hpp, instantiated per lmax in synth_inst_*.hip)
template <int LM>
static void synth_dispatch(int lmax, dim3 g, dim3 b, hipStream_t s, const AtomTables &at,
                           const double *x, const double *y, const double *z, long N,
                           const double *T, const double *aL, const double *aR, int acc,
                           int ext_mode, double *v) {
  if constexpr (LM > MAX_LMAX) {
    throw Error("lmax above the supported maximum " + std::to_string(MAX_LMAX));
  } else {
    if (lmax == LM)
      launch_synth_t<LM>(g, b, s, at, x, y, z, N, T, aL, aR, acc, ext_mode, v);
    else
      synth_dispatch<LM + 1>(lmax, g, b, s, at, x, y, z, N, T, aL, aR, acc, ext_mode, v);
  }
}
void launch_synth(const AtomTables &at, const double *x, const double *y, const double *z, long N,
                  const double *T, const double *ampL, const double *ampR, int lmax, int accumulate,
                  double *v, hipStream_t s, int ext_mode) {
  NAPMO_REQUIRE(lmax >= 0 && lmax <= MAX_LMAX, "lmax out of range for synthesis");
  if (N <= 0) return;
  synth_dispatch<0>(lmax, dim3(div_up(N, 256)), dim3(256), s, at, x, y, z, N, T, ampL, ampR,
                    accumulate, ext_mode, v);
  NAPMO_HIP(hipGetLastError());
}

// ----------------------------------------------------- bucketed synthesis support
__device__ inline int pair_bucket(const AtomTables &at, int A, double X, double Y, double Z) {
  const double dx = X - at.center[3 * A], dy = Y - at.center[3 * A + 1], dz = Z - at.center[3 * A + 2];
  const double d = sqrt(dx * dx + dy * dy + dz * dz);
  const int nr = at.nrad[A];
  int loc;
  if (d < at.first_x[A]) {
    loc = 0;
  } else if (d <= at.last_x[A]) {
    const int kind = at.rkind[A];
    const double t = kind == 0 ? -(acos((d - at.rp0[A]) / (d + at.rp0[A])) / at.rp1[A]) + nr
                               : (kind == 1 ? pow(d / at.rp0[A], 1.0 / at.rp1[A]) - 1 : d);
    int j = (int)floor(t);
    if (j >= nr - 1) j = nr - 2;
    if (j < 0) j = 0;
    loc = 1 + j;
  } else {
    loc = nr;
  }
  return A * (at.max_nrad + 1) + loc;
}

// Per workgroup (256 points, one centre): LDS histogram of the centre's local buckets,
// then one global atomic per non-empty bin (pair_bucket is A * (max_nrad + 1) + loc).
constexpr int PAIR_BINS = 1024;  // local buckets per centre (max_nrad + 1 <= PAIR_BINS)

__global__ void __launch_bounds__(256) k_pair_count(AtomTables at, const double *__restrict__ x,
                                                    const double *__restrict__ y,
                                                    const double *__restrict__ z, long N,
                                                    int *__restrict__ count) {
  __shared__ int hist[PAIR_BINS];
  const int A = blockIdx.y, nb = at.max_nrad + 1;
  for (int b = threadIdx.x; b < nb; b += blockDim.x) hist[b] = 0;
  __syncthreads();
  const long p = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (p < N) atomicAdd(&hist[pair_bucket(at, A, x[p], y[p], z[p]) - A * nb], 1);
  __syncthreads();
  for (int b = threadIdx.x; b < nb; b += blockDim.x)
    if (hist[b]) atomicAdd(&count[A * nb + b], hist[b]);
}

__global__ void __launch_bounds__(256) k_pair_fill(AtomTables at, const double *__restrict__ x,
                                                   const double *__restrict__ y,
                                                   const double *__restrict__ z, long N,
                                                   const long *__restrict__ off,
                                                   int *__restrict__ cursor,
                                                   int *__restrict__ list) {
  __shared__ int hist[PAIR_BINS], base[PAIR_BINS];
  const int A = blockIdx.y, nb = at.max_nrad + 1;
  for (int b = threadIdx.x; b < nb; b += blockDim.x) hist[b] = 0;
  __syncthreads();
  const long p = (long)blockIdx.x * blockDim.x + threadIdx.x;
  int loc = -1, rank = 0;
  if (p < N) {
    loc = pair_bucket(at, A, x[p], y[p], z[p]) - A * nb;
    rank = atomicAdd(&hist[loc], 1);
  }
  __syncthreads();
  for (int b = threadIdx.x; b < nb; b += blockDim.x)
    if (hist[b]) base[b] = atomicAdd(&cursor[A * nb + b], hist[b]);
  __syncthreads();
  if (loc >= 0) list[off[A * nb + loc] + base[loc] + rank] = (int)p;
}

void launch_pair_count(const AtomTables &at, const double *x, const double *y, const double *z,
                       long N, int *count, hipStream_t s) {
  NAPMO_REQUIRE(at.max_nrad + 1 <= PAIR_BINS, "too many radial points for the synthesis buckets");
  k_pair_count<<<dim3(div_up(N, 256), at.M), 256, 0, s>>>(at, x, y, z, N, count);
  NAPMO_HIP(hipGetLastError());
}

void launch_pair_fill(const AtomTables &at, const double *x, const double *y, const double *z,
                      long N, const long *off, int *cursor, int *list, hipStream_t s) {
  NAPMO_REQUIRE(at.max_nrad + 1 <= PAIR_BINS, "too many radial points for the synthesis buckets");
  k_pair_fill<<<dim3(div_up(N, 256), at.M), 256, 0, s>>>(at, x, y, z, N, off, cursor, list);
  NAPMO_HIP(hipGetLastError());
}

// One wavefront per 64-pair slot: the geometry each synthesis launch would otherwise form
// per pair (gathers of the point, distance, unit vector and the inverse radial transform),
// formed once per grid. Slots past a bucket's pairs (list entry -1) get a fixed finite
// geometry (unit distance along x, offset 0 in the interval) whose results are never used.
__global__ void __launch_bounds__(64) k_pair_geometry(AtomTables at, const double *__restrict__ px,
                                                      const double *__restrict__ py,
                                                      const double *__restrict__ pz,
                                                      const int *__restrict__ list,
                                                      const int *__restrict__ wave_bucket,
                                                      double *__restrict__ geo) {
  const long w = blockIdx.x;
  const int lane = threadIdx.x;
  const int gb = wave_bucket[w];
  const int A = gb / (at.max_nrad + 1), loc = gb - A * (at.max_nrad + 1);
  const int nr = at.nrad[A];
  const int reg = (loc == 0) ? 0 : (loc == nr ? 2 : 1);
  const int j = (reg == 1) ? loc - 1 : 0;
  const int p = list[w * 64 + lane];
  double *g = geo + w * 256 + lane;
  if (p < 0) {
    g[0] = (reg == 1) ? 0.0 : 1.0;
    g[64] = 1.0;
    g[128] = 0.0;
    g[192] = 0.0;
    return;
  }
  const double cx = at.center[3 * A], cy = at.center[3 * A + 1], cz = at.center[3 * A + 2];
  const double dx = px[p] - cx, dy = py[p] - cy, dz = pz[p] - cz;
  const double d = sqrt(dx * dx + dy * dy + dz * dz);
  const double inv_d = 1.0 / d;
  g[0] = (reg == 1) ? rtf_inv(at.rkind[A], at.rp0[A], at.rp1[A], nr, d) - j : d;
  g[64] = dx * inv_d;
  g[128] = dy * inv_d;
  g[192] = dz * inv_d;
}

void launch_pair_geometry(const AtomTables &at, const double *x, const double *y,
                          const double *z, const int *list, const int *wave_bucket, long nwaves,
                          double *geo, hipStream_t s) {
  if (nwaves <= 0) return;
  k_pair_geometry<<<dim3((unsigned)nwaves), 64, 0, s>>>(at, x, y, z, list, wave_bucket, geo);
  NAPMO_HIP(hipGetLastError());
}

template <int LM>
static void synth2_dispatch(int lmax, int np, hipStream_t s, const AtomTables &at,
                            const double *geo, long N,
                            const int *list, const int *wb, long nw, const double *T,
                            const double *aL, const double *aR, double *contrib) {
  if constexpr (LM > MAX_LMAX) {
    throw Error("lmax above the supported maximum " + std::to_string(MAX_LMAX));
  } else {
    if (lmax == LM)
      launch_synth2_t<LM>(np, s, at, geo, N, list, wb, nw, T, aL, aR, contrib);
    else
      synth2_dispatch<LM + 1>(lmax, np, s, at, geo, N, list, wb, nw, T, aL, aR, contrib);
  }
}

void launch_synth2(const AtomTables &at, const double *geo, long N,
                   const int *list, const int *wave_bucket, long nwaves, const double *T,
                   const double *ampL, const double *ampR, int lmax, double *contrib,
                   hipStream_t s, int np) {
  NAPMO_REQUIRE(lmax >= 0 && lmax <= MAX_LMAX, "lmax out of range for synthesis");
  NAPMO_REQUIRE(np == 1 || np == 2, "synthesis: 1 or 2 pairs per lane");
  NAPMO_REQUIRE(nwaves % (SYNTH_PAD / 64) == 0, "synthesis: pair lists must be padded to 128");
  if (nwaves <= 0) return;
  synth2_dispatch<0>(lmax, np, s, at, geo, N, list, wave_bucket, nwaves, T, ampL, ampR, contrib);
  NAPMO_HIP(hipGetLastError());
}

__global__ void k_contrib_reduce(const double *__restrict__ contrib, int M, long N, int accumulate,
                                 double scale, double *__restrict__ v) {
  const long p = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (p >= N) return;
  double s = 0.0;
  for (int A = 0; A < M; ++A) s += contrib[(long)A * N + p];
  v[p] = accumulate ? v[p] + scale * s : scale * s;
}

// v = sum_A contrib[A] and, in the same pass, sv = v wbw (zero for N <= p < Npad).
__global__ void k_contrib_reduce_scale(const double *__restrict__ contrib, int M, long N, long Npad,
                                       const double *__restrict__ wbw, double *__restrict__ v,
                                       double *__restrict__ sv) {
  const long p = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (p >= Npad) return;
  if (p >= N) {
    sv[p] = 0.0;
    return;
  }
  double s = 0.0;
  for (int A = 0; A < M; ++A) s += contrib[(long)A * N + p];
  const double vp = 1.0 * s;
  v[p] = vp;
  sv[p] = vp * wbw[p];
}

void launch_contrib_reduce(const double *contrib, int M, long N, int accumulate, double *v,
                           hipStream_t s, double scale) {
  if (N <= 0) return;
  k_contrib_reduce<<<div_up(N, 256), 256, 0, s>>>(contrib, M, N, accumulate, scale, v);
  NAPMO_HIP(hipGetLastError());
}

// One thread per (point, density) of a tile, 16 densities of a point adjacent: the sum over
// centres in index order, as k_contrib_reduce.
__global__ void k_contrib_reduce_tile(const double *__restrict__ tile, int M, long N, int nvalid,
                                      double scale, double *__restrict__ out, long ostride) {
  const long e = (long)blockIdx.x * blockDim.x + threadIdx.x;
  const long p = e >> 4;
  const int k = (int)(e & 15);
  if (p >= N || k >= nvalid) return;
  double s = 0.0;
  for (int A = 0; A < M; ++A) s += tile[((long)A * N + p) * 16 + k];
  out[k * ostride + p] = scale * s;
}

void launch_contrib_reduce_tile(const double *tile, int M, long N, int nvalid, double scale,
                                double *out, long ostride, hipStream_t s) {
  if (N <= 0 || nvalid <= 0) return;
  NAPMO_REQUIRE(nvalid <= 16, "tile reduction: at most 16 densities");
  k_contrib_reduce_tile<<<div_up(N * 16, 256), 256, 0, s>>>(tile, M, N, nvalid, scale, out, ostride);
  NAPMO_HIP(hipGetLastError());
}

__global__ void k_contrib_reduce_scale_group(const ScaleMember *__restrict__ mem, int nmem,
                                             const double *__restrict__ contrib,
                                             const long *__restrict__ cbase,
                                             const double *__restrict__ wbw,
                                             double *__restrict__ v) {
  const long g = blockIdx.x;
  const ScaleMember &m = mem[group_member(mem, nmem, g)];
  const long q = (g - m.block0) * blockDim.x + threadIdx.x;  // the member's own point index
  if (q >= m.Npad) return;
  if (q >= m.N) {
    m.s[q] = 0.0;
    return;
  }
  const long p = m.p0 + q;
  double s = 0.0;
  for (int A = m.A0; A < m.A1; ++A) s += contrib[cbase[A] + p];
  const double vp = 1.0 * s;
  v[p] = vp;
  m.s[q] = vp * wbw[p];
}

void launch_contrib_reduce_scale_group(const ScaleMember *d_mem, int nmem, long nblocks,
                                       const double *contrib, const long *cbase,
                                       const double *wbw, double *v, hipStream_t st) {
  if (nmem <= 0 || nblocks <= 0) return;
  k_contrib_reduce_scale_group<<<dim3((unsigned)nblocks), 256, 0, st>>>(d_mem, nmem, contrib, cbase,
                                                                        wbw, v);
  NAPMO_HIP(hipGetLastError());
}

__global__ void k_apmo_reduce_group(const ScaleMember *__restrict__ mem, int nmem,
                                    const SpeciesSum *__restrict__ sp,
                                    const double *__restrict__ contrib, long Nu,
                                    const double *__restrict__ wbw, double *__restrict__ vown,
                                    double *__restrict__ veff) {
  const long g = blockIdx.x;
  const int ms = group_member(mem, nmem, g);
  const ScaleMember &m = mem[ms];
  const long q = (g - m.block0) * blockDim.x + threadIdx.x;
  if (q >= m.Npad) return;
  if (q >= m.N) {
    m.s[q] = 0.0;
    return;
  }
  const long p = m.p0 + q;
  double own = 0.0, vc = 0.0;
  bool first = true;
  for (int t = 0; t < nmem; ++t) {
    double s = 0.0;
    for (int A = sp[t].A0; A < sp[t].A1; ++A) s += contrib[(long)A * Nu + p];
    if (t == ms) {
      own = 1.0 * s;
    } else {
      vc = first ? sp[t].q * s : vc + sp[t].q * s;
      first = false;
    }
  }
  const double qs = sp[ms].q;
  const double ve = first ? qs * qs * own : qs * qs * own + qs * vc;
  vown[p] = own;
  veff[p] = ve;
  m.s[q] = ve * wbw[p];
}

void launch_apmo_reduce_group(const ScaleMember *d_mem, int nmem, long nblocks,
                              const SpeciesSum *sp, const double *contrib, long Nu,
                              const double *wbw, double *vown, double *veff, hipStream_t st) {
  if (nmem <= 0 || nblocks <= 0) return;
  k_apmo_reduce_group<<<dim3((unsigned)nblocks), 256, 0, st>>>(d_mem, nmem, sp, contrib, Nu, wbw,
                                                               vown, veff);
  NAPMO_HIP(hipGetLastError());
}

__global__ void k_apmo_energy_group(const ApmoEnergyMember *__restrict__ mem, int ns) {
  const int s = threadIdx.x;
  if (s >= ns) return;
  const ApmoEnergyMember &e = mem[s];
  e.E[2] = e.q2 * e.E2[1];
  e.E[3] = e.E[1] - e.E[2];
}

void launch_apmo_energy_group(const ApmoEnergyMember *d_mem, int ns, hipStream_t st) {
  NAPMO_REQUIRE(ns >= 1 && ns <= 256, "APMO energies: 1 to 256 species");
  k_apmo_energy_group<<<1, 256, 0, st>>>(d_mem, ns);
  NAPMO_HIP(hipGetLastError());
}

void launch_contrib_reduce_scale(const double *contrib, int M, long N, long Npad, const double *wbw,
                                 double *v, double *sv, hipStream_t s) {
  if (Npad <= 0) return;
  k_contrib_reduce_scale<<<div_up(Npad, 256), 256, 0, s>>>(contrib, M, N, Npad, wbw, v, sv);
  NAPMO_HIP(hipGetLastError());
}

// V[p] = sum_A q_A / |p - R_A|, charges in list order (napmo/wavefunction/nnuclear.py:15-37).
__global__ void k_nuclear(const double *__restrict__ x, const double *__restrict__ y,
                          const double *__restrict__ z, long N, const double *__restrict__ q,
                          const double *__restrict__ o, int nq, double *__restrict__ V) {
  const long p = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (p >= N) return;
  double s = 0.0;
  for (int a = 0; a < nq; ++a) {
    const double dx = o[3 * a] - x[p], dy = o[3 * a + 1] - y[p], dz = o[3 * a + 2] - z[p];
    s += q[a] / sqrt(dx * dx + dy * dy + dz * dz);
  }
  V[p] = s;
}

void launch_nuclear(const double *x, const double *y, const double *z, long N, const double *q,
                    const double *o, int nq, double *V, hipStream_t s) {
  if (N <= 0) return;
  k_nuclear<<<div_up(N, 256), 256, 0, s>>>(x, y, z, N, q, o, nq, V);
  NAPMO_HIP(hipGetLastError());
}

// Exchange-potential helpers (napmo/wavefunction/psi_numeric.py:186-215).
// chi[l][p] = sum_k D[k][l] psi[k][p] (psi, chi [ndim x N] function-major).
__global__ void k_exchange_chi(const double *__restrict__ psi, const double *__restrict__ D,
                               int ndim, long N, double *__restrict__ chi) {
  const long p = (long)blockIdx.x * blockDim.x + threadIdx.x;
  const int l = blockIdx.y;
  if (p >= N) return;
  double s = 0.0;
  for (int k = 0; k < ndim; ++k) s += D[(long)k * ndim + l] * psi[(long)k * N + p];
  chi[(long)l * N + p] = s;
}

// Orbital pairs (s, v), v <= s, in order: pair t = s (s + 1) / 2 + v.
__host__ __device__ inline long pair_base(int s) { return (long)s * (s + 1) / 2; }

// dens[k] = psi_s psi_v of pair t0 + k (a launch per pair cost 2.6 us and its gap: 21 pairs of
// 121,000 points 54 -> 10 us).
__global__ void k_exchange_dens(const double *__restrict__ psi, long t0, long N, double *__restrict__ dens) {
  const long p = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (p >= N) return;
  const long t = t0 + blockIdx.y;
  int s = (int)((sqrt(8.0 * (double)t + 1.0) - 1.0) * 0.5);
  while (pair_base(s) > t) --s;
  while (pair_base(s + 1) <= t) ++s;
  dens[(long)blockIdx.y * N + p] = psi[(long)s * N + p] * psi[(t - pair_base(s)) * N + p];
}

// K[r] += sum over the pairs t0 .. t0 + cnt - 1 that hold r of aux chi[partner], in pair order
// (aux = V[psi_s psi_v]); the first batch writes K. A workgroup row per orbital keeps its K in a
// register: an aux row is read twice and K once a batch, where a launch per pair read and wrote
// two rows of K each time (21 pairs of 121,000 points 92 -> 11 us).
__global__ void k_exchange_acc(const double *__restrict__ aux, const double *__restrict__ chi, int ndim,
                               long t0, int cnt, long N, double *__restrict__ K) {
  const long p = (long)blockIdx.x * blockDim.x + threadIdx.x;
  const int r = blockIdx.y;
  if (p >= N) return;
  const long rb = pair_base(r), t1 = t0 + cnt;
  const int v0 = (int)max(0L, t0 - rb), v1 = (int)min((long)r + 1, t1 - rb);
  double acc = t0 == 0 ? 0.0 : K[(long)r * N + p];
#pragma unroll 4
  for (int v = v0; v < v1; ++v) acc += aux[(rb + v - t0) * N + p] * chi[(long)v * N + p];
  int s0 = r + 1;
  while (s0 < ndim && pair_base(s0) + r < t0) ++s0;
#pragma unroll 4
  for (int s = s0; s < ndim; ++s) {
    const long t = pair_base(s) + r;
    if (t >= t1) break;
    acc += aux[(t - t0) * N + p] * chi[(long)s * N + p];
  }
  K[(long)r * N + p] = acc;
}

void launch_exchange_chi(const double *psi, const double *D, int ndim, long N, double *chi,
                         hipStream_t st) {
  if (N <= 0 || ndim <= 0) return;
  k_exchange_chi<<<dim3((unsigned)div_up(N, 256), ndim), 256, 0, st>>>(psi, D, ndim, N, chi);
  NAPMO_HIP(hipGetLastError());
}
void launch_exchange_dens(const double *psi, long t0, int cnt, long N, double *dens, hipStream_t st) {
  if (N <= 0 || cnt <= 0) return;
  k_exchange_dens<<<dim3((unsigned)div_up(N, 256), cnt), 256, 0, st>>>(psi, t0, N, dens);
  NAPMO_HIP(hipGetLastError());
}
void launch_exchange_acc(const double *aux, const double *chi, int ndim, long t0, int cnt, long N,
                         double *K, hipStream_t st) {
  if (N <= 0 || ndim <= 0) return;
  k_exchange_acc<<<dim3((unsigned)div_up(N, 256), ndim), 256, 0, st>>>(aux, chi, ndim, t0, cnt, N, K);
  NAPMO_HIP(hipGetLastError());
}

// v[p] = a x[p] + b y[p]
__global__ void k_axpby(double a, const double *__restrict__ x, double b,
                        const double *__restrict__ y, long N, double *__restrict__ v) {
  const long p = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (p < N) v[p] = a * x[p] + b * y[p];
}

void launch_axpby(double a, const double *x, double b, const double *y, long N, double *v,
                  hipStream_t s) {
  if (N <= 0) return;
  k_axpby<<<div_up(N, 256), 256, 0, s>>>(a, x, b, y, N, v);
  NAPMO_HIP(hipGetLastError());
}

// ============================================ FP64 MFMA layout; density partial sums
// v_mfma_f64_16x16x4f64 operand layout (lane i of 64), as measured on gfx950:
//   A[16 x 4]:  lane i holds A[i % 16][i / 16]
//   B[4 x 16]:  lane i holds B[i / 16][i % 16]
//   D[16 x 16]: lane i holds D[(i / 16) + 4 r][i % 16] in accumulator element r = 0..3

__global__ void k_rho_reduce(const double *__restrict__ partial, int nt, long Npad, long N,
                             double scale, double *__restrict__ rho) {
  const long p = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (p >= N) return;
  double s = 0.0;
  for (int t = 0; t < nt; ++t) s += partial[(long)t * Npad + p];
  rho[p] = scale * s;
}

__global__ void k_rho_reduce_group(const RhoReduceMember *__restrict__ mem, int nmem) {
  const long g = blockIdx.x;
  const RhoReduceMember &r = mem[group_member(mem, nmem, g)];
  const long p = (g - r.block0) * blockDim.x + threadIdx.x;
  if (p >= r.N) return;
  double s = 0.0;
  for (int t = 0; t < r.ntile; ++t) s += r.partial[(long)t * r.Npad + p];
  r.rho[p] = 1.0 * s;
}

void launch_rho_reduce_group(const RhoReduceMember *d_mem, int nmem, long nblocks, hipStream_t st) {
  if (nmem <= 0 || nblocks <= 0) return;
  k_rho_reduce_group<<<dim3((unsigned)nblocks), 256, 0, st>>>(d_mem, nmem);
  NAPMO_HIP(hipGetLastError());
}

void launch_rho_reduce(const double *partial, int ntile, long Npad, long N, double *rho,
                       hipStream_t s, double scale) {
  if (N <= 0) return;
  k_rho_reduce<<<div_up(N, 256), 256, 0, s>>>(partial, ntile, Npad, N, scale, rho);
  NAPMO_HIP(hipGetLastError());
}

__global__ void k_scale3(const double *__restrict__ a, const double *__restrict__ b,
                         const double *__restrict__ c, long N, long Npad, double *__restrict__ out) {
  const long p = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (p >= Npad) return;
  out[p] = (p < N) ? (c ? a[p] * b[p] * c[p] : a[p] * b[p]) : 0.0;
}

void launch_scale3(const double *a, const double *b, const double *c, long N, long Npad, double *s,
                   hipStream_t st) {
  k_scale3<<<div_up(Npad, 256), 256, 0, st>>>(a, b, c, N, Npad, s);
  NAPMO_HIP(hipGetLastError());
}

// ============================================================ FP64 energy traces
// Two passes with a fixed reduction order (deterministic): per-block partial sums of
// P o F and w bw rho v, then one block adds the partials.
constexpr int TRACE_BLOCKS = 512;

// block g of nb blocks (256 threads)
__device__ __forceinline__ void traces_partial_body(const double *__restrict__ P,
                                                    const double *__restrict__ F, long nn,
                                                    const double *__restrict__ wbw,
                                                    const double *__restrict__ rho,
                                                    const double *__restrict__ v, long N,
                                                    double *__restrict__ part, int g, int nb) {
  __shared__ double sa[256], sb[256];
  const int tid = threadIdx.x;
  const long stride = (long)nb * 256;
  double a = 0.0, b = 0.0;
  if (P && F)
    for (long e = (long)g * 256 + tid; e < nn; e += stride) a += P[e] * F[e];
  if (wbw && rho && v)
    for (long p = (long)g * 256 + tid; p < N; p += stride) b += wbw[p] * rho[p] * v[p];
  sa[tid] = a;
  sb[tid] = b;
  __syncthreads();
  for (int w = 128; w > 0; w >>= 1) {
    if (tid < w) sa[tid] += sa[tid + w], sb[tid] += sb[tid + w];
    __syncthreads();
  }
  if (tid == 0) part[g] = sa[0], part[nb + g] = sb[0];
}

__global__ void __launch_bounds__(256) k_traces_partial(const double *__restrict__ P,
                                                        const double *__restrict__ F, long nn,
                                                        const double *__restrict__ wbw,
                                                        const double *__restrict__ rho,
                                                        const double *__restrict__ v, long N,
                                                        double *__restrict__ part) {
  traces_partial_body(P, F, nn, wbw, rho, v, N, part, blockIdx.x, gridDim.x);
}

__device__ __forceinline__ void traces_final_body(const double *__restrict__ part, int nb,
                                                  double *__restrict__ E) {
  __shared__ double sa[512], sb[512];
  const int tid = threadIdx.x;
  sa[tid] = tid < nb ? part[tid] : 0.0;
  sb[tid] = tid < nb ? part[nb + tid] : 0.0;
  __syncthreads();
  for (int w = 256; w > 0; w >>= 1) {
    if (tid < w) sa[tid] += sa[tid + w], sb[tid] += sb[tid + w];
    __syncthreads();
  }
  if (tid == 0) E[0] = 0.5 * sa[0], E[1] = 0.5 * sb[0];
}

__global__ void __launch_bounds__(512) k_traces_final(const double *__restrict__ part, int nb,
                                                      double *__restrict__ E) {
  traces_final_body(part, nb, E);
}

// grouped: member = blockIdx.y, TRACE_BLOCKS partial blocks each (the same sums as one plan)
__global__ void __launch_bounds__(256) k_traces_partial_group(const TraceMember *__restrict__ mem) {
  const TraceMember &t = mem[blockIdx.y];
  traces_partial_body(t.P, t.F, t.nn, t.wbw, t.rho, t.v, t.N, t.work, blockIdx.x, gridDim.x);
}

__global__ void __launch_bounds__(512) k_traces_final_group(const TraceMember *__restrict__ mem,
                                                            int nb) {
  const TraceMember &t = mem[blockIdx.x];
  traces_final_body(t.work, nb, t.E);
}

void launch_traces(const double *P, const double *F, int n, const double *wbw, const double *rho,
                   const double *v, long N, double *E, double *work, hipStream_t st) {
  k_traces_partial<<<TRACE_BLOCKS, 256, 0, st>>>(P, F, (long)n * n, wbw, rho, v, N, work);
  k_traces_final<<<1, 512, 0, st>>>(work, TRACE_BLOCKS, E);
  NAPMO_HIP(hipGetLastError());
}

void launch_traces_group(const TraceMember *d_mem, int nmem, hipStream_t st) {
  if (nmem <= 0) return;
  NAPMO_REQUIRE(nmem <= 65535, "grouped traces: too many members");
  k_traces_partial_group<<<dim3(TRACE_BLOCKS, nmem), 256, 0, st>>>(d_mem);
  k_traces_final_group<<<dim3(nmem), 512, 0, st>>>(d_mem, TRACE_BLOCKS);
  NAPMO_HIP(hipGetLastError());
}

}  // namespace napmo
