// Becke-Dickson orbital correction on the GPU (napmo/wavefunction/ndpsi.py:15-89 and the
// per-orbital steps of napmo/wavefunction/psi_optimization.py:175-203).
//
// Per orbital o, atom A and angular momentum l the correction solves, on A's radial grid,
//   u'' + (2/r) u' + a u = c mu_lm,  a = c (l(l+1)/r^2 + Vsph - oi - doi),  c = -2/m_inv,
// with u(r_0) = u(r_max) = 0, for the 2l+1 projected sources mu_lm of (phi doi - ri) bw.
// a depends on the orbital, so unlike the Poisson solve the matrix cannot be factored once
// per geometry: one wavefront per (A, l, o) assembles the Hermite finite-element matrix
// from per-grid tables and eliminates it as a band matrix with partial pivoting together
// with the 2l+1 right-hand sides, one lane per column of either.
#include "common.hpp"
#include "kernels.hpp"

namespace napmo {

namespace {

// out[o][p] = a[o][p] s[o] - b[o][p]
__global__ void k_scaled_diff(const double *__restrict__ a, const double *__restrict__ s,
                              const double *__restrict__ b, long N, double *__restrict__ out) {
  const long p = (long)blockIdx.x * blockDim.x + threadIdx.x;
  const int o = blockIdx.y;
  if (p < N) out[(long)o * N + p] = a[(long)o * N + p] * s[o] - b[(long)o * N + p];
}

// One block per (shell i, atom A, orbital o): sum_j (f bw) w / sum_j w.
__global__ void __launch_bounds__(64) k_shell_average(AtomTables at, const double *__restrict__ V,
                                                      long N, const double *__restrict__ w,
                                                      const double *__restrict__ bw,
                                                      long nrad_total, double *__restrict__ Vsph) {
  const int i = blockIdx.x, A = blockIdx.y, o = blockIdx.z;
  if (i >= at.nrad[A]) return;
  const int na = at.nang[A];
  const long p0 = at.point_off[A] + (long)i * na;
  const double *f = V + (long)o * N;
  double num = 0.0, den = 0.0;
  for (int j = threadIdx.x; j < na; j += 64) {
    const long p = p0 + j;
    num += (f[p] * bw[p]) * w[p];
    den += w[p];
  }
  for (int k = 32; k > 0; k >>= 1) {
    num += __shfl_xor(num, k);
    den += __shfl_xor(den, k);
  }
  if (threadIdx.x == 0) Vsph[(long)o * nrad_total + at.rad_off[A] + i] = num / den;
}

// A double of lane `src` (the same for the whole wave) in every lane.
__device__ __forceinline__ double lane_value(double v, int src) {
  const unsigned long long b = __builtin_bit_cast(unsigned long long, v);
  const unsigned lo = (unsigned)__builtin_amdgcn_readlane((int)(unsigned)b, src);
  const unsigned hi = (unsigned)__builtin_amdgcn_readlane((int)(unsigned)(b >> 32), src);
  return __builtin_bit_cast(double, ((unsigned long long)hi << 32) | lo);
}

// Columns of one pass: 8 lanes of the wave hold the matrix and one the coefficient a.
constexpr int HELM_MAX_COLS = 55;

// One wave solves one (atom, l, orbital) system of nfn = 2 nrad unknowns. Nothing here is
// bound by bandwidth or rate: it is a chain of nfn elimination and nfn substitution steps, so
// what counts is the latency of a step. LDS holds the augmented matrix, a row of P doubles
// per unknown: 8 slots of band (columns row - 3 .. row + 3), then up to mc right-hand sides.
// The elimination keeps its window, rows k .. k + 3, in four registers per lane: matrix column
// c in lane c % 8, right-hand side q in lane 8 + q. One instruction then updates the band and
// all right-hand sides, so the forward substitution costs nothing of its own, no multiplier
// or interchange is stored, and a step reads LDS only for row k + 5, ahead of its use. The
// pivot column reaches all lanes by readlane; the three multipliers and 1 / pivot are one
// division in four lanes. Row k of U replaces the band of row k: slots 0 .. 6 are columns
// k .. k + 6, slot 7 is 1 / pivot, with which the back substitution divides in three FMAs
// (quotient, remainder, correction: the rounding of a division).
// 100 radial points, 2 atoms, lmax 8: 356 -> 101 us; 50 points, 16 atoms, lmax 12, 40
// orbitals: 1.0 -> 0.40 ms (before: the band in LDS, two barriers and three LDS round trips
// per step, then up to three passes of columns).
__global__ void __launch_bounds__(64) k_helmholtz_radial(
    AtomTables at, HelmholtzTables ht, int L, long nrad_total, const double *__restrict__ Vsph,
    const double *__restrict__ oi, const double *__restrict__ doi, double mass_inv,
    const double *__restrict__ mu, int mc, double *__restrict__ Uy, double *__restrict__ Udt,
    int *__restrict__ status) {
  extern __shared__ double sm[];
  const int A = blockIdx.x, l = blockIdx.y, o = blockIdx.z;
  const int lane = threadIdx.x;
  const int nr = at.nrad[A], nfn = 2 * nr, nm = 2 * l + 1;
  const int P = 8 + mc;
  double *an = sm + (nfn + 5) * P;  // [nfn + 2] a at even, its slope at odd indices, zeros
  double *sinv = an + nfn + 2;      // [nr] 1 / pivots of the spline system
  double *supm = sinv + nr;         // [nr] its eliminated super-diagonal
  const long r0 = at.rad_off[A];
  const double c = -2.0 / mass_inv;
  const double e_o = oi[o], d_o = doi[o];
  const double *rr = at.r + r0, *j1 = ht.j1 + r0, *j2 = ht.j2 + r0;
  const double *C0 = ht.c0 + ht.c0_off[A], *OA = ht.oa + ht.oa_off[A];
  const double *O2 = ht.o2 + ht.o2_off[A];
  const long ubase = ((long)o * nrad_total + r0) * L + l * l;

  for (int m0 = 0; m0 < nm; m0 += mc) {
    const int cnt = min(mc, nm - m0);
    // The band slots hold the right-hand-side integrals first (0 .. 5) and the node's j1, j2
    // (6, 7); the columns hold mu at even rows. a = c (l(l+1)/r^2 + Vsph - oi - doi).
    {
      const int s = lane & 7, stride = s < 6 ? 6 : 1, half = s < 6 ? 0 : 1;
      const double *src = s < 6 ? O2 + s : s == 6 ? j1 : j2;
#pragma unroll 4
      for (int row = lane >> 3; row < nfn; row += 8) sm[row * P + s] = src[(row >> half) * stride];
    }
    if (lane < cnt) {
      const double *src = mu + ubase + m0 + lane;
#pragma unroll 8
      for (int i = 0; i < nr; ++i) sm[2 * i * P + 8 + lane] = src[(long)i * L];
    }
    for (int i = lane; i < nr; i += 64) {
      const double r2inv = 1.0 / (rr[i] * rr[i]);
      an[2 * i] = c * ((l * (l + 1.0) * r2inv) + (Vsph[(long)o * nrad_total + r0 + i] - e_o - d_o));
      sinv[i] = ht.sinv[r0 + i];
      supm[i] = ht.supm[r0 + i];
    }
    for (int t = lane; t < 5 * P; t += 64) sm[nfn * P + t] = 0.0;
    if (lane < 2) an[nfn + lane] = 0.0;
    __syncthreads();

    // Spline slopes on the t-axis of mu (a column per lane) and of a (the last lane): the
    // (2, 4, ..., 4, 2 | 1) system of src/horton/cubic_spline.cpp:54-79, eliminated in the
    // table: r_i = (rhs_i - r_{i-1}) / den_i forward, dt_i = r_i - upm_i dt_{i+1} back.
    // Four nodes at a time, the next four read before the slopes are stored.
    if (lane < cnt || lane == 63) {
      double *x = lane == 63 ? an : sm + 8 + lane;
      const int st = lane == 63 ? 1 : P;
      double yn[4], sn[4], yc = x[0], ym = yc, rprev = 0.0;
      for (int j = 0; j < 4; ++j) {
        yn[j] = x[2 * min(j + 1, nr - 1) * st];
        sn[j] = sinv[min(j, nr - 1)];
      }
      for (int i0 = 0; i0 < nr; i0 += 4) {
        double y4[4], s4[4], res[4];
        for (int j = 0; j < 4; ++j) {
          y4[j] = x[2 * min(i0 + j + 5, nr - 1) * st];
          s4[j] = sinv[min(i0 + j + 4, nr - 1)];
        }
        for (int j = 0; j < 4; ++j) {
          rprev = (3.0 * (yn[j] - ym) - rprev) * sn[j];
          ym = yc, yc = yn[j];
          res[j] = rprev;
        }
        for (int j = 0; j < 4; ++j)
          if (i0 + j < nr) x[(2 * (i0 + j) + 1) * st] = res[j];
        for (int j = 0; j < 4; ++j) yn[j] = y4[j], sn[j] = s4[j];
      }
      double dtn = x[(nfn - 1) * st];
      for (int j = 0; j < 4; ++j) {
        yn[j] = x[(2 * max(nr - 2 - j, 0) + 1) * st];
        sn[j] = supm[max(nr - 2 - j, 0)];
      }
      for (int i0 = nr - 2; i0 >= 0; i0 -= 4) {
        double y4[4], s4[4], res[4];
        for (int j = 0; j < 4; ++j) {
          y4[j] = x[(2 * max(i0 - j - 4, 0) + 1) * st];
          s4[j] = supm[max(i0 - j - 4, 0)];
        }
        for (int j = 0; j < 4; ++j) {
          dtn = yn[j] - sn[j] * dtn;
          res[j] = dtn;
        }
        for (int j = 0; j < 4; ++j)
          if (i0 >= j) x[(2 * (i0 - j) + 1) * st] = res[j];
        for (int j = 0; j < 4; ++j) yn[j] = y4[j], sn[j] = s4[j];
      }
    }
    __syncthreads();

    // a on the t-axis: a_y j1^2, (a_x j1^2 + 2 a_y j2) j1 (napmo/utilities/ode2.py:35-118)
    for (int i = lane; i < nr; i += 64) {
      const double j1i = sm[2 * i * P + 6], ay = an[2 * i], ad = an[2 * i + 1];
      an[2 * i] = ay * (j1i * j1i);
      an[2 * i + 1] = (ad * j1i + 2 * ay * sm[2 * i * P + 7]) * j1i;
    }
    // The source f = c (mu, mu_x) on the t-axis likewise; the right-hand side of rows 2i,
    // 2i + 1 is the sum of f over nodes i-1, i, i+1 times the node integrals (zero rows for
    // the value conditions), in place through a register window of the three nodes.
    if (lane < cnt) {
      double *x = sm + 8 + lane;
      double ny = x[0], nd = x[P], n1 = sm[6], n2 = sm[7];
      double w[12];
      double fa0 = 0.0, fa1 = 0.0, fb0 = 0.0, fb1 = 0.0;
      for (int i = -1; i < nr; ++i) {
        // f of node i + 1 from what was read a step ago
        const double fy = c * ny;
        double fc0 = fy * (n1 * n1), fc1 = (c * nd * n1 + 2 * fy * n2) * n1;
        if (i + 1 >= nr) fc0 = 0.0, fc1 = 0.0;
        const int in = min(i + 2, nr - 1), iw = min(i + 1, nr - 1);
        double wn[12];
        ny = x[2 * in * P], nd = x[(2 * in + 1) * P], n1 = sm[2 * in * P + 6], n2 = sm[2 * in * P + 7];
        for (int t = 0; t < 6; ++t) {
          wn[t] = sm[2 * iw * P + t];
          wn[6 + t] = sm[(2 * iw + 1) * P + t];
        }
        if (i >= 0)
          for (int r = 0; r < 2; ++r) {
            const double *w6 = w + 6 * r;
            x[(2 * i + r) * P] = fa0 * w6[0] + fa1 * w6[1] + fb0 * w6[2] + fb1 * w6[3] +
                                 fc0 * w6[4] + fc1 * w6[5];
          }
        fa0 = fb0, fa1 = fb1, fb0 = fc0, fb1 = fc1;
        for (int t = 0; t < 12; ++t) w[t] = wn[t];
      }
    }
    __syncthreads();

    // Galerkin matrix: c0 + sum_k a_k oa[k], a lane per band entry; rows 0 and nfn - 2 are
    // u = 0, slot 7 is empty
    {
      const int s = lane & 7;
#pragma unroll 4
      for (int row = lane >> 3; row < nfn; row += 8) {
        const int col = row + s - 3, entry = row * 7 + min(s, 6);
        const int begin = max(2 * (row / 2 - 1), 0), end = min(2 * (row / 2 + 2), nfn);
        double v = C0[entry];
        for (int kk = 0; kk < 6; ++kk) v += an[begin + kk] * OA[entry * 6 + kk];  // 0 past end
        if (s == 7 || col < begin || col >= end) v = 0.0;
        if (row == 0 || row == nfn - 2) v = s == 3 ? 1.0 : 0.0;
        sm[row * P + s] = v;
      }
    }
    __syncthreads();

    // Elimination with partial pivoting (pivot among rows k .. k + 3). Lanes past the last
    // column repeat it. A lane's band slot in row r is its column minus (r - 3). Eight steps
    // at a time: the lane of the pivot column and the slots are then known in each.
    const int own = min(lane, 7 + cnt);
    double w0, w1, w2, w3, wn;
    {
      auto first = [&](int r) {
        const int s = lane - r + 3;
        return lane >= 8 ? sm[r * P + own] : (lane < 7 && s < 7) ? sm[r * P + s] : 0.0;
      };
      w0 = first(0), w1 = first(1), w2 = first(2), w3 = first(3);
    }
    int at_slot[8];
    for (int j = 0; j < 8; ++j) at_slot[j] = lane < 8 ? (lane - j) & 7 : own;
    wn = sm[4 * P + at_slot[1]];
    double *row = sm;
    for (int k0 = 0; k0 < nfn; k0 += 8) {
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        if (k0 + j >= nfn) break;
        const double wnn = row[5 * P + at_slot[(j + 2) & 7]];
        // every lane looks for the pivot of its own column; lane j's column is k0 + j
        double big = fabs(w0);
        int p = 0;
        if (fabs(w1) > big) big = fabs(w1), p = 1;
        if (fabs(w2) > big) big = fabs(w2), p = 2;
        if (fabs(w3) > big) big = fabs(w3), p = 3;
        p = __builtin_amdgcn_readlane(p, j);
        double u0 = p == 1 ? w1 : w0;
        u0 = p == 2 ? w2 : u0;
        u0 = p == 3 ? w3 : u0;
        w1 = p == 1 ? w0 : w1;
        w2 = p == 2 ? w0 : w2;
        w3 = p == 3 ? w0 : w3;
        const double c1 = lane_value(w1, j), c2 = lane_value(w2, j), c3 = lane_value(w3, j);
        double num = lane == 0 ? c1 : 1.0;
        num = lane == 1 ? c2 : num;
        num = lane == 2 ? c3 : num;
        const double f = num / lane_value(u0, j);
        const double f1 = lane_value(f, 0), f2 = lane_value(f, 1), f3 = lane_value(f, 2);
        const double inv = lane_value(f, 3);
        row[at_slot[j]] = lane == ((j + 7) & 7) ? inv : u0;
        const bool retired = lane == j;  // the next column in this lane starts at row k + 4
        w0 = retired ? 0.0 : w1 - f1 * u0;
        w1 = retired ? 0.0 : w2 - f2 * u0;
        w2 = retired ? 0.0 : w3 - f3 * u0;
        w3 = wn;
        wn = wnn;
        row += P;
      }
    }
    __syncthreads();

    // Back substitution, window u = x[k + 1 .. k + 6], the rows of the next node read ahead.
    // The solution's value y is u at even rows, its slope on the t-axis u at odd rows.
    if (lane < cnt) {
      double u1 = 0.0, u2 = 0.0, u3 = 0.0, u4 = 0.0, u5 = 0.0, u6 = 0.0;
      bool singular = false;
      double ra[9], rb[9];
      auto row = [&](int k, double *t) {
        for (int s = 0; s < 8; ++s) t[s] = sm[k * P + s];
        t[8] = sm[k * P + 8 + lane];
      };
      auto step = [&](const double *t) {
        const double s = (((t[8] - t[6] * u6) - t[5] * u5) - t[4] * u4) - t[3] * u3;
        const double sn = (s - t[2] * u2) - t[1] * u1;
        const double q = sn * t[7];
        singular |= t[0] == 0.0;
        const double xs = fma(fma(-t[0], q, sn), t[7], q);
        u6 = u5, u5 = u4, u4 = u3, u3 = u2, u2 = u1, u1 = xs;
      };
      row(nfn - 1, ra);
      row(nfn - 2, rb);
      double *oy = Uy + ubase + m0 + lane, *od = Udt + ubase + m0 + lane;
      for (int i = nr - 1; i >= 0; --i) {
        double na[9], nb[9];
        const int in = max(i - 1, 0);
        row(2 * in + 1, na);
        row(2 * in, nb);
        step(ra);
        step(rb);
        od[(long)i * L] = u2;
        oy[(long)i * L] = u1;
        for (int s = 0; s < 9; ++s) ra[s] = na[s], rb[s] = nb[s];
      }
      if (singular) status[0] = 1;
    }
    __syncthreads();
  }
}

// R = T + V - e psi; per-block partial sums of R psi w bw, then a fixed-order final sum.
__global__ void __launch_bounds__(256) k_residual(const double *__restrict__ psi,
                                                  const double *__restrict__ T,
                                                  const double *__restrict__ V,
                                                  const double *__restrict__ e,
                                                  const double *__restrict__ wbw, long N,
                                                  double *__restrict__ R,
                                                  double *__restrict__ work) {
  __shared__ double red[4];
  const int o = blockIdx.y;
  const long base = (long)o * N;
  const double eo = e[o];
  double acc = 0.0;
  for (long p = (long)blockIdx.x * 256 + threadIdx.x; p < N; p += (long)gridDim.x * 256) {
    const double r = T[base + p] + V[base + p] - eo * psi[base + p];
    R[base + p] = r;
    acc += (r * psi[base + p]) * wbw[p];
  }
  for (int k = 32; k > 0; k >>= 1) acc += __shfl_xor(acc, k);
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = acc;
  __syncthreads();
  if (threadIdx.x == 0) work[(long)o * gridDim.x + blockIdx.x] = ((red[0] + red[1]) + red[2]) + red[3];
}

__global__ void k_residual_final(const double *__restrict__ work, int nblk, int norb,
                                 double *__restrict__ de) {
  const int o = blockIdx.x * blockDim.x + threadIdx.x;
  if (o >= norb) return;
  double s = 0.0;
  for (int b = 0; b < nblk; ++b) s += work[(long)o * nblk + b];
  de[o] = s;
}

}  // namespace

void launch_scaled_diff(const double *a, const double *s, const double *b, int norb, long N,
                        double *out, hipStream_t st) {
  if (norb <= 0 || N <= 0) return;
  k_scaled_diff<<<dim3((unsigned)div_up(N, 256), norb), 256, 0, st>>>(a, s, b, N, out);
  NAPMO_HIP(hipGetLastError());
}

void launch_shell_average(const AtomTables &at, const double *V, int norb, long N, const double *w,
                          const double *bw, long nrad_total, double *Vsph, hipStream_t st) {
  if (norb <= 0) return;
  k_shell_average<<<dim3(at.max_nrad, at.M, norb), 64, 0, st>>>(at, V, N, w, bw, nrad_total, Vsph);
  NAPMO_HIP(hipGetLastError());
}

void launch_helmholtz_radial(const AtomTables &at, const HelmholtzTables &ht, int lmax, int norb,
                             long nrad_total, const double *Vsph, const double *oi,
                             const double *doi, double mass_inv, const double *mu, double *Uy,
                             double *Udt, int *status, hipStream_t st) {
  if (norb <= 0) return;
  NAPMO_REQUIRE(at.max_nrad <= HELMHOLTZ_MAX_NRAD,
                "orbital correction: radial grids of more than " +
                    std::to_string(HELMHOLTZ_MAX_NRAD) + " points are not supported");
  NAPMO_REQUIRE(at.max_nrad >= 3, "orbital correction: radial grids need at least 3 points");
  const int L = (lmax + 1) * (lmax + 1);
  const long nr = at.max_nrad, nfn = 2L * nr, nm = 2L * lmax + 1;
  // Columns of one pass: every pass repeats the elimination, and the columns' LDS decides how
  // many systems a CU holds at once. Take the number of passes that is cheapest per system
  // resident, counting no more of them than the launch can fill.
  const long cap = (long)max_lds_per_block();
  auto lds = [&](long cols) { return ((nfn + 5) * (8 + cols) + 2 * nfn + 2) * (long)sizeof(double); };
  int dev = 0, cus = 0;
  NAPMO_HIP(hipGetDevice(&dev));
  NAPMO_HIP(hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev));
  const long need = div_up((long)at.M * (lmax + 1) * norb, (long)cus);
  long mc = 1;
  double best = 0.0;
  for (long pass = 1; pass <= nm; ++pass) {
    const long cols = div_up(nm, pass);
    if (cols > HELM_MAX_COLS || lds(cols) > cap) continue;
    const double cost = (double)pass / (double)std::min(need, cap / lds(cols));
    if (best == 0.0 || cost < best) best = cost, mc = cols;
  }
  const size_t bytes = (size_t)lds(mc);
  NAPMO_REQUIRE(bytes <= max_lds_per_block(), "orbital correction: radial system does not fit in LDS");
  // past 64 KB (about 230 radial points) the kernel needs the device's full LDS per block
  static int configured = -1;
  if (configured != dev) {
    NAPMO_HIP(hipFuncSetAttribute((const void *)k_helmholtz_radial, hipFuncAttributeMaxDynamicSharedMemorySize,
                                  (int)max_lds_per_block()));
    configured = dev;
  }
  k_helmholtz_radial<<<dim3(at.M, lmax + 1, norb), 64, bytes, st>>>(
      at, ht, L, nrad_total, Vsph, oi, doi, mass_inv, mu, (int)mc, Uy, Udt, status);
  NAPMO_HIP(hipGetLastError());
}

void launch_residual(const double *psi, const double *T, const double *V, const double *e,
                     const double *wbw, int norb, long N, double *R, double *de, double *work,
                     hipStream_t st) {
  if (norb <= 0) return;
  const int nblk = (int)std::max<long>(1, std::min<long>(RESID_BLOCKS, div_up(N, 256)));
  k_residual<<<dim3(nblk, norb), 256, 0, st>>>(psi, T, V, e, wbw, N, R, work);
  k_residual_final<<<div_up(norb, 64), 64, 0, st>>>(work, nblk, norb, de);
  NAPMO_HIP(hipGetLastError());
}

}  // namespace napmo
