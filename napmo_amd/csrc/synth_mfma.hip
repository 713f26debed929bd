// Synthesis of many densities at once on FP64 MFMA. The same sum as k_synth2n,
// v_s(p) = sum_A sum_q S^{A,s}_q(d) Y_q(p - R_A): inside one (centre, radial interval) bucket
// every pair shares the interval's spline coefficients, so with the pair's features
// f_qc = u^c Y_q the sum is the product F [pairs x 4 L] . T [4 L x densities]
// (src/horton/evaluate.cpp:129-223 evaluated for every density).
//
// A wavefront takes one 64-pair slot of a bucket (four 16-pair row blocks b) and up to
// 16 TW + 4 T4 densities: per q and row block one feature (lane % 16 the pair, lane / 16 the
// Horner power c) feeds TW products 16 x 16 x 4 and T4 products 4 x 4 x 4 (four blocks of four
// pairs, four densities), which take 64 and 16 cycles, so a last tile costs what its densities
// need in fours. FP64 MFMA holds the SIMD's VALU, so forming the features (about two FP64
// operations per q and row block) adds to the matrix time: two tiles per wave halve it. Bound by
// FP64 MFMA. Measured on 16 centres x 472,000 points at lmax 12: 40 densities 7.9 ms (32 in
// tiles of 16, one tile per wave, and 8 one at a time) -> 6.6 ms (62 TFLOP/s).
#include <hip/hip_runtime.h>

#include <algorithm>

#include "common.hpp"
#include "kernels.hpp"
#include "synth_rows.hpp"

namespace napmo {

typedef double smf_d4 __attribute__((ext_vector_type(4)));
typedef unsigned smf_u2 __attribute__((ext_vector_type(2)));

namespace {

constexpr int SMF_WPB = 4;  // waves per workgroup (independent, no LDS)
// coefficient loads in flight, in (l, m) steps: two long steps cover L2 as four short ones do
constexpr int smf_pd(int tw, int t4) { return tw == 2 && t4 > 0 ? 2 : 4; }

// beta(l, m) of the scaled recurrence at l (l + 1) / 2 + m, 0 for l < m + 2
struct BetaTable {
  double v[(MAX_LMAX + 1) * (MAX_LMAX + 2) / 2];
};
constexpr BetaTable make_beta() {
  BetaTable t = {};
  for (int l = 0; l <= MAX_LMAX; ++l)
    for (int m = 0; m <= l; ++m) t.v[l * (l + 1) / 2 + m] = l >= m + 2 ? pi_beta(l, m) : 0.0;
  return t;
}
__constant__ BetaTable SMF_BETA = make_beta();

// REG 1 (interval): feature u^c Y_q, coefficient T_j[q][c]. REG 0 / 2 (extrapolation): only
// c = 0 carries a term, d^l Y_q or d^-(l+1) Y_q with the amplitude of q (the rows c > 0 of the
// features are zero). row: wave-uniform coefficient row of q = 0, rows qstride doubles apart;
// tofs, qofs: this lane's byte offsets for the tiles and the fours. The harmonics are formed by
// the recurrences of synth_harmonics_np (Re / Im (x + i y)^m and the scaled PI_l^m(z)).
template <int TW, int T4, int REG>
__device__ __forceinline__ void smf_body(const double (&g0)[4], const double (&ux)[4], const double (&uy)[4],
                                         const double (&uz)[4], int c, int lmax, const double *row, long qstride,
                                         unsigned tofs, unsigned qofs, unsigned tstep, unsigned qstep,
                                         smf_d4 (&acc)[4][TW > 0 ? TW : 1], double (&acq)[4][T4 > 0 ? T4 : 1]) {
  constexpr int SMF_PD = smf_pd(TW, T4);
  const int L = (lmax + 1) * (lmax + 1), steps = (lmax + 1) * (lmax + 2) / 2;
  double w[4], base[4], pwm[4], Am[4], Bm[4], fa[4], fb[4], cur[4], prev[4], pw[4];
#pragma unroll
  for (int b = 0; b < 4; ++b) {
    if (REG == 1) {
      const double u = g0[b], u2 = u * u;
      w[b] = c == 0 ? 1.0 : (c == 1 ? u : (c == 2 ? u2 : u2 * u));
      base[b] = 1.0, pwm[b] = 1.0;
    } else {
      w[b] = c == 0 ? 1.0 : 0.0;
      base[b] = (REG == 0) ? g0[b] : 1.0 / g0[b];
      pwm[b] = (REG == 2) ? base[b] : 1.0;
    }
    Am[b] = 1.0, Bm[b] = 0.0, fa[b] = w[b], fb[b] = 0.0, cur[b] = 1.0, prev[b] = 0.0, pw[b] = pwm[b];
  }
  // coefficients of the next SMF_PD steps: rows q (cos) and q + 1 (sin; not used for m = 0),
  // through a buffer descriptor of the bucket's rows: lane offset + scalar offset, no address
  // arithmetic on the VALU. Past the last step the last row is read again, and its features are
  // zero.
  const __amdgpu_buffer_rsrc_t rsrc = __builtin_amdgcn_make_buffer_rsrc((void *)row, 0, (int)(L * qstride * 8), 0x00020000);
  const int qbytes = (int)qstride * 8, qlast = (L - 1) * qbytes;
  double rt[SMF_PD][2][TW > 0 ? TW : 1], rq[SMF_PD][2][T4 > 0 ? T4 : 1];
  SynthRows next;  // of the load stream
  auto fetch = [&](unsigned v, int so) {
    const smf_u2 r = __builtin_amdgcn_raw_buffer_load_b64(rsrc, (int)v, so, 0);
    return __builtin_bit_cast(double, r);
  };
  auto load = [&](int k) {
    const int so[2] = {next.cos_row(qlast), next.sin_row(qbytes, qlast)};
#pragma unroll
    for (int h = 0; h < 2; ++h) {
#pragma unroll
      for (int t = 0; t < TW; ++t) rt[k][h][t] = fetch(tofs + t * tstep, so[h]);
#pragma unroll
      for (int t = 0; t < T4; ++t) rq[k][h][t] = fetch(qofs + t * qstep, so[h]);
    }
    next.next(lmax, qbytes);
  };
  auto products = [&](const double (&f)[4], const double (&ct)[TW > 0 ? TW : 1], const double (&cq)[T4 > 0 ? T4 : 1]) {
#pragma unroll
    for (int b = 0; b < 4; ++b) {
#pragma unroll
      for (int t = 0; t < TW; ++t) acc[b][t] = __builtin_amdgcn_mfma_f64_16x16x4f64(f[b], ct[t], acc[b][t], 0, 0, 0);
#pragma unroll
      for (int t = 0; t < T4; ++t) acq[b][t] = __builtin_amdgcn_mfma_f64_4x4x4f64(f[b], cq[t], acq[b][t], 0, 0, 0);
    }
  };
#pragma unroll
  for (int k = 0; k < SMF_PD; ++k) {
    load(k);
    __builtin_amdgcn_sched_barrier(0);  // in this order, as in the loop
  }
  int l = 0, m = 0;
  double beta = 0.0;  // of the next l, read one step ahead
  // whole groups of SMF_PD steps (no early exit, so that the waits keep the loads in flight):
  // past the last step the features are zero
#pragma unroll 1
  for (int s = 0; s < steps; s += SMF_PD) {
#pragma unroll
    for (int k = 0; k < SMF_PD; ++k) {
      double f[4];
#pragma unroll
      for (int b = 0; b < 4; ++b) f[b] = REG == 1 ? fa[b] * cur[b] : fa[b] * cur[b] * pw[b];
      products(f, rt[k][0], rq[k][0]);
      if (m > 0) {
#pragma unroll
        for (int b = 0; b < 4; ++b) f[b] = REG == 1 ? fb[b] * cur[b] : fb[b] * cur[b] * pw[b];
        products(f, rt[k][1], rq[k][1]);
      }
      load(k);
      __builtin_amdgcn_sched_barrier(0);
      if (l == lmax) {
        l = ++m;
        beta = 0.0;
        const bool past = m > lmax;
#pragma unroll
        for (int b = 0; b < 4; ++b) {
          const double a2 = fma(ux[b], Am[b], -(uy[b] * Bm[b]));
          Bm[b] = fma(ux[b], Bm[b], uy[b] * Am[b]);
          Am[b] = a2;
          if (REG != 1) pwm[b] *= base[b];
          fa[b] = past ? 0.0 : w[b] * Am[b], fb[b] = past ? 0.0 : w[b] * Bm[b];
          cur[b] = 1.0, prev[b] = 0.0, pw[b] = past ? 0.0 : pwm[b];
        }
      } else {
        ++l;
#pragma unroll
        for (int b = 0; b < 4; ++b) {
          const double n = fma(uz[b], cur[b], -(beta * prev[b]));
          prev[b] = cur[b];
          cur[b] = n;
          if (REG != 1) pw[b] *= base[b];
        }
        const int ln = min(l + 1, lmax);
        beta = SMF_BETA.v[ln * (ln + 1) / 2 + min(m, ln)];
      }
    }
  }
}

// Unit = 64-pair slot; workgroups are dealt to the 8 XCDs round-robin, so slot ranges are
// remapped to be contiguous per XCD and the waves of one bucket share that XCD's L2 copy of the
// bucket's coefficient rows.
// Tables (density-interleaved, ndp columns): T [A][interval][q][ndp][4], ampL / ampR [A][q][ndp].
// Output: tile t at contrib + t * tstride, layout [A][N][16] (one 128-byte row of 16 densities
// per (centre, point)), the fours in tile TW; padding pairs (list entry < 0) are not written.
template <int TW, int T4>
__global__ void __launch_bounds__(64 * SMF_WPB, 2) k_synth_mfma(
    AtomTables at, int lmax, const double *__restrict__ geo, long N, const int *__restrict__ list,
    const int *__restrict__ wave_bucket, long nslots, int ndp, const double *__restrict__ T,
    const double *__restrict__ ampL, const double *__restrict__ ampR, long tstride,
    double *__restrict__ contrib) {
  const int L = (lmax + 1) * (lmax + 1);
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const long per_xcd = (long)(gridDim.x >> 3);
  const long wg = (long)(blockIdx.x & 7) * per_xcd + (blockIdx.x >> 3);
  const long slot = wg * SMF_WPB + wave;
  if (slot >= nslots) return;
  const int gb = __builtin_amdgcn_readfirstlane(wave_bucket[slot]);
  const int A = gb / (at.max_nrad + 1), loc = gb - A * (at.max_nrad + 1);
  const int nr = at.nrad[A];
  const int reg = (loc == 0) ? 0 : (loc == nr ? 2 : 1);
  const int i = lane & 15, c = lane >> 4;
  const double *gs = geo + slot * 256;
  double g0[4], ux[4], uy[4], uz[4];
#pragma unroll
  for (int b = 0; b < 4; ++b) {
    g0[b] = gs[16 * b + i];
    ux[b] = gs[64 + 16 * b + i];
    uy[b] = gs[128 + 16 * b + i];
    uz[b] = gs[192 + 16 * b + i];
  }
  const int pown = list[slot * 64 + lane];
  smf_d4 acc[4][TW > 0 ? TW : 1];
  double acq[4][T4 > 0 ? T4 : 1];
#pragma unroll
  for (int b = 0; b < 4; ++b) {
#pragma unroll
    for (int t = 0; t < (TW > 0 ? TW : 1); ++t) acc[b][t] = (smf_d4){0.0, 0.0, 0.0, 0.0};
#pragma unroll
    for (int t = 0; t < (T4 > 0 ? T4 : 1); ++t) acq[b][t] = 0.0;
  }
  const unsigned dq = 16 * TW + (lane & 3);
  if (reg == 1) {
    const double *row = T + ((long)A * (at.max_nrad - 1) + loc - 1) * L * ndp * 4;
    smf_body<TW, T4, 1>(g0, ux, uy, uz, c, lmax, row, (long)ndp * 4, (i * 4 + c) * 8, (dq * 4 + c) * 8, 16 * 32,
                        4 * 32, acc, acq);
  } else if (reg == 0) {
    smf_body<TW, T4, 0>(g0, ux, uy, uz, c, lmax, ampL + (long)A * L * ndp, ndp, i * 8, dq * 8, 16 * 8, 4 * 8, acc, acq);
  } else {
    smf_body<TW, T4, 2>(g0, ux, uy, uz, c, lmax, ampR + (long)A * L * ndp, ndp, i * 8, dq * 8, 16 * 8, 4 * 8, acc, acq);
  }
  // 16 x 16 x 4: element r of a lane is pair 16 b + lane / 16 + 4 r, density lane % 16;
  // 4 x 4 x 4: pair 16 b + 4 (lane / 4 % 4) + lane / 16, density lane % 4
  double *out = contrib + (long)A * N * 16;
#pragma unroll
  for (int b = 0; b < 4; ++b) {
    if (TW > 0) {
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int p = __shfl(pown, 16 * b + c + 4 * r);
        if (p >= 0)
#pragma unroll
          for (int t = 0; t < TW; ++t) out[(long)t * tstride + (long)p * 16 + i] = acc[b][t][r];
      }
    }
    if (T4 > 0) {
      const int p = __shfl(pown, 16 * b + 4 * ((lane >> 2) & 3) + c);
      if (p >= 0)
#pragma unroll
        for (int t = 0; t < T4; ++t) out[(long)TW * tstride + (long)p * 16 + 4 * t + (lane & 3)] = acq[b][t];
    }
  }
}

}  // namespace

void launch_synth_mfma(const AtomTables &at, const double *geo, long N, const int *list,
                       const int *wave_bucket, long nslots, int tiles, int fours, const double *T,
                       const double *ampL, const double *ampR, int lmax, double *contrib,
                       hipStream_t s) {
  NAPMO_REQUIRE(lmax >= 0 && lmax <= MAX_LMAX, "lmax out of range for synthesis");
  NAPMO_REQUIRE(tiles >= 0 && tiles <= 2 && fours >= 0 && fours <= 3 && tiles + fours > 0,
                "MFMA synthesis: up to two tiles of 16 densities and three of 4");
  if (nslots <= 0) return;
  const int ndp = 16 * (tiles + (fours > 0 ? 1 : 0));
  const long per_xcd = div_up(div_up(nslots, SMF_WPB), 8);
  const dim3 grid((unsigned)(8 * per_xcd)), block(64 * SMF_WPB);
  switch (tiles * 4 + fours) {
#define NAPMO_CASE(TW, T4)                                                                        \
  case TW * 4 + T4:                                                                               \
    k_synth_mfma<TW, T4><<<grid, block, 0, s>>>(at, lmax, geo, N, list, wave_bucket, nslots, ndp, \
                                                T, ampL, ampR, (long)at.M * N * 16, contrib);     \
    break;
    NAPMO_CASE(0, 1) NAPMO_CASE(0, 2) NAPMO_CASE(0, 3)
    NAPMO_CASE(1, 0) NAPMO_CASE(1, 1) NAPMO_CASE(1, 2) NAPMO_CASE(1, 3)
    NAPMO_CASE(2, 0) NAPMO_CASE(2, 1) NAPMO_CASE(2, 2) NAPMO_CASE(2, 3)
#undef NAPMO_CASE
  }
  NAPMO_HIP(hipGetLastError());
}

}  // namespace napmo
