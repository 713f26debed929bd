// Grid density on FP64 MFMA: X = Phi B, then rho from X
// (napmo/wavefunction/psi_hybrid.py:144-154 and napmo/wavefunction/psi_numeric.py:361-369).
//   P form:       rho_p = sum_c X_pc Phi_pc with B the fold of P onto its lower block triangle
//   orbital form: rho_p = sum_c X_pc^2 with B = C (k_density_tiles; k_density_orb_stream when C
//                 fits in LDS)
//   product:      X [Npad x ldb] itself (the gradient's Phi P; k_phi_times)
#include <algorithm>
#include <type_traits>

#include "common.hpp"
#include "kernels.hpp"

namespace napmo {

typedef double d4 __attribute__((ext_vector_type(4)));

// Smallest e with 2^e >= m (m > 0).
__device__ inline int dens_pow2_ceil_exp(double m) {
  int ex;
  const double mant = frexp(m, &ex);
  return mant == 0.5 ? ex - 1 : ex;
}
typedef double d2 __attribute__((ext_vector_type(2)));

namespace {

// Workgroup g runs on XCD g % 8 (round-robin dispatch); the column tiles of one point
// tile are given ids that are congruent mod 8, so they share that XCD's L2 and the point
// tile's Phi rows come from HBM once: g = 8 i + x, column tile i % nct, point tile
// (i / nct) * 8 + x.
__device__ inline bool xcd_tile(int g, int nct, int npt, int &pt, int &ct) {
  const int x = g & 7, i = g >> 3;
  ct = i % nct;
  pt = (i / nct) * 8 + x;
  return pt < npt;
}

// ------------------------------------------------------------------------ product X = Phi B
// Workgroup: 128 points x 64 columns, 4 waves; wave w owns points 32 w .. 32 w + 31 and all 64
// columns. K runs in stages of 16: the next stage's Phi rows and B rows are loaded into
// registers while the MFMAs of the current stage run, then stored to the other LDS buffer. LDS
// rows are padded so each 16 x 4 fragment read of a wave touches every bank once per half.
constexpr int DPT = 128, DKS = 16;
constexpr int ASTRIDE = DPT + 16, BSTRIDE = TILE + 16;

__global__ void __launch_bounds__(256) k_phi_times(const double *__restrict__ phi, int ld, long Npad,
                                                   const double *__restrict__ B, int ldb,
                                                   double *__restrict__ X) {
  __shared__ double As[2][DKS][ASTRIDE];  // As[.][k][m] = Phi[p0 + m][k0 + k]
  __shared__ double Bs[2][DKS][BSTRIDE];  // Bs[.][k][c] = B[k0 + k][c0 + c]
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  int pt, ct;
  if (!xcd_tile(blockIdx.x, ldb / TILE, (int)(Npad / DPT), pt, ct)) return;
  const long p0 = (long)pt * DPT;
  const int c0 = ct * TILE, am = tid >> 1, ak = (tid & 1) * 8;
  const double *arow = phi + (p0 + am) * ld + ak;
  d2 ra[4];
  double rb[4];
  auto load = [&](int k0) {
#pragma unroll
    for (int i = 0; i < 4; ++i) ra[i] = *(const d2 *)(arow + k0 + 2 * i);
#pragma unroll
    for (int q = 0; q < 4; ++q) rb[q] = B[(long)(k0 + (tid + q * 256) / TILE) * ldb + c0 + tid % TILE];
  };
  auto store = [&](int buf) {
#pragma unroll
    for (int i = 0; i < 4; ++i) As[buf][ak + 2 * i][am] = ra[i].x, As[buf][ak + 2 * i + 1][am] = ra[i].y;
#pragma unroll
    for (int q = 0; q < 4; ++q) Bs[buf][(tid + q * 256) / TILE][tid % TILE] = rb[q];
  };
  d4 acc[2][4];
#pragma unroll
  for (int a = 0; a < 2; ++a)
#pragma unroll
    for (int b = 0; b < 4; ++b) acc[a][b] = (d4){0, 0, 0, 0};
  const int kr = lane >> 4, mi = lane & 15;
  load(0);
  store(0);
  __syncthreads();
  for (int k0 = 0; k0 < ld; k0 += DKS) {
    const int buf = (k0 / DKS) & 1;
    if (k0 + DKS < ld) load(k0 + DKS);
#pragma unroll
    for (int ks = 0; ks < DKS; ks += 4) {
      double a[2], b[4];
#pragma unroll
      for (int i = 0; i < 2; ++i) a[i] = As[buf][ks + kr][wave * 32 + i * 16 + mi];
#pragma unroll
      for (int j = 0; j < 4; ++j) b[j] = Bs[buf][ks + kr][j * 16 + mi];
#pragma unroll
      for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j)
          acc[i][j] = __builtin_amdgcn_mfma_f64_16x16x4f64(a[i], b[j], acc[i][j], 0, 0, 0);
    }
    if (k0 + DKS < ld) store(buf ^ 1);
    __syncthreads();
  }
  // f64 16x16x4 output: lane i, element r -> row (i / 16) + 4 r, column i % 16
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const long p = p0 + wave * 32 + i * 16 + kr + 4 * r;
#pragma unroll
      for (int j = 0; j < 4; ++j) X[p * ldb + c0 + j * 16 + mi] = acc[i][j][r];
    }
}

// -------------------------------------------------------------- density over column tiles
// rho = diag(Phi P Phi^T) takes only the symmetric part of P, so P is folded onto the lower
// block triangle (16 x 16 blocks): Q_kc = P_kc + P_ck for block row k below block column c, P
// itself in the diagonal blocks, nothing above; rho_p = sum_c Phi_pc (Phi Q)_pc. Column tile ct
// (64 columns) then multiplies the functions from 64 ct on only, and inside its diagonal the
// blocks k >= c: nb (nb + 1) / 2 blocks instead of nb^2.
//
// The operand (Q, or C in the orbital form) is laid out in fragment order, per column tile and
// group of 16 k: [ct][g][j][h][lane][2], lane (kr, mi) of block j holding k = 16 g + 4 kr + 2 h
// + (0, 1), column 64 ct + 16 j + mi.
__host__ __device__ inline long operand_size(int groups, int ntile) { return (long)ntile * groups * 1024; }

__device__ __forceinline__ void density_operand_body(const double *__restrict__ src, int n, int ncol, int fold,
                                                     int groups, double *__restrict__ dst, long e) {
  const int t = (int)(e & 1), lane = (int)(e >> 1) & 63, h = (int)(e >> 7) & 1, j = (int)(e >> 8) & 3;
  const long gg = e >> 10;
  const int g = (int)(gg % groups), ct = (int)(gg / groups);
  const int k = 16 * g + 4 * (lane >> 4) + 2 * h + t, c = 64 * ct + 16 * j + (lane & 15);
  double v = 0.0;
  if (k < n && c < ncol) {
    if (!fold)
      v = src[(long)k * ncol + c];
    else if (g == 4 * ct + j)
      v = src[(long)k * n + c];
    else if (g > 4 * ct + j)
      v = src[(long)k * n + c] + src[(long)c * n + k];
  }
  dst[e] = v;
}

__global__ void __launch_bounds__(256) k_density_operand(const double *__restrict__ src, int n, int ncol,
                                                         int fold, int groups, long size,
                                                         double *__restrict__ dst) {
  const long e = (long)blockIdx.x * 256 + threadIdx.x;
  if (e < size) density_operand_body(src, n, ncol, fold, groups, dst, e);
}

__global__ void __launch_bounds__(256) k_density_operand_group(const OperandMember *__restrict__ mem, int nmem) {
  const long g = blockIdx.x;
  const OperandMember &m = mem[group_member(mem, nmem, g)];
  density_operand_body(m.P, m.n, m.n, 1, m.groups, m.dst, (g - m.block0) * 256 + threadIdx.x);
}

constexpr int DT_SG = 2;                     // k groups per LDS stage
constexpr int DT_STAGE = DT_SG * 1024;       // doubles

// Workgroup: 4 waves, wave w owns 16 RB rows of points and the tile's NB column blocks. Phi rows
// come straight from memory as MFMA operands (lane (kr, mi) loads Phi[row mi][16 g + 4 kr .. + 3],
// the next group's vectors in flight; the k order inside a group is permuted alike on both
// operands), the operand through double-buffered LDS shared by the waves. Per group a wave issues
// RB x NB x 4 products and RB + 2 NB loads, with constant offsets: FP64 MFMA holds the VALU, so
// the loop has next to no other arithmetic. Bound by FP64 MFMA and by the start and end of each
// workgroup. Measured: P form, n = 300, 472,000 points 1.95 -> 1.05 ms against 64-column tiles
// over the whole P staged through LDS on both sides; orbital form, n = 480, 90 orbitals,
// 1,062,000 points 2.62 -> 2.07 ms (96 columns instead of 128).
template <int RB, int NB, bool PFORM>
__device__ __forceinline__ void density_tile_body(const DensityMember &d, int pt, int ct, double *lds) {
  const int tid = threadIdx.x, lane = tid & 63, kr = lane >> 4, mi = lane & 15;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int ld = d.ld, G = d.groups, g0 = PFORM ? 4 * ct : 0;
  const long row0 = ((long)pt * 4 + wave) * 16 * RB;
  const char *abase = (const char *)(d.phi + row0 * ld);  // wave-uniform; lane offsets below
  unsigned aoff[RB];
#pragma unroll
  for (int rb = 0; rb < RB; ++rb) aoff[rb] = (unsigned)(((16 * rb + mi) * ld + 4 * kr) * 8);
  const double *src = d.B + (long)ct * G * 1024;
  d2 r[DT_SG * 2];
  auto load = [&](int g) {  // operand of groups g, g + 1 (the last group again past the end)
#pragma unroll
    for (int q = 0; q < DT_SG * 2; ++q) {
      const int gq = min(g + q / 2, G - 1);
      r[q] = ((const d2 *)(src + (long)gq * 1024))[(q & 1) * 256 + tid];
    }
  };
  auto store = [&](int buf) {
#pragma unroll
    for (int q = 0; q < DT_SG * 2; ++q) ((d2 *)(lds + buf * DT_STAGE))[q * 256 + tid] = r[q];
  };
  d4 acc[RB][NB], a[2][RB];
#pragma unroll
  for (int rb = 0; rb < RB; ++rb)
#pragma unroll
    for (int j = 0; j < NB; ++j) acc[rb][j] = (d4){0, 0, 0, 0};
  auto rows = [&](int s, int g) {
    const char *b = abase + (long)min(g, G - 1) * 128;
#pragma unroll
    for (int rb = 0; rb < RB; ++rb) a[s][rb] = *(const d4 *)(b + aoff[rb]);
  };
  // group gg of the stage, its first NJ column blocks
  auto group = [&](auto NJ, int buf, int gg) {
    constexpr int nj = decltype(NJ)::value < NB ? decltype(NJ)::value : NB;
    d2 b[nj][2];
#pragma unroll
    for (int j = 0; j < nj; ++j)
#pragma unroll
      for (int h = 0; h < 2; ++h)
        b[j][h] = ((const d2 *)(lds + buf * DT_STAGE + gg * 1024))[(j * 2 + h) * 64 + lane];
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int s = 0; s < 4; ++s)
#pragma unroll
      for (int rb = 0; rb < RB; ++rb)
#pragma unroll
        for (int j = 0; j < nj; ++j)
          acc[rb][j] = __builtin_amdgcn_mfma_f64_16x16x4f64(a[gg][rb][s], b[j][s >> 1][s & 1], acc[rb][j], 0, 0, 0);
    __builtin_amdgcn_sched_barrier(0);
  };
  auto stage = [&](auto NJ0, auto NJ1, int g, int buf) {
    load(g + 2);
    rows(1, g + 1);
    group(NJ0, buf, 0);
    rows(0, g + 2);
    if (g + 1 < G) group(NJ1, buf, 1);
    store(buf ^ 1);
    __syncthreads();
  };
  load(g0);
  rows(0, g0);
  store(0);
  __syncthreads();
  typedef std::integral_constant<int, 1> N1;
  typedef std::integral_constant<int, 2> N2;
  typedef std::integral_constant<int, 3> N3;
  typedef std::integral_constant<int, 4> N4;
  int g = g0, buf = 0;
  if (PFORM) {
    stage(N1(), N2(), g, 0);
    g += 2;
    if (g < G) {
      stage(N3(), N4(), g, 1);
      g += 2;
    }
  }
#pragma unroll 1
  for (; g < G; g += 2, buf ^= 1) stage(N4(), N4(), g, buf);
  // f64 16x16x4 output: lane i, element r -> row (i / 16) + 4 r, column i % 16
#pragma unroll
  for (int rb = 0; rb < RB; ++rb)
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const long p = row0 + rb * 16 + kr + 4 * q;
      double sum = 0.0;
#pragma unroll
      for (int j = 0; j < NB; ++j) {
        const double x = acc[rb][j][q];
        sum += PFORM ? x * d.phi[p * ld + 64 * ct + j * 16 + mi] : x * x;
      }
      sum += __shfl_xor(sum, 8);
      sum += __shfl_xor(sum, 4);
      sum += __shfl_xor(sum, 2);
      sum += __shfl_xor(sum, 1);
      if (mi == 0 && p < d.nvalid) d.partial[(long)ct * d.Npad + p] = d.scale * sum;
    }
}

template <int RB, bool PFORM>
__device__ __forceinline__ void density_tiles(const DensityMember &d, int g, double *lds) {
  int pt, ct;
  if (!xcd_tile(g, d.ntile, (int)(d.Npad / (64 * RB)), pt, ct)) return;
  if constexpr (PFORM) {
    density_tile_body<RB, 4, true>(d, pt, ct, lds);
  } else {
    // the last tile's own column blocks
    switch (min(4, (d.ncol - 64 * ct + 15) / 16)) {
      case 1: density_tile_body<RB, 1, false>(d, pt, ct, lds); break;
      case 2: density_tile_body<RB, 2, false>(d, pt, ct, lds); break;
      case 3: density_tile_body<RB, 3, false>(d, pt, ct, lds); break;
      default: density_tile_body<RB, 4, false>(d, pt, ct, lds);
    }
  }
}

template <int RB, bool PFORM>
__global__ void __launch_bounds__(256, RB == 4 ? 2 : 3) k_density_tiles(DensityMember d) {
  __shared__ double lds[2 * DT_STAGE];
  density_tiles<RB, PFORM>(d, blockIdx.x, lds);
}

// Many plans in one launch: workgroup blockIdx.x belongs to the member whose block range
// holds it (block0 multiples of 8, so the XCD-aware tile order of each member is kept).
__global__ void __launch_bounds__(256, 3) k_density_tiles_group(const DensityMember *__restrict__ mem, int nmem) {
  __shared__ double lds[2 * DT_STAGE];
  const long g = blockIdx.x;
  const DensityMember d = mem[group_member(mem, nmem, g)];
  density_tiles<2, true>(d, (int)(g - d.block0), lds);
}

// Orbital form with C resident in LDS: the whole zero-padded C [kend x 16 NB] is copied
// once per workgroup into fragment order, Cf[g][j][lane][s] = C[16 g + 4 (lane / 16) + s]
// [16 j + lane % 16], and every wave then streams its own Phi rows from HBM straight into
// MFMA operands with no LDS staging and no barrier: for K group g (16 functions) lane
// (kr, mi) loads Phi[row mi][16 g + 4 kr .. + 3] as one 32-byte vector, and step s of the
// group multiplies element s of it by Cf[g][j][lane][s] (the k order inside a group is
// permuted identically on both operands). A wave owns 16 RB rows at a time and walks the
// row tiles with a stride of all waves in the grid; two groups are in flight per wave.
//
// SCR (screening, sc.S > 0): phi is the plan's Phi with its columns in the order sc.perm
// (row k of C is C[sc.perm[k]]), sc.eT [Npad / 16][ld / 16] bounds every |Phi| of a 16-row,
// 16-function block by 2^eT, and each workgroup bounds sum over a group's functions of
// max_c |C| by 2^eC; the products of a 16-row tile and group with eT + eC <= -S (each of
// their terms of X below 2^-S) are neither loaded nor multiplied.
template <int NB, int RB, int WAVES, int PF, bool SCR>
__global__ void __launch_bounds__(64 * WAVES) k_density_orb_stream(
    const double *__restrict__ phi, int ld, long Npad, const double *__restrict__ C, int nrow,
    int ncol, int kend, double scale, long nvalid, long ntiles, double *__restrict__ out,
    DensityScreen sc) {
  extern __shared__ d4 Cf[];  // [G][NB][64] vectors of 4 steps (then, SCR: eC [G] int)
  const int G = kend / 16;
  // C [nrow x ncol] row-major as given; entries past it are the zero padding
  for (int e = threadIdx.x; e < G * NB * 256; e += 64 * WAVES) {
    const int st = e & 3, ln = (e >> 2) & 63, gj = e >> 8;
    const int j = gj % NB, g = gj / NB;
    const int k = 16 * g + 4 * (ln >> 4) + st, c = 16 * j + (ln & 15);
    const int kk = SCR && k < nrow ? sc.perm[k] : k;
    ((double *)Cf)[e] = (k < nrow && c < ncol) ? C[(long)kk * ncol + c] : 0.0;
  }
  int *eC = (int *)(Cf + G * NB * 64);
  if constexpr (SCR) {
    // eC[g]: exponent bounding sum over the group's 16 functions of max_c |C| (16 lanes each)
    for (int e = threadIdx.x; e < G * 16; e += 64 * WAVES) {
      const int k = e;  // 16 g + t
      double m = 0.0;
      if (k < nrow) {
        const double *row = C + (long)sc.perm[k] * ncol;
        for (int c = 0; c < ncol; ++c) m = fmax(m, fabs(row[c]));
      }
      m += __shfl_xor(m, 8);
      m += __shfl_xor(m, 4);
      m += __shfl_xor(m, 2);
      m += __shfl_xor(m, 1);
      if ((e & 15) == 0) eC[e >> 4] = m > 0.0 ? dens_pow2_ceil_exp(m) : -4000;
    }
  }
  __syncthreads();
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, kr = lane >> 4, mi = lane & 15;
  const long nw = (long)gridDim.x * WAVES;
  const long ntile16 = Npad / 16;
  const int ldg = ld / 16;
  // SCR: the block exponents of a wave's next tile are loaded one tile ahead
  auto tile_exp = [&](long t, int rb) -> int {
    const long t16 = min(t * RB + rb, ntile16 - 1);
    return lane < G ? (int)sc.eT[t16 * ldg + lane] : 0;
  };
  int eTn[RB];
  if constexpr (SCR) {
#pragma unroll
    for (int rb = 0; rb < RB; ++rb) eTn[rb] = tile_exp((long)blockIdx.x * WAVES + wave, rb);
  }
  for (long t = (long)blockIdx.x * WAVES + wave; t < ntiles; t += nw) {
    const long r0 = t * 16 * RB;
    const double *ap[RB];
#pragma unroll
    for (int rb = 0; rb < RB; ++rb) {
      const long row = min(r0 + rb * 16 + mi, Npad - 1);  // rows past Npad: read, never written
      ap[rb] = phi + row * ld + 4 * kr;
    }
    // SCR: bit g of live[rb] = the (16-row tile, group g) products are kept
    unsigned long long live[RB];
#pragma unroll
    for (int rb = 0; rb < RB; ++rb) {
      live[rb] = ~0ull;
      if constexpr (SCR) {
        const bool keep = lane < G && eTn[rb] + eC[lane] > -sc.S;
        live[rb] = __ballot(keep);
        eTn[rb] = tile_exp(t + nw, rb);
      }
    }
    d4 acc[RB][NB];
#pragma unroll
    for (int rb = 0; rb < RB; ++rb)
#pragma unroll
      for (int j = 0; j < NB; ++j) acc[rb][j] = (d4){0, 0, 0, 0};
    auto load = [&](d4 (&a)[RB], int g) {
#pragma unroll
      for (int rb = 0; rb < RB; ++rb)
        if (!SCR || ((live[rb] >> g) & 1)) a[rb] = *(const d4 *)(ap[rb] + 16 * g);
    };
    auto compute = [&](const d4 (&a)[RB], int g) {
      d4 b[NB];
#pragma unroll
      for (int j = 0; j < NB; ++j) b[j] = Cf[(g * NB + j) * 64 + lane];
      if constexpr (!SCR) {
#pragma unroll
        for (int st = 0; st < 4; ++st)
#pragma unroll
          for (int rb = 0; rb < RB; ++rb)
#pragma unroll
            for (int j = 0; j < NB; ++j)
              acc[rb][j] = __builtin_amdgcn_mfma_f64_16x16x4f64(a[rb][st], b[j][st], acc[rb][j], 0, 0, 0);
      } else {
#pragma unroll
        for (int rb = 0; rb < RB; ++rb)
          if ((live[rb] >> g) & 1) {
#pragma unroll
            for (int st = 0; st < 4; ++st)
#pragma unroll
              for (int j = 0; j < NB; ++j)
                acc[rb][j] = __builtin_amdgcn_mfma_f64_16x16x4f64(a[rb][st], b[j][st], acc[rb][j], 0, 0, 0);
          }
      }
    };
    d4 a[PF][RB];
    if constexpr (!SCR) {
      // a ring of PF groups in flight: slot i holds group g0 + i
#pragma unroll
      for (int i = 0; i < PF; ++i)
        if (i < G) load(a[i], i);
      for (int g0 = 0; g0 < G; g0 += PF) {
#pragma unroll
        for (int i = 0; i < PF; ++i) {
          const int g = g0 + i;
          if (g < G) {
            compute(a[i], g);
            if (g + PF < G) load(a[i], g + PF);
          }
        }
      }
    } else {
      // the ring walks only the groups some 16-row tile of this wave keeps, in increasing
      // order (each accumulator adds its kept groups in the same order as the full ring)
      unsigned long long rest = 0;
#pragma unroll
      for (int rb = 0; rb < RB; ++rb) rest |= live[rb];
      if (G < 64) rest &= (1ull << G) - 1;
      int gl[PF];
#pragma unroll
      for (int i = 0; i < PF; ++i) {
        gl[i] = rest ? (int)__builtin_ctzll(rest) : -1;
        rest &= rest - 1;
        if (gl[i] >= 0) load(a[i], gl[i]);
      }
      while (gl[0] >= 0) {
#pragma unroll
        for (int i = 0; i < PF; ++i) {
          if (gl[i] < 0) break;
          compute(a[i], gl[i]);
          gl[i] = rest ? (int)__builtin_ctzll(rest) : -1;
          rest &= rest - 1;
          if (gl[i] >= 0) load(a[i], gl[i]);
        }
      }
    }
    // f64 16x16x4 output: lane i, element r -> row (i / 16) + 4 r, column i % 16
#pragma unroll
    for (int rb = 0; rb < RB; ++rb)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const long p = r0 + rb * 16 + kr + 4 * r;
        double sum = 0.0;
#pragma unroll
        for (int j = 0; j < NB; ++j) sum += acc[rb][j][r] * acc[rb][j][r];
        sum += __shfl_xor(sum, 8);
        sum += __shfl_xor(sum, 4);
        sum += __shfl_xor(sum, 2);
        sum += __shfl_xor(sum, 1);
        if (mi == 0 && p < nvalid) out[p] = scale * sum;
      }
  }
}

template <int NB, int RB, int WAVES, int PF, bool SCR>
void launch_orb_stream_scr(const double *phi, int ld, long Npad, const double *C, int nrow, int ncol,
                           int kend, double scale, long nvalid, double *out, const DensityScreen &sc,
                           hipStream_t s) {
  constexpr int STREAM_RB = RB, STREAM_WAVES = WAVES;
  const size_t bytes = (size_t)kend * 16 * NB * sizeof(double) + (SCR ? 4 * (size_t)round_up(kend / 16, 4) : 0);
  const long ntiles = div_up(Npad, 16L * STREAM_RB);
  auto kern = k_density_orb_stream<NB, RB, WAVES, PF, SCR>;
  static thread_local int configured = -1;  // per instantiation: dynamic LDS above 64 KB
  int dev = 0;
  NAPMO_HIP(hipGetDevice(&dev));
  if (configured != dev) {
    NAPMO_HIP(hipFuncSetAttribute((const void *)kern, hipFuncAttributeMaxDynamicSharedMemorySize,
                                  (int)max_lds_per_block()));
    configured = dev;
  }
  int occ = 0, cus = 0;
  NAPMO_HIP(hipOccupancyMaxActiveBlocksPerMultiprocessor(&occ, kern, 64 * STREAM_WAVES, bytes));
  NAPMO_HIP(hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev));
  NAPMO_REQUIRE(occ >= 1, "density_orb_stream: no occupancy");
  const long blocks = std::min<long>((long)occ * cus, div_up(ntiles, STREAM_WAVES));
  kern<<<dim3((unsigned)blocks), dim3(64 * STREAM_WAVES), bytes, s>>>(phi, ld, Npad, C, nrow, ncol,
                                                                       kend, scale, nvalid, ntiles, out, sc);
  NAPMO_HIP(hipGetLastError());
}

template <int NB, int RB, int WAVES, int PF>
void launch_orb_stream_nb(const double *phi, int ld, long Npad, const double *C, int nrow, int ncol,
                          int kend, double scale, long nvalid, double *out, const DensityScreen &sc,
                          hipStream_t s) {
  if (sc.S > 0)
    launch_orb_stream_scr<NB, RB, WAVES, PF, true>(phi, ld, Npad, C, nrow, ncol, kend, scale, nvalid, out, sc, s);
  else
    launch_orb_stream_scr<NB, RB, WAVES, PF, false>(phi, ld, Npad, C, nrow, ncol, kend, scale, nvalid, out, sc, s);
}

}  // namespace

static DensityMember density_member(const double *phi, int ld, long Npad, const double *B, int n, int ncol,
                                    int ntile, double *partial, double scale, long nvalid) {
  NAPMO_REQUIRE(ld % TILE == 0 && Npad % 256 == 0 && n >= 1 && n <= ld, "density: padding mismatch");
  DensityMember d = {};
  d.phi = phi, d.B = B, d.partial = partial, d.Npad = Npad, d.nvalid = nvalid, d.scale = scale;
  d.ld = ld, d.groups = (int)div_up(n, 16), d.ntile = ntile, d.ncol = ncol;
  return d;
}

long density_operand_size(int n, int ncol) {
  return operand_size((int)div_up(n, 16), (int)div_up(ncol, 64));
}

void launch_density_operand(const double *src, int n, int ncol, bool fold, double *dst, hipStream_t s) {
  const long size = density_operand_size(n, ncol);
  k_density_operand<<<div_up(size, 256), 256, 0, s>>>(src, n, ncol, fold ? 1 : 0, (int)div_up(n, 16), size, dst);
  NAPMO_HIP(hipGetLastError());
}

long density_operand_group_fill(OperandMember &m, const double *P, int n, double *dst, long block0) {
  m.P = P, m.dst = dst, m.block0 = block0, m.n = n, m.groups = (int)div_up(n, 16);
  return density_operand_size(n, n) / 256;
}

void launch_density_operand_group(const OperandMember *d_mem, int nmem, long nblocks, hipStream_t st) {
  if (nmem <= 0 || nblocks <= 0) return;
  k_density_operand_group<<<dim3((unsigned)nblocks), 256, 0, st>>>(d_mem, nmem);
  NAPMO_HIP(hipGetLastError());
}

// Points per workgroup: 256 (64 per wave, the fewest operand reads per product) where that makes
// at least two rounds of the 512 workgroups the device holds, else 128.
template <bool PFORM>
static void launch_density_tiles(const DensityMember &d, hipStream_t s) {
  if (d.Npad / 256 * d.ntile >= 1024)
    k_density_tiles<4, PFORM><<<(unsigned)(round_up(d.Npad / 256, 8) * d.ntile), 256, 0, s>>>(d);
  else
    k_density_tiles<2, PFORM><<<(unsigned)(round_up(d.Npad / 128, 8) * d.ntile), 256, 0, s>>>(d);
  NAPMO_HIP(hipGetLastError());
}

long density_group_fill(DensityMember &d, const double *phi, int ld, long Npad, const double *operand,
                        double *partial, int n, long block0) {
  NAPMO_REQUIRE(block0 % 8 == 0, "grouped density: workgroup alignment");
  d = density_member(phi, ld, Npad, operand, n, n, (int)div_up(n, 64), partial, 1.0, Npad);
  d.block0 = block0;
  return round_up(Npad / 128, 8) * d.ntile;
}

void launch_density_group(const DensityMember *d_mem, int nmem, long nblocks, hipStream_t s) {
  if (nmem <= 0 || nblocks <= 0) return;
  k_density_tiles_group<<<dim3((unsigned)nblocks), 256, 0, s>>>(d_mem, nmem);
  NAPMO_HIP(hipGetLastError());
}

void launch_density_f64(const double *phi, int ld, long Npad, const double *operand, double *partial,
                        hipStream_t s, int n) {
  launch_density_tiles<true>(density_member(phi, ld, Npad, operand, n, n, (int)div_up(n, 64), partial, 1.0, Npad), s);
}

int density_orb_cols(int nocc) {
  const int c = (int)round_up(nocc, 16);
  return c <= 64 ? c : (int)round_up(nocc, 64);
}

void launch_density_orb_f64(const double *phi, int ld, long Npad, const double *operand, int n, int nocc,
                            double *partial, hipStream_t s, double scale, long nvalid) {
  const int ntile = (int)div_up(nocc, 64);
  NAPMO_REQUIRE(nvalid < 0 || ntile == 1, "density_orb: a direct (scaled) write needs one column tile");
  launch_density_tiles<false>(density_member(phi, ld, Npad, operand, n, nocc, ntile, partial, scale,
                                             nvalid < 0 ? Npad : nvalid), s);
}

bool density_orb_stream_supported(int ld, int ldc, int nreal) {
  if (ldc > 64 || ldc % 16 || ld % 16) return false;
  const int kend = (nreal > 0 && nreal < ld) ? (int)round_up(nreal, 16) : ld;
  return (size_t)kend * ldc * sizeof(double) <= max_lds_per_block();
}

template <int RB, int WAVES, int PF>
static void orb_stream_shape(int nb, const double *phi, int ld, long Npad, const double *C, int nrow,
                             int ncol, int kend, double scale, long nvalid, double *out,
                             const DensityScreen &sc, hipStream_t s) {
  switch (nb) {
    case 1: launch_orb_stream_nb<1, RB, WAVES, PF>(phi, ld, Npad, C, nrow, ncol, kend, scale, nvalid, out, sc, s); break;
    case 2: launch_orb_stream_nb<2, RB, WAVES, PF>(phi, ld, Npad, C, nrow, ncol, kend, scale, nvalid, out, sc, s); break;
    case 3: launch_orb_stream_nb<3, RB, WAVES, PF>(phi, ld, Npad, C, nrow, ncol, kend, scale, nvalid, out, sc, s); break;
    default: launch_orb_stream_nb<4, RB, WAVES, PF>(phi, ld, Npad, C, nrow, ncol, kend, scale, nvalid, out, sc, s); break;
  }
}

void launch_density_orb_stream(const double *phi, int ld, long Npad, const double *C, int nrow,
                               int ncol, double *out, hipStream_t s, double scale, long nvalid,
                               int shape, const DensityScreen &sc) {
  const int ldc = density_orb_cols(ncol);
  NAPMO_REQUIRE(nrow >= 1 && nrow <= ld && ncol >= 1, "density_orb_stream: bad C shape");
  NAPMO_REQUIRE(density_orb_stream_supported(ld, ldc, nrow) && Npad % 16 == 0,
                "density_orb_stream: C does not fit in LDS or bad padding");
  NAPMO_REQUIRE(sc.S <= 0 || (sc.perm && sc.eT && ld <= 1024),
                "density_orb_stream: screening needs the column order and block exponents");
  const int kend = (int)std::min<long>(ld, round_up(nrow, 16));
  if (nvalid < 0) nvalid = Npad;
  const int nb = ldc / 16;
  // shapes: rows per wave (16 RB), waves per workgroup, K groups in flight
  switch (shape) {
    case 2: orb_stream_shape<3, 8, 2>(nb, phi, ld, Npad, C, nrow, ncol, kend, scale, nvalid, out, sc, s); break;
    case 3: orb_stream_shape<3, 8, 3>(nb, phi, ld, Npad, C, nrow, ncol, kend, scale, nvalid, out, sc, s); break;
    default: orb_stream_shape<2, 12, 3>(nb, phi, ld, Npad, C, nrow, ncol, kend, scale, nvalid, out, sc, s); break;
  }
}

__global__ void k_phi_tile_exp(const double *__restrict__ phi, int ld, long ntile16,
                               signed char *__restrict__ out) {
  const long e = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (e >= ntile16 * ld) return;
  const long t = e / ld;
  const int f = (int)(e % ld);
  double m = 0.0;
  for (int r = 0; r < 16; ++r) m = fmax(m, fabs(phi[(16 * t + r) * ld + f]));
  out[e] = m > 0.0 ? (signed char)max(-127, min(127, dens_pow2_ceil_exp(m))) : (signed char)-128;
}

__global__ void k_permute_cols(const double *__restrict__ phi, int ld, long Npad, const int *__restrict__ perm,
                               double *__restrict__ out) {
  const long e = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (e >= Npad * ld) return;
  const long p = e / ld;
  const int k = (int)(e % ld);
  out[e] = phi[p * ld + perm[k]];
}

void launch_phi_tile_exp(const double *phi, int ld, long Npad, signed char *out, hipStream_t s) {
  NAPMO_REQUIRE(Npad % 16 == 0, "phi tile exponents: rows not a multiple of 16");
  const long ne = (Npad / 16) * ld;
  k_phi_tile_exp<<<div_up(ne, 256), 256, 0, s>>>(phi, ld, Npad / 16, out);
  NAPMO_HIP(hipGetLastError());
}

void launch_permute_cols(const double *phi, int ld, long Npad, const int *perm, double *out, hipStream_t s) {
  const long ne = Npad * ld;
  k_permute_cols<<<div_up(ne, 256), 256, 0, s>>>(phi, ld, Npad, perm, out);
  NAPMO_HIP(hipGetLastError());
}

void launch_phi_times(const double *phi, int ld, long Npad, const double *B, int ldb, double *X,
                      hipStream_t s) {
  NAPMO_REQUIRE(ld % TILE == 0 && ldb % TILE == 0 && Npad % DPT == 0, "phi_times: padding");
  k_phi_times<<<(unsigned)(round_up(Npad / DPT, 8) * (ldb / TILE)), 256, 0, s>>>(phi, ld, Npad, B, ldb, X);
  NAPMO_HIP(hipGetLastError());
}

}  // namespace napmo
