// HIP kernels of the PECS per-time-step IMEX path for gfx950 (CDNA4).
//
// Per step (SolarCell.cpp:2057-2075):
//   k_rhs_carrier   assemble_{semiconductor,electrolyte}_rhs, both regions in
//                   one launch: geometry rebuilt from the 4 vertices
//                   (MappingQ1), old densities, Poisson field (Piola) and
//                   lagged traces of the other region at QGauss(k+2) points,
//                   contracted on FP64 MFMA; stores W = mu A^{-1} f_p in
//                   place of the current part f_p.
//   k_schur_rhs     g = f_v + B^T W (cell, face neighbours, hanging faces), a
//                   lane per density DoF.
//   k_fwd_gather / k_sweep  supernodal triangular solves
//                   with S = L L^T of both regions, level by level on the
//                   elimination forest:
//                   row tiles of dense [Linv; L21 Linv] panels, vector chunks
//                   staged in LDS, W lanes per row (deterministic, no atomics).
//   k_schur_recover q = W - A^{-1} B u; writes [Jx | Jy | u].
//   k_poisson_*     hybridised mixed Poisson: cell condensation, face
//                   assembly, multiplier solve, cell recovery.
// Batches of instances sharing the factors: k_sweep_mfma (FP64 MFMA) with
// RHS-interleaved vectors and their gathers.  FP32 variants (*_f32) of the
// Schur and Poisson cell kernels, a thread per cell on wave-uniform cell lists
// (table entries as scalar operands), serve the mixed-precision mode.
#include <hip/hip_runtime.h>

#include "kernels.hpp"

#include <algorithm>

namespace pecs {

namespace {

constexpr int WAVE = 64;

__device__ __forceinline__ double wave_sum(double x) {
#pragma unroll
  for (int o = WAVE / 2; o > 0; o >>= 1) x += __shfl_xor(x, o, WAVE);
  return x;
}

struct GeoD {
  double x, y, J00, J01, J10, J11, det;
};

__device__ __forceinline__ GeoD bilin(const double* v, double xi, double eta) {
  GeoD g;
  const double a = (1 - xi) * (1 - eta), b = xi * (1 - eta), c = (1 - xi) * eta, d = xi * eta;
  g.x = v[0] * a + v[2] * b + v[4] * c + v[6] * d;
  g.y = v[1] * a + v[3] * b + v[5] * c + v[7] * d;
  g.J00 = (v[2] - v[0]) * (1 - eta) + (v[6] - v[4]) * eta;
  g.J10 = (v[3] - v[1]) * (1 - eta) + (v[7] - v[5]) * eta;
  g.J01 = (v[4] - v[0]) * (1 - xi) + (v[6] - v[2]) * xi;
  g.J11 = (v[5] - v[1]) * (1 - xi) + (v[7] - v[3]) * xi;
  g.det = g.J00 * g.J11 - g.J01 * g.J10;
  return g;
}

__device__ __forceinline__ void face_nrm(const double* v, int f, double& nx, double& ny, double& len) {
  int a, b;
  if (f == 0) { a = 0; b = 2; }
  else if (f == 1) { a = 1; b = 3; }
  else if (f == 2) { a = 0; b = 1; }
  else { a = 2; b = 3; }
  const double tx = v[2 * b] - v[2 * a], ty = v[2 * b + 1] - v[2 * a + 1];
  len = sqrt(tx * tx + ty * ty);
  if (f == 1 || f == 2) { nx = ty / len; ny = -tx / len; }
  else { nx = -ty / len; ny = tx / len; }
}

template <int K>
struct Sz {
  static constexpr int NB = (K + 1) * (K + 1);
  static constexpr int NQ = (K + 2) * (K + 2);
  static constexpr int NF = K + 2;
  static constexpr int NRT = 2 * K * (K + 1);
  static constexpr int NRTX = K * (K + 1);
  static constexpr int NPHI = K * K;
  static constexpr int NL = NRT + NPHI;
};

typedef double v4d __attribute__((ext_vector_type(4)));

// doubles per type of the Schur kernels' operator tables (ctab)
template <int K>
constexpr int schur_tab() {
  return 3 * Sz<K>::NB * Sz<K>::NB + 8 * (K + 1) * (K + 1);
}

// local RT index of face node m of face f (RT_{K-1} nodal basis)
template <int K>
__device__ __forceinline__ int rt_face(int f, int m) {
  if (f == 0) return (K + 1) * m;
  if (f == 1) return K + (K + 1) * m;
  if (f == 2) return Sz<K>::NRTX + m;
  return Sz<K>::NRTX + m + K * K;
}

// ------------------------------------------------------------------------
// Carrier right-hand sides (SolarCell.cpp:1073-1414 and 1451-1726)
// ------------------------------------------------------------------------
// Both regions in one launch; a wave takes 16 cells of one region, lane
// l = 16 kq + col cell col, and the element contractions run on FP64 MFMA
// (16x16x4): values at the quadrature points from the DoFs, and the DoF rows
// from the pointwise integrands.  The result layout (lane l, register r: row
// kq + 4 r, cell col) of the first is the operand layout (k = kq of step r) of
// the second, so a lane computes the integrands of its own points
// q = 16 qb + 4 r + kq in registers and nothing moves between lanes.  The
// faces on the boundary and the interface take the same two steps over the
// face points, skipped where no cell of the wave has one.
// W (wmode): the current part is multiplied by mu A^{-1} before it is stored
// (what the Schur kernels read), one (cell, DoF) per thread from LDS.
// One thread per cell with the whole quadrature loop (255 VGPRs, about 4000
// dependent FP64 operations) took 36 + 36 us at refinement 8, k = 2, and
// 58 + 74 us at refinement 4, k = 3, the regions one after the other.
template <int K>
__global__ __launch_bounds__(256) void k_rhs_carrier(RhsPair A, DevPoisson P, DevTabs T,
                                                     const DevPhys* __restrict__ phs, const double* __restrict__ pvec,
                                                     int64_t sP) {
  using S = Sz<K>;
  constexpr int NB = S::NB, NQ = S::NQ, NF = S::NF, NX = S::NRTX;
  constexpr int SA = (NB + 3) / 4, SX = (NX + 3) / 4, QB = (NQ + 15) / 16, SF = (NF + 3) / 4;
  __shared__ double sf[4][64 * NB];  // [carrier, component][cell][DoF] (wmode)
  const bool first = (int)blockIdx.x < A.nblk0;
  const RhsSide& R = first ? A.side[0] : A.side[1];
  const bool semi = R.semi != 0;
  const int c0 = ((int)blockIdx.x - (first ? 0 : A.nblk0)) * 64;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
  const int col = lane & 15, kq = lane >> 4;
  const int cw = c0 + 16 * wave + col, nc = R.ncell;
  const bool on = cw < nc;
  const int c = on ? cw : nc - 1;  // (lanes past the last cell repeat it and store nothing)
  const int64_t inst = blockIdx.y;
  const DevPhys ph = phs[inst];
  const double* __restrict__ u1 = R.u[0] + inst * R.s;
  const double* __restrict__ u2 = R.u[1] + inst * R.s;
  pvec += inst * sP;
  const size_t nn = (size_t)nc * NB, uo = 2 * nn + (size_t)c * NB;
  double v[8];
#pragma unroll
  for (int t = 0; t < 8; ++t) v[t] = R.V[8 * (size_t)c + t];
  double d1[SA], d2[SA];
#pragma unroll
  for (int t = 0; t < SA; ++t) {
    const int a = 4 * t + kq;
    d1[t] = a < NB ? u1[uo + a] : 0.0;
    d2[t] = a < NB ? u2[uo + a] : 0.0;
  }
  const int* __restrict__ id = P.idx + (size_t)(semi ? c : P.ncell_semi + c) * P.nloc;
  double ex[SX], ey[SX];
#pragma unroll
  for (int t = 0; t < SX; ++t) {
    const int i = 4 * t + kq;
    ex[t] = i < NX ? pvec[id[i]] : 0.0;
    ey[t] = i < NX ? pvec[id[NX + i]] : 0.0;
  }
  const v4d zero = {0.0, 0.0, 0.0, 0.0};
  v4d ax1 = zero, ay1 = zero, av1 = zero, ax2 = zero, ay2 = zero, av2 = zero;
  const double inv_perm = 1.0 / (semi ? ph.eps_s : ph.eps_e), idt = 1.0 / ph.dt;
#pragma unroll
  for (int qb = 0; qb < QB; ++qb) {
    v4d n1 = zero, n2 = zero, hx = zero, hy = zero;
    const int qr = 16 * qb + col;  // this lane's row of the first operand
#pragma unroll
    for (int t = 0; t < SA; ++t) {
      const int a = 4 * t + kq;
      const double f = (qr < NQ && a < NB) ? T.phi[a * NQ + qr] : 0.0;
      n1 = __builtin_amdgcn_mfma_f64_16x16x4f64(f, d1[t], n1, 0, 0, 0);
      n2 = __builtin_amdgcn_mfma_f64_16x16x4f64(f, d2[t], n2, 0, 0, 0);
    }
#pragma unroll
    for (int t = 0; t < SX; ++t) {
      const int i = 4 * t + kq;
      const bool in = qr < NQ && i < NX;
      const double fx = in ? T.psix[i * NQ + qr] : 0.0, fy = in ? T.psiy[(NX + i) * NQ + qr] : 0.0;
      hx = __builtin_amdgcn_mfma_f64_16x16x4f64(fx, ex[t], hx, 0, 0, 0);
      hy = __builtin_amdgcn_mfma_f64_16x16x4f64(fy, ey[t], hy, 0, 0, 0);
    }
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      if (16 * qb + 4 * r >= NQ) continue;
      const int q = 16 * qb + 4 * r + kq;
      const bool in = q < NQ;
      const int qc = in ? q : NQ - 1;
      const GeoD g = bilin(v, T.qx[qc], T.qy[qc]);
      const double jxw = T.qw[qc] * g.det;
      const double Ex = (g.J00 * hx[r] + g.J01 * hy[r]) / g.det;
      const double Ey = (g.J10 * hx[r] + g.J11 * hy[r]) / g.det;
      double src = 0.0;
      if (semi) {
        if (ph.gen_mode == 0) src = ph.alpha * ph.G0 * exp(ph.alpha * (g.y - ph.H));
        else if (ph.gen_mode == 1) src = ph.G0 * exp(-ph.alpha * g.x);
        if (ph.srh)
          src += (ph.ni * ph.ni - n1[r] * n2[r]) / (ph.tau_n * (n1[r] + ph.ni) + ph.tau_p * (n2[r] + ph.ni));
      }
      if (R.msrc) src += R.msrc[(size_t)c * NQ + qc];
      // (selected, not multiplied by zero: rows past the last point may hold no number)
      const double sv1 = in ? jxw * (n1[r] * idt + src) : 0.0, sv2 = in ? jxw * (n2[r] * idt + src) : 0.0;
      const double cp1 = -inv_perm * n1[r] * jxw, cp2 = inv_perm * n2[r] * jxw;
      const double x1 = in ? cp1 * Ex : 0.0, y1 = in ? cp1 * Ey : 0.0;
      const double x2 = in ? cp2 * Ex : 0.0, y2 = in ? cp2 * Ey : 0.0;
      const double f = (in && col < NB) ? T.phi[col * NQ + q] : 0.0;
      av1 = __builtin_amdgcn_mfma_f64_16x16x4f64(f, sv1, av1, 0, 0, 0);
      av2 = __builtin_amdgcn_mfma_f64_16x16x4f64(f, sv2, av2, 0, 0, 0);
      ax1 = __builtin_amdgcn_mfma_f64_16x16x4f64(f, x1, ax1, 0, 0, 0);
      ay1 = __builtin_amdgcn_mfma_f64_16x16x4f64(f, y1, ay1, 0, 0, 0);
      ax2 = __builtin_amdgcn_mfma_f64_16x16x4f64(f, x2, ax2, 0, 0, 0);
      ay2 = __builtin_amdgcn_mfma_f64_16x16x4f64(f, y2, ay2, 0, 0, 0);
    }
  }
  const double hc = R.h[c];
  for (int f = 0; f < 4; ++f) {
    const int bid = R.bid[4 * (size_t)c + f];
    const int e = bid == 0 ? R.sigma_nb[c] : -1;
    const bool flux = R.mflux && (bid == 0 || bid == 2);  // manufactured data: prescribed normal flux, -<v, h>
    const bool dir = bid == 1, iface = bid == 0 && e >= 0, sch = semi && bid == 3;
    if (!__any(flux || dir || iface || sch)) continue;  // wave-uniform
    const double* fph = T.fphi + (size_t)f * NB * NF;
    const double* foph = T.fphi + (size_t)(f ^ 1) * NB * NF;
    v4d t1 = zero, t2 = zero, o1 = zero, o2 = zero;  // own and other side's traces
    if (__any(iface || sch)) {
      const size_t ob = 2 * (size_t)R.ncell_o * NB + (size_t)(e < 0 ? 0 : e) * NB;
      const double* __restrict__ ou1 = R.ou[0] + inst * R.so;
      const double* __restrict__ ou2 = R.ou[1] + inst * R.so;
#pragma unroll
      for (int t = 0; t < SA; ++t) {
        const int a = 4 * t + kq;
        const bool in = col < NF && a < NB;
        const double fo = in ? fph[a * NF + col] : 0.0, fe = in ? foph[a * NF + col] : 0.0;
        t1 = __builtin_amdgcn_mfma_f64_16x16x4f64(fo, d1[t], t1, 0, 0, 0);
        t2 = __builtin_amdgcn_mfma_f64_16x16x4f64(fo, d2[t], t2, 0, 0, 0);
        const bool ld = iface && a < NB;
        o1 = __builtin_amdgcn_mfma_f64_16x16x4f64(fe, ld ? ou1[ob + a] : 0.0, o1, 0, 0, 0);
        o2 = __builtin_amdgcn_mfma_f64_16x16x4f64(fe, ld ? ou2[ob + a] : 0.0, o2, 0, 0, 0);
      }
    }
    double nx, ny, len;
    face_nrm(v, f, nx, ny, len);
#pragma unroll
    for (int r = 0; r < SF; ++r) {
      const int q = 4 * r + kq;
      const bool in = q < NF;
      const int qc = in ? q : NF - 1;
      const double jw = T.fw[qc] * len;
      double w1 = 0.0, w2 = 0.0, x1 = 0.0, y1 = 0.0, x2 = 0.0, y2 = 0.0;
      if (flux) w1 = w2 = -R.mflux[(4 * (size_t)c + f) * NF + qc] * jw;
      if (dir) {  // Dirichlet
        const double pen = ph.penalty / hc;
        const double md = R.mdir ? R.mdir[(4 * (size_t)c + f) * NF + qc] : 0.0;
        const double e1 = jw * (R.mdir ? md : semi ? ph.ne : ph.rinf), e2 = jw * (R.mdir ? md : semi ? ph.pe : ph.oinf);
        x1 = -nx * e1;
        y1 = -ny * e1;
        w1 = pen * e1;
        x2 = -nx * e2;
        y2 = -ny * e2;
        w2 = pen * e2;
      } else if (iface) {
        if (semi) {
          w1 += -ph.k_et * (t1[r] - ph.ne) * o2[r] * jw;  // -v k_et (n - n^e) o
          w2 += ph.k_ht * (t2[r] - ph.pe) * o1[r] * jw;   // +v k_ht (p - p^e) r
        } else {
          const double cur = (-ph.k_et * (o1[r] - ph.ne) * t2[r] + ph.k_ht * (o2[r] - ph.pe) * t1[r]) * jw;
          w1 += cur;
          w2 -= cur;
        }
      } else if (sch) {  // Schottky (SolarCell.cpp:1348-1402)
        w1 += -ph.v_rec_n * (t1[r] - ph.ne) * jw;
        w2 += ph.v_rec_p * (t2[r] - ph.pe) * jw;
      }  // Neumann: nothing (SolarCell.cpp:1403-1406)
      if (!in) w1 = w2 = x1 = y1 = x2 = y2 = 0.0;
      const double fa = (in && col < NB) ? fph[col * NF + q] : 0.0;
      av1 = __builtin_amdgcn_mfma_f64_16x16x4f64(fa, w1, av1, 0, 0, 0);
      av2 = __builtin_amdgcn_mfma_f64_16x16x4f64(fa, w2, av2, 0, 0, 0);
      if (__any(dir)) {
        ax1 = __builtin_amdgcn_mfma_f64_16x16x4f64(fa, x1, ax1, 0, 0, 0);
        ay1 = __builtin_amdgcn_mfma_f64_16x16x4f64(fa, y1, ay1, 0, 0, 0);
        ax2 = __builtin_amdgcn_mfma_f64_16x16x4f64(fa, x2, ax2, 0, 0, 0);
        ay2 = __builtin_amdgcn_mfma_f64_16x16x4f64(fa, y2, ay2, 0, 0, 0);
      }
    }
  }
  double* __restrict__ b1 = R.b[0] + inst * R.s;
  double* __restrict__ b2 = R.b[1] + inst * R.s;
  const bool wm = A.wmode != 0;
#pragma unroll
  for (int r = 0; r < (NB + 3) / 4; ++r) {
    const int a = 4 * r + kq;
    if (a >= NB || !on) continue;
    const size_t at = (size_t)c * NB + a;
    b1[2 * nn + at] = av1[r];
    b2[2 * nn + at] = av2[r];
    if (wm) {
      const int l = (16 * wave + col) * NB + a;
      sf[0][l] = ax1[r];
      sf[1][l] = ay1[r];
      sf[2][l] = ax2[r];
      sf[3][l] = ay2[r];
    } else {
      b1[at] = ax1[r];
      b1[nn + at] = ay1[r];
      b2[at] = ax2[r];
      b2[nn + at] = ay2[r];
    }
  }
  if (!wm) return;
  __syncthreads();
  const int last = min(64, nc - c0) * NB;
  for (int l = threadIdx.x; l < last; l += 256) {
    const int lc = l / NB, a = l % NB;
    const double* tb = R.tab + (size_t)R.type[c0 + lc] * schur_tab<K>() + a * NB;
    double w[4] = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
    for (int q = 0; q < NB; ++q) {
      const double m = tb[q];
#pragma unroll
      for (int h = 0; h < 4; ++h) w[h] += m * sf[h][lc * NB + q];
    }
    const size_t at = (size_t)c0 * NB + l;
    b1[at] = R.mu[0] * w[0];
    b1[nn + at] = R.mu[0] * w[1];
    b2[at] = R.mu[1] * w[2];
    b2[nn + at] = R.mu[1] * w[3];
  }
}

// ------------------------------------------------------------------------
// Schur complement transforms
// ------------------------------------------------------------------------
// W_M = mu A_M^{-1} f_p,M of cell M (the current part of carrier RHS b):
// the cell-local inverse mass block times the cell's two current components.
template <int K>
__device__ __forceinline__ void schur_w(const DevRegion& R, const double* __restrict__ b, double mu, int M,
                                        int ty, double* w) {
  constexpr int NB = Sz<K>::NB;
  const size_t nc = R.ncell;
  const double* Minv = R.table + (size_t)ty * R.stride;
  double fx[NB], fy[NB];
#pragma unroll
  for (int a = 0; a < NB; ++a) {
    fx[a] = b[(size_t)M * NB + a];
    fy[a] = b[nc * NB + (size_t)M * NB + a];
  }
#pragma unroll
  for (int a = 0; a < NB; ++a) {
    double sx = 0.0, sy = 0.0;
#pragma unroll
    for (int t = 0; t < NB; ++t) {
      const double m = Minv[a * NB + t];
      sx += m * fx[t];
      sy += m * fy[t];
    }
    w[a] = mu * sx;
    w[NB + a] = mu * sy;
  }
}

// Cell of thread t on a wave-uniform cell list: cells grouped so that every
// wave's cells share the operator types the kernel reads (groups padded to
// whole waves with -1), so that the table offsets are wave-uniform and the
// table entries are fetched once per wave through the scalar cache.
__device__ __forceinline__ int schur_cell(const int* __restrict__ list, int n, int t) { return t < n ? list[t] : -1; }

__device__ __forceinline__ int wave_type(const DevRegion& R, int M) {
  return __builtin_amdgcn_readfirstlane(R.type[M]);
}

// The FP64 Schur kernels: one lane per (cell, density DoF a), NB = (K + 1)^2
// lanes per cell, 256 / NB cells per workgroup, both regions in one launch.
//
// They read W = mu A^{-1} f_p (k_carrier_w) in the place of the current part
// of the right-hand side, and compact operator tables (ctab): per type Minv,
// Bself and, per face f, the face's 2 (K + 1) x (K + 1) block of B: the trace
// DoFs of the cell's own currents against the neighbour's trace DoFs, all
// that is not zero of the 2 NB x NB block.  Per cell and right-hand side that
// is 2 NB^2 + 8 (K + 1)^2 products and 5 NB + 8 (K + 1) loads for the
// transform where whole blocks with W recomputed for 5 cells took 20 NB^2.
// A lane keeps its rows of the tables in registers and runs over `per`
// instances of a batch; a cell's W, u and s pass between its lanes in LDS.
// A lane's node lies on at most two faces: one of x = 0, 1 and one of y = 0, 1.
// HANG: the couplings across hanging faces, whole blocks, by the lanes of the
// few cells that have one (kernels of their own, a cell per thread, took 25 +
// 25 us and 23 + 22 us per step on the boundary-layer mesh at
// refinement 5; the step 354 -> 256 us).  The loop costs up to 70
// registers, so a system without hanging faces has its own variant.
// One thread per cell with whole blocks (its chain of 700 to 4000 dependent
// products and, on conic meshes, 9.7 KB of table per cell set the time) ->
// this, per step: refinement 4, k = 3, distinct mobilities 344 -> 236 us;
// refinement 7 conic 822 -> 594 us; 16 bias points at refinement 6 conic
// 940 -> 686 us; refinement 8 planar 1627 -> 1608 us.
template <int K>
struct SchurLane {
  static constexpr int NB = Sz<K>::NB, N1 = K + 1, CPB = 256 / NB;
  static constexpr int TAB = schur_tab<K>();
  static constexpr int FACE = 3 * NB * NB;
  __device__ static __forceinline__ int node(int f, int m) {
    return f == 0 ? N1 * m : f == 1 ? K + N1 * m : f == 2 ? m : N1 * K + m;
  }
};

// the region of this workgroup and its first cell
template <int K>
__device__ __forceinline__ const SchurSide& schur_side(const SchurPair& P, int& c0) {
  const bool first = (int)blockIdx.x < P.nblk0;
  c0 = ((int)blockIdx.x - (first ? 0 : P.nblk0)) * SchurLane<K>::CPB;
  return first ? P.side[0] : P.side[1];
}

// W = mu A^{-1} f_p of every cell (the current part of a carrier right-hand
// side): the cell-local inverse mass block times the two current components.
// In place when w == b.
template <int K>
__global__ __launch_bounds__(256) void k_carrier_w(SchurPair P, int nrhs, int ninst, int per) {
  using S = SchurLane<K>;
  constexpr int NB = S::NB, CPB = S::CPB;
  __shared__ double sf[2][CPB * NB];
  int c0;
  const SchurSide& R = schur_side<K>(P, c0);
  const int t = threadIdx.x, lc = t / NB, a = t % NB, c = c0 + lc;
  const bool on = lc < CPB && c < R.ncell;
  const size_t nb = (size_t)R.ncell * NB, at = (size_t)c * NB + a;
  double m[NB];
  if (on) {
    const double* tb = R.tab + (size_t)R.type[c] * S::TAB + a * NB;
#pragma unroll
    for (int q = 0; q < NB; ++q) m[q] = tb[q];
  }
  const int i1 = min(ninst, ((int)blockIdx.y + 1) * per);
  for (int i = blockIdx.y * per; i < i1; ++i)
    for (int h = 0; h < nrhs; ++h) {
      const double* b = R.b[h] + i * R.sb;
      double* w = R.w[h] + i * R.sb;
      if (on) {
        sf[0][t] = b[at];
        sf[1][t] = b[nb + at];
      }
      __syncthreads();
      if (on) {
        double x = 0.0, y = 0.0;
#pragma unroll
        for (int q = 0; q < NB; ++q) {
          x += m[q] * sf[0][lc * NB + q];
          y += m[q] * sf[1][lc * NB + q];
        }
        w[at] = R.mu[h] * x;
        w[nb + at] = R.mu[h] * y;
      }
      __syncthreads();
    }
}

// g = f_v + B^T W: the cell's own block and its face neighbours' traces of W
template <int K, int NRHS, bool HANG>
__global__ __launch_bounds__(256) void k_schur_rhs(SchurPair P, int ninst, int per) {
  using S = SchurLane<K>;
  constexpr int NB = S::NB, N1 = S::N1, CPB = S::CPB;
  __shared__ double sw[2][NRHS][2][CPB * NB];  // two buffers: one barrier per instance
  int c0;
  const SchurSide& R = schur_side<K>(P, c0);
  const int t = threadIdx.x, lc = t / NB, a = t % NB, c = c0 + lc;
  const bool on = lc < CPB && c < R.ncell;
  const size_t nb = (size_t)R.ncell * NB, at = (size_t)c * NB + a;
  const int ax = a % N1, ay = a / N1;
  double bs[2 * NB], bf[2][2 * N1];
  int M[2] = {-1, -1}, fc[2];
  fc[0] = ax == 0 ? 0 : 1;
  fc[1] = ay == 0 ? 2 : 3;
  size_t pm = 0;
  if (on) {
    const double* tb = R.tab + (size_t)R.type[c] * S::TAB + NB * NB + a;
#pragma unroll
    for (int i = 0; i < 2 * NB; ++i) bs[i] = tb[i * NB];
    if (ax == 0 || ax == K) M[0] = R.nbr[4 * (size_t)c + fc[0]];
    if (ay == 0 || ay == K) M[1] = R.nbr[4 * (size_t)c + fc[1]];
#pragma unroll
    for (int e = 0; e < 2; ++e) {
      if (M[e] < 0) continue;
      // the neighbour's block on its side of the face, this node's column
      const double* fb = R.tab + (size_t)R.type[M[e]] * S::TAB + S::FACE + (fc[e] ^ 1) * 2 * N1 * N1 + (e ? ax : ay);
#pragma unroll
      for (int i = 0; i < 2 * N1; ++i) bf[e][i] = fb[i * N1];
    }
    pm = R.perm[at];
  }
  const bool hg = HANG && on && R.hx_all;
  const int h0 = hg ? R.hx_all[c] : 0, h1 = hg ? R.hx_all[c + 1] : 0;
  int buf = 0;
  const int i1 = min(ninst, ((int)blockIdx.y + 1) * per);
  for (int i = blockIdx.y * per; i < i1; ++i, buf ^= 1) {
    double acc[NRHS];
    if (on) {
#pragma unroll
      for (int h = 0; h < NRHS; ++h) {
        const double* w = R.w[h] + i * R.sb;
        sw[buf][h][0][t] = w[at];
        sw[buf][h][1][t] = w[nb + at];
        acc[h] = R.b[h][i * R.sb + 2 * nb + at];
      }
#pragma unroll
      for (int e = 0; e < 2; ++e) {
        if (M[e] < 0) continue;
#pragma unroll
        for (int h = 0; h < NRHS; ++h) {
          const double* wm = R.w[h] + i * R.sb + (size_t)M[e] * NB;
#pragma unroll
          for (int m = 0; m < N1; ++m) {
            const int n = S::node(fc[e] ^ 1, m);
            acc[h] += bf[e][m] * wm[n] + bf[e][N1 + m] * wm[nb + n];
          }
        }
      }
      for (int e = h0; HANG && e < h1; ++e) {  // hanging faces
        const double* B = R.hblk + (size_t)R.hx_blk[e] * 2 * NB * NB + a;
#pragma unroll
        for (int h = 0; h < NRHS; ++h) {
          const double* wm = R.w[h] + i * R.sb + (size_t)R.hx_src[e] * NB;
#pragma unroll
          for (int q = 0; q < NB; ++q) acc[h] += B[q * NB] * wm[q] + B[(NB + q) * NB] * wm[nb + q];
        }
      }
    }
    __syncthreads();
    if (on) {
#pragma unroll
      for (int h = 0; h < NRHS; ++h) {
#pragma unroll
        for (int q = 0; q < NB; ++q)
          acc[h] += bs[q] * sw[buf][h][0][lc * NB + q] + bs[NB + q] * sw[buf][h][1][lc * NB + q];
        R.g[h][i * R.sg + pm] = acc[h];
      }
    }
  }
}

// q = W - mu A^{-1} B u; writes [Jx | Jy | u]
template <int K, int NRHS, bool HANG>
__global__ __launch_bounds__(256, K == 2 && !HANG ? 4 : 1) void k_schur_recover(SchurPair P, int ninst, int per) {
  using S = SchurLane<K>;
  constexpr int NB = S::NB, N1 = S::N1, CPB = S::CPB;
  __shared__ double su[NRHS][CPB * NB], ss[NRHS][2][CPB * NB];
  int c0;
  const SchurSide& R = schur_side<K>(P, c0);
  const int t = threadIdx.x, lc = t / NB, a = t % NB, c = c0 + lc;
  const bool on = lc < CPB && c < R.ncell;
  const size_t nb = (size_t)R.ncell * NB, at = (size_t)c * NB + a;
  const int ax = a % N1, ay = a / N1;
  double mi[NB], bs[2][NB], bf[2][2][N1];
  int M[2] = {-1, -1}, fc[2], pn[2][N1];
  fc[0] = ax == 0 ? 0 : 1;
  fc[1] = ay == 0 ? 2 : 3;
  size_t pm = 0;
  if (on) {
    const double* tb = R.tab + (size_t)R.type[c] * S::TAB;
#pragma unroll
    for (int q = 0; q < NB; ++q) {
      mi[q] = tb[a * NB + q];
      bs[0][q] = tb[NB * NB + a * NB + q];
      bs[1][q] = tb[NB * NB + (NB + a) * NB + q];
    }
    if (ax == 0 || ax == K) M[0] = R.nbr[4 * (size_t)c + fc[0]];
    if (ay == 0 || ay == K) M[1] = R.nbr[4 * (size_t)c + fc[1]];
#pragma unroll
    for (int e = 0; e < 2; ++e) {
      if (M[e] < 0) continue;
      const double* fb = tb + S::FACE + fc[e] * 2 * N1 * N1 + (e ? ax : ay) * N1;
#pragma unroll
      for (int j = 0; j < N1; ++j) {
        bf[e][0][j] = fb[j];
        bf[e][1][j] = fb[N1 * N1 + j];
        pn[e][j] = R.perm[(size_t)M[e] * NB + S::node(fc[e] ^ 1, j)];
      }
    }
    pm = R.perm[at];
  }
  const bool hg = HANG && on && R.hm_all;
  const int h0 = hg ? R.hm_all[c] : 0, h1 = hg ? R.hm_all[c + 1] : 0;
  const int i1 = min(ninst, ((int)blockIdx.y + 1) * per);
  for (int i = blockIdx.y * per; i < i1; ++i) {
    double s0[NRHS], s1[NRHS], w0[NRHS], w1[NRHS];
    if (on) {
#pragma unroll
      for (int h = 0; h < NRHS; ++h) {
        const double u = R.g[h][i * R.sg + pm];
        su[h][t] = u;
        R.o[h][i * R.so + 2 * nb + at] = u;
        w0[h] = R.w[h][i * R.sb + at];
        w1[h] = R.w[h][i * R.sb + nb + at];
        s0[h] = s1[h] = 0.0;
      }
#pragma unroll
      for (int e = 0; e < 2; ++e) {
        if (M[e] < 0) continue;
#pragma unroll
        for (int h = 0; h < NRHS; ++h)
#pragma unroll
          for (int j = 0; j < N1; ++j) {
            const double v = R.g[h][i * R.sg + pn[e][j]];
            s0[h] += bf[e][0][j] * v;
            s1[h] += bf[e][1][j] * v;
          }
      }
      for (int e = h0; HANG && e < h1; ++e) {  // hanging faces
        const int* px = R.perm + (size_t)R.hm_dst[e] * NB;
        const double* B = R.hblk + (size_t)R.hm_blk[e] * 2 * NB * NB + a * NB;
#pragma unroll
        for (int q = 0; q < NB; ++q)
#pragma unroll
          for (int h = 0; h < NRHS; ++h) {
            const double v = R.g[h][i * R.sg + px[q]];
            s0[h] += B[q] * v;
            s1[h] += B[NB * NB + q] * v;
          }
      }
    }
    __syncthreads();
    if (on) {
#pragma unroll
      for (int h = 0; h < NRHS; ++h) {
#pragma unroll
        for (int q = 0; q < NB; ++q) {
          const double v = su[h][lc * NB + q];
          s0[h] += bs[0][q] * v;
          s1[h] += bs[1][q] * v;
        }
        ss[h][0][t] = s0[h];
        ss[h][1][t] = s1[h];
      }
    }
    __syncthreads();
    if (on) {
#pragma unroll
      for (int h = 0; h < NRHS; ++h) {
        double q0 = 0.0, q1 = 0.0;
#pragma unroll
        for (int q = 0; q < NB; ++q) {
          q0 += mi[q] * ss[h][0][lc * NB + q];
          q1 += mi[q] * ss[h][1][lc * NB + q];
        }
        R.o[h][i * R.so + at] = w0[h] - R.mu[h] * q0;
        R.o[h][i * R.so + nb + at] = w1[h] - R.mu[h] * q1;
      }
    }
  }
}

// ------------------------------------------------------------------------
// Mixed precision (FP32 element contractions, FP64 vectors and solves)
// ------------------------------------------------------------------------
// The cell-local contractions with the cell-type tables run in FP32 on an
// FP32 copy of the table, with FP32 accumulation; inputs are read and
// results written in FP64, and the terms that are not contractions (the
// density part f_v of the Schur right-hand side, the difference f - B u
// before the recovery's inverse mass) stay FP64.  Wave-uniform cell lists
// only (planar meshes): the table entries are scalar operands.
template <int K>
__device__ __forceinline__ void schur_rhs_one_f32(const DevRegion& R, const double* __restrict__ b, double mu,
                                                  double* __restrict__ g, int X) {
  constexpr int NB = Sz<K>::NB;
  const size_t nc = R.ncell;
  const float muf = (float)mu;
  float acc[NB];
#pragma unroll
  for (int a = 0; a < NB; ++a) acc[a] = 0.0f;
  for (int f = -1; f < 4; ++f) {
    const int M = f < 0 ? X : R.nbr[4 * (size_t)X + f];
    if (M < 0) continue;
    const int ty = wave_type(R, M);
    const float* Minv = R.table_f + (size_t)ty * R.stride;
    const float* B = Minv + NB * NB + (f < 0 ? 0 : 2 * NB * NB + (f ^ 1) * 2 * NB * NB);
    float fx[NB], fy[NB], w[2 * NB];
#pragma unroll
    for (int a = 0; a < NB; ++a) {
      fx[a] = (float)b[(size_t)M * NB + a];
      fy[a] = (float)b[nc * NB + (size_t)M * NB + a];
    }
#pragma unroll
    for (int a = 0; a < NB; ++a) {
      float sx = 0.0f, sy = 0.0f;
#pragma unroll
      for (int t = 0; t < NB; ++t) {
        sx += Minv[a * NB + t] * fx[t];
        sy += Minv[a * NB + t] * fy[t];
      }
      w[a] = muf * sx;
      w[NB + a] = muf * sy;
    }
    for (int i = 0; i < 2 * NB; ++i) {
#pragma unroll
      for (int a = 0; a < NB; ++a) acc[a] += B[i * NB + a] * w[i];
    }
  }
  const int* __restrict__ pm = R.perm + (size_t)X * NB;
#pragma unroll
  for (int a = 0; a < NB; ++a) g[pm[a]] = b[2 * nc * NB + (size_t)X * NB + a] + (double)acc[a];
}

template <int K, int NRHS>
__global__ __launch_bounds__(64) void k_schur_rhs_f32(DevRegion R, const double* __restrict__ b1,
                                                      const double* __restrict__ b2, double mu1, double mu2,
                                                      double* __restrict__ g1, double* __restrict__ g2, int64_t sb,
                                                      int64_t sg) {
  const int X = schur_cell(R.ucell_nbh, R.nu_nbh, blockIdx.x * blockDim.x + threadIdx.x);
  if (X < 0) return;
  const int64_t i = blockIdx.y;
  schur_rhs_one_f32<K>(R, b1 + i * sb, mu1, g1 + i * sg, X);
  if (NRHS > 1) schur_rhs_one_f32<K>(R, b2 + i * sb, mu2, g2 + i * sg, X);
}

template <int K>
__device__ __forceinline__ void schur_recover_one_f32(const DevRegion& R, const float* tb,
                                                      const double* __restrict__ b, const double* __restrict__ x,
                                                      double mu, double* __restrict__ o, int M) {
  constexpr int NB = Sz<K>::NB;
  const size_t nc = R.ncell;
  float s[2 * NB], u[NB];
  double ud[NB];
  const int* __restrict__ pm = R.perm + (size_t)M * NB;
#pragma unroll
  for (int a = 0; a < NB; ++a) {
    ud[a] = x[pm[a]];
    u[a] = (float)ud[a];
  }
  for (int i = 0; i < 2 * NB; ++i) {
    float t = 0.0f;
#pragma unroll
    for (int a = 0; a < NB; ++a) t += tb[NB * NB + i * NB + a] * u[a];
    s[i] = t;
  }
  for (int f = 0; f < 4; ++f) {
    const int X = R.nbr[4 * (size_t)M + f];
    if (X < 0) continue;
    const int* __restrict__ px = R.perm + (size_t)X * NB;
    float v[NB];
#pragma unroll
    for (int a = 0; a < NB; ++a) v[a] = (float)x[px[a]];
    const float* B = tb + NB * NB + 2 * NB * NB + f * 2 * NB * NB;
    for (int i = 0; i < 2 * NB; ++i) {
      float t = 0.0f;
#pragma unroll
      for (int a = 0; a < NB; ++a) t += B[i * NB + a] * v[a];
      s[i] += t;
    }
  }
  // q = mu A^{-1} (f_q - B u): the difference in FP64, the inverse mass in FP32
  const float muf = (float)mu;
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    float d[NB];
#pragma unroll
    for (int t = 0; t < NB; ++t) d[t] = (float)(b[(size_t)h * nc * NB + (size_t)M * NB + t] - (double)s[h * NB + t]);
#pragma unroll
    for (int a = 0; a < NB; ++a) {
      float t1 = 0.0f;
#pragma unroll
      for (int t = 0; t < NB; ++t) t1 += tb[a * NB + t] * d[t];
      o[(size_t)h * nc * NB + (size_t)M * NB + a] = (double)(muf * t1);
    }
  }
#pragma unroll
  for (int a = 0; a < NB; ++a) o[2 * nc * NB + (size_t)M * NB + a] = ud[a];
}

template <int K, int NRHS>
__global__ __launch_bounds__(64) void k_schur_recover_f32(DevRegion R, const double* __restrict__ b1,
                                                          const double* __restrict__ b2,
                                                          const double* __restrict__ x1,
                                                          const double* __restrict__ x2, double mu1, double mu2,
                                                          double* __restrict__ o1, double* __restrict__ o2,
                                                          int64_t sb, int64_t sx, int64_t so) {
  const int M = schur_cell(R.ucell_own, R.nu_own, blockIdx.x * blockDim.x + threadIdx.x);
  if (M < 0) return;
  const int64_t i = blockIdx.y;
  const float* tb = R.table_f + (size_t)wave_type(R, M) * R.stride;
  schur_recover_one_f32<K>(R, tb, b1 + i * sb, x1 + i * sx, mu1, o1 + i * so, M);
  if (NRHS > 1) schur_recover_one_f32<K>(R, tb, b2 + i * sb, x2 + i * sx, mu2, o2 + i * so, M);
}

// ------------------------------------------------------------------------
// Supernodal triangular solves (S = L L^T), level by level
// ------------------------------------------------------------------------
// One workgroup per tile of rows of one supernode.  The vector the rows are
// dotted with is staged in LDS in chunks of CW entries per right-hand side;
// W lanes share a row (256/W rows per pass), partial sums stay in registers
// across chunks.
//   forward  (FWD): vector t_own (= b_own - updates z owed by descendants,
//                   from k_fwd_gather), rows of [Linv; W21]; outputs
//                   y_own -> Y, z -> Z.
//   backward:       vector [y_own; x at the panel rows], rows
//                   [Linv^T(j, j:) | -W21^T(j, :)]; outputs x_own -> X.
constexpr int CW = 1024;

template <int W>
__device__ __forceinline__ double group_sum(double x) {
#pragma unroll
  for (int o = W / 2; o > 0; o >>= 1) x += __shfl_xor(x, o, W);
  return x;
}

// W lanes per row, 256/W rows per pass, MAXR passes: a tile holds at most
// (256/W) * MAXR rows of one supernode.
template <int W, int MAXR_>
struct SweepShape {
  static constexpr int R = 256 / W;
  static constexpr int MAXR = MAXR_;
  static constexpr int RB = R * MAXR;
};

// forward, part 1: t_p = b_p - sum of the updates z owed to row p, into X.
// Vectors are h-major (b[h n + p]); with two right-hand sides the updates are
// pair-interleaved (Z[2 z + h]), so one 16-byte load fetches both.  L lanes
// per row (L = 1, or 8 on levels with few rows: their rows collect many
// descendants' contributions); the lanes' partial sums are combined by
// shuffles in a fixed order.
template <int L, int NRHS>
__global__ __launch_bounds__(256) void k_fwd_gather(DevFactor F, const int* __restrict__ lrows, int nrow,
                                                    const double* __restrict__ b) {
  const int t = blockIdx.x * blockDim.x + threadIdx.x;
  const int i = t / L, lane = t % L;
  if (i >= nrow) return;  // nrow * L threads: whole L-groups exit together
  const int p = lrows[i];
  const int64_t c1 = F.cptr[p + 1];
  double z0 = 0.0, z1 = 0.0;
  for (int64_t c = F.cptr[p] + lane; c < c1; c += L) {
    if (NRHS == 2) {
      const double2 z = *reinterpret_cast<const double2*>(F.Z + 2 * F.czidx[c]);
      z0 += z.x;
      z1 += z.y;
    } else {
      z0 += F.Z[F.czidx[c]];
    }
  }
#pragma unroll
  for (int o = L / 2; o > 0; o >>= 1) {
    z0 += __shfl_xor(z0, o, L);
    if (NRHS == 2) z1 += __shfl_xor(z1, o, L);
  }
  if (lane == 0) {
    F.X[p] = b[p] - z0;
    if (NRHS == 2) F.X[(int64_t)F.n + p] = b[(int64_t)F.n + p] - z1;
  }
}

// PF: the factor loads of the next pair of positions are issued before this
// pair's products (unconditional loads from clamped positions, masked at use,
// two register sets in turn).  Costlier in registers and issue slots, it
// pays on the levels with few tiles, whose time is the latency of each
// lane's chain of loads; the tuner picks it per level.
template <int NRHS, int W, int MAXR_, bool FWD, bool PF = false>
__global__ __launch_bounds__(256) void k_sweep(DevFactor F, const int4* __restrict__ tiles,
                                               const double* __restrict__ b0, const double* __restrict__ b1,
                                               double* __restrict__ Y0, double* __restrict__ Y1) {
  using SS = SweepShape<W, MAXR_>;
  constexpr int R = SS::R, MAXR = SS::MAXR;
  __shared__ double vec[NRHS][CW];
  const int4 tl = tiles[blockIdx.x];
  const int s = tl.x, row0 = tl.y, nr = tl.z;
  const int ns = F.ns[s], ms = F.ms[s], p0 = F.p0[s];
  const int VL = FWD ? ns : ns + ms;
  const int g = threadIdx.x / W, sl = threadIdx.x % W;
  const double* __restrict__ base = FWD ? F.fwd + F.fwd_off[s] : F.bwd + F.bwd_off[s];
  // The group's MAXR rows are walked together: every column step issues one
  // load per row, so each lane keeps 2*MAXR independent loads in flight and
  // reads each staged vector entry from LDS once for all its rows.  Row q
  // holds vector positions [rs[q], re[q]), its element at position p at
  // base[off[q] + p].
  int64_t off[MAXR];
  int rs[MAXR], re[MAXR];
  int lo = VL, hi = 0;
#pragma unroll
  for (int q = 0; q < MAXR; ++q) {
    const int lr = row0 + g + q * R;
    if (lr < row0 + nr) {
      if (FWD) {
        rs[q] = 0;
        if (lr < ns) {
          off[q] = (int64_t)lr * (lr + 1) / 2;
          re[q] = lr + 1;
        } else {
          off[q] = (int64_t)ns * (ns + 1) / 2 + (int64_t)(lr - ns) * ns;
          re[q] = ns;
        }
      } else {
        off[q] = (int64_t)lr * (ns + ms) - (int64_t)lr * (lr - 1) / 2 - lr;
        rs[q] = lr;
        re[q] = ns + ms;
      }
      lo = min(lo, rs[q]);
      hi = max(hi, re[q]);
    } else {
      off[q] = 0;
      rs[q] = 0;
      re[q] = 0;
    }
  }
  double acc[MAXR][NRHS];
#pragma unroll
  for (int q = 0; q < MAXR; ++q)
#pragma unroll
    for (int h = 0; h < NRHS; ++h) acc[q][h] = 0.0;
  // backward rows start at their own index, so no row of the tile uses
  // positions below row0
  const int tlo = FWD ? 0 : row0;
  for (int c0 = tlo; c0 < VL; c0 += CW) {
    const int cl = min(CW, VL - c0);
    __syncthreads();
    for (int i = threadIdx.x; i < cl; i += 256) {
      const int pos = c0 + i;
      if (FWD) {  // t from X, or straight from the right-hand side b0 (leaf level: nothing to gather)
        const double* __restrict__ xs = b0 ? b0 : F.X;
        vec[0][i] = xs[p0 + pos];
        if (NRHS > 1) vec[NRHS - 1][i] = xs[F.n + p0 + pos];
      } else if (pos < ns) {
        vec[0][i] = Y0[p0 + pos];
        if (NRHS > 1) vec[NRHS - 1][i] = Y1[p0 + pos];
      } else {  // x at the panel rows: rows of ancestors, solved by earlier launches
        const int64_t p = F.rows[F.rows_off[s] + (pos - ns)];
        vec[0][i] = F.X[p];
        if (NRHS > 1) vec[NRHS - 1][i] = F.X[F.n + p];
      }
    }
    __syncthreads();
    const int e = min(hi, c0 + cl);
    if constexpr (PF) {
      auto ld = [&](int p, double (&L)[MAXR]) {
#pragma unroll
        for (int q = 0; q < MAXR; ++q) {
          const int pc = re[q] > rs[q] ? min(max(p, rs[q]), re[q] - 1) : 0;
          L[q] = __builtin_nontemporal_load(base + off[q] + pc);
        }
      };
      auto fma_pair = [&](int pa, const double (&La)[MAXR], const double (&Lb)[MAXR]) {
        const int pb = pa + W;
        const bool okb = pb < e;
        const int ib = okb ? pb - c0 : 0;
        const double va0 = vec[0][pa - c0];
        const double vb0 = okb ? vec[0][ib] : 0.0;
        const double va1 = NRHS > 1 ? vec[NRHS - 1][pa - c0] : 0.0;
        const double vb1 = NRHS > 1 && okb ? vec[NRHS - 1][ib] : 0.0;
#pragma unroll
        for (int q = 0; q < MAXR; ++q) {
          const double a = (pa >= rs[q] && pa < re[q]) ? La[q] : 0.0;
          const double b = (pb >= rs[q] && pb < re[q]) ? Lb[q] : 0.0;
          acc[q][0] += a * va0 + b * vb0;
          if (NRHS > 1) acc[q][NRHS - 1] += a * va1 + b * vb1;
        }
      };
      int pa = max(lo, c0) + sl;
      if (pa < e) {
        double La[MAXR], Lb[MAXR], Ma[MAXR], Mb[MAXR];
        ld(pa, La);
        ld(pa + W, Lb);
        for (; pa < e; pa += 4 * W) {
          ld(pa + 2 * W, Ma);
          ld(pa + 3 * W, Mb);
          __builtin_amdgcn_sched_barrier(0);
          fma_pair(pa, La, Lb);
          __builtin_amdgcn_sched_barrier(0);
          ld(pa + 4 * W, La);
          ld(pa + 5 * W, Lb);
          __builtin_amdgcn_sched_barrier(0);
          if (pa + 2 * W < e) fma_pair(pa + 2 * W, Ma, Mb);
          __builtin_amdgcn_sched_barrier(0);
        }
      }
      continue;
    }
    for (int pa = max(lo, c0) + sl; pa < e; pa += 2 * W) {
      const int pb = pa + W;
      const bool okb = pb < e;
      double La[MAXR], Lb[MAXR];
#pragma unroll
      for (int q = 0; q < MAXR; ++q) {
        La[q] = (pa >= rs[q] && pa < re[q]) ? __builtin_nontemporal_load(base + off[q] + pa) : 0.0;
        Lb[q] = (okb && pb >= rs[q] && pb < re[q]) ? __builtin_nontemporal_load(base + off[q] + pb) : 0.0;
      }
      const double va0 = vec[0][pa - c0];
      const double vb0 = okb ? vec[0][pb - c0] : 0.0;
#pragma unroll
      for (int q = 0; q < MAXR; ++q) acc[q][0] += La[q] * va0 + Lb[q] * vb0;
      if (NRHS > 1) {
        const double va1 = vec[NRHS - 1][pa - c0];
        const double vb1 = okb ? vec[NRHS - 1][pb - c0] : 0.0;
#pragma unroll
        for (int q = 0; q < MAXR; ++q) acc[q][NRHS - 1] += La[q] * va1 + Lb[q] * vb1;
      }
    }
  }
#pragma unroll
  for (int q = 0; q < MAXR; ++q) {
    const int lr = row0 + g + q * R;
    double r0 = group_sum<W>(acc[q][0]);
    double r1 = (NRHS > 1) ? group_sum<W>(acc[q][NRHS - 1]) : 0.0;
    if (lr >= row0 + nr || sl != 0) continue;
    if (FWD) {
      if (lr < ns) {
        Y0[p0 + lr] = r0;
        if (NRHS > 1) Y1[p0 + lr] = r1;
      } else {
        const int64_t z = F.z_off[s] + (lr - ns);
        if (NRHS > 1) {
          *reinterpret_cast<double2*>(F.Z + 2 * z) = double2{r0, r1};
        } else {
          F.Z[z] = r0;
        }
      }
    } else {
      F.X[p0 + lr] = r0;
      if (NRHS > 1) F.X[F.n + p0 + lr] = r1;
    }
  }
}

// Many right-hand sides (a batch of instances sharing the factor): the row
// tile times the vector block is a skinny GEMM, done with FP64 MFMA
// (v_mfma_f64_16x16x4f64).  These solves keep their vectors RHS-interleaved
// (entry p of right-hand side h at [p * NRP + h], NRP = 16 or 32 padded
// right-hand sides, the padding zero), so the B operand of a 16-column step is
// four 128-byte rows straight from L2: no LDS staging and no barriers.  Each
// wave owns MB blocks of 16 rows; per step a lane loads 4 consecutive entries
// of one row (lane l: row l%16, columns 4(l/16)..4(l/16)+3) and issues 4 MFMAs
// whose B operand holds the vector at the same columns (lane l: column
// 4(l/16)+e, right-hand side l%16), so the k order of A and B agree.
// Accumulator lane l, register r holds row l/16 + 4r, right-hand side l%16.
// The interleaved vectors from and to one vector per right-hand side (entry
// p of right-hand side h at [h * n + p]): a tile of IL_TP rows passes through
// LDS, so that the per-right-hand-side side moves IL_TP consecutive rows
// (256 bytes) per wave access and the interleaved side whole rows of NRP
// entries.  The padding columns (h >= nrhs) are written as zeros.
constexpr int IL_TP = 32;

template <int NRP>
__global__ __launch_bounds__(256) void k_pack_il(DevFactor F, const double* __restrict__ v, int nrhs, int pb, int pe) {
  __shared__ double s[NRP * (IL_TP + 1)];
  const int64_t n = F.n, p0 = pb + (int64_t)blockIdx.x * IL_TP;
  for (int e = threadIdx.x; e < NRP * IL_TP; e += 256) {
    const int h = e / IL_TP, pp = e % IL_TP;
    s[h * (IL_TP + 1) + pp] = (h < nrhs && p0 + pp < pe) ? v[(int64_t)h * n + p0 + pp] : 0.0;
  }
  __syncthreads();
  for (int e = threadIdx.x; e < IL_TP * NRP / 2; e += 256) {
    const int pp = e / (NRP / 2), h = 2 * (e % (NRP / 2));
    if (p0 + pp < pe)
      *reinterpret_cast<double2*>(F.X + (p0 + pp) * NRP + h) =
          double2{s[h * (IL_TP + 1) + pp], s[(h + 1) * (IL_TP + 1) + pp]};
  }
}

template <int NRP>
__global__ __launch_bounds__(256) void k_unpack_il(DevFactor F, double* __restrict__ v, int nrhs, int pb, int pe) {
  __shared__ double s[NRP * (IL_TP + 1)];
  const int64_t n = F.n, p0 = pb + (int64_t)blockIdx.x * IL_TP;
  for (int e = threadIdx.x; e < IL_TP * NRP / 2; e += 256) {
    const int pp = e / (NRP / 2), h = 2 * (e % (NRP / 2));
    if (p0 + pp < pe) {
      const double2 x = *reinterpret_cast<const double2*>(F.X + (p0 + pp) * NRP + h);
      s[h * (IL_TP + 1) + pp] = x.x;
      s[(h + 1) * (IL_TP + 1) + pp] = x.y;
    }
  }
  __syncthreads();
  for (int e = threadIdx.x; e < nrhs * IL_TP; e += 256) {
    const int h = e / IL_TP, pp = e % IL_TP;
    if (p0 + pp < pe) v[(int64_t)h * n + p0 + pp] = s[h * (IL_TP + 1) + pp];
  }
}

// t_p = b_p - sum of the updates z owed to row p, in place on the packed
// right-hand sides (X holds b on entry; rows owed nothing are left alone).
// A thread takes two adjacent right-hand sides (16-byte loads and stores).
template <int NRP>
__global__ __launch_bounds__(256) void k_fwd_gather_il(DevFactor F, const int* __restrict__ lrows, int nrow,
                                                       int nrhs) {
  constexpr int NP = NRP / 2;
  const int64_t e = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  if (e >= (int64_t)nrow * NP) return;
  const int i = (int)(e / NP), h = 2 * (int)(e % NP);
  const int p = lrows[i];
  const int64_t c0 = F.cptr[p], c1 = F.cptr[p + 1];
  if (c0 == c1 || h >= nrhs) return;
  double2* x = reinterpret_cast<double2*>(F.X + (int64_t)p * NRP + h);
  double2 a = *x;
  // four contributions' loads in flight at a time, subtracted in order
  int64_t c = c0;
  for (; c + 4 <= c1; c += 4) {
    double2 z[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) z[u] = *reinterpret_cast<const double2*>(F.Z + F.czidx[c + u] * NRP + h);
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      a.x -= z[u].x;
      a.y -= z[u].y;
    }
  }
  for (; c < c1; ++c) {
    const double2 z = *reinterpret_cast<const double2*>(F.Z + F.czidx[c] * NRP + h);
    a.x -= z.x;
    a.y -= z.y;
  }
  if (h + 1 >= nrhs) a.y = 0.0;
  *x = a;
}

template <int NRP>
__global__ __launch_bounds__(256) void k_bwd_gather_il(DevFactor F, const int64_t* __restrict__ idx, int nidx) {
  constexpr int NP = NRP / 2;
  const int64_t e = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  if (e >= (int64_t)nidx * NP) return;
  const int i = (int)(e / NP), h = 2 * (int)(e % NP);
  const int64_t q = idx[i];
  *reinterpret_cast<double2*>(F.Z + q * NRP + h) =
      *reinterpret_cast<const double2*>(F.X + (int64_t)F.rows[q] * NRP + h);
}

// ks > 0: the tile is column segment tl.w (columns [tl.w ks, (tl.w + 1) ks))
// of its row tile and writes its partial sums to Part (slot tbase + tile, rows
// relative to row0, 64 MB rows per slot); k_sweep_reduce adds the segments.
// Single-block tiles (MB = 1) with up to 32 right-hand sides ask for 4 waves
// per SIMD: the forward sweep then fits its accumulators in the VGPRs (111,
// no spills) instead of taking 130 registers with AGPRs, which allowed only 3
// waves; the backward sweep goes from 4 to 5 waves the same way.  With 64 or
// 128 right-hand sides the accumulators (NRP / 4 doubles per block) and the
// double-buffered vector operands need the full register file.
// HPW < NRP / 16 splits the right-hand-side groups of a row block over
// NRP / 16 / HPW waves (each loads the row block's factor and its own groups'
// vector entries): a workgroup then covers 64 MB HPW 16 / NRP rows, with
// fewer registers per wave and so more waves in flight.
constexpr int mfma_waves_per_eu(int nrp, int mb, int hpw) {
  if (hpw == nrp / 16) return mb == 1 && nrp <= 32 ? 4 : 1;
  return hpw == 1 ? (mb == 1 ? 6 : mb == 2 ? 4 : 2) : (mb == 4 ? 2 : 1);
}

// Workgroups are dispatched to the 8 XCDs round-robin (workgroup b to XCD
// b % 8), each XCD with its own L2.  Tile of workgroup b such that every XCD
// takes a contiguous run of the tile list: the tiles of one node (which
// stage the same vector rows) then share an L2.  A bijection on [0, n).
__device__ __forceinline__ int xcd_tile(int b, int n) {
  const int q = n / 8, r = n % 8, x = b % 8;
  return x * q + min(x, r) + b / 8;
}

template <int NRP, int MB, bool FWD, int HPW = NRP / 16>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(mfma_waves_per_eu(NRP, MB, HPW)))) void k_sweep_mfma(
    DevFactor F, const int4* __restrict__ tiles, double* __restrict__ Y, int ks, double* __restrict__ Part, int tbase) {
  constexpr int NH = HPW;                  // right-hand-side groups of this wave
  constexpr int WPR = NRP / 16 / HPW;      // waves per row block
  static_assert(WPR >= 1 && 4 % WPR == 0, "a row block's waves must divide the workgroup");
  const int ti = xcd_tile(blockIdx.x, gridDim.x);
  const int4 tl = tiles[ti];
  const int s = tl.x, row0 = tl.y, nr = tl.z;  // row0 is a multiple of 16
  const int ns = F.ns[s], ms = F.ms[s], p0 = F.p0[s];
  const int VL = FWD ? ns : ns + ms;
  // the wave index through readfirstlane: everything derived from it (rows,
  // column range, step count) is then scalar and the step loop's control flow
  // is uniform, so the compiler counts outstanding loads exactly
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
  const int ri = lane & 15, kq = lane >> 4;
  const int hg0 = (wave % WPR) * HPW;                    // this wave's first right-hand-side group
  const int first = row0 + (wave / WPR) * MB * 16;       // wave-uniform
  if (first >= row0 + nr) return;                        // no rows for this wave (no barriers below)
  const int last = min(row0 + nr, first + MB * 16) - 1;
  const int lo = FWD ? 0 : first;
  const int hi = FWD ? (last < ns ? last + 1 : ns) : ns + ms;
  // the wave's blocks in the MFMA-blocked copy: data base, first column, steps
  const double* __restrict__ blk = FWD ? F.fblk : F.bblk;
  const int64_t* __restrict__ boff = FWD ? F.fblk_off : F.bblk_off;
  const int bnode = FWD ? F.fblk0[s] : F.bblk0[s];
  int64_t bbase[MB];
  int bclo[MB], bsteps[MB];
#pragma unroll
  for (int mb = 0; mb < MB; ++mb) {
    const int b = first / 16 + mb;
    bbase[mb] = 0;
    bclo[mb] = 0;
    bsteps[mb] = 0;
    if (first + mb * 16 < row0 + nr) {
      bbase[mb] = boff[bnode + b];
      bclo[mb] = FWD ? 0 : 16 * b;
      bsteps[mb] = (int)((boff[bnode + b + 1] - bbase[mb]) >> 8);
    }
  }
  v4d acc[MB][NH];
#pragma unroll
  for (int mb = 0; mb < MB; ++mb)
#pragma unroll
    for (int hg = 0; hg < NH; ++hg) acc[mb][hg] = v4d{0.0, 0.0, 0.0, 0.0};
  // vector entry at column col of right-hand side h (interleaved storage).
  // Columns past the rows' last one (col >= VL, in the last step) read the
  // last column's entry instead: the factor's entries there are zero and the
  // vector entries are finite, so the products vanish.  The loads then carry
  // no per-lane branch, and the compiler issues them back to back instead of
  // waiting on each one to select between it and zero.
  const int64_t zrow = FWD ? 0 : F.rows_off[s] - ns;
  auto vecv = [&](int col, int h) -> double {
    const int c = min(col, VL - 1);
    if (FWD) return F.X[(int64_t)(p0 + c) * NRP + h];
    const double* src = c < ns ? Y + (int64_t)(p0 + c) * NRP : F.Z + (zrow + c) * NRP;
    return src[h];
  };
  int c0 = (lo >> 4) << 4, cend = hi;
  if (ks > 0) {  // this tile's column segment (ks and the segment start are multiples of 16)
    c0 = max(c0, tl.w * ks);
    cend = min(cend, (tl.w + 1) * ks);
  }
  const int nstep = cend > c0 ? (cend - c0 + 15) >> 4 : 0;
  // Step st's operands.  Every load is unconditional: a block outside its
  // stored columns at this step (only with MB > 1) loads its nearest stored
  // step and is masked to zero where the MFMA uses it (inb), so no load waits
  // behind a select.
  auto load = [&](int st, double (&L)[MB][4], double (&Bv)[4][NH], bool (&inb)[MB]) {
    const int cc = c0 + 16 * st;
#pragma unroll
    for (int mb = 0; mb < MB; ++mb) {
      const int idx = (cc - bclo[mb]) >> 4;  // the block's own step (wave-uniform)
      inb[mb] = cc >= bclo[mb] && idx < bsteps[mb];
      // a block past the tile's rows (bsteps 0) reads block 0's first step,
      // which exists: the wave has rows, so block 0 has at least one step
      const int ic = min(max(idx, 0), max(bsteps[mb] - 1, 0));
      const double* src = blk + (bsteps[mb] > 0 ? bbase[mb] + (int64_t)ic * 256 : bbase[0]) + lane;
#pragma unroll
      for (int q = 0; q < 4; ++q) L[mb][q] = __builtin_nontemporal_load(src + q * 64);
    }
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const int col = cc + 4 * kq + q;
#pragma unroll
      for (int hg = 0; hg < NH; ++hg) Bv[q][hg] = vecv(col, (hg0 + hg) * 16 + ri);
    }
  };
  auto mma = [&](const double (&L)[MB][4], const double (&Bv)[4][NH], const bool (&inb)[MB]) {
#pragma unroll
    for (int q = 0; q < 4; ++q)
#pragma unroll
      for (int hg = 0; hg < NH; ++hg)
#pragma unroll
        for (int mb = 0; mb < MB; ++mb)
          acc[mb][hg] = __builtin_amdgcn_mfma_f64_16x16x4f64(MB == 1 || inb[mb] ? L[mb][q] : 0.0, Bv[q][hg],
                                                             acc[mb][hg], 0, 0, 0);
  };
  // loads run one step ahead of the MFMAs that use them (two register sets);
  // past the last step they repeat it (unused), so the loop body has no
  // conditional loads
  double LA[MB][4], LB[MB][4], BA[4][NH], BB[4][NH];
  bool IA[MB], IB[MB];
  // (sched_barrier keeps each step's loads ahead of the previous step's MFMAs:
  // left alone, the scheduler sinks them next to their use)
  if (nstep > 0) {
    load(0, LA, BA, IA);
    for (int st = 0; st < nstep; st += 2) {
      load(min(st + 1, nstep - 1), LB, BB, IB);
      __builtin_amdgcn_sched_barrier(0);
      mma(LA, BA, IA);
      __builtin_amdgcn_sched_barrier(0);
      load(min(st + 2, nstep - 1), LA, BA, IA);
      __builtin_amdgcn_sched_barrier(0);
      if (st + 1 < nstep) mma(LB, BB, IB);
      __builtin_amdgcn_sched_barrier(0);
    }
  }
#pragma unroll
  for (int mb = 0; mb < MB; ++mb)
#pragma unroll
    for (int hg = 0; hg < NH; ++hg)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int lr = first + mb * 16 + kq + 4 * r;
        const int h = (hg0 + hg) * 16 + ri;
        if (lr >= row0 + nr) continue;
        const double v = acc[mb][hg][r];
        if (ks > 0) {
          Part[((int64_t)(tbase + ti) * (64 * MB) + (lr - row0)) * NRP + h] = v;
        } else if (FWD) {
          if (lr < ns) Y[(int64_t)(p0 + lr) * NRP + h] = v;
          else F.Z[(F.z_off[s] + (lr - ns)) * NRP + h] = v;
        } else {
          F.X[(int64_t)(p0 + lr) * NRP + h] = v;
        }
      }
}

// The MFMA sweep with the vector operand staged in LDS once per workgroup:
// its 4 waves each own MBL consecutive 16-row blocks of the tile (64 MBL
// rows) and all right-hand-side groups, and step through the union of their
// column ranges together.  Per 16-column step the workgroup loads the step's
// 16 x NRP vector entries once (NRP / 16 per thread, 16-byte pieces), stores them
// in LDS and every wave reads its B operands there, each B operand serving
// the wave's MBL blocks: the vector bytes leaving L2 drop to 1 / (4 MBL) of
// per-block loads.  The next step's vector entries (and the factor operands
// of the step after it) are loaded into registers while this step's MFMAs
// run, with one barrier per step (double-buffered LDS).  The tile order is
// XCD-aware (xcd_tile).  A
// block contributes zero on steps outside its stored columns (masked factor
// operand), and a wave skips the steps none of its blocks stores (wave-uniform
// through readfirstlane); a wave without rows still loads, stores and meets
// every barrier.
template <int NRP, bool FWD, int MBL>
__global__ __launch_bounds__(256) void k_sweep_mfma_lds(DevFactor F, const int4* __restrict__ tiles,
                                                        double* __restrict__ Y, int ks,
                                                        double* __restrict__ Part, int tbase) {
  constexpr int NH = NRP / 16;
  constexpr int S = NRP + 4;   // LDS row stride (doubles): the 4 column groups of a read fall in 2 bank halves
  constexpr int K = NRP / 16;  // staged entries per thread per step
  __shared__ __align__(16) double sB[2][16 * S];
  const int ti = xcd_tile(blockIdx.x, gridDim.x);
  const int4 tl = tiles[ti];
  const int s = tl.x, row0 = tl.y, nr = tl.z;  // row0 is a multiple of 16
  const int ns = F.ns[s], ms = F.ms[s], p0 = F.p0[s];
  const int VL = FWD ? ns : ns + ms;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
  const int ri = lane & 15, kq = lane >> 4;
  const int first = row0 + wave * 16 * MBL;
  const int last_t = row0 + nr - 1;  // the tile's last row
  // the workgroup's column range (the union of its blocks')
  const int lo = FWD ? 0 : row0;
  const int hi = FWD ? (last_t < ns ? last_t + 1 : ns) : ns + ms;
  int c0 = (lo >> 4) << 4, cend = hi;
  if (ks > 0) {
    c0 = max(c0, tl.w * ks);
    cend = min(cend, (tl.w + 1) * ks);
  }
  const int nstep = cend > c0 ? (cend - c0 + 15) >> 4 : 0;
  // this wave's blocks in the MFMA-blocked copy
  const double* __restrict__ blk = FWD ? F.fblk : F.bblk;
  const int64_t* __restrict__ boff = FWD ? F.fblk_off : F.bblk_off;
  const int bnode = FWD ? F.fblk0[s] : F.bblk0[s];
  bool rows[MBL];
  int64_t bbase[MBL];
  int bclo[MBL], bsteps[MBL];
#pragma unroll
  for (int j = 0; j < MBL; ++j) {
    const int b = first / 16 + j;
    rows[j] = first + 16 * j < row0 + nr;  // wave-uniform
    bbase[j] = rows[j] ? boff[bnode + b] : boff[bnode];
    bclo[j] = rows[j] ? (FWD ? 0 : 16 * b) : 0;
    bsteps[j] = rows[j] ? (int)((boff[bnode + b + 1] - bbase[j]) >> 8) : 0;
  }
  const int64_t zrow = FWD ? 0 : F.rows_off[s] - ns;
  // staged entries of thread t at step st: column c = t / 16 of the step,
  // right-hand-side pairs 2 (t % 16) + 32 jj (jj < K / 2), so that each
  // 16-lane group moves 256 contiguous bytes per instruction, from the
  // interleaved vector and into LDS (no bank conflicts on the stores); past
  // the rows' last column the last column's entries (finite; the factor is
  // zero there).  The backward sweep reads its panel columns (the
  // ancestors' rows, solved by earlier launches) straight from x through the
  // row index: no gathered copy.
  const int sc = threadIdx.x >> 4, sl = 2 * (threadIdx.x & 15);
  auto stage_load = [&](int st, double (&R)[K]) {
    const int col = min(c0 + 16 * st + sc, VL - 1);
    const double* src;
    if (FWD) src = F.X + (int64_t)(p0 + col) * NRP + sl;
    else src = col < ns ? Y + (int64_t)(p0 + col) * NRP + sl : F.X + (int64_t)F.rows[zrow + col] * NRP + sl;
#pragma unroll
    for (int j = 0; j < K; j += 2) {
      const double2 v = *reinterpret_cast<const double2*>(src + 16 * j);
      R[j] = v.x;
      R[j + 1] = v.y;
    }
  };
  auto stage_store = [&](int buf, const double (&R)[K]) {
#pragma unroll
    for (int j = 0; j < K; j += 2)
      *reinterpret_cast<double2*>(&sB[buf][sc * S + sl + 16 * j]) = double2{R[j], R[j + 1]};
  };
  // the factor operands of step st (clamped into each block's stored steps;
  // in[j] = whether the step is one of block j's, wave-uniform)
  auto a_load = [&](int st, double (&L)[MBL][4], int (&in)[MBL]) {
#pragma unroll
    for (int j = 0; j < MBL; ++j) {
      const int idx = (c0 + 16 * st - bclo[j]) >> 4;
      in[j] = __builtin_amdgcn_readfirstlane((int)(rows[j] && idx >= 0 && idx < bsteps[j]));
      const int ic = min(max(idx, 0), max(bsteps[j] - 1, 0));
      const double* src = blk + bbase[j] + (int64_t)ic * 256 + lane;
      // (a block without rows reads its node's first block: a valid
      // address, skipped by in)
#pragma unroll
      for (int q = 0; q < 4; ++q) L[j][q] = __builtin_nontemporal_load(src + q * 64);
    }
  };
  v4d acc[MBL][NH];
#pragma unroll
  for (int j = 0; j < MBL; ++j)
#pragma unroll
    for (int hg = 0; hg < NH; ++hg) acc[j][hg] = v4d{0.0, 0.0, 0.0, 0.0};
  auto mma = [&](int buf, const double (&L)[MBL][4], const int (&in)[MBL]) {
    int any = 0;
#pragma unroll
    for (int j = 0; j < MBL; ++j) any |= in[j];
    if (!any) return;
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const double* row = &sB[buf][(4 * kq + q) * S + ri];
#pragma unroll
      for (int hg = 0; hg < NH; ++hg) {
        const double bv = row[hg * 16];
#pragma unroll
        for (int j = 0; j < MBL; ++j)
          acc[j][hg] = __builtin_amdgcn_mfma_f64_16x16x4f64(in[j] ? L[j][q] : 0.0, bv, acc[j][hg], 0, 0, 0);
      }
    }
  };
  if (nstep > 0) {
    // the factor operands are loaded two steps ahead, into three register
    // sets that rotate (step s uses set s % 3 and loads step s + 2 into the
    // set step s - 1 used); the staged vector one step ahead, through the
    // two LDS buffers (step s reads buffer s % 2)
    double R[K], LA[MBL][4], LB[MBL][4], LC[MBL][4];
    int IA[MBL], IB[MBL], IC[MBL];
    auto step = [&](int st, int buf, const double (&Lu)[MBL][4], const int (&Iu)[MBL], double (&Ln)[MBL][4],
                    int (&In)[MBL]) {
      stage_load(min(st + 1, nstep - 1), R);
      a_load(min(st + 2, nstep - 1), Ln, In);
      __builtin_amdgcn_sched_barrier(0);
      mma(buf, Lu, Iu);
      __builtin_amdgcn_sched_barrier(0);
      if (st + 1 < nstep) stage_store(buf ^ 1, R);
      __syncthreads();
      return st + 1 < nstep;
    };
    stage_load(0, R);
    a_load(0, LA, IA);
    a_load(min(1, nstep - 1), LB, IB);
    stage_store(0, R);
    __syncthreads();
    for (int st = 0;; st += 6) {
      if (!step(st, 0, LA, IA, LC, IC)) break;
      if (!step(st + 1, 1, LB, IB, LA, IA)) break;
      if (!step(st + 2, 0, LC, IC, LB, IB)) break;
      if (!step(st + 3, 1, LA, IA, LC, IC)) break;
      if (!step(st + 4, 0, LB, IB, LA, IA)) break;
      if (!step(st + 5, 1, LC, IC, LB, IB)) break;
    }
  }
#pragma unroll
  for (int j = 0; j < MBL; ++j) {
    if (!rows[j]) continue;  // after the last barrier
#pragma unroll
    for (int hg = 0; hg < NH; ++hg)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int lr = first + 16 * j + kq + 4 * r;
        const int h = hg * 16 + ri;
        if (lr >= row0 + nr) continue;
        const double v = acc[j][hg][r];
        if (ks > 0) {
          Part[((int64_t)(tbase + ti) * (64 * MBL) + (lr - row0)) * NRP + h] = v;
        } else if (FWD) {
          if (lr < ns) Y[(int64_t)(p0 + lr) * NRP + h] = v;
          else F.Z[(F.z_off[s] + (lr - ns)) * NRP + h] = v;
        } else {
          F.X[(int64_t)(p0 + lr) * NRP + h] = v;
        }
      }
  }
}

// workgroups per row tile in k_sweep_reduce (a level has a few hundred split
// row tiles: one workgroup each would leave most SIMDs idle)
constexpr int REDUCE_SPLIT = 8;

// Sum of the column segments of split row tiles, in segment order: row tile
// rt = (node, row0, nrows, 64 * first tile + nseg); partial sums of tile t at
// Part[(t * cap + r) * NRP + h] (cap = 64 MB rows per slot).
template <int NRP, bool FWD>
__global__ __launch_bounds__(256) void k_sweep_reduce(DevFactor F, const int4* __restrict__ rtiles, int cap,
                                                      const double* __restrict__ Part, double* __restrict__ Y) {
  const int4 rt = rtiles[blockIdx.x];
  const int s = rt.x, row0 = rt.y, nr = rt.z, t0 = rt.w >> 6, nseg = rt.w & 63;
  const int ns = F.ns[s], p0 = F.p0[s];
  // gridDim.y workgroups share a row tile's entries; each entry's segments
  // are added in segment order, four loads in flight at a time
  for (int e = blockIdx.y * blockDim.x + threadIdx.x; e < nr * NRP; e += gridDim.y * blockDim.x) {
    const int r = e / NRP, h = e % NRP;
    const double* pp = Part + ((int64_t)t0 * cap + r) * NRP + h;
    const int64_t seg = (int64_t)cap * NRP;
    double v = 0.0;
    int k = 0;
    for (; k + 4 <= nseg; k += 4) {
      double q[4];
#pragma unroll
      for (int u = 0; u < 4; ++u) q[u] = pp[(k + u) * seg];
#pragma unroll
      for (int u = 0; u < 4; ++u) v += q[u];
    }
    for (; k < nseg; ++k) v += pp[k * seg];
    const int lr = row0 + r;
    if (FWD) {
      if (lr < ns) Y[(int64_t)(p0 + lr) * NRP + h] = v;
      else F.Z[(F.z_off[s] + (lr - ns)) * NRP + h] = v;
    } else {
      F.X[(int64_t)(p0 + lr) * NRP + h] = v;
    }
  }
}

// ------------------------------------------------------------------------
// Hybridised mixed Poisson
// ------------------------------------------------------------------------
template <int K>
__device__ __forceinline__ void poisson_fphi(const DevPoisson& P, const DevTabs& T, const DevPhys& ph, int Kc,
                                             const double* un, const double* up, const double* ur,
                                             const double* uo, int ncs, int nce, double* fphi) {
  using S = Sz<K>;
  constexpr int NB = S::NB, NQ = S::NQ, NPHI = S::NPHI;
  const bool semi = Kc < ncs;
  const int c = semi ? Kc : Kc - ncs;
  const int nc = semi ? ncs : nce;
  const double* u1 = semi ? un : ur;
  const double* u2 = semi ? up : uo;
  const double rho0 = semi ? (ph.ne - ph.pe) : 0.0;  // N_D - N_A (SolarCell.cpp:542-548)
  double v[8];
#pragma unroll
  for (int t = 0; t < 8; ++t) v[t] = P.V[8 * (size_t)Kc + t];
  double d1[NB], d2[NB];
  const size_t ub = 2 * (size_t)nc * NB + (size_t)c * NB;
#pragma unroll
  for (int a = 0; a < NB; ++a) {
    d1[a] = u1[ub + a];
    d2[a] = u2[ub + a];
  }
#pragma unroll
  for (int l = 0; l < NPHI; ++l) fphi[l] = 0.0;
  for (int q = 0; q < NQ; ++q) {
    const GeoD g = bilin(v, T.qx[q], T.qy[q]);
    const double jxw = T.qw[q] * g.det;
    double n1 = 0.0, n2 = 0.0;
#pragma unroll
    for (int a = 0; a < NB; ++a) {
      n1 += d1[a] * T.phi[a * NQ + q];
      n2 += d2[a] * T.phi[a * NQ + q];
    }
    double rho = rho0 + (-1.0 * n1 + 1.0 * n2);
    if (P.msrc) rho += P.msrc[(size_t)Kc * NQ + q];
#pragma unroll
    for (int l = 0; l < NPHI; ++l) fphi[l] -= T.phiP[l * NQ + q] * rho * jxw;
  }
}

// constant Dirichlet / Schottky data of D row i from the cell's unit parts
template <int K>
__device__ __forceinline__ double poisson_bias(const double* tb, const DevPhys& ph, int i) {
  constexpr int NL = Sz<K>::NL, NRT = Sz<K>::NRT;
  const double* U = tb + NL * NL;
  return ph.phi_bi * U[i] - ph.phi_app * U[NRT + i] - ph.phi_sch * U[2 * NRT + i];
}

// D rows of the cell's right-hand side from manufactured Dirichlet data:
// -<psi_i . n, g> over its Dirichlet faces (the same integral as the unit
// bias parts, with g given at the face points)
template <int K>
__device__ __forceinline__ void poisson_mdir(const DevPoisson& P, const DevTabs& T, int Kc, double* f) {
  constexpr int NRT = Sz<K>::NRT, NF = Sz<K>::NF;
  double v[8];
#pragma unroll
  for (int t = 0; t < 8; ++t) v[t] = P.V[8 * (size_t)Kc + t];
  for (int fc = 0; fc < 4; ++fc) {
    if (P.pbid[4 * (size_t)Kc + fc] != 1) continue;  // Dirichlet faces only
    double nx, ny, len;
    face_nrm(v, fc, nx, ny, len);
    for (int q = 0; q < NF; ++q) {
      const double s = T.fs[q];
      const double xi = fc == 0 ? 0.0 : fc == 1 ? 1.0 : s, eta = fc == 2 ? 0.0 : fc == 3 ? 1.0 : s;
      const GeoD g = bilin(v, xi, eta);
      const double w = -P.mdir[(4 * (size_t)Kc + fc) * NF + q] * T.fw[q] * len;
#pragma unroll
      for (int i = 0; i < NRT; ++i) {
        const double hx = T.fpsix[(fc * NRT + i) * NF + q], hy = T.fpsiy[(fc * NRT + i) * NF + q];
        f[i] += ((g.J00 * hx + g.J01 * hy) * nx + (g.J10 * hx + g.J11 * hy) * ny) / g.det * w;
      }
    }
  }
}

// face DoF ownership for the continuous D layout: left/bottom faces belong to
// the cell; right/top faces only on the right/top boundary.
template <int K>
__device__ __forceinline__ int face_of_local(int i, int& m) {
  constexpr int NRTX = Sz<K>::NRTX;
  if (i < NRTX) {
    const int a = i % (K + 1), b = i / (K + 1);
    m = b;
    if (a == 0) return 0;
    if (a == K) return 1;
    return -1;
  }
  const int ii = i - NRTX, a = ii % K, b = ii / K;
  m = a;
  if (b == 0) return 2;
  if (b == K) return 3;
  return -1;
}

template <int K>
__device__ __forceinline__ bool owns_face(const DevPoisson& P, int Kc, int f) {
  return (P.own[Kc] >> f) & 1;
}

// y = A^{-1} f of cells whose f is in LDS, or (assemble) f into the global
// right-hand side
template <int K, int IG, int NC>
__device__ __forceinline__ void poisson_store(const DevPoisson& P, const double (&sf)[IG][NC][Sz<K>::NL], int c0, int i0,
                                              int ninst, double* __restrict__ y, int64_t sy, int assemble) {
  constexpr int NL = Sz<K>::NL, NRT = Sz<K>::NRT;
  for (int e = threadIdx.x; e < NC * NL; e += 256) {
    const int i = e % NL, lc = e / NL, Kc = c0 + lc;
    if (Kc >= P.ncell) break;
    if (assemble) {
      int m;
      const int fc = i < NRT ? face_of_local<K>(i, m) : -1;
      if (fc < 0 || owns_face<K>(P, Kc, fc)) y[P.idx[(size_t)Kc * NL + i]] = sf[0][lc][i];
      continue;
    }
    const double* __restrict__ tb = P.tab_t + (size_t)P.type[Kc] * NL * NL + i;
    double s[IG];
#pragma unroll
    for (int g = 0; g < IG; ++g) s[g] = 0.0;
#pragma unroll
    for (int j = 0; j < NL; ++j) {
      const double a = tb[j * NL];
#pragma unroll
      for (int g = 0; g < IG; ++g) s[g] += a * sf[g][lc][j];
    }
#pragma unroll
    for (int g = 0; g < IG; ++g)
      if (i0 + g < ninst) y[(i0 + g) * sy + (size_t)Kc * NL + i] = s[g];
  }
}

// Cell right-hand side f (D rows: bias data; Phi rows: -<phi, rho>) and, unless
// `assemble`, its condensation y = A^{-1} f (into y); assemble: f itself into
// the global right-hand side y.  A wave takes 16 cells of one instance: the
// charge at the quadrature points and its moments are FP64 MFMA products, as in
// k_rhs_carrier; then a thread takes a (cell, row) and applies A^{-1} from LDS,
// its table row (A^{-1} transposed: coalesced over the rows) for all IG
// instances.  IG 4: 16 cells of 4 instances per workgroup, else 64 cells.
// One thread per cell took 26 us at refinement 8, k = 2 and 20 us at
// refinement 4, k = 3.
template <int K, int IG>
__global__ __launch_bounds__(256) void k_poisson_cell(DevPoisson P, DevTabs T, const DevPhys* __restrict__ phs,
                                                      const double* __restrict__ un, const double* __restrict__ up,
                                                      const double* __restrict__ ur, const double* __restrict__ uo,
                                                      int ncs, int nce, double* __restrict__ y, int64_t ss, int64_t se,
                                                      int64_t sy, int ninst, int assemble) {
  using S = Sz<K>;
  constexpr int NB = S::NB, NQ = S::NQ, NRT = S::NRT, NL = S::NL, NPHI = S::NPHI;
  constexpr int SA = (NB + 3) / 4, QB = (NQ + 15) / 16, NC = 64 / IG;
  __shared__ double sf[IG][NC][NL];
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
  const int col = lane & 15, kq = lane >> 4;
  const int c0 = blockIdx.x * NC, i0 = blockIdx.y * IG;
  {
    const int ig = IG > 1 ? wave : 0, lc = (IG > 1 ? 0 : 16 * wave) + col;
    const int i = min(i0 + ig, ninst - 1);  // (instances and cells past the last repeat it and store nothing)
    const int Kc = min(c0 + lc, P.ncell - 1);
    const bool semi = Kc < ncs;
    const int c = semi ? Kc : Kc - ncs, nc = semi ? ncs : nce;
    const double* __restrict__ u1 = semi ? un + i * ss : ur + i * se;
    const double* __restrict__ u2 = semi ? up + i * ss : uo + i * se;
    const double rho0 = semi ? phs[i].ne - phs[i].pe : 0.0;  // N_D - N_A (SolarCell.cpp:542-548)
    const size_t ub = 2 * (size_t)nc * NB + (size_t)c * NB;
    double v[8], d[SA];
#pragma unroll
    for (int t = 0; t < 8; ++t) v[t] = P.V[8 * (size_t)Kc + t];
#pragma unroll
    for (int t = 0; t < SA; ++t) {
      const int a = 4 * t + kq;
      d[t] = a < NB ? u2[ub + a] - u1[ub + a] : 0.0;
    }
    v4d f = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
    for (int qb = 0; qb < QB; ++qb) {
      v4d rho = {0.0, 0.0, 0.0, 0.0};
      const int qr = 16 * qb + col;
#pragma unroll
      for (int t = 0; t < SA; ++t) {
        const int a = 4 * t + kq;
        rho = __builtin_amdgcn_mfma_f64_16x16x4f64((qr < NQ && a < NB) ? T.phi[a * NQ + qr] : 0.0, d[t], rho, 0, 0, 0);
      }
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        if (16 * qb + 4 * r >= NQ) continue;
        const int q = 16 * qb + 4 * r + kq;
        const bool in = q < NQ;
        const int qc = in ? q : NQ - 1;
        const GeoD g = bilin(v, T.qx[qc], T.qy[qc]);
        double w = rho0 + rho[r];
        if (P.msrc) w += P.msrc[(size_t)Kc * NQ + qc];
        w = in ? -w * T.qw[qc] * g.det : 0.0;
        f = __builtin_amdgcn_mfma_f64_16x16x4f64((in && col < NPHI) ? T.phiP[col * NQ + q] : 0.0, w, f, 0, 0, 0);
      }
    }
#pragma unroll
    for (int r = 0; r < (NPHI + 3) / 4; ++r)
      if (4 * r + kq < NPHI) sf[ig][lc][NRT + 4 * r + kq] = f[r];
  }
  for (int e = threadIdx.x; e < IG * NC * NRT; e += 256) {  // D rows
    const int i = e % NRT, lc = e / NRT % NC, ig = e / (NRT * NC);
    const int Kc = min(c0 + lc, P.ncell - 1);
    sf[ig][lc][i] = poisson_bias<K>(P.table + (size_t)P.type[Kc] * P.stride, phs[min(i0 + ig, ninst - 1)], i);
  }
  __syncthreads();
  if (P.mdir) {
    for (int lc = threadIdx.x; lc < NC; lc += 256) {
      double f[NRT];
#pragma unroll
      for (int i = 0; i < NRT; ++i) f[i] = 0.0;
      if (c0 + lc < P.ncell) poisson_mdir<K>(P, T, c0 + lc, f);
      for (int ig = 0; ig < IG; ++ig)
        for (int i = 0; i < NRT; ++i) sf[ig][lc][i] += f[i];
    }
    __syncthreads();
  }
  poisson_store<K, IG, NC>(P, sf, c0, i0, ninst, y, sy, assemble);
}

// condensation of a given right-hand side b (in the global layout)
template <int K>
__global__ __launch_bounds__(256) void k_poisson_cell_from_b(DevPoisson P, const double* __restrict__ b,
                                                             double* __restrict__ y) {
  constexpr int NL = Sz<K>::NL, NRT = Sz<K>::NRT, NC = 16;
  __shared__ double sf[1][NC][NL];
  const int c0 = blockIdx.x * NC;
  for (int e = threadIdx.x; e < NC * NL; e += 256) {
    const int i = e % NL, lc = e / NL, Kc = c0 + lc;
    if (Kc >= P.ncell) break;
    int m;
    const int fc = (i < NRT) ? face_of_local<K>(i, m) : -1;
    sf[0][lc][i] = (fc < 0 || owns_face<K>(P, Kc, fc)) ? b[P.idx[(size_t)Kc * NL + i]] : 0.0;
  }
  __syncthreads();
  poisson_store<K, 1, NC>(P, sf, c0, 0, 1, y, 0, 0);
}

__global__ __launch_bounds__(256) void k_poisson_face(DevPoisson P, const double* __restrict__ y,
                                                      double* __restrict__ r, int64_t sy, int64_t sr) {
  const int m = blockIdx.x * blockDim.x + threadIdx.x;
  if (m >= P.nmult) return;
  y += blockIdx.y * sy;
  r += blockIdx.y * sr;
  double s = 0.0;
  for (int e = 0; e < 2; ++e) {
    const int c = P.mcell[2 * m + e];
    if (c >= 0) s += P.mcoef[2 * m + e] * y[(size_t)c * P.nloc + P.mloc[2 * m + e]];
  }
  const int h = P.mhang ? P.mhang[m] : -1;
  if (h >= 0) {  // the coarse side of a hanging face
    const int k = P.nphi == 1 ? 1 : P.nphi == 4 ? 2 : 3, f = P.h_face[h];
    const double* E = P.hE + (P.h_sub[h] * k + m - P.h_mbase[h]) * k;
    const double* yc = y + (size_t)P.h_cell[h] * P.nloc;
    double t = 0.0;
    for (int j = 0; j < k; ++j)
      t += E[j] * yc[k == 1 ? rt_face<1>(f, j) : k == 2 ? rt_face<2>(f, j) : rt_face<3>(f, j)];
    s += (f == 1 || f == 3) ? t : -t;
  }
  r[P.mult_perm[m]] = s;
}

// x_K = y - A^{-1} E^T lambda, a (cell, row) per thread, 32 cells per
// workgroup, the cell's weighted multipliers in LDS, the table entries for all
// IG instances of the workgroup.
template <int K, int IG>
__global__ __launch_bounds__(256) void k_poisson_recover(DevPoisson P, const double* __restrict__ lam,
                                                         const double* __restrict__ y, double* __restrict__ out,
                                                         int64_t sl, int64_t sy, int64_t so, int ninst) {
  constexpr int NL = Sz<K>::NL, NRT = Sz<K>::NRT, NC = 32, NE = 4 * K;
  __shared__ double se[IG][NC][NE];
  const int c0 = blockIdx.x * NC, i0 = blockIdx.y * IG;
  for (int e = threadIdx.x; e < NC * NE; e += 256) {
    const int fm = e % NE, lc = e / NE, Kc = c0 + lc, f = fm / K, m = fm - f * K;
    if (Kc >= P.ncell) break;
    const int base = P.mult_face[4 * (size_t)Kc + f];
    const double w = (f == 1 || f == 3) ? P.gw[m] : -P.gw[m];
    const int p = base < 0 ? 0 : P.mult_perm[base + m];
#pragma unroll
    for (int g = 0; g < IG; ++g) se[g][lc][fm] = base < 0 ? 0.0 : w * lam[min(i0 + g, ninst - 1) * sl + p];
    if (P.hc_all) {  // the coarse side of hanging faces: the fine faces' multipliers against this DoF
      for (int q = P.hc_all[Kc]; q < P.hc_all[Kc + 1]; ++q) {
        if (P.h_face[q] != f) continue;
        for (int mm = 0; mm < K; ++mm) {
          const double c = P.hE[(P.h_sub[q] * K + mm) * K + m];
          const int pp = P.mult_perm[P.h_mbase[q] + mm];
#pragma unroll
          for (int g = 0; g < IG; ++g) {
            const double l = lam[min(i0 + g, ninst - 1) * sl + pp];
            se[g][lc][fm] += c * ((f == 1 || f == 3) ? l : -l);
          }
        }
      }
    }
  }
  __syncthreads();
  for (int e = threadIdx.x; e < NC * NL; e += 256) {
    const int i = e % NL, lc = e / NL, Kc = c0 + lc;
    if (Kc >= P.ncell) break;
    bool zero = false;
    if (i < NRT) {
      int m;
      const int fc = face_of_local<K>(i, m);
      if (fc >= 0) {
        if (!owns_face<K>(P, Kc, fc)) continue;
        zero = P.pbid[4 * (size_t)Kc + fc] == 2;  // Neumann D.n = 0 (Poisson.cpp:41-47)
      }
    }
    const double* __restrict__ tb = P.tab_t + (size_t)P.type[Kc] * NL * NL + i;
    double s[IG];
#pragma unroll
    for (int g = 0; g < IG; ++g) s[g] = y[min(i0 + g, ninst - 1) * sy + (size_t)Kc * NL + i];
#pragma unroll
    for (int f = 0; f < 4; ++f)
#pragma unroll
      for (int m = 0; m < K; ++m) {
        const double a = tb[rt_face<K>(f, m) * NL];
#pragma unroll
        for (int g = 0; g < IG; ++g) s[g] -= a * se[g][lc][f * K + m];
      }
    const int id = P.idx[(size_t)Kc * NL + i];
#pragma unroll
    for (int g = 0; g < IG; ++g)
      if (i0 + g < ninst) out[(i0 + g) * so + id] = zero ? 0.0 : s[g];
  }
}

// Mixed precision: the cell condensation y = A^{-1} f and the recovery's
// correction A^{-1} E^T lambda contract in FP32 with the FP32 table (the
// right-hand side f, y and the results stay FP64); wave-uniform lists only.
template <int K>
__global__ __launch_bounds__(64) void k_poisson_cell_f32(DevPoisson P, DevTabs T, const DevPhys* __restrict__ phs,
                                                         const double* __restrict__ un,
                                                         const double* __restrict__ up,
                                                         const double* __restrict__ ur,
                                                         const double* __restrict__ uo, int ncs, int nce,
                                                         double* __restrict__ y, int64_t ss, int64_t se,
                                                         int64_t sy) {
  const DevPhys ph = phs[blockIdx.y];
  {
    const int64_t i = blockIdx.y;
    un += i * ss;
    up += i * ss;
    ur += i * se;
    uo += i * se;
    y += i * sy;
  }
  using S = Sz<K>;
  constexpr int NRT = S::NRT, NL = S::NL;
  const int t0 = blockIdx.x * blockDim.x + threadIdx.x;
  const int Kc = t0 < P.nucell ? P.ucell[t0] : -1;
  if (Kc < 0) return;
  const int ty = __builtin_amdgcn_readfirstlane(P.type[Kc]);
  const double* tb = P.table + (size_t)ty * P.stride;
  const float* tf = P.table_f + (size_t)ty * P.stride;
  double f[NL];
#pragma unroll
  for (int i = 0; i < NRT; ++i) f[i] = poisson_bias<K>(tb, ph, i);
  if (P.mdir) poisson_mdir<K>(P, T, Kc, f);
  poisson_fphi<K>(P, T, ph, Kc, un, up, ur, uo, ncs, nce, f + NRT);
  float ff[NL];
#pragma unroll
  for (int j = 0; j < NL; ++j) ff[j] = (float)f[j];
  for (int i = 0; i < NL; ++i) {
    float s = 0.0f;
#pragma unroll
    for (int j = 0; j < NL; ++j) s += tf[i * NL + j] * ff[j];
    y[(size_t)Kc * NL + i] = (double)s;
  }
}

template <int K>
__global__ __launch_bounds__(64) void k_poisson_recover_f32(DevPoisson P, const double* __restrict__ lam,
                                                            const double* __restrict__ y, double* __restrict__ out,
                                                            int64_t sl, int64_t sy, int64_t so) {
  constexpr int NL = Sz<K>::NL, NRT = Sz<K>::NRT;
  const int t0 = blockIdx.x * blockDim.x + threadIdx.x;
  const int Kc = t0 < P.nucell ? P.ucell[t0] : -1;
  if (Kc < 0) return;
  lam += blockIdx.y * sl;
  y += blockIdx.y * sy;
  out += blockIdx.y * so;
  float e[4 * K];
#pragma unroll
  for (int f = 0; f < 4; ++f) {
    const int base = P.mult_face[4 * (size_t)Kc + f];
    const double sf = (f == 1 || f == 3) ? 1.0 : -1.0;
#pragma unroll
    for (int m = 0; m < K; ++m)
      e[f * K + m] = base < 0 ? 0.0f : (float)(sf * P.gw[m] * lam[P.mult_perm[base + m]]);
  }
  const float* tf = P.table_f + (size_t)__builtin_amdgcn_readfirstlane(P.type[Kc]) * P.stride;
  const int* id = P.idx + (size_t)Kc * NL;
  for (int i = 0; i < NL; ++i) {
    float c = 0.0f;
#pragma unroll
    for (int f = 0; f < 4; ++f)
#pragma unroll
      for (int m = 0; m < K; ++m) c += tf[i * NL + rt_face<K>(f, m)] * e[f * K + m];
    double s = y[(size_t)Kc * NL + i] - (double)c;
    if (i < NRT) {
      int m;
      const int fc = face_of_local<K>(i, m);
      if (fc >= 0) {
        if (!owns_face<K>(P, Kc, fc)) continue;
        if (P.pbid[4 * (size_t)Kc + fc] == 2) s = 0.0;  // Neumann D.n = 0 (Poisson.cpp:41-47)
      }
    }
    out[id[i]] = s;
  }
}

// dst = src of up to 5 vectors, one launch (blockIdx.y: the vector)
__global__ __launch_bounds__(256) void k_copy(VecPairs v) {
  const double* __restrict__ src = v.a[blockIdx.y];
  double* __restrict__ dst = v.b[blockIdx.y];
  const int64_t n = v.n[blockIdx.y];
  for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < n; i += (int64_t)gridDim.x * 256) dst[i] = src[i];
}

// Steady-residual norms without atomics (the sums are bitwise reproducible):
// block (g, j, i) of k_diff_norms writes its partial sums of |a - b|^2 and
// |b|^2 over part g of vector j of instance i to part[2 ((i nvec + j) parts +
// g)]; k_sum_partials then adds each instance's partials in a fixed order.
// One launch for every vector and instance: a launch per vector and instance
// was 320 launches, 1.1 ms, at the end of a step call with 64 instances.
__device__ __forceinline__ void block_sum2(double& d, double& o) {
  __shared__ double s0[4], s1[4];
  d = wave_sum(d);
  o = wave_sum(o);
  if ((threadIdx.x & 63) == 0) {
    s0[threadIdx.x >> 6] = d;
    s1[threadIdx.x >> 6] = o;
  }
  __syncthreads();
  d = (s0[0] + s0[1]) + (s0[2] + s0[3]);
  o = (s1[0] + s1[1]) + (s1[2] + s1[3]);
}

__global__ __launch_bounds__(256) void k_diff_norms(VecPairs v, double* __restrict__ part) {
  const int j = blockIdx.y, i = blockIdx.z;
  const double* __restrict__ a = v.a[j] + i * v.stride[j];
  const double* __restrict__ b = v.b[j] + i * v.stride[j];
  double d = 0.0, o = 0.0;
  for (int64_t e = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; e < v.n[j]; e += (int64_t)gridDim.x * blockDim.x) {
    const double t = a[e] - b[e];
    d += t * t;
    o += b[e] * b[e];
  }
  block_sum2(d, o);
  if (threadIdx.x == 0) {
    double* p = part + 2 * (((int64_t)i * gridDim.y + j) * gridDim.x + blockIdx.x);
    p[0] = d;
    p[1] = o;
  }
}

// One block per instance: acc[2 i], acc[2 i + 1] = sums of the instance's
// nparts partial pairs at part + 2 nparts i.
__global__ __launch_bounds__(256) void k_sum_partials(const double* __restrict__ part, int nparts,
                                                      double* __restrict__ acc) {
  const double* p = part + 2 * (int64_t)nparts * blockIdx.x;
  double d = 0.0, o = 0.0;
  for (int i = threadIdx.x; i < nparts; i += 256) {
    d += p[2 * i];
    o += p[2 * i + 1];
  }
  block_sum2(d, o);
  if (threadIdx.x == 0) {
    acc[2 * blockIdx.x] = d;
    acc[2 * blockIdx.x + 1] = o;
  }
}

// ------------------------------------------------------------------------
// Density fields on a regular grid (the warm-start network's output space)
// ------------------------------------------------------------------------
// A region's cells are the logical grid (i, j) = Morton decode of c, cell
// (i, j) covering logical [i, i+1] / N x [j, j+1] / N with its reference
// coordinates along i and j (the mesh is a uniform logical subdivision of
// the region's coarse quadrilateral).
__device__ __forceinline__ int morton_code(int i, int j, int r) {
  int c = 0;
  for (int b = 0; b < r; ++b) c |= (((i >> b) & 1) << (2 * b)) | (((j >> b) & 1) << (2 * b + 1));
  return c;
}

// Lagrange basis of the K+1 equispaced nodes on [0, 1], node a, at x
template <int K>
__device__ __forceinline__ double lagrange_eq(int a, double x) {
  double v = 1.0;
#pragma unroll
  for (int m = 0; m <= K; ++m)
    if (m != a) v *= (x - (double)m / K) / ((double)(a - m) / K);
  return v;
}

// out[b G + a] = density of carrier vector u at logical ((a + 1/2) / G, (b + 1/2) / G)
template <int K>
__global__ __launch_bounds__(256) void k_grid_sample(const double* __restrict__ u, int r, int G,
                                                     double* __restrict__ out) {
  constexpr int NB = (K + 1) * (K + 1);
  const int e = blockIdx.x * 256 + threadIdx.x;
  if (e >= G * G) return;
  const int N = 1 << r, nc = N * N;
  const int a = e % G, b = e / G;
  const double s = (a + 0.5) / G * N, t = (b + 0.5) / G * N;
  const int i = min((int)s, N - 1), j = min((int)t, N - 1);
  const double xi = s - i, eta = t - j;
  const double* d = u + 2 * (size_t)nc * NB + (size_t)morton_code(i, j, r) * NB;
  double v = 0.0;
#pragma unroll
  for (int q = 0; q <= K; ++q) {
    const double ly = lagrange_eq<K>(q, eta);
#pragma unroll
    for (int p = 0; p <= K; ++p) v += d[p + (K + 1) * q] * lagrange_eq<K>(p, xi) * ly;
  }
  out[e] = v;
}

// Density block of carrier vector u from a G x G grid of values at the
// logical cell centres ((a + 1/2) / G, (b + 1/2) / G): each nodal DoF takes
// the bilinear interpolant of the grid at its logical position (constant
// continuation in the half-cell band along the region's edges).
template <int K>
__global__ __launch_bounds__(256) void k_grid_project(const double* __restrict__ grid, int G, int r,
                                                      double* __restrict__ u) {
  constexpr int NB = (K + 1) * (K + 1);
  const int N = 1 << r, nc = N * N;
  const int e = blockIdx.x * 256 + threadIdx.x;
  if (e >= nc * NB) return;
  const int c = e / NB, m = e % NB;
  int i = 0, j = 0;
  for (int b = 0; b < r; ++b) {
    i |= ((c >> (2 * b)) & 1) << b;
    j |= ((c >> (2 * b + 1)) & 1) << b;
  }
  const double s = ((double)i + (double)(m % (K + 1)) / K) / N, t = ((double)j + (double)(m / (K + 1)) / K) / N;
  const double gx = fmin(fmax(s * G - 0.5, 0.0), (double)(G - 1)), gy = fmin(fmax(t * G - 0.5, 0.0), (double)(G - 1));
  const int x0 = min((int)gx, G - 2 < 0 ? 0 : G - 2), y0 = min((int)gy, G - 2 < 0 ? 0 : G - 2);
  const int x1 = min(x0 + 1, G - 1), y1 = min(y0 + 1, G - 1);
  const double fx = gx - x0, fy = gy - y0;
  const double v = (1.0 - fy) * ((1.0 - fx) * grid[y0 * G + x0] + fx * grid[y0 * G + x1]) +
                   fy * ((1.0 - fx) * grid[y1 * G + x0] + fx * grid[y1 * G + x1]);
  u[2 * (size_t)nc * NB + e] = v;
}

inline int nblk(int64_t n, int b) { return (int)((n + b - 1) / b); }

}  // namespace

#define PECS_DISPATCH_K(k, CALL) \
  switch (k) {                   \
    case 1: { constexpr int KK = 1; CALL; } break; \
    case 2: { constexpr int KK = 2; CALL; } break; \
    case 3: { constexpr int KK = 3; CALL; } break; \
    default: return (int)hipErrorInvalidValue;      \
  }

// ------------------------------------------------------------------------
// Hanging faces of boundary-layer refinement
// ------------------------------------------------------------------------
// The mixed-precision kernels leave out the couplings across hanging faces
// (those faces are absent from the neighbour lists); these kernels add them
// afterwards, in FP64, one thread per cell that has such a coupling.  Both are
// linear in the terms they add, so the sum equals the one over all couplings.
template <int K, int NRHS>
__global__ __launch_bounds__(64) void k_schur_rhs_hang(DevRegion R, const double* __restrict__ b1,
                                                       const double* __restrict__ b2, double mu1, double mu2,
                                                       double* __restrict__ g1, double* __restrict__ g2, int64_t sb,
                                                       int64_t sg) {
  constexpr int NB = Sz<K>::NB;
  const int t = blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= R.nhx) return;
  {
    const int64_t i = blockIdx.y;
    b1 += i * sb;
    b2 += i * sb;
    g1 += i * sg;
    g2 += i * sg;
  }
  double a1[NB], a2[NB];
#pragma unroll
  for (int a = 0; a < NB; ++a) a1[a] = a2[a] = 0.0;
  for (int e = R.hx_ptr[t]; e < R.hx_ptr[t + 1]; ++e) {
    const int M = R.hx_src[e];
    const double* B = R.hblk + (size_t)R.hx_blk[e] * 2 * NB * NB;
    const int ty = R.type[M];
    double w1[2 * NB], w2[2 * NB];
    schur_w<K>(R, b1, mu1, M, ty, w1);
    if (NRHS > 1) schur_w<K>(R, b2, mu2, M, ty, w2);
    for (int i = 0; i < 2 * NB; ++i) {
#pragma unroll
      for (int a = 0; a < NB; ++a) {
        a1[a] += B[i * NB + a] * w1[i];
        if (NRHS > 1) a2[a] += B[i * NB + a] * w2[i];
      }
    }
  }
  const int* __restrict__ pm = R.perm + (size_t)R.hx_cell[t] * NB;
#pragma unroll
  for (int a = 0; a < NB; ++a) {
    g1[pm[a]] += a1[a];
    if (NRHS > 1) g2[pm[a]] += a2[a];
  }
}

template <int K, int NRHS>
__global__ __launch_bounds__(64) void k_schur_recover_hang(DevRegion R, const double* __restrict__ x1,
                                                           const double* __restrict__ x2, double mu1, double mu2,
                                                           double* __restrict__ o1, double* __restrict__ o2,
                                                           int64_t sx, int64_t so) {
  constexpr int NB = Sz<K>::NB;
  const int t = blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= R.nhm) return;
  {
    const int64_t i = blockIdx.y;
    x1 += i * sx;
    x2 += i * sx;
    o1 += i * so;
    o2 += i * so;
  }
  const int M = R.hm_cell[t];
  const size_t nc = R.ncell;
  double s1[2 * NB], s2[2 * NB];
#pragma unroll
  for (int i = 0; i < 2 * NB; ++i) s1[i] = s2[i] = 0.0;
  for (int e = R.hm_ptr[t]; e < R.hm_ptr[t + 1]; ++e) {
    const double* B = R.hblk + (size_t)R.hm_blk[e] * 2 * NB * NB;
    const int* __restrict__ px = R.perm + (size_t)R.hm_dst[e] * NB;
    double v1[NB], v2[NB];
#pragma unroll
    for (int a = 0; a < NB; ++a) {
      v1[a] = x1[px[a]];
      v2[a] = (NRHS > 1) ? x2[px[a]] : 0.0;
    }
    for (int i = 0; i < 2 * NB; ++i) {
#pragma unroll
      for (int a = 0; a < NB; ++a) {
        s1[i] += B[i * NB + a] * v1[a];
        if (NRHS > 1) s2[i] += B[i * NB + a] * v2[a];
      }
    }
  }
  const double* Minv = R.table + (size_t)R.type[M] * R.stride;
#pragma unroll
  for (int h = 0; h < 2; ++h)
#pragma unroll
    for (int a = 0; a < NB; ++a) {
      double t1 = 0.0, t2 = 0.0;
#pragma unroll
      for (int q = 0; q < NB; ++q) {
        t1 += Minv[a * NB + q] * s1[h * NB + q];
        if (NRHS > 1) t2 += Minv[a * NB + q] * s2[h * NB + q];
      }
      const size_t off = (size_t)h * nc * NB + (size_t)M * NB + a;
      o1[off] -= mu1 * t1;
      if (NRHS > 1) o2[off] -= mu2 * t2;
    }
}

// Recovery in mixed precision: x_K -= A_K^{-1} E_K^T lambda over the coarse
// cell's hanging faces (with the same write rules as k_poisson_recover)
template <int K>
__global__ __launch_bounds__(64) void k_poisson_recover_hang(DevPoisson P, const double* __restrict__ lam,
                                                             double* __restrict__ out, int64_t sl, int64_t so) {
  constexpr int NL = Sz<K>::NL, NRT = Sz<K>::NRT;
  const int t = blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= P.nhc) return;
  lam += blockIdx.y * sl;
  out += blockIdx.y * so;
  const int Kc = P.hc_cell[t];
  double e[4 * K];
#pragma unroll
  for (int i = 0; i < 4 * K; ++i) e[i] = 0.0;
  for (int q = P.hc_ptr[t]; q < P.hc_ptr[t + 1]; ++q) {
    const int f = P.h_face[q], sub = P.h_sub[q], mb = P.h_mbase[q];
    const double sf = (f == 1 || f == 3) ? 1.0 : -1.0;
    for (int m = 0; m < K; ++m) {
      const double l = sf * lam[P.mult_perm[mb + m]];
#pragma unroll
      for (int j = 0; j < K; ++j) e[f * K + j] += P.hE[(sub * K + m) * K + j] * l;
    }
  }
  const double* tb = P.table + (size_t)P.type[Kc] * P.stride;
  const int* id = P.idx + (size_t)Kc * NL;
  for (int i = 0; i < NL; ++i) {
    if (i < NRT) {
      int m;
      const int fc = face_of_local<K>(i, m);
      if (fc >= 0 && (!owns_face<K>(P, Kc, fc) || P.pbid[4 * (size_t)Kc + fc] == 2)) continue;
    }
    double c = 0.0;
#pragma unroll
    for (int f = 0; f < 4; ++f)
#pragma unroll
      for (int j = 0; j < K; ++j) c += tb[i * NL + rt_face<K>(f, j)] * e[f * K + j];
    out[id[i]] -= c;
  }
}

static inline int nblk1(int64_t n, int b) { return (int)((n + b - 1) / b); }

RhsSide rhs_side_of(const DevRegion& R, const DevRegion& O, bool semi, const double* u1, const double* u2,
                    const double* ou1, const double* ou2, double* b1, double* b2, double mu1, double mu2, int64_t s,
                    int64_t so) {
  return RhsSide{R.ncell, O.ncell, semi ? 1 : 0, R.V,   R.h,          R.bid,        R.type, R.sigma_nb, R.ctab,
                 R.msrc,  R.mdir,  R.mflux,      {u1, u2}, {ou1, ou2}, {b1, b2},    {mu1, mu2}, s,      so};
}

int launch_rhs_carrier(int k, RhsPair A, const DevPoisson& P, const DevTabs& T, const DevPhys* phs, const double* pvec,
                       hipStream_t s, int nb, int64_t sP) {
  A.nblk0 = nblk1(A.side[0].ncell, 64);
  const int n = A.nblk0 + nblk1(A.side[1].ncell, 64);
  if (n == 0) return 0;
  PECS_DISPATCH_K(k, (k_rhs_carrier<KK><<<dim3(n, nb), 256, 0, s>>>(A, P, T, phs, pvec, sP)));
  return (int)hipGetLastError();
}

// Instances of a batch per workgroup of the Schur kernels: enough that the
// table rows a lane loads are used again, few enough that the launch still
// has several thousand workgroups.
static int schur_per(int nblk, int nb) {
  int per = 1;
  while (per < 16 && per < nb && (int64_t)nblk * nblk1(nb, 2 * per) >= 4096) per *= 2;
  return per;
}

int schur_ctab_size(int k) { return 3 * (k + 1) * (k + 1) * (k + 1) * (k + 1) + 8 * (k + 1) * (k + 1); }

#define PECS_SCHUR_LAUNCH(KERNEL, ARGS)                                                      \
  do {                                                                                       \
    P.nblk0 = nblk1(P.side[0].ncell, 256 / ((k + 1) * (k + 1)));                             \
    const int n = P.nblk0 + nblk1(P.side[1].ncell, 256 / ((k + 1) * (k + 1)));               \
    if (n == 0) return 0;                                                                    \
    const int per = schur_per(n, nb);                                                        \
    PECS_DISPATCH_K(k, (KERNEL<<<dim3(n, nblk1(nb, per)), 256, 0, s>>>ARGS));                \
    return (int)hipGetLastError();                                                           \
  } while (0)
#define PECS_SCHUR_CASE(KERNEL, NRHS, HANG)                                                  \
  if (nrhs == NRHS && hang == HANG) PECS_SCHUR_LAUNCH((KERNEL<KK, NRHS, HANG>), (P, nb, per))
#define PECS_SCHUR_CASES(KERNEL)                                                             \
  PECS_SCHUR_CASE(KERNEL, 1, false);                                                         \
  PECS_SCHUR_CASE(KERNEL, 2, false);                                                         \
  PECS_SCHUR_CASE(KERNEL, 1, true);                                                          \
  PECS_SCHUR_CASE(KERNEL, 2, true);                                                          \
  return (int)hipErrorInvalidValue

int launch_carrier_w(int k, SchurPair P, int nrhs, hipStream_t s, int nb) {
  PECS_SCHUR_LAUNCH((k_carrier_w<KK>), (P, nrhs, nb, per));
}

static int launch_schur_rhs_main(int k, SchurPair P, int nrhs, hipStream_t s, int nb) {
  const bool hang = P.side[0].hx_all || P.side[1].hx_all;
  PECS_SCHUR_CASES(k_schur_rhs);
}

static int launch_schur_recover_main(int k, SchurPair P, int nrhs, hipStream_t s, int nb) {
  const bool hang = P.side[0].hm_all || P.side[1].hm_all;
  PECS_SCHUR_CASES(k_schur_recover);
}
#undef PECS_SCHUR_CASES
#undef PECS_SCHUR_CASE
#undef PECS_SCHUR_LAUNCH

template <int NRHS, bool FWD>
static int sweep_dispatch(const DevFactor& F, const int4* tl, int nt, int w, int maxr, const double* v0,
                          const double* v1, double* t0, double* t1, hipStream_t s, bool pf) {
#define PECS_SWEEP_CASE(WW, MM)                                                          \
  if (w == WW && maxr == MM) {                                                           \
    if (pf) k_sweep<NRHS, WW, MM, FWD, true><<<nt, 256, 0, s>>>(F, tl, v0, v1, t0, t1);  \
    else k_sweep<NRHS, WW, MM, FWD><<<nt, 256, 0, s>>>(F, tl, v0, v1, t0, t1);           \
    return 0;                                                                            \
  }
  PECS_SWEEP_CASE(8, 1) PECS_SWEEP_CASE(8, 2) PECS_SWEEP_CASE(8, 4)
  PECS_SWEEP_CASE(16, 1) PECS_SWEEP_CASE(16, 2) PECS_SWEEP_CASE(16, 4)
  PECS_SWEEP_CASE(32, 1) PECS_SWEEP_CASE(32, 2) PECS_SWEEP_CASE(32, 4)
  PECS_SWEEP_CASE(64, 1) PECS_SWEEP_CASE(64, 2) PECS_SWEEP_CASE(64, 4)
  PECS_SWEEP_CASE(32, 8) PECS_SWEEP_CASE(64, 8)
#undef PECS_SWEEP_CASE
  return (int)hipErrorInvalidValue;
}

template <bool FWD>
static int sweep_mfma_dispatch(const DevFactor& F, const int4* tl, int nt, int mb, int nrp, bool split, double* Y,
                               int ks, const int4* rtl, int nrt, hipStream_t s, int tbase) {
  if (ks > 0 && (!rtl || !F.Part)) return (int)hipErrorInvalidValue;
#define PECS_MFMA_CASE(NN, MM)                                                              \
  if (!split && nrp == NN && mb == MM) {                                                    \
    k_sweep_mfma<NN, MM, FWD><<<nt, 256, 0, s>>>(F, tl, Y, ks, F.Part, tbase);                   \
    if (ks > 0 && nrt > 0) k_sweep_reduce<NN, FWD><<<dim3(nrt, REDUCE_SPLIT), 256, 0, s>>>(F, rtl, 64 * MM, F.Part, Y); \
    return 0;                                                                               \
  }
#define PECS_MFMA_SPLIT(NN, MM, HH)                                                         \
  if (split && nrp == NN && mb == MM) {                                                     \
    k_sweep_mfma<NN, MM, FWD, HH><<<nt, 256, 0, s>>>(F, tl, Y, ks, F.Part, tbase);               \
    if (ks > 0 && nrt > 0) k_sweep_reduce<NN, FWD><<<dim3(nrt, REDUCE_SPLIT), 256, 0, s>>>(F, rtl, 64 * MM, F.Part, Y); \
    return 0;                                                                               \
  }
  PECS_MFMA_CASE(16, 1) PECS_MFMA_CASE(16, 2) PECS_MFMA_CASE(16, 4)
  PECS_MFMA_CASE(32, 1) PECS_MFMA_CASE(32, 2) PECS_MFMA_CASE(32, 4)
  PECS_MFMA_CASE(64, 1) PECS_MFMA_CASE(64, 2) PECS_MFMA_CASE(64, 4)
  PECS_MFMA_CASE(128, 1) PECS_MFMA_CASE(128, 2)
  PECS_MFMA_SPLIT(32, 1, 1) PECS_MFMA_SPLIT(32, 2, 1) PECS_MFMA_SPLIT(32, 4, 1)
  PECS_MFMA_SPLIT(64, 1, 1) PECS_MFMA_SPLIT(64, 2, 1) PECS_MFMA_SPLIT(64, 4, 1)
  PECS_MFMA_SPLIT(128, 1, 2) PECS_MFMA_SPLIT(128, 2, 2) PECS_MFMA_SPLIT(128, 4, 2)
#undef PECS_MFMA_SPLIT
#undef PECS_MFMA_CASE
  return (int)hipErrorInvalidValue;
}

int mfma_rhs_pad(int nrhs) { return nrhs <= 16 ? 16 : nrhs <= 32 ? 32 : nrhs <= 64 ? 64 : 128; }

// 4 blocks per wave at 128 right-hand sides only with the groups split over
// waves (2 groups per wave): unsplit, their accumulators and operands would
// not fit the register file
bool mfma_shape_ok(int nrp, int mb, bool split) { return mb == 1 || mb == 2 || (mb == 4 && (nrp <= 64 || split)); }

int mfma_tile_rows(int nrp, int mb, bool split) {
  if (!split || nrp <= 16) return 64 * mb;
  const int hpw = nrp >= 128 ? 2 : 1, wpr = nrp / 16 / hpw;
  return 4 / wpr * 16 * mb;
}

int launch_sweep(const DevFactor& F, const int4* tiles, int nt, int w, int maxr, bool fwd, int nrhs,
                 double* t, hipStream_t s, int ks, const int4* rtiles, int nrt, const double* src, bool pf,
                 int tbase) {
  if (nt <= 0) return 0;
  if (w <= 0) {  // 0: MFMA sweep, -1: its right-hand-side groups split over waves, -2: LDS-staged vector
    if (nrhs > MAX_MFMA_RHS) return (int)hipErrorInvalidValue;
    const int nrp = mfma_rhs_pad(nrhs);
    // a factor tuned for many right-hand sides and solved with 16 or fewer
    // (single solves on a batched context): the LDS-staged shape runs as the
    // plain MFMA sweep, whose tiles of 64 maxr rows and partial-sum slots
    // are the same
    if (w == -2 && nrp < 32) w = 0;
    if (w == -2) {
      if ((maxr != 1 && maxr != 2) || (ks > 0 && (!rtiles || !F.Part))) return (int)hipErrorInvalidValue;
#define PECS_MFMA_LDS(NN, MM)                                                                    \
  if (nrp == NN && maxr == MM) {                                                                 \
    if (fwd) {                                                                                   \
      k_sweep_mfma_lds<NN, true, MM><<<nt, 256, 0, s>>>(F, tiles, t, ks, F.Part, tbase);                \
      if (ks > 0 && nrt > 0) k_sweep_reduce<NN, true><<<dim3(nrt, REDUCE_SPLIT), 256, 0, s>>>(F, rtiles, 64 * MM, F.Part, t); \
    } else {                                                                                     \
      k_sweep_mfma_lds<NN, false, MM><<<nt, 256, 0, s>>>(F, tiles, t, ks, F.Part, tbase);               \
      if (ks > 0 && nrt > 0) k_sweep_reduce<NN, false><<<dim3(nrt, REDUCE_SPLIT), 256, 0, s>>>(F, rtiles, 64 * MM, F.Part, t); \
    }                                                                                            \
    return (int)hipGetLastError();                                                               \
  }
      PECS_MFMA_LDS(32, 1) PECS_MFMA_LDS(64, 1) PECS_MFMA_LDS(128, 1)
      PECS_MFMA_LDS(32, 2) PECS_MFMA_LDS(64, 2) PECS_MFMA_LDS(128, 2)
#undef PECS_MFMA_LDS
      return (int)hipErrorInvalidValue;
    }
    const bool split = w < 0 && nrp > 16;
    return fwd ? sweep_mfma_dispatch<true>(F, tiles, nt, maxr, nrp, split, t, ks, rtiles, nrt, s, tbase)
               : sweep_mfma_dispatch<false>(F, tiles, nt, maxr, nrp, split, t, ks, rtiles, nrt, s, tbase);
  }
  if (nrhs > 2 || ks > 0) return (int)hipErrorInvalidValue;
  const double* v0 = fwd ? src : nullptr;
  double* t1 = nrhs == 2 ? t + F.n : t;
  if (fwd) {
    return nrhs == 2 ? sweep_dispatch<2, true>(F, tiles, nt, w, maxr, v0, v0, t, t1, s, pf)
                     : sweep_dispatch<1, true>(F, tiles, nt, w, maxr, v0, v0, t, t1, s, pf);
  }
  return nrhs == 2 ? sweep_dispatch<2, false>(F, tiles, nt, w, maxr, v0, v0, t, t1, s, pf)
                   : sweep_dispatch<1, false>(F, tiles, nt, w, maxr, v0, v0, t, t1, s, pf);
}

// The tiles (rows, row tiles) of level l: of one system, or of all (sys -1).
struct LevelRange {
  int at, n, base;
  LevelRange(const int* off, const FactorLevels& L, int l, int sys) {
    base = off[l * L.nsys];
    at = sys < 0 ? base : off[l * L.nsys + sys];
    n = off[sys < 0 ? (l + 1) * L.nsys : l * L.nsys + sys + 1] - at;
  }
};

template <int NRP>
static int chol_solve_il(const DevFactor& F, const FactorLevels& L, double* v, double* t, int nrhs, hipStream_t s,
                         int sys) {
  const int pb = sys < 0 ? 0 : L.sys_p0[sys], pe = sys < 0 ? F.n : L.sys_p0[sys + 1];
  k_pack_il<NRP><<<nblk(pe - pb, IL_TP), 256, 0, s>>>(F, v, nrhs, pb, pe);
  // the leaf level's rows are owed nothing (pack_layout checks it)
  for (int l = 0; l < L.nlevels; ++l) {
    const LevelRange g(L.goff, L, l, sys), f(L.foff, L, l, sys), r(L.froff, L, l, sys);
    if (l > 0 && g.n > 0)
      k_fwd_gather_il<NRP><<<nblk((int64_t)g.n * NRP / 2, 256), 256, 0, s>>>(F, F.lrows + g.at, g.n, nrhs);
    if (L.fw[l] > 0) return (int)hipErrorInvalidValue;
    const int e = launch_sweep(F, F.ftiles + f.at, f.n, L.fw[l], L.fm[l], true, nrhs, t, s, L.fks[l], F.frtiles + r.at,
                               r.n, nullptr, false, f.at - f.base);
    if (e) return e;
  }
  for (int l = L.nlevels - 1; l >= 0; --l) {
    const LevelRange x(L.xoff, L, l, sys), b(L.boff, L, l, sys), r(L.broff, L, l, sys);
    // (the LDS-staged sweep, 32 or more right-hand sides, reads the panel
    // columns through the row index)
    if (x.n > 0 && !(L.bw[l] == -2 && NRP >= 32))
      k_bwd_gather_il<NRP><<<nblk((int64_t)x.n * NRP / 2, 256), 256, 0, s>>>(F, F.xidx + x.at, x.n);
    if (L.bw[l] > 0) return (int)hipErrorInvalidValue;
    const int e = launch_sweep(F, F.btiles + b.at, b.n, L.bw[l], L.bm[l], false, nrhs, t, s, L.bks[l], F.brtiles + r.at,
                               r.n, nullptr, false, b.at - b.base);
    if (e) return e;
  }
  k_unpack_il<NRP><<<nblk(pe - pb, IL_TP), 256, 0, s>>>(F, v, nrhs, pb, pe);
  return (int)hipGetLastError();
}

int launch_chol_solve(const DevFactor& F, const FactorLevels& L, double* v, double* t, int nrhs, hipStream_t s,
                      int sys) {
  if (L.nlevels > 0 && L.fw[0] <= 0) {  // MFMA-shaped factor: interleaved vectors
    if (nrhs > MAX_MFMA_RHS) return (int)hipErrorInvalidValue;
    switch (mfma_rhs_pad(nrhs)) {
      case 16: return chol_solve_il<16>(F, L, v, t, nrhs, s, sys);
      case 32: return chol_solve_il<32>(F, L, v, t, nrhs, s, sys);
      case 64: return chol_solve_il<64>(F, L, v, t, nrhs, s, sys);
      default: return chol_solve_il<128>(F, L, v, t, nrhs, s, sys);
    }
  }
  if (nrhs > 2) return (int)hipErrorInvalidValue;
  for (int l = 0; l < L.nlevels; ++l) {
    // level 0 (leaves) owes nothing to its rows: its sweep reads the right-hand side itself
    const LevelRange g(L.goff, L, l, sys), f(L.foff, L, l, sys);
    if (l > 0 && g.n > 0) {
      const int* lr = F.lrows + g.at;
      if (g.n >= 16384) {
        if (nrhs == 2) k_fwd_gather<1, 2><<<nblk(g.n, 256), 256, 0, s>>>(F, lr, g.n, v);
        else k_fwd_gather<1, 1><<<nblk(g.n, 256), 256, 0, s>>>(F, lr, g.n, v);
      } else {
        if (nrhs == 2) k_fwd_gather<8, 2><<<nblk(8 * (int64_t)g.n, 256), 256, 0, s>>>(F, lr, g.n, v);
        else k_fwd_gather<8, 1><<<nblk(8 * (int64_t)g.n, 256), 256, 0, s>>>(F, lr, g.n, v);
      }
    }
    const int e = launch_sweep(F, F.ftiles + f.at, f.n, L.fw[l], L.fm[l], true, nrhs, t, s, 0, nullptr, 0,
                               l == 0 ? v : nullptr, L.fpf && L.fpf[l]);
    if (e) return e;
  }
  for (int l = L.nlevels - 1; l >= 0; --l) {
    // the backward sweep reads the panel rows' x straight from X (no gather)
    const LevelRange b(L.boff, L, l, sys);
    const int e = launch_sweep(F, F.btiles + b.at, b.n, L.bw[l], L.bm[l], false, nrhs, t, s, 0, nullptr, 0, nullptr,
                               L.bpf && L.bpf[l]);
    if (e) return e;
  }
  return (int)hipGetLastError();
}

int launch_poisson_cell(int k, const DevPoisson& P, const DevTabs& T, const DevPhys* phs, const double* un,
                        const double* up, const double* ur, const double* uo, int ncs, int nce, double* y,
                        hipStream_t s, int nb, int64_t ss, int64_t se, int64_t sy) {
  if (P.table_f && P.ucell) {  // mixed precision
    PECS_DISPATCH_K(k, (k_poisson_cell_f32<KK><<<dim3(nblk(P.nucell, 64), nb), 64, 0, s>>>(
                           P, T, phs, un, up, ur, uo, ncs, nce, y, ss, se, sy)));
    return (int)hipGetLastError();
  }
  if (nb >= 4) {
    PECS_DISPATCH_K(k, (k_poisson_cell<KK, 4><<<dim3(nblk(P.ncell, 16), nblk(nb, 4)), 256, 0, s>>>(
                           P, T, phs, un, up, ur, uo, ncs, nce, y, ss, se, sy, nb, 0)));
  } else {
    PECS_DISPATCH_K(k, (k_poisson_cell<KK, 1><<<dim3(nblk(P.ncell, 64), nb), 256, 0, s>>>(
                           P, T, phs, un, up, ur, uo, ncs, nce, y, ss, se, sy, nb, 0)));
  }
  return (int)hipGetLastError();
}

int launch_poisson_cell_from_b(const DevPoisson& P, const double* b, double* y, hipStream_t s) {
  const int k = (P.nphi == 1) ? 1 : (P.nphi == 4 ? 2 : 3);
  PECS_DISPATCH_K(k, (k_poisson_cell_from_b<KK><<<nblk(P.ncell, 16), 256, 0, s>>>(P, b, y)));
  return (int)hipGetLastError();
}

int launch_poisson_face(const DevPoisson& P, const double* y, double* r, hipStream_t s, int nb, int64_t sy,
                        int64_t sr) {
  k_poisson_face<<<dim3(nblk(P.nmult, 256), nb), 256, 0, s>>>(P, y, r, sy, sr);
  return (int)hipGetLastError();
}

static int launch_poisson_recover_main(int k, const DevPoisson& P, const double* lam, const double* y, double* out,
                           hipStream_t s, int nb, int64_t sl, int64_t sy, int64_t so) {
  if (P.table_f && P.ucell) {  // mixed precision
    PECS_DISPATCH_K(k, (k_poisson_recover_f32<KK><<<dim3(nblk(P.nucell, 64), nb), 64, 0, s>>>(P, lam, y, out, sl, sy,
                                                                                              so)));
    return (int)hipGetLastError();
  }
  if (nb >= 4) {
    PECS_DISPATCH_K(k, (k_poisson_recover<KK, 4><<<dim3(nblk(P.ncell, 32), nblk(nb, 4)), 256, 0, s>>>(
                           P, lam, y, out, sl, sy, so, nb)));
  } else {
    PECS_DISPATCH_K(k, (k_poisson_recover<KK, 1><<<dim3(nblk(P.ncell, 32), nb), 256, 0, s>>>(P, lam, y, out, sl, sy, so,
                                                                                             nb)));
  }
  return (int)hipGetLastError();
}

SchurSide schur_side_of(const DevRegion& R, const double* b1, const double* b2, double* w1, double* w2, double mu1,
                        double mu2, double* g1, double* g2, double* o1, double* o2, int64_t sb, int64_t sg, int64_t so) {
  return SchurSide{R.ncell,   R.nbr,    R.type,   R.perm,     R.ctab, {b1, b2}, {w1, w2},
                   {g1, g2},  {o1, o2}, {mu1, mu2}, sb,       sg,     so,       R.hx_all,
                   R.hx_src,  R.hx_blk, R.hm_all, R.hm_dst,   R.hm_blk, R.hblk};
}

int launch_schur_rhs(int k, const DevRegion* const* R, const SchurPair& P, int nrhs, hipStream_t s, int nb) {
  bool f32 = false;
  for (int r = 0; r < 2; ++r) f32 = f32 || (R[r] && R[r]->table_f);
  if (!f32) {
    const int rc = launch_schur_rhs_main(k, P, nrhs, s, nb);
    if (rc) return rc;
  }
  for (int r = 0; r < 2; ++r) {
    if (!R[r] || P.side[r].ncell == 0) continue;
    const SchurSide& S = P.side[r];
    if (f32) {  // mixed precision
      const dim3 g(nblk(R[r]->nu_nbh, 64), nb);
      if (nrhs == 2) {
        PECS_DISPATCH_K(k, (k_schur_rhs_f32<KK, 2><<<g, 64, 0, s>>>(*R[r], S.b[0], S.b[1], S.mu[0], S.mu[1], S.g[0],
                                                                    S.g[1], S.sb, S.sg)));
      } else {
        PECS_DISPATCH_K(k, (k_schur_rhs_f32<KK, 1><<<g, 64, 0, s>>>(*R[r], S.b[0], S.b[0], S.mu[0], S.mu[0], S.g[0],
                                                                    S.g[0], S.sb, S.sg)));
      }
    }
    if (!f32 || R[r]->nhx == 0) continue;
    const dim3 g(nblk(R[r]->nhx, 64), nb);
    if (nrhs == 2) {
      PECS_DISPATCH_K(k, (k_schur_rhs_hang<KK, 2><<<g, 64, 0, s>>>(*R[r], S.b[0], S.b[1], S.mu[0], S.mu[1], S.g[0],
                                                                   S.g[1], S.sb, S.sg)));
    } else {
      PECS_DISPATCH_K(k, (k_schur_rhs_hang<KK, 1><<<g, 64, 0, s>>>(*R[r], S.b[0], S.b[0], S.mu[0], S.mu[0], S.g[0],
                                                                   S.g[0], S.sb, S.sg)));
    }
  }
  return (int)hipGetLastError();
}

int launch_schur_recover(int k, const DevRegion* const* R, const SchurPair& P, int nrhs, hipStream_t s, int nb) {
  bool f32 = false;
  for (int r = 0; r < 2; ++r) f32 = f32 || (R[r] && R[r]->table_f);
  if (!f32) {
    const int rc = launch_schur_recover_main(k, P, nrhs, s, nb);
    if (rc) return rc;
  }
  for (int r = 0; r < 2; ++r) {
    if (!R[r] || P.side[r].ncell == 0) continue;
    const SchurSide& S = P.side[r];
    const int h = nrhs - 1;
    if (f32) {  // mixed precision
      const dim3 g(nblk(R[r]->nu_own, 64), nb);
      if (nrhs == 2) {
        PECS_DISPATCH_K(k, (k_schur_recover_f32<KK, 2><<<g, 64, 0, s>>>(*R[r], S.b[0], S.b[1], S.g[0], S.g[1], S.mu[0],
                                                                        S.mu[1], S.o[0], S.o[1], S.sb, S.sg, S.so)));
      } else {
        PECS_DISPATCH_K(k, (k_schur_recover_f32<KK, 1><<<g, 64, 0, s>>>(*R[r], S.b[0], S.b[0], S.g[0], S.g[0], S.mu[0],
                                                                        S.mu[0], S.o[0], S.o[0], S.sb, S.sg, S.so)));
      }
    }
    if (!f32 || R[r]->nhm == 0) continue;
    const dim3 g(nblk(R[r]->nhm, 64), nb);
    if (nrhs == 2) {
      PECS_DISPATCH_K(k, (k_schur_recover_hang<KK, 2><<<g, 64, 0, s>>>(*R[r], S.g[0], S.g[1], S.mu[0], S.mu[1], S.o[0],
                                                                       S.o[1], S.sg, S.so)));
    } else {
      PECS_DISPATCH_K(k, (k_schur_recover_hang<KK, 1><<<g, 64, 0, s>>>(*R[r], S.g[h], S.g[h], S.mu[h], S.mu[h],
                                                                       S.o[h], S.o[h], S.sg, S.so)));
    }
  }
  return (int)hipGetLastError();
}

int launch_poisson_recover(int k, const DevPoisson& P, const double* lam, const double* y, double* out,
                           hipStream_t s, int nb, int64_t sl, int64_t sy, int64_t so) {
  const int rc = launch_poisson_recover_main(k, P, lam, y, out, s, nb, sl, sy, so);
  if (rc || P.nhc == 0 || !P.table_f) return rc;
  PECS_DISPATCH_K(k, (k_poisson_recover_hang<KK><<<dim3(nblk(P.nhc, 64), nb), 64, 0, s>>>(P, lam, out, sl, so)));
  return (int)hipGetLastError();
}

int launch_poisson_rhs_assemble(int k, const DevPoisson& P, const DevTabs& T, const DevPhys* phs, const double* un,
                                const double* up, const double* ur, const double* uo, int ncs, int nce, double* b,
                                hipStream_t s) {
  PECS_DISPATCH_K(k, (k_poisson_cell<KK, 1><<<dim3(nblk(P.ncell, 64), 1), 256, 0, s>>>(P, T, phs, un, up, ur, uo, ncs,
                                                                                       nce, b, 0, 0, 0, 1, 1)));
  return (int)hipGetLastError();
}

int launch_copy(const VecPairs& v, hipStream_t s) {
  int64_t n = 0;
  for (int j = 0; j < v.nvec; ++j) n = std::max(n, v.n[j]);
  if (n <= 0) return 0;
  k_copy<<<dim3((unsigned)std::min<int64_t>(nblk(n, 256), 2048), v.nvec), 256, 0, s>>>(v);
  return (int)hipGetLastError();
}

int launch_norms(const VecPairs& v, double* part, double* acc, int ninst, hipStream_t s) {
  int64_t n = 1;
  for (int j = 0; j < v.nvec; ++j) n = std::max(n, v.n[j]);
  // 8 entries per thread and vector, at most RES_PARTS blocks
  const int parts = (int)std::min<int64_t>(nblk(n, 2048), RES_PARTS);
  k_diff_norms<<<dim3(parts, v.nvec, ninst), 256, 0, s>>>(v, part);
  k_sum_partials<<<ninst, 256, 0, s>>>(part, v.nvec * parts, acc);
  return (int)hipGetLastError();
}

int launch_grid_sample(int k, const double* u, int r, int G, double* out, hipStream_t s) {
  PECS_DISPATCH_K(k, (k_grid_sample<KK><<<nblk((int64_t)G * G, 256), 256, 0, s>>>(u, r, G, out)));
  return (int)hipGetLastError();
}

int launch_grid_project(int k, const double* grid, int G, int r, double* u, hipStream_t s) {
  const int64_t n = ((int64_t)1 << (2 * r)) * (k + 1) * (k + 1);
  PECS_DISPATCH_K(k, (k_grid_project<KK><<<nblk(n, 256), 256, 0, s>>>(grid, G, r, u)));
  return (int)hipGetLastError();
}

}  // namespace pecs
