// Gauge molecular dynamics on the device (FP64): Wilson gauge force, link
// update, reunitarisation, plaquette and kinetic energy.
//
// wilson_gauge_force : library/forces.cpp:262-283 + staples.cpp:82-107
// update_links       : library/update.cpp:228-247 + suNa.cpp:113-134 (exp)
// reunitarize        : library/suNg.cpp:171-359
// plaquette          : library/wilsonloop.cpp:58-133 (avr_wilson(1,1))
// improved_gauge_force: library/forces.cpp:285-310 + staples.cpp:7-80
// avr_wilson(h, w)   : library/wilsonloop.cpp:58-133 (rectangle weights of
//                      bcs.cpp:30-31, 72-120)
// hamiltonian (P^2)  : library/update.cpp:201-216
// Fundamental links are kept as component planes (the layout of the
// represented links): a wave of 64 consecutive sites of one parity and one
// direction reads each element as one contiguous 1 KB segment.  Host
// transfers in the reference layout (4*id+mu, re plane then im plane) are
// transposed through LDS.  Momenta are SoA mom[(mu * NG + a) * V + id].  Periodic, open and
// SF gauge boundaries (bcs.cpp: boundary plaquette weights, fixed links).
#include <algorithm>
#include "yh_internal.hpp"
#include "yh_reduce.hpp"

namespace yh {

typedef Cx<double> cd;

// diagonal phases of the SF boundary links (bcs.cpp:208-232)
struct SfPhases {
  double c1[4], c2[4];
};

template <int NC>
struct M {
  cd m[NC][NC];
};

template <int NC>
__device__ __forceinline__ M<NC> ld(const double2* fund, int id, int mu, const Geom& g) {
  M<NC> u;
  const double2* p = fund + fund_at<NC>(id, mu, g);
#pragma unroll
  for (int e = 0; e < NC * NC; e++) {
    const double2 v = p[(size_t)e * g.VHpad];
    u.m[e / NC][e % NC] = cd(v.x, v.y);
  }
  return u;
}

// conjugate transpose of the link
template <int NC>
__device__ __forceinline__ M<NC> ldd(const double2* fund, int id, int mu, const Geom& g) {
  M<NC> u;
  const double2* p = fund + fund_at<NC>(id, mu, g);
#pragma unroll
  for (int e = 0; e < NC * NC; e++) {
    const double2 v = p[(size_t)e * g.VHpad];
    u.m[e % NC][e / NC] = cd(v.x, -v.y);
  }
  return u;
}

template <int NC>
__device__ __forceinline__ void st(double2* fund, int id, int mu, const M<NC>& u, const Geom& g) {
  double2* p = fund + fund_at<NC>(id, mu, g);
#pragma unroll
  for (int e = 0; e < NC * NC; e++)
    p[(size_t)e * g.VHpad] = make_double2(u.m[e / NC][e % NC].re, u.m[e / NC][e % NC].im);
}

// host layout <-> component planes for the n sites from site i0 (full EO
// index; aos holds those sites only): a block moves S of them through LDS, so
// that both sides are coalesced.  16 sites keep 256-byte segments of the planes
// and spread a small lattice over the chip (SU(3), 8^4, to page-locked memory:
// 62 us, 64 with 64 sites; 50 for the copy alone).
template <int NC>
struct AosTile {
  static constexpr int S = 16;           // sites
  static constexpr int W = 8 * NC * NC;  // doubles of a site's four links
};

template <int NC, bool TO_AOS>
__global__ void __launch_bounds__(256) k_fund_aos(double* __restrict__ aos, double2* __restrict__ fund, Geom g, int i0,
                                                  int n) {
  typedef AosTile<NC> A;
  constexpr int NN = NC * NC;
  __shared__ double tile[A::S * (A::W + 1)];  // the odd site stride spreads the banks
  const int j0 = blockIdx.x * A::S;
  const int ns = min(A::S, n - j0);
  double* base = aos + (size_t)j0 * A::W;
  if (!TO_AOS) {
    for (int i = threadIdx.x; i < ns * A::W; i += 256) tile[(i / A::W) * (A::W + 1) + i % A::W] = base[i];
    __syncthreads();
  }
  for (int j = threadIdx.x; j < 4 * NN * A::S; j += 256) {
    const int s = j % A::S, mu = j / A::S / NN, e = j / A::S % NN;
    if (s >= ns) continue;
    double2* f = fund + fund_at<NC>(i0 + j0 + s, mu, g) + (size_t)e * g.VHpad;
    double* t = tile + s * (A::W + 1) + mu * 2 * NN + e;
    if (TO_AOS) {
      const double2 v = *f;
      t[0] = v.x;
      t[NN] = v.y;
    } else {
      *f = make_double2(t[0], t[NN]);
    }
  }
  if (TO_AOS) {
    __syncthreads();
    for (int i = threadIdx.x; i < ns * A::W; i += 256) base[i] = tile[(i / A::W) * (A::W + 1) + i % A::W];
  }
}

template <int NC>
__device__ __forceinline__ M<NC> mul(const M<NC>& a, const M<NC>& b) {
  M<NC> r;
#pragma unroll
  for (int i = 0; i < NC; i++)
#pragma unroll
    for (int j = 0; j < NC; j++) {
      cd s(0, 0);
#pragma unroll
      for (int k = 0; k < NC; k++) cmac(s, a.m[i][k], b.m[k][j]);
      r.m[i][j] = s;
    }
  return r;
}

// a * b^+
template <int NC>
__device__ __forceinline__ M<NC> muld(const M<NC>& a, const M<NC>& b) {
  M<NC> r;
#pragma unroll
  for (int i = 0; i < NC; i++)
#pragma unroll
    for (int j = 0; j < NC; j++) {
      cd s(0, 0);
#pragma unroll
      for (int k = 0; k < NC; k++) cmac(s, a.m[i][k], conj(b.m[j][k]));
      r.m[i][j] = s;
    }
  return r;
}

// a^+ * b
template <int NC>
__device__ __forceinline__ M<NC> dmul(const M<NC>& a, const M<NC>& b) {
  M<NC> r;
#pragma unroll
  for (int i = 0; i < NC; i++)
#pragma unroll
    for (int j = 0; j < NC; j++) {
      cd s(0, 0);
#pragma unroll
      for (int k = 0; k < NC; k++) cmac_conj(s, a.m[k][i], b.m[k][j]);
      r.m[i][j] = s;
    }
  return r;
}

// anti-Hermitian matrix of an algebra vector (library/suNg.cpp:15-58)
template <int NC>
__device__ __forceinline__ M<NC> alg(const double* mom, int V, int mu, int id) {
  constexpr int NG = NC * NC - 1;
  M<NC> r;
#pragma unroll
  for (int i = 0; i < NC; i++)
#pragma unroll
    for (int j = 0; j < NC; j++) r.m[i][j] = cd(0, 0);
  int n = 0;
#pragma unroll
  for (int i = 0; i < NC; i++)
#pragma unroll
    for (int j = 0; j < NC; j++) {
      if (i > j) {
        double v = mom[(size_t)(mu * NG + n) * V + id];
        r.m[i][j].im += v;
        r.m[j][i].im += v;
        n++;
      } else if (i < j) {
        double v = mom[(size_t)(mu * NG + n) * V + id];
        r.m[i][j].re += v;
        r.m[j][i].re -= v;
        n++;
      } else if (i > 0) {
        double v = mom[(size_t)(mu * NG + n) * V + id];
        double w = sqrt(2.0 / (i * (i + 1)));
        for (int k = 0; k < i; k++) r.m[k][k].im += w * v;
        r.m[i][i].im -= i * w * v;
        n++;
      }
    }
  return r;
}

// determinant by Gaussian elimination with partial pivoting (the row swaps
// are selects, so every index stays static); the reference uses an
// unpivoted LU (suNg.cpp:296-330) for the same value
template <int NC>
__device__ __forceinline__ cd det_gauss(M<NC> m) {
  cd det(1, 0);
#pragma unroll
  for (int c = 0; c < NC; c++) {
#pragma unroll
    for (int i = c + 1; i < NC; i++) {
      const double ai = m.m[i][c].re * m.m[i][c].re + m.m[i][c].im * m.m[i][c].im;
      const double ac = m.m[c][c].re * m.m[c][c].re + m.m[c][c].im * m.m[c][c].im;
      const bool sw = ai > ac;
#pragma unroll
      for (int j = 0; j < NC; j++) {
        const cd a = m.m[c][j], b = m.m[i][j];
        m.m[c][j] = sw ? b : a;
        m.m[i][j] = sw ? a : b;
      }
      det = sw ? cd(-det.re, -det.im) : det;
    }
    const cd p = m.m[c][c];
    det = det * p;
    const double n = 1.0 / (p.re * p.re + p.im * p.im);
    const cd inv(p.re * n, -p.im * n);
#pragma unroll
    for (int i = c + 1; i < NC; i++) {
      const cd f = m.m[i][c] * inv;
#pragma unroll
      for (int j = c; j < NC; j++) m.m[i][j] = m.m[i][j] - f * m.m[c][j];
    }
  }
  return det;
}

// suNg::reunitarize (library/suNg.cpp:171-359); a zero row returns the
// input unchanged (the reference returns early there, with the rows before
// it already processed in the general branch)
//   NC = 2: normalise row 0, row 1 = (-conj r01, conj r00)
//   NC = 3: normalise row 0, orthogonalise and normalise row 1,
//           row 2 = conj(r0 x r1)
//   other:  modified Gram-Schmidt over all rows, then the last row times
//           exp(-i arg det) so that det = 1
template <int NC>
__device__ __forceinline__ void reunit(M<NC>& u) {
  if constexpr (NC == 2 || NC == 3) {
    double n0 = 0;
#pragma unroll
    for (int j = 0; j < NC; j++) n0 += u.m[0][j].re * u.m[0][j].re + u.m[0][j].im * u.m[0][j].im;
    if (n0 == 0.0) return;
    n0 = 1.0 / sqrt(n0);
#pragma unroll
    for (int j = 0; j < NC; j++) u.m[0][j] = n0 * u.m[0][j];
    if constexpr (NC == 2) {
      u.m[1][0] = cd(-u.m[0][1].re, u.m[0][1].im);
      u.m[1][1] = conj(u.m[0][0]);
    } else {
      cd p(0, 0);
#pragma unroll
      for (int j = 0; j < NC; j++) cmac_conj(p, u.m[0][j], u.m[1][j]);
#pragma unroll
      for (int j = 0; j < NC; j++) u.m[1][j] = u.m[1][j] - p * u.m[0][j];
      double n1 = 0;
#pragma unroll
      for (int j = 0; j < NC; j++) n1 += u.m[1][j].re * u.m[1][j].re + u.m[1][j].im * u.m[1][j].im;
      n1 = 1.0 / sqrt(n1);
#pragma unroll
      for (int j = 0; j < NC; j++) u.m[1][j] = n1 * u.m[1][j];
      u.m[2][0] = conj(u.m[0][1] * u.m[1][2] - u.m[0][2] * u.m[1][1]);
      u.m[2][1] = conj(u.m[0][2] * u.m[1][0] - u.m[0][0] * u.m[1][2]);
      u.m[2][2] = conj(u.m[0][0] * u.m[1][1] - u.m[0][1] * u.m[1][0]);
    }
  } else {
    const M<NC> orig = u;
    bool zero = false;
#pragma unroll
    for (int i = 0; i < NC; i++) {
      double n = 0;
#pragma unroll
      for (int j = 0; j < NC; j++) n += u.m[i][j].re * u.m[i][j].re + u.m[i][j].im * u.m[i][j].im;
      zero = zero || n == 0.0;
      n = n == 0.0 ? 1.0 : 1.0 / sqrt(n);
#pragma unroll
      for (int j = 0; j < NC; j++) u.m[i][j] = n * u.m[i][j];
#pragma unroll
      for (int k = i + 1; k < NC; k++) {
        cd p(0, 0);
#pragma unroll
        for (int j = 0; j < NC; j++) cmac_conj(p, u.m[i][j], u.m[k][j]);
#pragma unroll
        for (int j = 0; j < NC; j++) u.m[k][j] = u.m[k][j] - p * u.m[i][j];
      }
    }
    if (zero) {
      u = orig;
      return;
    }
    const cd d = det_gauss<NC>(u);
    const double inv = 1.0 / sqrt(d.re * d.re + d.im * d.im);
    const cd ph(d.re * inv, -d.im * inv);
#pragma unroll
    for (int j = 0; j < NC; j++) u.m[NC - 1][j] = u.m[NC - 1][j] * ph;
  }
}

// Open and SF boundaries of the gauge field (library/bcs.cpp:28-130, 166-262):
// spatial plaquettes based on the boundary slices (open: t = 0 and T-1; SF:
// t = 0 and T-2) count half in the action and its force, and the links the
// boundary fixes (open: U_0 at t = T-1; SF: the spatial links at t = 0, every
// link at t = T-2 and T-1) keep their values: their momenta are zeroed.
__device__ __forceinline__ double plaq_w(int t, int mu, int nu, const Geom& g) {
  if (mu == 0 || nu == 0) return 1.0;
  if (g.bc == BC_OPEN && (t == 0 || t == g.L[0] - 1)) return 0.5;
  if (g.bc == BC_SF && (t == 0 || t == g.L[0] - 2)) return 0.5;
  return 1.0;
}

__device__ __forceinline__ bool link_fixed(int t, int mu, const Geom& g) {
  if (g.bc == BC_OPEN) return t == g.L[0] - 1 && mu == 0;
  if (g.bc == BC_SF) return (t == 0 && mu > 0) || t == g.L[0] - 2 || t == g.L[0] - 1;
  return false;
}

// rect_weight(id, a, b) of the 1 x 2 rectangle based on time slice t with
// its short side along a and long side along b: open boundaries use the
// plaquette weights (bcs.cpp:31); SF weights 0 for the spatial a < b
// rectangles on t = 0 and T-2 and 1.5 for a = 0 on t = 0 and T-3
// (bcs.cpp:89-116)
__device__ __forceinline__ double rect_w(int t, int a, int b, const Geom& g) {
  if (g.bc == BC_OPEN) return plaq_w(t, a, b, g);
  if (g.bc != BC_SF) return 1.0;
  if ((t == 0 || t == g.L[0] - 2) && a >= 1 && a < b) return 0.0;
  if ((t == 0 || t == g.L[0] - 3) && a == 0 && b >= 1) return 1.5;
  return 1.0;
}

// one step of a path on coordinates c: forward (d, +1) multiplies P by
// U(c, d) and moves to c + d; backward (d, -1) moves to c - d and multiplies
// by U(c - d, d)^+
template <int NC>
__device__ __forceinline__ void path_step(M<NC>& P, const double2* fund, int (&c)[4], int d, bool fw, const Geom& g) {
  if (fw) {
    P = mul<NC>(P, ld<NC>(fund, full_index(c[0], c[1], c[2], c[3], g), d, g));
    c[d] = c[d] + 1 == g.L[d] ? 0 : c[d] + 1;
  } else {
    c[d] = c[d] == 0 ? g.L[d] - 1 : c[d] - 1;
    P = muld<NC>(P, ld<NC>(fund, full_index(c[0], c[1], c[2], c[3], g), d, g));
  }
}

template <int NC>
__device__ __forceinline__ M<NC> unit_matrix() {
  M<NC> r;
#pragma unroll
  for (int i = 0; i < NC; i++)
#pragma unroll
    for (int j = 0; j < NC; j++) r.m[i][j] = cd(i == j ? 1.0 : 0.0, 0.0);
  return r;
}

// apply_bcs_on_momentum_field (bcs.cpp:166-199)
__global__ void __launch_bounds__(256) k_mom_bcs(double* __restrict__ mom, int NG, Geom g) {
  int t = blockIdx.x * 256 + threadIdx.x;
  if (t >= 4 * g.V) return;
  int id = t >> 2, mu = t & 3;
  int c[4];
  full_coords(id, g, c);
  if (!link_fixed(c[0], mu, g)) return;
  for (int a = 0; a < NG; a++) mom[(size_t)(mu * NG + a) * g.V + id] = 0.0;
}

// apply_bcs_on_gauge_field (bcs.cpp:201-262): the fixed links take their
// boundary values: zero, or the SF matrices diag(exp(i c1_k)), diag(exp(i c2_k))
template <int NC>
__global__ void __launch_bounds__(256) k_gauge_bcs(double2* __restrict__ fund, Geom g, SfPhases ph) {
  const int id = blockIdx.x * 256 + threadIdx.x, mu = blockIdx.y;
  if (id >= g.V) return;
  int c[4];
  full_coords(id, g, c);
  if (!link_fixed(c[0], mu, g)) return;
  M<NC> u;
#pragma unroll
  for (int i = 0; i < NC; i++)
#pragma unroll
    for (int j = 0; j < NC; j++) u.m[i][j] = cd(0, 0);
  if (g.bc == BC_SF && mu > 0 && (c[0] == 0 || c[0] == g.L[0] - 2)) {
    const double* v = c[0] == 0 ? ph.c1 : ph.c2;
#pragma unroll
    for (int i = 0; i < NC; i++) u.m[i][i] = cd(cos(v[i]), sin(v[i]));
  }
  st<NC>(fund, id, mu, u, g);
}

template <int NC>
__device__ __forceinline__ void axpy(M<NC>& s, double w, const M<NC>& a) {
#pragma unroll
  for (int i = 0; i < NC; i++)
#pragma unroll
    for (int j = 0; j < NC; j++) {
      s.m[i][j].re = fma(w, a.m[i][j].re, s.m[i][j].re);
      s.m[i][j].im = fma(w, a.m[i][j].im, s.m[i][j].im);
    }
}

template <int NC>
__device__ __forceinline__ M<NC> scaled(double w, const M<NC>& a) {
  M<NC> r;
#pragma unroll
  for (int i = 0; i < NC; i++)
#pragma unroll
    for (int j = 0; j < NC; j++) r.m[i][j] = w * a.m[i][j];
  return r;
}

// an opaque zero once every element of m is final: link indices that it is
// added to are loaded after m, so that the loads of a chain of products are
// not all issued (and held in registers) at its start
template <int NC>
__device__ __forceinline__ int settled(M<NC>& m) {
#pragma unroll
  for (int i = 0; i < NC; i++)
#pragma unroll
    for (int j = 0; j < NC; j++) __asm__ volatile("" : "+v"(m.m[i][j].re), "+v"(m.m[i][j].im));
  int z;
  __asm__ volatile("v_mov_b32 %0, 0" : "=v"(z));
  return z;
}

// Re Tr(iT_a F) of every generator, in the reference's order
// (suNa.cpp:102-111): each has two entries, or the i + 1 of a diagonal one
template <int NC>
__device__ __forceinline__ void project(double (&out)[NC * NC - 1], const M<NC>& F) {
  int a = 0;
#pragma unroll
  for (int i = 0; i < NC; i++)
#pragma unroll
    for (int j = 0; j < NC; j++) {
      if (i > j) {
        out[a++] = -F.m[j][i].im - F.m[i][j].im;
      } else if (i < j) {
        out[a++] = F.m[j][i].re - F.m[i][j].re;
      } else if (i > 0) {
        double re = i * F.m[i][i].im;
#pragma unroll
        for (int k = 0; k < i; k++) re -= F.m[k][k].im;
        out[a++] = re * sqrt(2.0 / (i * (i + 1)));
      }
    }
}

// Work order of the gauge-force kernels: mu fastest, then parity, then blocks
// of 64 sites, so that the workgroups that share links run side by side; each
// XCD takes 64 consecutive workgroups in turn, which keeps the time
// neighbours of its sites closer than one contiguous slab per XCD does
// (SU(3) Wilson force at 32^4, calls back to back: 690 us, one slab per XCD
// 746).
struct ForceItem {
  int mu, p, k;  // direction, parity, half index (may lie past the end)
};
__device__ __forceinline__ ForceItem force_item() {
  const int b = xcd_block(gridDim.x, 64);
  return ForceItem{b & 3, (b >> 2) & 1, (b >> 3) * 64 + (int)(threadIdx.x & 63)};
}

// The tail of a gauge-force workgroup: the waves' staples S meet in LDS and
// are added in a fixed order, and wave 0 projects U(x, mu) S onto the momenta.
template <int NC, int NW>
__device__ __forceinline__ void force_tail(M<NC>& S, const double2* fund, double* mom, double f, int w, int lane,
                                           const ForceItem& it, const Geom& g) {
  constexpr int NN = NC * NC, NG = NN - 1;
  __shared__ double2 ex[NW - 1][NN][64];
  if (w > 0) {
#pragma unroll
    for (int e = 0; e < NN; e++) ex[w - 1][e][lane] = make_double2(S.m[e / NC][e % NC].re, S.m[e / NC][e % NC].im);
  }
  __syncthreads();
  if (w > 0 || it.k >= g.VH) return;
#pragma unroll
  for (int q = 0; q < NW - 1; q++)
#pragma unroll
    for (int e = 0; e < NN; e++) {
      const double2 v = ex[q][e][lane];
      S.m[e / NC][e % NC] = S.m[e / NC][e % NC] + cd(v.x, v.y);
    }
  const int id = it.p * g.VH + it.k;
  double a[NG];
  project<NC>(a, mul<NC>(ld<NC>(fund, id, it.mu, g), S));
#pragma unroll
  for (int n = 0; n < NG; n++) mom[(size_t)(it.mu * NG + n) * g.V + id] += f * a[n];
}

// Wilson gauge force: mom -= algebra_project(U staple, dt beta / NC), the
// staples weighted by their plaquettes' weights (forces.cpp:262-283,
// staples.cpp:82-107).  A workgroup takes 64 consecutive sites of one parity
// and one mu, one wave per nu.  Bound by the 19 link reads per (x, mu) from
// L2: 728 us at 32^4 among the kernels of a leapfrog step, 690 back to back
// (15.7 and 16.6 TB/s of link reads; 1,614 us in the step with the links as an
// array of 144-byte structures, where every load of a wave touches 64 or
// more cache lines, and one thread per link).  Measured and not kept: one
// wave per plane forming the plaquettes that serve two links each (fewer
// reads, but 217 registers and two waves per SIMD: 923 us), and one wave per
// (nu, side) (1,015 us).
template <int NC>
__global__ void __launch_bounds__(192) k_wilson_force(const double2* __restrict__ fund, double* __restrict__ mom,
                                                      double f, Geom g) {
  const ForceItem it = force_item();
  const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int kk = min(it.k, g.VH - 1);  // lanes past the end compute on the last site and write nothing
  const int id = it.p * g.VH + kk, mu = it.mu, nu = w + (w >= mu);
  int c[4], cb[4], q[4];
  site_coords(kk, it.p, g, c);
  const int om = neighbour(c, mu, 1, g, q), on = neighbour(c, nu, 1, g, q);
  const int bn = neighbour(c, nu, -1, g, cb), bnm = neighbour(cb, mu, 1, g, q);
  auto L = [&](int i, int d) { return ld<NC>(fund, i, d, g); };
  M<NC> S = scaled(plaq_w(c[0], mu, nu, g), muld(L(om, nu), mul(L(id, nu), L(on, mu))));
  axpy(S, plaq_w(cb[0], nu, mu, g), dmul(mul(L(bn, mu), L(bnm, nu)), L(bn, nu)));
  force_tail<NC, 3>(S, fund, mom, f, w, lane, it, g);
}

// the weighted staples of the link (x, mu) on one side (UP: +nu) of it,
// paths from x + mu back to x.  With A = U(x+mu, nu), B = U(x+nu, mu)^+,
// C = U(x, nu)^+ (down: the links around the plaquette at x - nu) the
// plaquette staple is A B C, and each of the three 1 x 2 rectangles on this
// side replaces one of the three links by its own staple: A P C (long side
// along nu), Q B C and A B R (long side along mu).  Summed as
//   A (w0 B C + wP P C + wR B R) + wQ Q (B C):
// 11 products, against 17 for the four paths taken one by one.
template <int NC, bool UP>
__device__ __forceinline__ M<NC> side_staple(const double2* fund, const int (&c)[4], int id, int mu, int nu, double c0,
                                             double c1, const Geom& g) {
  auto L = [&](int i, int d) { return ld<NC>(fund, i, d, g); };
  auto D = [&](int i, int d) { return ldd<NC>(fund, i, d, g); };
  int cn[4], cm[4], cmn[4], q[4], r[4];
  const int om = neighbour(c, mu, 1, g, cm);
  const int on = neighbour(c, nu, UP ? 1 : -1, g, cn);    // x +- nu
  const int omn = neighbour(cn, mu, 1, g, cmn);           // x + mu +- nu
  const int dt = nu == 0 ? (UP ? 0 : -1) : 0;             // time of the base corner of the plaquette, less t
  auto wrap = [&](int t) { return t < 0 ? t + g.L[0] : t; };
  const double w0 = plaq_w(wrap(c[0] + dt), mu, nu, g);
  const double wP = c1 * rect_w(wrap(c[0] + 2 * dt), mu, nu, g);
  const double wQ = c1 * rect_w(wrap(c[0] + dt), nu, mu, g);
  const double wR = c1 * rect_w(wrap(c[0] + dt - (mu == 0)), nu, mu, g);
  const M<NC> B = D(on, mu);
  const M<NC> C = UP ? D(id, nu) : L(on, nu);
  const M<NC> BC = mul(B, C);
  M<NC> T = scaled(w0 * c0, BC);
  {
    // P: the staple of (x +- nu, mu) one step further along nu
    const int z = settled(T);
    const int o2n = neighbour(cn, nu, UP ? 1 : -1, g, q) + z;   // x +- 2 nu
    const int om2n = neighbour(q, mu, 1, g, r) + z;             // x + mu +- 2 nu
    M<NC> P = UP ? muld(L(omn + z, nu), L(o2n, mu)) : mul(D(om2n, nu), D(o2n, mu));
    P = UP ? muld(P, L(on + z, nu)) : mul(P, L(o2n, nu));
    axpy(T, wP, mul(P, C));
  }
  {
    // R: around the plaquette at x - mu (+- nu)
    const int z = settled(T);
    const int ob = neighbour(c, mu, -1, g, q) + z;              // x - mu
    const int obn = neighbour(cn, mu, -1, g, r) + z;            // x - mu +- nu
    M<NC> R = mul(D(obn, mu), UP ? D(ob, nu) : L(obn, nu));
    R = mul(R, L(ob, mu));
    axpy(T, wR, mul(B, R));
  }
  const int z = settled(T);
  M<NC> S = mul(UP ? L(om + z, nu) : D(omn + z, nu), T);
  {
    // Q: around the plaquette at x + mu (+- nu)
    const int z2 = settled(S);
    const int o2m = neighbour(cm, mu, 1, g, q) + z2;            // x + 2 mu
    const int o2mn = neighbour(cmn, mu, 1, g, r) + z2;          // x + 2 mu +- nu
    M<NC> Q = UP ? mul(L(om + z2, mu), L(o2m, nu)) : muld(L(om + z2, mu), L(o2mn, nu));
    Q = muld(Q, L(omn + z2, mu));
    axpy(S, wQ, mul(Q, BC));
  }
  return S;
}

// Improved gauge force: mom -= algebra_project(U staple, dt beta / NC) with
// staple = c0 S_plaq + c1 S_rect, S_rect the six weighted rectangles through
// the link for each nu (forces.cpp:285-310, staples.cpp:7-80).
// A workgroup takes 64 consecutive sites of one parity and one mu; its waves
// share out the six (nu, side), add their staples through LDS in a fixed
// order, and wave 0 multiplies by the link and projects.
// waves of a workgroup (SU(4) keeps both sides in a wave: the exchange of six takes 80 KB of LDS)
constexpr int rect_waves(int nc) { return nc < 4 ? 6 : 3; }

template <int NC>
__global__ void __launch_bounds__((64 * rect_waves(NC))) k_rect_force(const double2* __restrict__ fund,
                                                                     double* __restrict__ mom, double f, double c0,
                                                                     double c1, Geom g) {
  constexpr int NW = rect_waves(NC);
  const ForceItem it = force_item();
  const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int kk = min(it.k, g.VH - 1);  // lanes past the end compute on the last site and write nothing
  const int id = it.p * g.VH + kk, mu = it.mu;
  int c[4];
  site_coords(kk, it.p, g, c);
  const int j = NW == 6 ? w >> 1 : w;
  const int nu = j + (j >= mu);
  M<NC> S;
  if constexpr (NW == 6) {
    if (w & 1) S = side_staple<NC, false>(fund, c, id, mu, nu, c0, c1, g);
    else S = side_staple<NC, true>(fund, c, id, mu, nu, c0, c1, g);
  } else {
    S = side_staple<NC, true>(fund, c, id, mu, nu, c0, c1, g);
    axpy(S, 1.0, side_staple<NC, false>(fund, c, id + settled(S), mu, nu, c0, c1, g));
  }
  force_tail<NC, NW>(S, fund, mom, f, w, lane, it, g);
}

// U <- exp(eps P) U, Taylor series to |X^k/k!|^2 < 1e-24 then reunitarised
template <int NC>
__global__ void __launch_bounds__(128) k_update_links(double2* __restrict__ fund, const double* __restrict__ mom,
                                                      double eps, Geom g) {
  const int id = blockIdx.x * 128 + threadIdx.x, mu = blockIdx.y;
  if (id >= g.V) return;
  M<NC> X = alg<NC>(mom, g.V, mu, id);
  M<NC> R, Xk;
#pragma unroll
  for (int i = 0; i < NC; i++)
#pragma unroll
    for (int j = 0; j < NC; j++) {
      R.m[i][j] = cd(i == j ? 1.0 : 0.0, 0);
      Xk.m[i][j] = R.m[i][j];
    }
  double err = 1.0;
  for (int k = 1; k < 64 && err > 1e-24; k++) {
    Xk = mul<NC>(Xk, X);
    double f = eps / k;
    err = 0;
#pragma unroll
    for (int i = 0; i < NC; i++)
#pragma unroll
      for (int j = 0; j < NC; j++) {
        Xk.m[i][j] = f * Xk.m[i][j];
        R.m[i][j] = R.m[i][j] + Xk.m[i][j];
        err += Xk.m[i][j].re * Xk.m[i][j].re + Xk.m[i][j].im * Xk.m[i][j].im;
      }
  }
  reunit<NC>(R);
  st<NC>(fund, id, mu, mul<NC>(R, ld<NC>(fund, id, mu, g)), g);
}

template <int NC>
__global__ void __launch_bounds__(128) k_reunitarize(double2* __restrict__ fund, Geom g) {
  const int id = blockIdx.x * 128 + threadIdx.x, mu = blockIdx.y;
  if (id >= g.V) return;
  M<NC> u = ld<NC>(fund, id, mu, g);
  reunit<NC>(u);
  st<NC>(fund, id, mu, u, g);
}

// sum over planes of Re Tr of the plaquette
template <int NC>
__global__ void __launch_bounds__(256) k_plaquette(const double2* __restrict__ fund, double* partials, unsigned* ticket,
                                                   double* out, Geom g) {
  int id = blockIdx.x * 256 + threadIdx.x;
  double v[1] = {0.0};
  if (id < g.V) {
    int c[4];
    full_coords(id, g, c);
    for (int mu = 1; mu < 4; mu++)
      for (int nu = 0; nu < mu; nu++) {
        int o[4];
        const int a = neighbour(c, mu, 1, g, o), b = neighbour(c, nu, 1, g, o);
        M<NC> one = mul<NC>(ld<NC>(fund, id, mu, g), ld<NC>(fund, a, nu, g));
        M<NC> two = mul<NC>(ld<NC>(fund, id, nu, g), ld<NC>(fund, b, mu, g));
        M<NC> P = muld<NC>(one, two);
        double tr = 0.0;
#pragma unroll
        for (int i = 0; i < NC; i++) tr += P.m[i][i].re;
        v[0] += plaq_w(c[0], mu, nu, g) * tr;
      }
  }
  block_reduce_finish<1, 256>(v, partials, gridDim.x, blockIdx.x, ticket, out);
}

// sum over planes mu > nu of the weighted Re Tr of the h x w loop based at
// each site: h links along mu, w along nu, back along mu, back along nu
// (wilson_loop, wilsonloop.cpp:58-113)
template <int NC>
__global__ void __launch_bounds__(256) k_wilson_loop(const double2* __restrict__ fund, int h, int w, double* partials,
                                                     unsigned* ticket, double* out, Geom g) {
  int id = blockIdx.x * 256 + threadIdx.x;
  double v[1] = {0.0};
  if (id < g.V) {
    int c[4];
    full_coords(id, g, c);
    for (int mu = 1; mu < 4; mu++)
      for (int nu = 0; nu < mu; nu++) {
        int p[4] = {c[0], c[1], c[2], c[3]};
        M<NC> P = unit_matrix<NC>();
        for (int k = 0; k < h; k++) path_step<NC>(P, fund, p, mu, true, g);
        for (int k = 0; k < w; k++) path_step<NC>(P, fund, p, nu, true, g);
        for (int k = 0; k < h; k++) path_step<NC>(P, fund, p, mu, false, g);
        for (int k = 0; k < w; k++) path_step<NC>(P, fund, p, nu, false, g);
        double tr = 0.0;
#pragma unroll
        for (int i = 0; i < NC; i++) tr += P.m[i][i].re;
        if (h == 1 && w == 1) tr *= plaq_w(c[0], mu, nu, g);
        else if (h == 1 && w == 2) tr *= rect_w(c[0], mu, nu, g);
        else if (h == 2 && w == 1) tr *= rect_w(c[0], nu, mu, g);
        v[0] += tr;
      }
  }
  block_reduce_finish<1, 256>(v, partials, gridDim.x, blockIdx.x, ticket, out);
}

__global__ void __launch_bounds__(256) k_sumsq(const double* __restrict__ a, long n, double* partials, unsigned* ticket,
                                               double* out) {
  long i0 = (long)blockIdx.x * 256 + threadIdx.x;
  double v[1] = {0.0};
  for (long i = i0; i < n; i += (long)gridDim.x * 256) v[0] += a[i] * a[i];
  block_reduce_finish<1, 256>(v, partials, gridDim.x, blockIdx.x, ticket, out);
}

// ---------------------------------------------------------------------------
#define YH_NC_SWITCH(...)                                     \
  switch (c->nc) {                                            \
    case 2: { constexpr int NC_ = 2; __VA_ARGS__; } break;    \
    case 3: { constexpr int NC_ = 3; __VA_ARGS__; } break;    \
    case 4: { constexpr int NC_ = 4; __VA_ARGS__; } break;    \
    default: set_error("unsupported NC"); return YH_ERR_UNSUPPORTED; \
  }

// sites whose links the staging buffer holds (a whole number of blocks unless
// it holds the lattice)
static int fund_stage_sites(const Ctx* c) {
  const size_t site = sizeof(double) * 8 * c->nc * c->nc;
  return (int)std::min<size_t>(c->g.V, FUND_STAGE_BYTES / site / 16 * 16);
}

size_t fund_stage_bytes(const Ctx* c) { return sizeof(double) * 8 * c->nc * c->nc * (size_t)fund_stage_sites(c); }

template <int NC, bool TO_AOS>
static void fund_aos_launch(Ctx* c, int i0, int n) {
  static_assert(AosTile<NC>::S == 16, "fund_stage_sites");
  hipLaunchKernelGGL((k_fund_aos<NC, TO_AOS>), dim3((n + AosTile<NC>::S - 1) / AosTile<NC>::S), dim3(256), 0, c->stream,
                     c->fund_stage, c->fund, c->g, i0, n);
}

// Host transfers go through the staging buffer piece by piece: the stream
// keeps a piece's copy and transposition in order with the next one's.  A
// piece costs about 20 us beyond its copy, so pieces are large (SU(3), 32^4,
// to page-locked memory: 11.16 ms with 32 MiB a piece, 10.88 with 128 and
// 10.80 in one; 10.58 for the copy alone).
int gauge_upload(Ctx* c, const double* host) {
  const size_t site = 8 * (size_t)c->nc * c->nc;
  const int step = fund_stage_sites(c);
  for (int i0 = 0, n; i0 < c->g.V; i0 += n) {
    n = std::min(step, c->g.V - i0);
    YH_HIP(hipMemcpyAsync(c->fund_stage, host + site * i0, sizeof(double) * site * n, hipMemcpyHostToDevice, c->stream));
    YH_NC_SWITCH((fund_aos_launch<NC_, false>(c, i0, n)));
    YH_HIP(hipGetLastError());
  }
  return YH_OK;
}

int gauge_download(Ctx* c, double* host) {
  const size_t site = 8 * (size_t)c->nc * c->nc;
  const int step = fund_stage_sites(c);
  for (int i0 = 0, n; i0 < c->g.V; i0 += n) {
    n = std::min(step, c->g.V - i0);
    YH_NC_SWITCH((fund_aos_launch<NC_, true>(c, i0, n)));
    YH_HIP(hipGetLastError());
    YH_HIP(hipMemcpyAsync(host + site * i0, c->fund_stage, sizeof(double) * site * n, hipMemcpyDeviceToHost, c->stream));
  }
  YH_HIP(hipStreamSynchronize(c->stream));
  return YH_OK;
}

int md_gauge_force(Ctx* c, double dt, double beta) {
  int rc;
  if ((rc = force_alloc(c))) return rc;
  dim3 grid((c->g.VH + 63) / 64 * 8);
  YH_NC_SWITCH(hipLaunchKernelGGL((k_wilson_force<NC_>), grid, dim3(192), 0, c->stream, c->fund, c->mom,
                                  dt * beta / c->nc * 0.5, c->g));
  YH_HIP(hipGetLastError());
  return YH_OK;
}

int md_improved_gauge_force(Ctx* c, double dt, double beta, double c0, double c1) {
  int rc;
  if ((rc = force_alloc(c))) return rc;
  dim3 grid((c->g.VH + 63) / 64 * 8);
  YH_NC_SWITCH(hipLaunchKernelGGL((k_rect_force<NC_>), grid, dim3(64 * rect_waves(NC_)), 0, c->stream, c->fund, c->mom,
                                  dt * beta / c->nc * 0.5, c0, c1, c->g));
  YH_HIP(hipGetLastError());
  return YH_OK;
}

static bool gauge_bcs(const Ctx* c) { return c->g.bc == BC_OPEN || c->g.bc == BC_SF; }

static int mom_bcs(Ctx* c) {
  if (!gauge_bcs(c)) return YH_OK;
  hipLaunchKernelGGL(k_mom_bcs, dim3((4 * c->g.V + 255) / 256), dim3(256), 0, c->stream, c->mom, c->nc * c->nc - 1, c->g);
  YH_HIP(hipGetLastError());
  return YH_OK;
}

// the `volume` the plaquette is normalised by (bcs.cpp:32, 76; geometry.cpp:1150)
static double gauge_volume(const Ctx* c) {
  const double v3 = (double)c->g.V / c->g.L[0];
  if (c->g.bc == BC_OPEN) return (c->g.L[0] - 1) * v3;
  if (c->g.bc == BC_SF) return (c->g.L[0] - 2) * v3;
  return (double)c->g.V;
}

int md_apply_gauge_bcs(Ctx* c) {
  if (!gauge_bcs(c)) return YH_OK;
  SfPhases ph = {};
  if (c->g.bc == BC_SF) {
    // bcs.cpp:208-232: phases v1 / L, v2 / L with L = 2 NC L_X
    const double pi = 3.14159265358979323846;
    const double L = 2.0 * c->nc * c->g.L[1];
    if (c->nc == 2) {
      ph.c1[0] = -pi / L; ph.c1[1] = pi / L;
      ph.c2[0] = -3 * pi / L; ph.c2[1] = 3 * pi / L;
    } else if (c->nc == 3) {
      ph.c1[0] = -pi / L; ph.c1[1] = 0; ph.c1[2] = pi / L;
      ph.c2[0] = -5 * pi / L; ph.c2[1] = 2 * pi / L; ph.c2[2] = 3 * pi / L;
    } else {
      set_error("SF boundary values are defined for NC = 2 and 3");
      return YH_ERR_UNSUPPORTED;
    }
  }
  dim3 grid((c->g.V + 255) / 256, 4);
  YH_NC_SWITCH(hipLaunchKernelGGL((k_gauge_bcs<NC_>), grid, dim3(256), 0, c->stream, c->fund, c->g, ph));
  YH_HIP(hipGetLastError());
  return YH_OK;
}

int md_update_links(Ctx* c, double eps) {
  int rc;
  if ((rc = force_alloc(c))) return rc;
  // the fixed links' momenta are zeroed, so exp(0) U leaves them as they are
  // (update.cpp:231-243 zeroes them, updates, and sets the fixed links again)
  if ((rc = mom_bcs(c))) return rc;
  dim3 grid((c->g.V + 127) / 128, 4);
  YH_NC_SWITCH(hipLaunchKernelGGL((k_update_links<NC_>), grid, dim3(128), 0, c->stream, c->fund, c->mom, eps, c->g));
  YH_HIP(hipGetLastError());
  return YH_OK;
}

int md_reunitarize(Ctx* c) {
  dim3 grid((c->g.V + 127) / 128, 4);
  YH_NC_SWITCH(hipLaunchKernelGGL((k_reunitarize<NC_>), grid, dim3(128), 0, c->stream, c->fund, c->g));
  YH_HIP(hipGetLastError());
  return YH_OK;
}

int md_plaquette(Ctx* c, double* out) {
  dim3 grid((c->g.V + 255) / 256);
  double* dst = &c->sc->red[0];
  YH_NC_SWITCH(hipLaunchKernelGGL((k_plaquette<NC_>), grid, dim3(256), 0, c->stream, c->fund, c->partials, c->ticket,
                                  dst, c->g));
  YH_HIP(hipGetLastError());
  double v;
  YH_HIP(hipMemcpyAsync(&v, dst, sizeof(double), hipMemcpyDeviceToHost, c->stream));
  YH_HIP(hipStreamSynchronize(c->stream));
  *out = v / (c->nc * 6.0 * gauge_volume(c));
  return YH_OK;
}

int md_avr_wilson(Ctx* c, int h, int w, double* out) {
  dim3 grid((c->g.V + 255) / 256);
  double* dst = &c->sc->red[0];
  YH_NC_SWITCH(hipLaunchKernelGGL((k_wilson_loop<NC_>), grid, dim3(256), 0, c->stream, c->fund, h, w, c->partials,
                                  c->ticket, dst, c->g));
  YH_HIP(hipGetLastError());
  double v;
  YH_HIP(hipMemcpyAsync(&v, dst, sizeof(double), hipMemcpyDeviceToHost, c->stream));
  YH_HIP(hipStreamSynchronize(c->stream));
  *out = v / (c->nc * 6.0 * gauge_volume(c));
  return YH_OK;
}

int md_kinetic(Ctx* c, double* out) {
  int rc;
  if ((rc = force_alloc(c))) return rc;
  // hamiltonian() applies the momentum BCs first (update.cpp:201-206)
  if ((rc = mom_bcs(c))) return rc;
  long n = 4L * c->g.V * (c->nc * c->nc - 1);
  int grid = (int)std::min<long>((n + 255) / 256, (long)c->nblk);
  double* dst = &c->sc->red[0];
  hipLaunchKernelGGL(k_sumsq, dim3(grid), dim3(256), 0, c->stream, c->mom, n, c->partials, c->ticket, dst);
  YH_HIP(hipGetLastError());
  double v;
  YH_HIP(hipMemcpyAsync(&v, dst, sizeof(double), hipMemcpyDeviceToHost, c->stream));
  YH_HIP(hipStreamSynchronize(c->stream));
  *out = v;  // TF / 2 = 1
  return YH_OK;
}

}  // namespace yh

// ---------------------------------------------------------------------------
using namespace yh;

static int md_check(Ctx* c) {
  if (!c) { set_error("null argument"); return YH_ERR_ARG; }
  if (!c->gauge_set) { set_error("no gauge field"); return YH_ERR_STATE; }
  if (c->g.bc == YH_BC_SF && c->nc > 3) {
    set_error("SF boundary values are defined for NC = 2 and 3");
    return YH_ERR_UNSUPPORTED;
  }
  YH_HIP(hipSetDevice(c->device));
  return YH_OK;
}

static int md_sync(Ctx* c, int rc) {
  if (rc) return rc;
  YH_HIP(hipStreamSynchronize(c->stream));
  return YH_OK;
}

extern "C" {

int yh_get_gauge(yh_ctx* c, double* links) {
  if (!c || !links) { set_error("null argument"); return YH_ERR_ARG; }
  if (!c->gauge_set) { set_error("no gauge field"); return YH_ERR_STATE; }
  YH_HIP(hipSetDevice(c->device));
  return gauge_download(c, links);
}

int yh_represent_gauge_field(yh_ctx* c) {
  if (!c) { set_error("null argument"); return YH_ERR_ARG; }
  if (!c->gauge_set) { set_error("no gauge field"); return YH_ERR_STATE; }
  YH_HIP(hipSetDevice(c->device));
  int rc;
  if ((rc = gauge_represent(c))) return rc;
  if ((rc = clover_build(c))) return rc;
  return md_sync(c, YH_OK);
}

int yh_wilson_gauge_force(yh_ctx* c, double dt, double beta) {
  int rc = md_check(c);
  if (rc) return rc;
  return md_sync(c, md_gauge_force(c, dt, beta));
}

int yh_improved_gauge_force(yh_ctx* c, double dt, double beta, double c0, double c1) {
  int rc = md_check(c);
  if (rc) return rc;
  return md_sync(c, md_improved_gauge_force(c, dt, beta, c0, c1));
}

int yh_avr_wilson(yh_ctx* c, int height, int width, double* out) {
  if (!out) { set_error("null argument"); return YH_ERR_ARG; }
  if (height < 1 || width < 1 || height > 16 || width > 16) { set_error("avr_wilson: loop sides must be 1..16"); return YH_ERR_ARG; }
  int rc = md_check(c);
  if (rc) return rc;
  return md_avr_wilson(c, height, width, out);
}

int yh_update_links(yh_ctx* c, double eps) {
  int rc = md_check(c);
  if (rc) return rc;
  return md_sync(c, md_update_links(c, eps));
}

int yh_reunitarize(yh_ctx* c) {
  int rc = md_check(c);
  if (rc) return rc;
  return md_sync(c, md_reunitarize(c));
}

int yh_plaquette(yh_ctx* c, double* out) {
  if (!out) { set_error("null argument"); return YH_ERR_ARG; }
  int rc = md_check(c);
  if (rc) return rc;
  return md_plaquette(c, out);
}

int yh_apply_bcs_on_gauge_field(yh_ctx* c) {
  int rc = md_check(c);
  if (rc) return rc;
  return md_sync(c, md_apply_gauge_bcs(c));
}

int yh_momenta_energy(yh_ctx* c, double* out) {
  if (!c || !out) { set_error("null argument"); return YH_ERR_ARG; }
  YH_HIP(hipSetDevice(c->device));
  return md_kinetic(c, out);
}

}  // extern "C"
