// Gauge-side kernels (FP64): representation of the links, clover term,
// odd-site clover inverse and log det, and the derived low-precision copies.
//
// represent  : library/repr.cpp:107-280 (written as the action of U on the
//              representation basis, repr.cpp:25-61)
// clover     : library/wilsonloop.cpp:5-31 + library/clover.cpp:93-168
// inverse    : library/clover.cpp:25-91 + library/solver.cpp:97-142 (the
//              same unpivoted LDL^+ factorisation, then the explicit
//              Hermitian inverse is stored instead of the factors, so the
//              apply is one Hermitian mat-vec)
// logdet     : library/clover.cpp:281-305
#include <math.h>
#include <string.h>
#include <type_traits>
#include <vector>
#include "yh_internal.hpp"

namespace yh {

// representation basis b_n (DR <= 15, NC <= 4): the context's table
// tab_basis[n * 16 + row * NC + col]

static const double kSqrtHalf = 0.70710678118654752440;

// anti-Hermitian generator matrix for algebra vector e_n
// (library/suNg.cpp:15-58)
static void alg_unit(int nc, int n, std::vector<double2>& m) {
  m.assign(nc * nc, make_double2(0, 0));
  int k = 0;
  for (int i = 0; i < nc; i++)
    for (int j = 0; j < nc; j++) {
      if (i > j) {
        if (k == n) { m[i * nc + j].y += 1; m[j * nc + i].y += 1; }
        k++;
      } else if (i < j) {
        if (k == n) { m[i * nc + j].x += 1; m[j * nc + i].x -= 1; }
        k++;
      } else if (i > 0) {
        if (k == n) {
          double v = sqrt(2.0 / (i * (i + 1)));
          for (int q = 0; q < i; q++) m[q * nc + q].y += v;
          m[i * nc + i].y -= i * v;
        }
        k++;
      }
    }
}

int gauge_init_basis(Ctx* c) {
  int nc = c->nc, dr = c->dr;
  std::vector<double2> b(15 * 16, make_double2(0, 0));
  if (c->repr == YH_REPR_SYMMETRIC) {
    for (int i = 0, n = 0; i < nc; i++)
      for (int j = 0; j <= i; j++, n++) {
        if (i == j) b[n * 16 + i * nc + i].x = 1;
        else { b[n * 16 + i * nc + j].x = kSqrtHalf; b[n * 16 + j * nc + i].x = kSqrtHalf; }
      }
  } else if (c->repr == YH_REPR_ANTISYMMETRIC) {
    for (int i = 0, n = 0; i < nc; i++)
      for (int j = 0; j < i; j++, n++) {
        b[n * 16 + j * nc + i].x = kSqrtHalf;
        b[n * 16 + i * nc + j].x = -kSqrtHalf;
      }
  } else if (c->repr == YH_REPR_ADJOINT) {
    std::vector<double2> g;
    for (int n = 0; n < dr; n++) {
      alg_unit(nc, n, g);
      // (-i / sqrt 2) * g
      for (int k = 0; k < nc * nc; k++) b[n * 16 + k] = make_double2(kSqrtHalf * g[k].y, -kSqrtHalf * g[k].x);
    }
  }
  return upload_table(c, c->tab_basis, b.data(), b.size());
}

typedef Cx<double> cd;

template <int NC>
__device__ __forceinline__ void load_fund(cd (&u)[NC][NC], const double2* fund, int id, int mu, const Geom& g) {
  const double2* p = fund + fund_at<NC>(id, mu, g);
#pragma unroll
  for (int e = 0; e < NC * NC; e++) {
    const double2 v = p[(size_t)e * g.VHpad];
    u[e / NC][e % NC] = cd(v.x, v.y);
  }
}

template <int NC>
__device__ __forceinline__ void mm(cd (&r)[NC][NC], const cd (&a)[NC][NC], const cd (&b)[NC][NC]) {
#pragma unroll
  for (int i = 0; i < NC; i++)
#pragma unroll
    for (int j = 0; j < NC; j++) {
      cd s(0, 0);
#pragma unroll
      for (int k = 0; k < NC; k++) cmac(s, a[i][k], b[k][j]);
      r[i][j] = s;
    }
}
// r = a * b^+
template <int NC>
__device__ __forceinline__ void mmd(cd (&r)[NC][NC], const cd (&a)[NC][NC], const cd (&b)[NC][NC]) {
#pragma unroll
  for (int i = 0; i < NC; i++)
#pragma unroll
    for (int j = 0; j < NC; j++) {
      cd s(0, 0);
#pragma unroll
      for (int k = 0; k < NC; k++) cmac(s, a[i][k], conj(b[j][k]));
      r[i][j] = s;
    }
}
// r = a^+ * b
template <int NC>
__device__ __forceinline__ void mdm(cd (&r)[NC][NC], const cd (&a)[NC][NC], const cd (&b)[NC][NC]) {
#pragma unroll
  for (int i = 0; i < NC; i++)
#pragma unroll
    for (int j = 0; j < NC; j++) {
      cd s(0, 0);
#pragma unroll
      for (int k = 0; k < NC; k++) cmac_conj(s, a[k][i], b[k][j]);
      r[i][j] = s;
    }
}

// index pair (i >= j, or i > j) of element n of the two-index basis
// (repr.cpp:25-61)
template <bool SYM>
constexpr int pair_row(int n) {
  int i = SYM ? 0 : 1;
  while (n > i - (SYM ? 0 : 1)) n -= (i++) + (SYM ? 1 : 0);
  return i;
}
template <bool SYM>
constexpr int pair_col(int n) {
  const int i = pair_row<SYM>(n);
  return n - (SYM ? i * (i + 1) / 2 : i * (i - 1) / 2);
}

// element (N, M) of the two-index representation of U, in closed form: the
// basis elements have one or two entries, so with n = (i, j), m = (k, l)
//   R_nm = U_ik U_jl + U_il U_jk  (symmetric; sqrt 2 less for each of n, m
//   that is diagonal),   U_ik U_jl - U_il U_jk  (antisymmetric)
// - 2 complex products, where conjugating with every basis matrix takes 108
// a column
template <int NC, bool SYM, int N, int M>
__device__ __forceinline__ cd two_index(const cd (&U)[NC][NC]) {
  constexpr int i = pair_row<SYM>(N), j = pair_col<SYM>(N), k = pair_row<SYM>(M), l = pair_col<SYM>(M);
  constexpr double s2 = 1.41421356237309504880;
  if constexpr (SYM && i == j && k == l) return U[i][k] * U[i][k];
  else if constexpr (SYM && i == j) return s2 * (U[i][k] * U[i][l]);
  else if constexpr (SYM && k == l) return s2 * (U[i][k] * U[j][k]);
  else {
    cd r = U[i][k] * U[j][l];
    const cd a = SYM ? U[i][l] : cd(-U[i][l].re, -U[i][l].im);
    cmac(r, a, U[j][k]);
    return r;
  }
}
static_assert(pair_row<true>(4) == 2 && pair_col<true>(4) == 1 && pair_row<false>(4) == 3 && pair_col<false>(4) == 1,
              "two-index pair order");

// calls f.template operator()<I>() for I = 0 .. N - 1
template <int I, int N, typename F>
__device__ __forceinline__ void static_for(F&& f) {
  if constexpr (I < N) {
    f(std::integral_constant<int, I>());
    static_for<I + 1, N>(f);
  }
}

// R(U) for the fermion representation
template <int NC, int REPR, int D>
__device__ __forceinline__ void represent(cd (&R)[D][D], const cd (&U)[NC][NC], const double2* __restrict__ basis) {
  if constexpr (REPR == YH_REPR_FUNDAMENTAL) {
#pragma unroll
    for (int i = 0; i < NC; i++)
#pragma unroll
      for (int j = 0; j < NC; j++) R[i][j] = U[i][j];
  } else if constexpr (REPR != YH_REPR_ADJOINT) {
    static_for<0, D * D>([&](auto e) {
      constexpr int n = e() / D, m = e() % D;
      R[n][m] = two_index<NC, REPR == YH_REPR_SYMMETRIC, n, m>(U);
    });
  } else {
    for (int m = 0; m < D; m++) {
      // X = U b_m U^+,  R_nm = Tr(b_n X)
      cd W[NC][NC], X[NC][NC];
#pragma unroll
      for (int a = 0; a < NC; a++)
#pragma unroll
        for (int d = 0; d < NC; d++) {
          cd s(0, 0);
#pragma unroll
          for (int q = 0; q < NC; q++) {
            double2 bb = basis[m * 16 + q * NC + d];
            cmac(s, U[a][q], cd(bb.x, bb.y));
          }
          W[a][d] = s;
        }
      mmd<NC>(X, W, U);
      for (int n = 0; n < D; n++) {
        cd s(0, 0);
#pragma unroll
        for (int a = 0; a < NC; a++)
#pragma unroll
          for (int b = 0; b < NC; b++) {
            double2 bb = basis[n * 16 + b * NC + a];
            cmac(s, cd(bb.x, bb.y), X[a][b]);
          }
        R[n][m] = s;
      }
    }
  }
}

// the represented links in every storage precision (no BC sign)
struct LinkCopies {
  double2* f64;
  float2* f32;
  unsigned* f16;
  float4* f32r12;   // the 12-real copies: SU(3) fundamental only (FP64
                    // reads the first two rows of the 18-real planes)
  uint2* f16r12;
};

// fundamental links -> represented links, every copy written from registers
template <int NC, int REPR, int D>
__global__ void k_represent(const double2* __restrict__ fund, LinkCopies out, Geom g,
                            const double2* __restrict__ basis) {
  const int id = blockIdx.x * blockDim.x + threadIdx.x, mu = blockIdx.y;
  if (id >= g.V) return;
  cd U[NC][NC], R[D][D];
  load_fund<NC>(U, fund, id, mu, g);
  represent<NC, REPR, D>(R, U, basis);
  const int p = id >= g.VH;
  const size_t k = id - p * g.VH, S = g.VHpad, dir = p * 4 + mu;
#pragma unroll
  for (int e = 0; e < D * D; e++) {
    const cd v = R[e / D][e % D];
    const size_t o = (dir * D * D + e) * S + k;
    out.f64[o] = make_double2(v.re, v.im);
    out.f32[o] = make_float2((float)v.re, (float)v.im);
    out.f16[o] = f2q((float)v.re) | (f2q((float)v.im) << 16);
  }
  if constexpr (NC == 3 && REPR == YH_REPR_FUNDAMENTAL) {
#pragma unroll
    for (int v = 0; v < 3; v++) {
      const cd a = R[2 * v / 3][2 * v % 3], b = R[(2 * v + 1) / 3][(2 * v + 1) % 3];
      out.f32r12[(dir * 3 + v) * S + k] = make_float4((float)a.re, (float)a.im, (float)b.re, (float)b.im);
      out.f16r12[(dir * 3 + v) * S + k] = make_uint2(f2q((float)a.re) | (f2q((float)a.im) << 16),
                                                     f2q((float)b.re) | (f2q((float)b.im) << 16));
    }
  }
}

__device__ __forceinline__ void coords_of(int id, const Geom& g, int c[4]) { full_coords(id, g, c); }

__device__ __forceinline__ int shift(const int c[4], int mu, int d, const Geom& g) {
  int n[4] = {c[0], c[1], c[2], c[3]};
  n[mu] = (n[mu] + d + g.L[mu]) % g.L[mu];
  return full_index(n[0], n[1], n[2], n[3], g);
}

// packed Hermitian store: n reals then strictly-lower triangle
template <int N>
__device__ __forceinline__ void store_packed(double2* base, int stride, int site, int vec0, const cd (&M)[N][N]) {
  double v[N * N];
  int o = 0;
#pragma unroll
  for (int i = 0; i < N; i++) v[o++] = M[i][i].re;
#pragma unroll
  for (int i = 1; i < N; i++)
#pragma unroll
    for (int j = 0; j < i; j++) { v[o++] = M[i][j].re; v[o++] = M[i][j].im; }
#pragma unroll
  for (int k = 0; k < N * N / 2; k++) base[(size_t)(vec0 + k) * stride + site] = make_double2(v[2 * k], v[2 * k + 1]);
}

template <int N>
__device__ __forceinline__ void load_packed(cd (&M)[N][N], const double2* base, int stride, int site, int vec0) {
  double v[N * N];
#pragma unroll
  for (int k = 0; k < N * N / 2; k++) {
    double2 w = base[(size_t)(vec0 + k) * stride + site];
    v[2 * k] = w.x;
    v[2 * k + 1] = w.y;
  }
  int o = 0;
#pragma unroll
  for (int i = 0; i < N; i++) M[i][i] = cd(v[o++], 0);
#pragma unroll
  for (int i = 1; i < N; i++)
#pragma unroll
    for (int j = 0; j < i; j++) {
      M[i][j] = cd(v[o], v[o + 1]);
      M[j][i] = cd(v[o], -v[o + 1]);
      o += 2;
    }
}

// ---------------------------------------------------------------------------
// Clover term per site -> packed blocks [parity][2 blocks * n^2/2 vec][site]
// (library/clover.cpp:120-168; the dense form is -(c_sw/16) sum_{mu<nu}
// (1/2)[g_mu, g_nu] (x) f_mu_nu, f = Q - Q^+, Q_mu_nu the represented sum of
// the four plaquette leaves, wilsonloop.cpp:5-31), in every storage
// precision.
//
// k_clover_planes (fundamental and two-index representations): S sites per
// workgroup, one thread per (site, plane).  Only the anti-Hermitian part of
// the leaf sum is needed, so in the fundamental the leaves pair up:
//   f = G - G^+,  G = U_mu(x) W(x) + W(x-mu) U_mu(x-mu),
//   W(y) = [upper - lower staple of the link (y, mu) along nu]
// (10 products a plane where the four leaves take 12).  A two-index
// representation forms each leaf and adds R(L) - R(L)^+ entry by entry
// (two_index).  The lower triangles of the six f meet in LDS; then the
// threads of the workgroup share out the packed vectors, in pairs: FP64 and
// FP32 copies from registers, and the 16-bit copy once the block maxima have
// met in LDS too.
// Measured (clover term and represented links of SU(3) at 32^4): 1.97 ms with
// 64 sites, whose six waves fit a CU once at 170 registers; 1.41 ms with 32
// sites (three waves) and three waves per SIMD asked for; 4.7 ms for the
// clover term alone as a group of D_R lanes per site over links stored as
// 144-byte structures.  SU(4) spills at that bound: 64 sites and no bound
// (171 us at 16^4; 195 us with 32 sites).
template <int NC, int REPR>
constexpr int clover_sites() { return REPR == YH_REPR_FUNDAMENTAL && NC == 4 ? 64 : 32; }
template <int NC, int REPR>
constexpr int clover_waves() { return REPR == YH_REPR_FUNDAMENTAL && NC == 3 ? 3 : 1; }

struct CloverCopies {
  double2* f64;
  float4* f32;
  uint2* q16;
  float* nrm;
};

// the packed vector v of an N x N Hermitian block: rows of the diagonal
// entries (2v, 2v + 1) for v < N / 2, else entry (r, c) of the lower triangle
__device__ __forceinline__ void packed_entry(int N, int v, int& r, int& c) {
  int q = v - N / 2;
  r = 1;
  while (q >= r) q -= r++;
  c = q;
}

template <int NC, int REPR, int D>
__global__ void __launch_bounds__((6 * clover_sites<NC, REPR>()), (clover_waves<NC, REPR>())) k_clover_planes(const double2* __restrict__ fund,
                                                                                 CloverCopies out, Geom g, double csw) {
  constexpr int S = clover_sites<NC, REPR>(), N = 2 * D, NT = D * (D + 1) / 2;
  __shared__ double2 F[6][NT][S];       // f_rc, r >= c, of the planes 03, 12, 01, 02, 13, 23
  __shared__ double mx[6][2][S];        // largest |real| of each block, by thread group
  const int pl = S == 64 ? __builtin_amdgcn_readfirstlane(threadIdx.x / S) : threadIdx.x / S;
  const int s = threadIdx.x % S;
  const int b0 = xcd_block(gridDim.x, 64);
  const int p = b0 & 1, k = (b0 >> 1) * S + s;
  const int kk = min(k, g.VH - 1);  // threads past the end compute on the last site and write nothing
  const int id = p * g.VH + kk;
  int c[4];
  site_coords(kk, p, g, c);
  {
    const int mu = pl == 0 || pl == 2 || pl == 3 ? 0 : pl == 5 ? 2 : 1;
    const int nu = pl == 2 ? 1 : pl == 1 || pl == 3 ? 2 : 3;
    int cm[4], cn[4], cb[4], q[4];
    auto L = [&](cd (&u)[NC][NC], int i, int d) { load_fund<NC>(u, fund, i, d, g); };
    if constexpr (REPR == YH_REPR_FUNDAMENTAL) {
      // W of the link (y, mu), y with coordinates cy
      auto W = [&](cd (&w)[NC][NC], const int (&cy)[4], int y) {
        cd a[NC][NC], b[NC][NC], t[NC][NC];
        L(a, y, nu);
        L(b, neighbour(cy, nu, 1, g, q), mu);
        mm<NC>(t, a, b);
        L(a, neighbour(cy, mu, 1, g, q), nu);
        mmd<NC>(w, a, t);
        const int yb = neighbour(cy, nu, -1, g, cb);
        L(a, yb, mu);
        L(b, neighbour(cb, mu, 1, g, q), nu);
        mm<NC>(t, a, b);
        L(a, yb, nu);
        mdm<NC>(b, t, a);
#pragma unroll
        for (int i = 0; i < NC; i++)
#pragma unroll
          for (int j = 0; j < NC; j++) w[i][j] = w[i][j] - b[i][j];
      };
      cd G[NC][NC], w[NC][NC], u[NC][NC];
      W(w, c, id);
      L(u, id, mu);
      mm<NC>(G, u, w);
      // the second half's loads wait for the first half (an opaque zero)
      int z;
#pragma unroll
      for (int i = 0; i < NC; i++)
#pragma unroll
        for (int j = 0; j < NC; j++) __asm__ volatile("" : "+v"(G[i][j].re), "+v"(G[i][j].im));
      __asm__ volatile("v_mov_b32 %0, 0" : "=v"(z));
      const int xb = neighbour(c, mu, -1, g, cm) + z;
      W(w, cm, xb);
      L(u, xb, mu);
#pragma unroll
      for (int i = 0; i < NC; i++)
#pragma unroll
        for (int j = 0; j < NC; j++)
#pragma unroll
          for (int q2 = 0; q2 < NC; q2++) cmac(G[i][j], w[i][q2], u[q2][j]);
#pragma unroll
      for (int i = 0; i < NC; i++)
#pragma unroll
        for (int j = 0; j <= i; j++)
          F[pl][i * (i + 1) / 2 + j][s] = make_double2(G[i][j].re - G[j][i].re, G[i][j].im + G[j][i].im);
    } else {
      const int xm = neighbour(c, mu, 1, g, q), xn = neighbour(c, nu, 1, g, q);
      const int bm = neighbour(c, mu, -1, g, cm), bn = neighbour(c, nu, -1, g, cn);
      const int bm_pn = neighbour(cm, nu, 1, g, q), bm_mn = neighbour(cm, nu, -1, g, q);
      const int bn_pm = neighbour(cn, mu, 1, g, q);
      double fr[NT], fi[NT];
#pragma unroll
      for (int e = 0; e < NT; e++) fr[e] = fi[e] = 0.0;
#pragma unroll 1
      for (int leaf = 0; leaf < 4; leaf++) {
        cd a[NC][NC], b[NC][NC], t[NC][NC], l[NC][NC];
        // the two halves of the leaf, each a product of two links
        if (leaf == 0) {
          L(a, id, nu); L(b, xn, mu); mm<NC>(t, a, b);
          L(a, id, mu); L(b, xm, nu); mm<NC>(l, a, b);
          mmd<NC>(a, l, t);
        } else if (leaf == 1) {
          L(a, id, nu); L(b, bm_pn, mu); mmd<NC>(l, a, b);
          L(a, bm, nu); L(b, bm, mu); mdm<NC>(t, a, b);
          mm<NC>(a, l, t);
        } else if (leaf == 2) {
          L(a, bm_mn, nu); L(b, bm, mu); mm<NC>(l, a, b);
          L(a, bm_mn, mu); L(b, bn, nu); mm<NC>(t, a, b);
          mdm<NC>(a, l, t);
        } else {
          L(a, bn, nu); L(b, bn, mu); mdm<NC>(l, a, b);
          L(a, bn_pm, nu); L(b, id, mu); mmd<NC>(t, a, b);
          mm<NC>(a, l, t);
        }
        static_for<0, D * D>([&](auto e) {
          constexpr int r = e() / D, m = e() % D;
          if constexpr (m <= r) {
            const cd x = two_index<NC, REPR == YH_REPR_SYMMETRIC, r, m>(a);
            const cd y = two_index<NC, REPR == YH_REPR_SYMMETRIC, m, r>(a);
            fr[r * (r + 1) / 2 + m] += x.re - y.re;
            fi[r * (r + 1) / 2 + m] += x.im + y.im;
          }
        });
      }
#pragma unroll
      for (int e = 0; e < NT; e++) F[pl][e][s] = make_double2(fr[e], fi[e]);
    }
  }
  __syncthreads();
  bool zero = csw == 0.0;
  if (g.bc == BC_SF) zero = zero || c[0] == 0 || c[0] == g.L[0] - 1 || c[0] == g.L[0] - 2;
  if (g.bc == BC_OPEN) zero = zero || c[0] == 0 || c[0] == g.L[0] - 1;
  const double cc = zero ? 0.0 : -csw / 16.0;
  // f_rc of plane q
  auto f = [&](int q, int r, int m) -> cd {
    const double2 v = r >= m ? F[q][r * (r + 1) / 2 + m][s] : F[q][m * (m + 1) / 2 + r][s];
    return r >= m ? cd(v.x, v.y) : cd(-v.x, v.y);
  };
  // entry (r, m) of the diagonal D x D block of chiral block b (its lower
  // right one is the negative), clover.cpp:149-165
  auto diag = [&](int b, int r, int m) -> cd {
    const cd x = f(0, r, m), y = f(1, r, m);
    return b == 0 ? cd(cc * (x.im - y.im), cc * (y.re - x.re)) : cd(-cc * (x.im + y.im), cc * (y.re + x.re));
  };
  // entry (D + r, m): the conjugate of entry (m, r) of the upper right block
  auto off = [&](int b, int r, int m) -> cd {
    const cd x = f(2, m, r), y = f(3, m, r), u = f(4, m, r), w = f(5, m, r);
    const cd ct(x.im - y.re, -x.re - y.im), dt(u.re + w.im, u.im - w.re);
    return b == 0 ? cd(cc * (ct.re - dt.re), -cc * (ct.im - dt.im)) : cd(-cc * (ct.re + dt.re), cc * (ct.im + dt.im));
  };
  auto packed = [&](int b, int v) -> cd {
    int r, m;
    if (v < N / 2) {
      r = 2 * v;
      const double x = diag(b, r % D, r % D).re, y = diag(b, (r + 1) % D, (r + 1) % D).re;
      return cd(r < D ? x : -x, r + 1 < D ? y : -y);
    }
    packed_entry(N, v, r, m);
    if (r < D) return diag(b, r, m);
    if (m >= D) {
      const cd x = diag(b, r - D, m - D);
      return cd(-x.re, -x.im);
    }
    return off(b, r - D, m);
  };
  constexpr int PB = N * N / 4, NP = 2 * PB, MP = (NP + 5) / 6;  // vector pairs of a block, of a site, of a thread
  double v[MP][4];
  double m0 = 0.0, m1 = 0.0;
  const size_t stride = g.VHpad;
  const bool on = k < g.VH;
#pragma unroll
  for (int i = 0; i < MP; i++) {
    const int pr = pl + 6 * i;
    if (pr < NP) {
      const int b = pr >= PB, u = pr - b * PB;
      const cd x = packed(b, 2 * u), y = packed(b, 2 * u + 1);
      v[i][0] = x.re; v[i][1] = x.im; v[i][2] = y.re; v[i][3] = y.im;
      const double w = fmax(fmax(fabs(x.re), fabs(x.im)), fmax(fabs(y.re), fabs(y.im)));
      if (b) m1 = fmax(m1, w);
      else m0 = fmax(m0, w);
      if (on) {
        const size_t o = (size_t)p * NP + pr;
        out.f64[2 * o * stride + k] = make_double2(x.re, x.im);
        out.f64[(2 * o + 1) * stride + k] = make_double2(y.re, y.im);
        out.f32[o * stride + k] = make_float4((float)x.re, (float)x.im, (float)y.re, (float)y.im);
      }
    }
  }
  mx[pl][0][s] = m0;
  mx[pl][1][s] = m1;
  __syncthreads();
  if (!on) return;
  m0 = m1 = 0.0;
#pragma unroll
  for (int q = 0; q < 6; q++) {
    m0 = fmax(m0, mx[q][0][s]);
    m1 = fmax(m1, mx[q][1][s]);
  }
  if (pl == 0) {
    out.nrm[(size_t)(2 * p) * stride + k] = (float)m0;
    out.nrm[(size_t)(2 * p + 1) * stride + k] = (float)m1;
  }
  const double i0 = m0 > 0.0 ? 1.0 / (double)(float)m0 : 0.0, i1 = m1 > 0.0 ? 1.0 / (double)(float)m1 : 0.0;
#pragma unroll
  for (int i = 0; i < MP; i++) {
    const int pr = pl + 6 * i;
    if (pr < NP) {
      const double inv = pr >= PB ? i1 : i0;
      out.q16[((size_t)p * NP + pr) * stride + k] = make_uint2(
          pack_q2((float)(v[i][0] * inv), (float)(v[i][1] * inv)), pack_q2((float)(v[i][2] * inv), (float)(v[i][3] * inv)));
    }
  }
}

// Adjoint representation, where row i of R(L) takes a product with every
// basis matrix: a group of D_R lanes per site, lane i computing row i of
// every D_R x D_R matrix, so that no lane holds more than a few rows.  Per
// plane, lanes 0..3 of the group each form one leaf in the fundamental as a
// product of four links, L = F1 F2 F3 F4, and put it in LDS; every lane then
// adds row i of R(L) for the four leaves:
//   R[i][m] = sum_cd Y_cd (b_m)_dc,  Y = L^+ b_i L
// (follows from represent()).  The at/bt/ct/dt combinations need column
// i of the plane sum too, which the group exchanges through LDS.  The block
// is one wave; LDS traffic needs only wavefront-scope fences (a wave's LDS
// operations execute in order).
// LDS exchange between lanes of one wave: a wavefront-scope fence (the
// wave's LDS operations execute in order, so it emits no wait; it keeps the
// compiler from moving LDS accesses across it)
__device__ __forceinline__ void cb_fence() { __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront"); }

template <int NC, int D>
__global__ void __launch_bounds__(64) k_clover_build_rows(const double2* __restrict__ fund, double2* __restrict__ out,
                                                         Geom g, double csw, const double2* __restrict__ basis) {
  constexpr int G = 64 / D, N = 2 * D, NN = NC * NC;
  __shared__ double2 lv[G][4][NN];  // the plane's four leaves
  __shared__ double2 qx[G][D * D];  // row exchange
  __shared__ double2 bl[D * 16];    // the representation basis
  const int lane = threadIdx.x;
  for (int e = lane; e < D * 16; e += 64) bl[e] = basis[e];
  cb_fence();
  const int gi = min(lane / D, G - 1);
  const int i = lane % D;
  const int grp = blockIdx.x * G + gi;
  const bool on = lane < G * D && grp < g.V;
  const int id = grp < g.V ? grp : g.V - 1;  // tail lanes compute on a valid site and write nothing
  int c[4];
  full_coords(id, g, c);
  bool zero = csw == 0.0;
  if (g.bc == BC_SF) zero = zero || c[0] == 0 || c[0] == g.L[0] - 1 || c[0] == g.L[0] - 2;
  if (g.bc == BC_OPEN) zero = zero || c[0] == 0 || c[0] == g.L[0] - 1;
  cd r1[D], r2[D];  // at, bt rows, then ct, dt rows
  const double cc = -csw / 16.0;
  const int p = id >= g.VH, k = id - p * g.VH;
  double2* base = out + (size_t)p * (N * N) * g.VHpad;
  // output addresses are formed where they are stored (from an opaque base:
  // hoisted out of the plane loop they would hold dozens of registers)
  double2* ob = base;
  auto put_re = [&](int vec0, int o, double v) {
    if (on) ((double*)(ob + (size_t)(vec0 + o / 2) * g.VHpad + k))[o & 1] = v;
  };
  auto put_cx = [&](int vec0, int o, cd v) {  // o even
    if (on) ob[(size_t)(vec0 + o / 2) * g.VHpad + k] = make_double2(v.re, v.im);
  };
  auto lo = [](int r, int s) { return N + 2 * (r * (r - 1) / 2 + s); };  // packed index of (r, s), r > s
  // planes 03, 12, 01, 02, 13, 23 (clover.cpp:135-156)
#pragma unroll 1
  for (int pl = 0; pl < 6; pl++) {
    const int mu = pl == 0 ? 0 : pl == 1 ? 1 : pl == 2 ? 0 : pl == 3 ? 0 : pl == 4 ? 1 : 2;
    const int nu = pl == 0 ? 3 : pl == 1 ? 2 : pl == 2 ? 1 : pl == 3 ? 2 : pl == 4 ? 3 : 3;
    // leaves: lane q < 4 of the group forms leaf q
    for (int q = i; q < 4; q += D) {
      int xm = shift(c, mu, 1, g), xn = shift(c, nu, 1, g);
      int bm = shift(c, mu, -1, g), bn = shift(c, nu, -1, g);
      int cb[4], cn[4];
      coords_of(bm, g, cb);
      coords_of(bn, g, cn);
      const int bm_pn = shift(cb, nu, 1, g), bm_mn = shift(cb, nu, -1, g), bn_pm = shift(cn, mu, 1, g);
      // the four leaves as products F1 F2 F3 F4 (leaf 0: U(x,mu) U(x+mu,nu)
      // U(x+nu,mu)^+ U(x,nu)^+, and the others around x)
      int s[4], d[4];
      bool h[4];
      if (q == 0) {
        s[0] = id; d[0] = mu; h[0] = false; s[1] = xm; d[1] = nu; h[1] = false;
        s[2] = xn; d[2] = mu; h[2] = true; s[3] = id; d[3] = nu; h[3] = true;
      } else if (q == 1) {
        s[0] = id; d[0] = nu; h[0] = false; s[1] = bm_pn; d[1] = mu; h[1] = true;
        s[2] = bm; d[2] = nu; h[2] = true; s[3] = bm; d[3] = mu; h[3] = false;
      } else if (q == 2) {
        s[0] = bm; d[0] = mu; h[0] = true; s[1] = bm_mn; d[1] = nu; h[1] = true;
        s[2] = bm_mn; d[2] = mu; h[2] = false; s[3] = bn; d[3] = nu; h[3] = false;
      } else {
        s[0] = bn; d[0] = nu; h[0] = true; s[1] = bn; d[1] = mu; h[1] = false;
        s[2] = bn_pm; d[2] = nu; h[2] = false; s[3] = id; d[3] = mu; h[3] = true;
      }
      // L = F1 F2 F3 F4, each factor a link or its dagger, multiplied in
      // place row by row
      cd L[NC][NC], F[NC][NC];
      auto ldf = [&](cd (&u)[NC][NC], int st, int dr, bool dg) {
        const double2* pf = fund + fund_at<NC>(st, dr, g);
#pragma unroll
        for (int a = 0; a < NC; a++)
#pragma unroll
          for (int b = 0; b < NC; b++) {
            const double2 v = pf[(size_t)(a * NC + b) * g.VHpad];
            u[a][b] = cd(v.x, dg ? -v.y : v.y);
          }
        // a dagger is transposed in registers: the lanes of a wave, some of
        // which take it and some not, read the same component plane at a time
        // (SU(3) adjoint, 24^4: represented links and clover term 7.66 ms; by
        // transposed addresses 9.25)
#pragma unroll
        for (int a = 0; a < NC; a++)
#pragma unroll
          for (int b = 0; b < a; b++) {
            const cd v = u[a][b], w = u[b][a];
            u[a][b] = dg ? w : v;
            u[b][a] = dg ? v : w;
          }
      };
      ldf(L, s[0], d[0], h[0]);
#pragma unroll
      for (int f = 1; f < 4; f++) {
        ldf(F, s[f], d[f], h[f]);
#pragma unroll
        for (int a = 0; a < NC; a++) {
          cd row[NC];
#pragma unroll
          for (int b = 0; b < NC; b++) {
            cd t(0, 0);
#pragma unroll
            for (int kk = 0; kk < NC; kk++) cmac(t, L[a][kk], F[kk][b]);
            row[b] = t;
          }
#pragma unroll
          for (int b = 0; b < NC; b++) L[a][b] = row[b];
        }
      }
#pragma unroll
      for (int a = 0; a < NC; a++)
#pragma unroll
        for (int b = 0; b < NC; b++) lv[gi][q][a * NC + b] = make_double2(L[a][b].re, L[a][b].im);
    }
    cb_fence();
    // row i of the plane sum Q = sum_leaves R(L)
    cd qr[D];
#pragma unroll
    for (int m = 0; m < D; m++) qr[m] = cd(0, 0);
#pragma unroll 1
    for (int q = 0; q < 4; q++) {
      cd L[NC][NC];
#pragma unroll
      for (int a = 0; a < NC; a++)
#pragma unroll
        for (int b = 0; b < NC; b++) {
          const double2 v = lv[gi][q][a * NC + b];
          L[a][b] = cd(v.x, v.y);
        }
      // column dd of T = b_i L and of Y = L^+ T, and its terms of row i of R(L)
#pragma unroll
      for (int dd = 0; dd < NC; dd++) {
        // basis from LDS through an opaque zero per column, so that the
        // compiler neither hoists the reads out of the loops nor issues them
        // all at once
        int z = 0;
        __asm__ volatile("" : "+v"(z));
        const double2* bs = bl + z;
        cd tc[NC], yc[NC];
#pragma unroll
        for (int a = 0; a < NC; a++) {
          cd t(0, 0);
#pragma unroll
          for (int b = 0; b < NC; b++) {
            const double2 v = bs[i * 16 + a * NC + b];
            cmac(t, cd(v.x, v.y), L[b][dd]);
          }
          tc[a] = t;
        }
#pragma unroll
        for (int cc2 = 0; cc2 < NC; cc2++) {
          cd y(0, 0);
#pragma unroll
          for (int a = 0; a < NC; a++) {
            cmac_conj(y, L[a][cc2], tc[a]);
          }
          yc[cc2] = y;
        }
#pragma unroll
        for (int m = 0; m < D; m++) {
#pragma unroll
          for (int cc2 = 0; cc2 < NC; cc2++) {
            const double2 bb = bs[m * 16 + dd * NC + cc2];
            cmac(qr[m], yc[cc2], cd(bb.x, bb.y));
          }
        }
      }
    }
    // column i through LDS
    cb_fence();
#pragma unroll
    for (int m = 0; m < D; m++) qx[gi][i * D + m] = make_double2(qr[m].re, qr[m].im);
    cb_fence();
    cd qc[D];
#pragma unroll
    for (int m = 0; m < D; m++) {
      const double2 v = qx[gi][m * D + i];
      qc[m] = cd(v.x, v.y);
    }
    cb_fence();
    // Q[i][j] = qr[j], Q[j][i] = qc[j] (clover.cpp:149-156)
#pragma unroll
    for (int j = 0; j < D; j++) {
      const cd a = qr[j], b = qc[j];
      if (pl == 0) r1[j] = cd(a.im + b.im, b.re - a.re);                    // at
      else if (pl == 1) r2[j] = cd(a.im + b.im, a.re - b.re);               // bt
      else if (pl == 2) r1[j] = cd(a.im + b.im, b.re - a.re);               // ct
      else if (pl == 3) r1[j] = r1[j] + cd(-a.re + b.re, -a.im - b.im);     // ct
      else if (pl == 4) r2[j] = cd(a.re - b.re, a.im + b.im);               // dt
      else r2[j] = r2[j] + cd(a.im + b.im, -a.re + b.re);                   // dt
    }
    if (pl == 1 || pl == 5) {
      int z = 0;
      __asm__ volatile("" : "+v"(z));
      ob = base + z;
    }
    if (pl == 1) {
      // A = cc (at - bt) (block 0, diagonal blocks), C (block 1)
#pragma unroll
      for (int j = 0; j < D; j++) {
        const cd at = r1[j], bt = r2[j];
        cd A(cc * (at.re - bt.re), cc * (at.im + bt.im));
        cd C(-cc * (at.re + bt.re), cc * (bt.im - at.im));
        if (zero) A = C = cd(0, 0);
        if (j == i) {
          put_re(0, i, A.re);
          put_re(0, D + i, -A.re);
          put_re(N * N / 2, i, C.re);
          put_re(N * N / 2, D + i, -C.re);
        } else if (j < i) {
          put_cx(0, lo(i, j), A);
          put_cx(0, lo(D + i, D + j), cd(-A.re, -A.im));
          put_cx(N * N / 2, lo(i, j), C);
          put_cx(N * N / 2, lo(D + i, D + j), cd(-C.re, -C.im));
        }
      }
    } else if (pl == 5) {
      // B (block 0) and D (block 1) off-diagonal blocks, stored as their
      // conjugates in the lower left
#pragma unroll
      for (int j = 0; j < D; j++) {
        const cd ct = r1[j], dt = r2[j];
        cd B(cc * (ct.re - dt.re), cc * (ct.im - dt.im));
        cd Dm(-cc * (ct.re + dt.re), -cc * (ct.im + dt.im));
        if (zero) B = Dm = cd(0, 0);
        put_cx(0, lo(D + j, i), conj(B));
        put_cx(N * N / 2, lo(D + j, i), conj(Dm));
      }
    }
  }
}

// Odd-site inverse of sigma + c_f shift + clover, per chiral block, and its
// log det (the reference factors with an unpivoted LDL^+, solver.cpp:97-117),
// in every storage precision.
// k_clover_sweep (D_R <= 6): one thread per (site, block), the packed lower
// triangle (N^2 reals) in registers, inverted in place by the Hermitian sweep
// without pivoting: step k takes a_ij -= a_ik conj(a_jk) / d, a_ik /= d,
// a_kk = -1 / d, and N steps leave minus the inverse.  Its pivots d are the
// d_i of the unpivoted LDL^+ (both are the ratios of the leading principal
// minors), so log det = sum log |d_i|.  Every load and store is a whole
// component plane segment; the group-of-lanes kernel below, which it replaces
// at these sizes, writes 16-byte pieces.
template <int D>
__global__ void __launch_bounds__(128) k_clover_sweep(const double2* __restrict__ clov, CloverCopies out,
                                                      double* __restrict__ logdet, Geom g, double sigma) {
  constexpr int N = 2 * D, NV = N * N / 2;
  __shared__ double ld1[64];
  const int s = threadIdx.x & 63, b = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int k = blockIdx.x * 64 + s;
  const int kk = min(k, g.VH - 1);  // threads past the end compute on the last site and write nothing
  int c[4];
  site_coords(kk, 1, g, c);
  const size_t stride = g.VHpad;
  const double2* src = clov + ((size_t)N * N + b * NV) * stride + kk;  // odd parity
  double d[N];
  cd l[N * (N - 1) / 2];  // (i, j), i > j, at i (i - 1) / 2 + j
  const double sh = sigma + bc_cf_shift(c[0], g);
#pragma unroll
  for (int v = 0; v < N / 2; v++) {
    const double2 x = src[(size_t)v * stride];
    d[2 * v] = x.x + sh;
    d[2 * v + 1] = x.y + sh;
  }
#pragma unroll
  for (int v = 0; v < N * (N - 1) / 2; v++) {
    const double2 x = src[(size_t)(N / 2 + v) * stride];
    l[v] = cd(x.x, x.y);
  }
  double ld = 0.0;
#pragma unroll
  for (int q = 0; q < N; q++) {
    ld += log(fabs(d[q]));
    const double ip = 1.0 / d[q];
    cd col[N];  // a_iq
#pragma unroll
    for (int i = 0; i < N; i++)
      if (i != q) col[i] = i > q ? l[i * (i - 1) / 2 + q] : conj(l[q * (q - 1) / 2 + i]);
#pragma unroll
    for (int i = 0; i < N; i++) {
      if (i == q) continue;
      const cd w(-ip * col[i].re, -ip * col[i].im);
      d[i] = fma(w.im, col[i].im, fma(w.re, col[i].re, d[i]));
#pragma unroll
      for (int j = 0; j < i; j++)
        if (j != q) {
          cd& a = l[i * (i - 1) / 2 + j];
          a.re = fma(w.im, col[j].im, fma(w.re, col[j].re, a.re));
          a.im = fma(-w.re, col[j].im, fma(w.im, col[j].re, a.im));
        }
      if (i > q) l[i * (i - 1) / 2 + q] = cd(-w.re, -w.im);
      else l[q * (q - 1) / 2 + i] = cd(-w.re, w.im);
    }
    d[q] = -ip;
  }
  if (b) ld1[s] = ld;
  __syncthreads();
  if (k >= g.VH) return;
  if (!b) logdet[k] = ld + ld1[s];
  auto vec = [&](int v) -> cd {  // packed vector v of the inverse
    if (v < N / 2) return cd(-d[2 * v], -d[2 * v + 1]);
    return cd(-l[v - N / 2].re, -l[v - N / 2].im);
  };
  double mx = 0.0;
#pragma unroll
  for (int v = 0; v < NV; v++) {
    const cd x = vec(v);
    mx = fmax(mx, fmax(fabs(x.re), fabs(x.im)));
    out.f64[((size_t)b * NV + v) * stride + k] = make_double2(x.re, x.im);
  }
  const double inv = mx > 0.0 ? 1.0 / (double)(float)mx : 0.0;
  out.nrm[(size_t)b * stride + k] = (float)mx;
#pragma unroll
  for (int u = 0; u < NV / 2; u++) {
    const cd x = vec(2 * u), y = vec(2 * u + 1);
    const size_t o = ((size_t)b * NV / 2 + u) * stride + k;
    out.f32[o] = make_float4((float)x.re, (float)x.im, (float)y.re, (float)y.im);
    out.q16[o] = make_uint2(pack_q2((float)(x.re * inv), (float)(x.im * inv)),
                            pack_q2((float)(y.re * inv), (float)(y.im * inv)));
  }
}

// The same for D_R = 8, whose 256 reals a block do not fit one thread: a
// group of N = 2 D_R lanes per odd site, lane r holding row r of the
// block: in-place Gauss-Jordan without pivoting (the same pivots).  Each
// step's normalised pivot row reaches the group through LDS (the block is
// one wave: a wave's LDS operations execute in order, wavefront-scope
// fences suffice).  The two chiral blocks of a site run one after the other in
// the same group, which then sums the 2N log |d_i| in fixed order.
template <int D>
__global__ void __launch_bounds__(64) k_clover_invert_rows(const double2* __restrict__ clov, double2* __restrict__ inv,
                                                          double* __restrict__ logdet, Geom g, double sigma) {
  constexpr int N = 2 * D, G = 64 / N;
  __shared__ double2 pr[G][N];   // pivot row
  __shared__ double lds_ld[G][N];
  const int lane = threadIdx.x;
  const int gi = min(lane / N, G - 1);
  const int r = lane % N;
  const int grp = blockIdx.x * G + gi;
  const bool on = lane < G * N && grp < g.VH;
  const int k = grp < g.VH ? grp : g.VH - 1;  // tail lanes compute on a valid site and write nothing
  int c[4];
  site_coords(k, 1, g, c);
  const double s = sigma + bc_cf_shift(c[0], g);
  const double2* src = clov + (size_t)1 * (N * N) * g.VHpad;  // odd parity
  auto lo = [](int a, int b) { return N + 2 * (a * (a - 1) / 2 + b); };  // packed real index of (a, b), a > b
  auto get = [&](const double2* base, int vec0, int o) -> double {
    return ((const double*)(base + (size_t)(vec0 + o / 2) * g.VHpad + k))[o & 1];
  };
  double ld = 0.0;
#pragma unroll 1
  for (int blk = 0; blk < 2; blk++) {
    const int vec0 = blk * N * N / 2;
    // row r of sigma + clover
    cd a[N];
#pragma unroll
    for (int j = 0; j < N; j++) {
      if (j == r) a[j] = cd(get(src, vec0, r) + s, 0.0);
      else if (j < r) a[j] = cd(get(src, vec0, lo(r, j)), get(src, vec0, lo(r, j) + 1));
      else a[j] = cd(get(src, vec0, lo(j, r)), -get(src, vec0, lo(j, r) + 1));
    }
#pragma unroll
    for (int kk = 0; kk < N; kk++) {
      if (r == kk) {
        const double d = a[kk].re;  // real for a Hermitian block, as the LDL^+ d
        const double ip = 1.0 / d;
        ld += log(fabs(d));
#pragma unroll
        for (int j = 0; j < N; j++) a[j] = j == kk ? cd(ip, 0.0) : ip * a[j];
#pragma unroll
        for (int j = 0; j < N; j++) pr[gi][j] = make_double2(a[j].re, a[j].im);
      }
      cb_fence();
      if (r != kk) {
        const cd f = a[kk];
#pragma unroll
        for (int j = 0; j < N; j++) {
          const double2 v = pr[gi][j];
          const cd pj(v.x, v.y);
          a[j] = j == kk ? cd(0.0, 0.0) - f * pj : a[j] - f * pj;
        }
      }
      cb_fence();
    }
    // row r of the inverse: diagonal and strictly lower part, packed
    if (on) {
      double2* base = inv;
      double dr = 0.0;  // a[r] without indexing the register array by a lane value
#pragma unroll
      for (int j = 0; j < N; j++) dr = j == r ? a[j].re : dr;
      ((double*)(base + (size_t)(vec0 + r / 2) * g.VHpad + k))[r & 1] = dr;
#pragma unroll
      for (int j = 0; j < N; j++)
        if (j < r) base[(size_t)(vec0 + lo(r, j) / 2) * g.VHpad + k] = make_double2(a[j].re, a[j].im);
    }
  }
  // log det of both blocks: lane r holds the log |d| of pivot r of each
  lds_ld[gi][r] = ld;
  cb_fence();
  if (r == 0) {
    double t = 0.0;
#pragma unroll
    for (int j = 0; j < N; j++) t += lds_ld[gi][j];
    if (on) logdet[k] = t;
  }
}

// packed clover F64 double2[vec] -> F32 float4[vec/2] (same real order)
__global__ void k_clover_to_f32(const double2* __restrict__ src, float4* __restrict__ dst, int nvec4, int VHpad, int VH) {
  int k = blockIdx.x * blockDim.x + threadIdx.x;
  if (k >= VH) return;
  int v = blockIdx.y;
  if (v >= nvec4) return;
  double2 a = src[(size_t)(2 * v) * VHpad + k], b = src[(size_t)(2 * v + 1) * VHpad + k];
  dst[(size_t)v * VHpad + k] = make_float4((float)a.x, (float)a.y, (float)b.x, (float)b.y);
}

// packed clover F64 -> 16-bit fixed point: per site and block the largest
// |real| becomes the block scale, 4 reals per uint2 (same real order)
__global__ void k_clover_to_q16(const double2* __restrict__ src, uint2* __restrict__ dst, float* __restrict__ nrm,
                                int n2, int VHpad, int VH) {
  int k = blockIdx.x * blockDim.x + threadIdx.x;
  if (k >= VH) return;
  for (int blk = 0; blk < 2; blk++) {
    const double2* s = src + (size_t)blk * (n2 / 2) * VHpad + k;
    double mx = 0.0;
    for (int v = 0; v < n2 / 2; v++) {
      double2 a = s[(size_t)v * VHpad];
      mx = fmax(mx, fmax(fabs(a.x), fabs(a.y)));
    }
    const float sc = (float)mx;
    const double inv = mx > 0.0 ? 1.0 / (double)sc : 0.0;
    nrm[(size_t)blk * VHpad + k] = sc;
    uint2* d = dst + (size_t)blk * (n2 / 4) * VHpad + k;
    for (int v = 0; v < n2 / 4; v++) {
      double2 a = s[(size_t)(2 * v) * VHpad], b = s[(size_t)(2 * v + 1) * VHpad];
      d[(size_t)v * VHpad] = make_uint2(pack_q2((float)(a.x * inv), (float)(a.y * inv)),
                                        pack_q2((float)(b.x * inv), (float)(b.y * inv)));
    }
  }
}

// ---------------------------------------------------------------------------
// host wrappers
// ---------------------------------------------------------------------------
#define YH_DISPATCH_MODEL(NCV, REPRV, DV, ...) \
  if (c->nc == NCV && c->repr == REPRV) { constexpr int NC_ = NCV, REPR_ = REPRV, D_ = DV; __VA_ARGS__; return YH_OK; }

#define YH_PLANE_MODELS(...)                                   \
  YH_DISPATCH_MODEL(3, YH_REPR_FUNDAMENTAL, 3, __VA_ARGS__)    \
  YH_DISPATCH_MODEL(2, YH_REPR_FUNDAMENTAL, 2, __VA_ARGS__)    \
  YH_DISPATCH_MODEL(4, YH_REPR_FUNDAMENTAL, 4, __VA_ARGS__)    \
  YH_DISPATCH_MODEL(3, YH_REPR_SYMMETRIC, 6, __VA_ARGS__)      \
  YH_DISPATCH_MODEL(2, YH_REPR_SYMMETRIC, 3, __VA_ARGS__)      \
  YH_DISPATCH_MODEL(3, YH_REPR_ANTISYMMETRIC, 3, __VA_ARGS__)  \
  YH_DISPATCH_MODEL(4, YH_REPR_ANTISYMMETRIC, 6, __VA_ARGS__)

#define YH_ALL_MODELS(...)                                     \
  YH_PLANE_MODELS(__VA_ARGS__)                                 \
  YH_DISPATCH_MODEL(2, YH_REPR_ADJOINT, 3, __VA_ARGS__)        \
  YH_DISPATCH_MODEL(3, YH_REPR_ADJOINT, 8, __VA_ARGS__)

static int grid1(long n) { return (int)((n + 255) / 256); }
static int grid_bs(long n, int bs) { return (int)((n + bs - 1) / bs); }

int gauge_represent(Ctx* c) {
  const bool r12 = c->nc == 3 && c->repr == YH_REPR_FUNDAMENTAL;
  const size_t per = (size_t)8 * c->g.VHpad;  // (parity, direction) planes
  auto alloc = [&](int prec, int recon, size_t bytes) -> int {
    if (!c->links[prec][recon]) YH_HIP(hipMalloc(&c->links[prec][recon], per * bytes));
    return YH_OK;
  };
  const size_t n = (size_t)c->dr * c->dr;
  int rc;
  if ((rc = alloc(PREC_F64, RECON_18, n * sizeof(double2))) || (rc = alloc(PREC_F32, RECON_18, n * sizeof(float2))) ||
      (rc = alloc(PREC_F16, RECON_18, n * sizeof(unsigned))))
    return rc;
  if (r12) {
    c->links[PREC_F64][RECON_12] = c->links[PREC_F64][RECON_18];
    if ((rc = alloc(PREC_F32, RECON_12, 3 * sizeof(float4))) || (rc = alloc(PREC_F16, RECON_12, 3 * sizeof(uint2))))
      return rc;
  }
  const LinkCopies out = {(double2*)c->links[PREC_F64][RECON_18], (float2*)c->links[PREC_F32][RECON_18],
                          (unsigned*)c->links[PREC_F16][RECON_18], (float4*)c->links[PREC_F32][RECON_12],
                          (uint2*)c->links[PREC_F16][RECON_12]};
  YH_ALL_MODELS(hipLaunchKernelGGL((k_represent<NC_, REPR_, D_>), dim3(grid1(c->g.V), 4), dim3(256), 0, c->stream,
                                   c->fund, out, c->g, c->tab_basis);
                YH_HIP(hipGetLastError()));
  set_error("unsupported (nc, repr) model");
  return YH_ERR_UNSUPPORTED;
}

int clover_build(Ctx* c) {
  // per site and parity: two N x N Hermitian blocks = 2 N^2 reals
  //   FP64: N^2 double2 vectors, FP32: N^2 / 2 float4 vectors
  int N = 2 * c->dr;
  size_t bytes = (size_t)2 * N * N * c->g.VHpad * sizeof(double2);
  if (!c->clov[PREC_F64]) YH_HIP(hipMalloc(&c->clov[PREC_F64], bytes));
  if (!c->clov[PREC_F32]) YH_HIP(hipMalloc(&c->clov[PREC_F32], bytes / 2));
  if (!c->clov[PREC_F16]) YH_HIP(hipMalloc(&c->clov[PREC_F16], bytes / 4));
  if (!c->clov_nrm) YH_HIP(hipMalloc(&c->clov_nrm, sizeof(float) * 4 * c->g.VHpad));
  const CloverCopies out = {(double2*)c->clov[PREC_F64], (float4*)c->clov[PREC_F32], (uint2*)c->clov[PREC_F16],
                            c->clov_nrm};
  c->cl_sigma = 0xF00F;  // invalidate the inverse (clover.cpp:337)
  if (c->repr != YH_REPR_ADJOINT) {
    YH_PLANE_MODELS(constexpr int S_ = clover_sites<NC_, REPR_>();
                    hipLaunchKernelGGL((k_clover_planes<NC_, REPR_, D_>), dim3((c->g.VH + S_ - 1) / S_ * 2),
                                       dim3(6 * S_), 0, c->stream, c->fund, out, c->g, c->csw);
                    YH_HIP(hipGetLastError()));
    set_error("unsupported (nc, repr) model");
    return YH_ERR_UNSUPPORTED;
  }
  // a group of D_R lanes per site
  if (c->nc == 2)
    hipLaunchKernelGGL((k_clover_build_rows<2, 3>), dim3(grid_bs(c->g.V, 64 / 3)), dim3(64), 0, c->stream, c->fund,
                       out.f64, c->g, c->csw, c->tab_basis);
  else if (c->nc == 3)
    hipLaunchKernelGGL((k_clover_build_rows<3, 8>), dim3(grid_bs(c->g.V, 64 / 8)), dim3(64), 0, c->stream, c->fund,
                       out.f64, c->g, c->csw, c->tab_basis);
  else {
    set_error("unsupported (nc, repr) model");
    return YH_ERR_UNSUPPORTED;
  }
  // FP32 and 16-bit copies (both parities)
  for (int p = 0; p < 2; p++) {
    dim3 grid(grid1(c->g.VH), N * N / 2);
    const double2* src = out.f64 + (size_t)p * (N * N) * c->g.VHpad;
    hipLaunchKernelGGL(k_clover_to_f32, grid, dim3(256), 0, c->stream, src,
                       out.f32 + (size_t)p * (N * N / 2) * c->g.VHpad, N * N / 2, c->g.VHpad, c->g.VH);
    hipLaunchKernelGGL(k_clover_to_q16, dim3(grid1(c->g.VH)), dim3(256), 0, c->stream, src,
                       out.q16 + (size_t)p * (N * N / 2) * c->g.VHpad, out.nrm + (size_t)p * 2 * c->g.VHpad, N * N,
                       c->g.VHpad, c->g.VH);
  }
  YH_HIP(hipGetLastError());
  return YH_OK;
}

// the inverse buffers of every precision, allocated once per context (at
// yh_set_gauge), so that solves never allocate
int clover_reserve_inverse(Ctx* c) {
  int N = 2 * c->dr;
  size_t bytes = (size_t)N * N * c->g.VHpad * sizeof(double2);  // odd sites only
  if (!c->clinv[PREC_F64]) YH_HIP(hipMalloc(&c->clinv[PREC_F64], bytes));
  if (!c->logdet_site) YH_HIP(hipMalloc(&c->logdet_site, sizeof(double) * c->g.VHpad));
  size_t b32 = (size_t)(N * N / 2) * c->g.VHpad * sizeof(float4);
  if (!c->clinv[PREC_F32]) YH_HIP(hipMalloc(&c->clinv[PREC_F32], b32));
  size_t b16 = (size_t)(N * N / 2) * c->g.VHpad * sizeof(uint2);
  if (!c->clinv[PREC_F16]) YH_HIP(hipMalloc(&c->clinv[PREC_F16], b16));
  if (!c->clinv_nrm) YH_HIP(hipMalloc(&c->clinv_nrm, sizeof(float) * 2 * c->g.VHpad));
  return YH_OK;
}

int clover_invert(Ctx* c, double sigma) {
  if (sigma == c->cl_sigma) return YH_OK;  // clover.cpp:314-321
  int N = 2 * c->dr;
  int rc = clover_reserve_inverse(c);
  if (rc) return rc;
  const double2* src = (const double2*)c->clov[PREC_F64];
  double2* inv = (double2*)c->clinv[PREC_F64];
  const CloverCopies out = {inv, (float4*)c->clinv[PREC_F32], (uint2*)c->clinv[PREC_F16], c->clinv_nrm};
  const dim3 grid((c->g.VH + 63) / 64);
#define YH_SWEEP(DD) \
  hipLaunchKernelGGL(k_clover_sweep<DD>, grid, dim3(128), 0, c->stream, src, out, c->logdet_site, c->g, sigma)
  switch (c->dr) {
    case 2: YH_SWEEP(2); break;
    case 3: YH_SWEEP(3); break;
    case 4: YH_SWEEP(4); break;
    case 6: YH_SWEEP(6); break;
    case 8: {
      hipLaunchKernelGGL(k_clover_invert_rows<8>, dim3(grid_bs(c->g.VH, 64 / 16)), dim3(64), 0, c->stream, src, inv,
                         c->logdet_site, c->g, sigma);
      hipLaunchKernelGGL(k_clover_to_f32, dim3(grid1(c->g.VH), N * N / 2), dim3(256), 0, c->stream, inv, out.f32,
                         N * N / 2, c->g.VHpad, c->g.VH);
      hipLaunchKernelGGL(k_clover_to_q16, dim3(grid1(c->g.VH)), dim3(256), 0, c->stream, inv, out.q16, out.nrm, N * N,
                         c->g.VHpad, c->g.VH);
      break;
    }
    default: set_error("unsupported representation dimension"); return YH_ERR_UNSUPPORTED;
  }
#undef YH_SWEEP
  YH_HIP(hipGetLastError());
  c->cl_sigma = sigma;
  return YH_OK;
}

// reference AoS layouts for read-back
__global__ void k_repr_to_aos(const double2* __restrict__ src, double* __restrict__ dst, Geom g, int D) {
  int t = blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= 4 * g.V) return;
  int id = t >> 2, mu = t & 3;
  int p = id >= g.VH, k = id - p * g.VH;
  int c[4];
  site_coords(k, p, g, c);
  double sgn = (g.bc == BC_ANTIPERIODIC && mu == 0 && c[0] == 0) ? -1.0 : 1.0;
  double* o = dst + (size_t)t * 2 * D * D;
  for (int e = 0; e < D * D; e++) {
    double2 v = src[((size_t)(p * 4 + mu) * D * D + e) * g.VHpad + k];
    o[e] = sgn * v.x;
    o[D * D + e] = sgn * v.y;
  }
}

__global__ void k_clover_to_aos(const double2* __restrict__ src, double* __restrict__ dst, Geom g, int D) {
  int id = blockIdx.x * blockDim.x + threadIdx.x;
  if (id >= g.V) return;
  int p = id >= g.VH, k = id - p * g.VH;
  int N = 2 * D;
  const double2* base = src + (size_t)p * (N * N) * g.VHpad;
  for (int blk = 0; blk < 2; blk++) {
    // unpack into A (or C) = M[i][j], B (or D) = M[i][D + j]
    double v[16 * 16];
    for (int q = 0; q < N * N / 2; q++) {
      double2 w = base[(size_t)(blk * N * N / 2 + q) * g.VHpad + k];
      v[2 * q] = w.x;
      v[2 * q + 1] = w.y;
    }
    auto get = [&](int i, int j, double& re, double& im) {
      if (i == j) { re = v[i]; im = 0; return; }
      bool lower = i > j;
      int a = lower ? i : j, b = lower ? j : i;
      int o = N + 2 * (a * (a - 1) / 2 + b);
      re = v[o];
      im = lower ? v[o + 1] : -v[o + 1];
    };
    double* A = dst + (size_t)(4 * id + 2 * blk) * 2 * D * D;
    double* B = dst + (size_t)(4 * id + 2 * blk + 1) * 2 * D * D;
    for (int i = 0; i < D; i++)
      for (int j = 0; j < D; j++) {
        get(i, j, A[i * D + j], A[D * D + i * D + j]);
        get(i, D + j, B[i * D + j], B[D * D + i * D + j]);
      }
  }
}

int gauge_download_repr(Ctx* c, double* host) {
  size_t n = (size_t)4 * c->g.V * 2 * c->dr * c->dr;
  double* d;
  YH_HIP(hipMalloc(&d, n * sizeof(double)));
  hipLaunchKernelGGL(k_repr_to_aos, dim3(grid1(4L * c->g.V)), dim3(256), 0, c->stream,
                     (const double2*)c->links[PREC_F64][RECON_18], d, c->g, c->dr);
  hipError_t e = hipMemcpyAsync(host, d, n * sizeof(double), hipMemcpyDeviceToHost, c->stream);
  if (e == hipSuccess) e = hipStreamSynchronize(c->stream);
  hipFree(d);
  if (e != hipSuccess) { set_error(hipGetErrorString(e)); return YH_ERR_HIP; }
  return YH_OK;
}

int clover_download(Ctx* c, double* host) {
  size_t n = (size_t)4 * c->g.V * 2 * c->dr * c->dr;
  double* d;
  YH_HIP(hipMalloc(&d, n * sizeof(double)));
  hipLaunchKernelGGL(k_clover_to_aos, dim3(grid_bs(c->g.V, 64)), dim3(64), 0, c->stream, (const double2*)c->clov[PREC_F64],
                     d, c->g, c->dr);
  hipError_t e = hipMemcpyAsync(host, d, n * sizeof(double), hipMemcpyDeviceToHost, c->stream);
  if (e == hipSuccess) e = hipStreamSynchronize(c->stream);
  hipFree(d);
  if (e != hipSuccess) { set_error(hipGetErrorString(e)); return YH_ERR_HIP; }
  return YH_OK;
}

}  // namespace yh
