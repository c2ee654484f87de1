// UFEM Navier-Stokes element assembly fused with a deterministic, atomic-free scatter into the LSS
// block-CSR matrix (gfx950).
//
// Work decomposition (row owner): a kAsmThreads-thread workgroup owns a contiguous range of node rows
// and all their incidences (element e, local node a).  Each thread takes one incidence, gathers the
// element's nodes from packed node records (double4: coordinates, state (u.., p), advection velocity
// and viscosity), computes the element quantities it needs, then produces the element row block
// M(a, b) = invdt*T(a,b) + theta*A'(a,b) one column node b at a time.  Per pass b the blocks are
// staged in LDS at rows sorted by target CSR block (precomputed staging map); the accumulator threads
// of every CSR block (one, or a few for blocks with many contributions) sum its run of rows, and the
// partial sums are added in thread order when the block is written: a sorted segmented reduction
// with a fixed order, so results are deterministic and no floating-point atomics are used.  Every
// CSR value and rhs entry is written exactly once, the values with coalesced stores.
//
// The specialised simplices take another route to the same row-owner sums, by block lists (assemble_lists_wg);
// the staged reduction above serves the generic expression, and specialised systems whose plan does not fit.
//
// Element mathematics (reference files relative to the coolfluid3 tree):
//   specialised P1 triangle / tetrahedron: plugins/UFEM/src/UFEM/NavierStokesSpecializations.hpp:38-303
//     (incl. the vk for wk substitution of lines 224-226 and 236-238 and tau from the velocity u)
//   generic expression (use_specializations = false): NavierStokesAssembly.hpp:44-66, order-2 Gauss
//   tau METRIC / TEZDUYAR: plugins/UFEM/src/UFEM/SUPG.hpp:141-219 (gij = J^-T J^-1 = Gram matrix of
//     the shape-function gradients of nodes 1..d for affine elements)
//   combine: NavierStokesAssembly.hpp:69-71 (rhs = -A x + a before the p rows are divided by theta;
//     theta * (A_p / theta) is formed as (theta * (1/theta)) * A_p, equal to within one rounding)
#include <algorithm>

#include "assembly_common.hpp"

// Multiply-adds are fused only within one source expression (a * b + c), never across statements:
// the rounding then follows the source, so a kernel body inlined into different kernels (the
// single-system and the batched persistent assembly) yields the same bits.
#pragma clang fp contract(on)

namespace cf3hip {

using namespace asmk;

namespace {

// ---------------------------------------------------------------------------------------------
// Specialised P1 simplex (D = 2 triangle, D = 3 tetrahedron) in arithmetic type R
// ---------------------------------------------------------------------------------------------
template<int D, typename R>
struct SpecP1 {
  static constexpr int K = D + 1, NEQ = D + 1, NN = NEQ * NEQ;
  uint32_t cn[K];
  R n[K][D];        // reference face normals (area vectors for D = 3, rotated edges for D = 2)
  R ua[D];          // mean advection velocity u_avg
  R na[D];          // normal of the row node a
  R Q[D];           // velocity-row coefficient: skew-symmetric advection + stress diffusion + bulk
  R tsdV, nudV, visc, m0dt;   // element: tau / (D^2 V), nu / (D^2 V), nu / (3 D^2 V) + tau_bulk / (D^2 V), V / (12|20 dt)
  R tsu;
  R cc, cpres, pn, pp, tdo, tdd, tpc;
  int a;

  // geometry in type T: normals and volume
  template<typename T>
  __device__ __forceinline__ static void geometry(const T X[K][D], T nrm[K][D], T& vol)
  {
    if constexpr(D == 2) {
      nrm[0][0] = X[1][1] - X[2][1]; nrm[0][1] = X[2][0] - X[1][0];
      nrm[1][0] = X[2][1] - X[0][1]; nrm[1][1] = X[0][0] - X[2][0];
      nrm[2][0] = X[0][1] - X[1][1]; nrm[2][1] = X[1][0] - X[0][0];
      vol = T(0.5) * ((X[1][0] - X[0][0]) * (X[2][1] - X[0][1]) - (X[2][0] - X[0][0]) * (X[1][1] - X[0][1]));
    } else {
      // NavierStokesSpecializations.hpp:162-173
      nrm[0][0] = T(0.5) * ((X[3][1]-X[1][1])*(X[2][2]-X[1][2]) - (X[2][1]-X[1][1])*(X[3][2]-X[1][2]));
      nrm[0][1] = T(0.5) * ((X[3][2]-X[1][2])*(X[2][0]-X[1][0]) - (X[2][2]-X[1][2])*(X[3][0]-X[1][0]));
      nrm[0][2] = T(0.5) * ((X[3][0]-X[1][0])*(X[2][1]-X[1][1]) - (X[2][0]-X[1][0])*(X[3][1]-X[1][1]));
      nrm[1][0] = T(0.5) * ((X[2][1]-X[0][1])*(X[3][2]-X[0][2]) - (X[3][1]-X[0][1])*(X[2][2]-X[0][2]));
      nrm[1][1] = T(0.5) * ((X[2][2]-X[0][2])*(X[3][0]-X[0][0]) - (X[3][2]-X[0][2])*(X[2][0]-X[0][0]));
      nrm[1][2] = T(0.5) * ((X[2][0]-X[0][0])*(X[3][1]-X[0][1]) - (X[3][0]-X[0][0])*(X[2][1]-X[0][1]));
      nrm[2][0] = T(0.5) * ((X[3][1]-X[0][1])*(X[1][2]-X[0][2]) - (X[1][1]-X[0][1])*(X[3][2]-X[0][2]));
      nrm[2][1] = T(0.5) * ((X[3][2]-X[0][2])*(X[1][0]-X[0][0]) - (X[1][2]-X[0][2])*(X[3][0]-X[0][0]));
      nrm[2][2] = T(0.5) * ((X[3][0]-X[0][0])*(X[1][1]-X[0][1]) - (X[1][0]-X[0][0])*(X[3][1]-X[0][1]));
      nrm[3][0] = T(0.5) * ((X[1][1]-X[0][1])*(X[2][2]-X[0][2]) - (X[2][1]-X[0][1])*(X[1][2]-X[0][2]));
      nrm[3][1] = T(0.5) * ((X[1][2]-X[0][2])*(X[2][0]-X[0][0]) - (X[2][2]-X[0][2])*(X[1][0]-X[0][0]));
      nrm[3][2] = T(0.5) * ((X[1][0]-X[0][0])*(X[2][1]-X[0][1]) - (X[2][0]-X[0][0])*(X[1][1]-X[0][1]));
      // det J = 2 (x3 - x0) . n_3 ; V = det / 6
      vol = (T(2) * ((X[3][0]-X[0][0])*nrm[3][0] + (X[3][1]-X[0][1])*nrm[3][1] + (X[3][2]-X[0][2])*nrm[3][2]))
            * T(1.0 / 6.0);
    }
  }

  // METRIC tau from the velocity at the centroid (SUPG.hpp:176-190); gij = n_i.n_l / (D^2 V^2).
  // s = 1 / (D V).  c1 = 1, c2 = 16, alpha = 1 on the specialised path.
  template<typename T>
  __device__ __forceinline__ static void tau_metric(const T nrm[K][D], T s, const T uc[D], T nu, T f4dt2, T& t_su, T& t_bu)
  {
    T gn[D][D];   // grad N of nodes 1..D
    for(int i = 0; i < D; ++i)
      for(int d = 0; d < D; ++d) gn[i][d] = nrm[i + 1][d] * s;
    T adv = T(0);
    for(int d = 0; d < D; ++d) {
      T acc = T(0);
      for(int i = 0; i < D; ++i) acc += uc[i] * gn[i][d];
      adv += acc * acc;
    }
    T gsq = T(0), tr = T(0);
    for(int i = 0; i < D; ++i)
      for(int l = i; l < D; ++l) {
        T gil = T(0);
        for(int d = 0; d < D; ++d) gil += gn[i][d] * gn[l][d];
        gsq += (i == l ? T(1) : T(2)) * gil * gil;
        if(i == l) tr += gil;
      }
    const T sq = sqrt(f4dt2 + adv + T(16) * (nu * nu * gsq));
    t_su = T(1) / sq;
    t_bu = sq / tr;
  }

  __device__ __forceinline__ void prepare(const AsmArgs& g, uint32_t e, int a_)
  {
    load_conn<K>(g.conn, e, cn);
    prepare_element(g, [&](uint32_t nd, double* x, double* u, double* w, double& nu) {
      double xp[4], st[4], ad[4];
      unpack(g.xp[nd], xp);
      unpack(g.st[nd], st);
      unpack(g.ad[nd], ad);
#pragma unroll
      for(int d = 0; d < D; ++d) { x[d] = xp[d]; u[d] = st[d]; w[d] = ad[d]; }
      nu = ad[3];
    });
    prepare_row(g, a_);
  }

  // element quantities from the coordinates, velocity, advection velocity and viscosity that node(cn[m], ...)
  // gives
  template<class Node>
  __device__ __forceinline__ void prepare_element(const AsmArgs& g, Node node)
  {
    double X[K][D];
    double uc[D];
    double nus = 0.;
    R uas[D];
    for(int d = 0; d < D; ++d) { uc[d] = 0.; uas[d] = R(0); }
#pragma unroll
    for(int m = 0; m < K; ++m) {
      double u[D], w[D], nun;
      node(cn[m], X[m], u, w, nun);
#pragma unroll
      for(int d = 0; d < D; ++d) {
        uc[d] += u[d];
        uas[d] += (R)w[d];
      }
      nus += nun;
    }
    for(int d = 0; d < D; ++d) {
      uc[d] = uc[d] * (1.0 / K);
      ua[d] = uas[d] * R(1.0 / K);
    }
    const double nu_mean = fabs(nus * (1.0 / K));
    const R nu = (R)nu_mean;
    R V = R(0), invV, tbu;
    bool fp64_geom = sizeof(R) == sizeof(double);
    if constexpr(sizeof(R) != sizeof(double)) {
      // coordinates relative to node 0, formed in FP64: the FP32 differences of absolute coordinates
      // would lose log2(1/h) bits (the normals and the volume are translation invariant)
      R Xr[K][D];
      for(int m = 0; m < K; ++m)
        for(int d = 0; d < D; ++d) Xr[m][d] = (R)(X[m][d] - X[0][d]);
      geometry<R>(Xr, n, V);
      // strongly skewed elements: geometry and tau in FP64.  Criterion from the face normals already
      // formed, S = sum |n_i|^2: tetrahedra V^2 < 1.4e-3 S^(3/2) (regular Kuhn tetrahedron 1.5e-2;
      // aspect ratio (longest edge / smallest height) 15 and more falls below ~7e-4, aspect ratio 8
      // and less stays above ~2.7e-3); triangles V < S / 240 (rotated edges: |V| < 0.0125 l_rms^2).
      R S = R(0);
      for(int m = 0; m < K; ++m)
        for(int d = 0; d < D; ++d) S += n[m][d] * n[m][d];
      if constexpr(D == 3) {
        if(V * V < R(1.4e-3) * S * sqrt(S)) fp64_geom = true;
      } else {
        if(fabs(V) < S * R(1.0 / 240.0)) fp64_geom = true;
      }
    }
    if(fp64_geom) {
      double n64[K][D], V64, ts, tb;
      geometry<double>(X, n64, V64);
      const double iv = 1. / V64;
      tau_metric<double>(n64, iv * (1.0 / D), uc, nu_mean, g.f4dt2, ts, tb);
      for(int m = 0; m < K; ++m)
        for(int d = 0; d < D; ++d) n[m][d] = (R)n64[m][d];
      V = (R)V64; invV = (R)iv; tsu = (R)ts; tbu = (R)tb;
      if(!(V64 > 0.)) g.status[0] = 1;   // every writer stores the same flag value
      if constexpr(D == 3 && sizeof(R) == sizeof(double)) {
        // the element terms take the reference's volume (NavierStokesSpecializations.hpp:156), tau above
        // det J of the Jacobian, as the reference's ComputeTau does (SUPG.hpp:178, ElementData.hpp:302-314)
        const double Vr = tet_volume_ref(X);
        V = Vr;
        invV = 1. / Vr;
      }
    } else {
      R ucr[D];
      for(int d = 0; d < D; ++d) ucr[d] = (R)uc[d];
      invV = R(1) / V;
      tau_metric<R>(n, invV * R(1.0 / D), ucr, nu, (R)g.f4dt2, tsu, tbu);
      if(!(V > R(0))) g.status[0] = 1;
    }
    const R rdV = invV * R(1.0 / (D * D));
    tsdV = tsu * rdV;
    nudV = nu * rdV;
    visc = nudV * R(1.0 / 3.0) + tbu * rdV;
    m0dt = (R)g.invdt * (V * R(D == 2 ? 1.0 / 12.0 : 1.0 / 20.0));
  }

  // coefficients of the row of local node a_
  __device__ __forceinline__ void prepare_row(const AsmArgs& g, int a_)
  {
    a = a_;
    // normal of the row node, selected without dynamic register indexing
#pragma unroll
    for(int d = 0; d < D; ++d) na[d] = n[0][d];
#pragma unroll
    for(int m = 1; m < K; ++m)
      if(m == a)
#pragma unroll
        for(int d = 0; d < D; ++d) na[d] = n[m][d];
    // per-row (node a) coefficients (NavierStokesSpecializations.hpp:66-145 / 196-301)
    const R c0 = R(D == 2 ? 1.0 / 6.0 : 1.0 / 12.0);
    R u_ni = R(0);
    for(int d = 0; d < D; ++d) u_ni += ua[d] * na[d];
    const R cskew = R(0.5) * c0 + R(0.5) * tsdV * u_ni;
    cc = c0 + tsdV * u_ni;
    const R inv_rho = (R)g.inv_rho;
    cpres = cc * inv_rho;
    const R time_ii = tsu * c0 * u_ni;
    // n_i . u~ with the tetrahedron substitution of vk for wk (lines 236-238)
    R ni_ut = na[0] * ua[0] + na[1] * ua[1];
    if constexpr(D == 3) ni_ut += na[2] * ua[1];
#pragma unroll
    for(int r = 0; r < D; ++r) {
      const R uk = ua[(D == 3 && r == 2) ? 1 : r];   // W rows use vk (lines 224-226)
      Q[r] = cskew * uk + visc * na[r];
    }
    pn = R(0.5) * tsdV * ni_ut + c0;   // tau_ps = tau_su
    pp = tsdV * inv_rho;
    const R invdt = (R)g.invdt;
    tdo = m0dt + invdt * time_ii;
    tdd = tdo + m0dt;
    tpc = invdt * tsu * c0;
  }

  // block (a, B): M = invdt*T + theta*A' into m[NN] (row-major); with RHS, rhs -= A x_B
  template<int B, bool RHS, typename VR>
  __device__ __forceinline__ void block(const AsmArgs& g, VR* m, R* rhs, const R* xb) const
  {
    const R* nj = n[B];
    R uknj = R(0), ninj = R(0);
#pragma unroll
    for(int d = 0; d < D; ++d) { uknj += ua[d] * nj[d]; ninj += na[d] * nj[d]; }
    const R dsum = uknj * cc + nudV * ninj;   // convection (std + SUPG) + diffusion n_a.n_b
    const R td = a == B ? tdd : tdo;
    const R th = (R)g.theta, thq = (R)g.thq;
#pragma unroll
    for(int r = 0; r < D; ++r) {
      R Ar[NEQ];
#pragma unroll
      for(int c = 0; c < D; ++c) Ar[c] = Q[r] * nj[c] + (r == c ? dsum : R(0));
      Ar[D] = cpres * nj[r];
      if constexpr(RHS) {
        R s = R(0);
#pragma unroll
        for(int c = 0; c < NEQ; ++c) s += Ar[c] * xb[c];
        rhs[r] -= s;
      }
#pragma unroll
      for(int c = 0; c < D; ++c) m[r * NEQ + c] = (VR)(th * Ar[c] + (r == c ? td : R(0)));
      m[r * NEQ + D] = (VR)(th * Ar[D]);
    }
    {
      R Ar[NEQ];
#pragma unroll
      for(int c = 0; c < D; ++c) Ar[c] = uknj * (tsdV * na[c]) + pn * nj[c];
      Ar[D] = pp * ninj;
      if constexpr(RHS) {
        R s = R(0);
#pragma unroll
        for(int c = 0; c < NEQ; ++c) s += Ar[c] * xb[c];
        rhs[D] -= s;
      }
#pragma unroll
      for(int c = 0; c < D; ++c) m[D * NEQ + c] = (VR)(tpc * na[c] + thq * Ar[c]);
      m[D * NEQ + D] = (VR)(thq * Ar[D]);
    }
  }

  __device__ __forceinline__ void rhs_source(const AsmArgs&, R*) const {}
};

// ---------------------------------------------------------------------------------------------
// Generic expression for P1 simplices (use_specializations = false): NavierStokesAssembly.hpp:44-66
// with tau from u_adv and the order-2 Gauss rule; gradients constant over the element.
// ---------------------------------------------------------------------------------------------
template<int D>
struct GenericP1 {
  typedef double R;
  static constexpr int K = D + 1, NEQ = D + 1, NN = NEQ * NEQ, NQ = D == 2 ? 3 : 4;
  uint32_t cn[K];
  R G[D][K];         // physical gradients
  R Ga[D];           // gradient of the row node a
  R detw;            // |J| (weights applied per point)
  R ua_n[K][D];      // nodal advection velocity
  R nu_n[K];
  R tps, tsu, tbu;
  R oh[K];           // one-hot of the row node a
  int a;

  __device__ __forceinline__ static void gauss(int q, R xi[D], R& w)
  {
    if constexpr(D == 2) {
      xi[0] = q == 2 ? 0.0 : 0.5;
      xi[1] = q == 0 ? 0.0 : 0.5;
      w = 1.0 / 6.0;
    } else {
      const R mu = 0.13819660112501051517954131656;
      xi[0] = q == 1 ? 1. - 3. * mu : mu;
      xi[1] = q == 2 ? 1. - 3. * mu : mu;
      xi[2] = q == 3 ? 1. - 3. * mu : mu;
      w = 0.04166666666666666666666666666666666667;
    }
  }

  __device__ __forceinline__ static void shape(const R xi[D], R N[K])
  {
    R s = 1.;
#pragma unroll
    for(int d = 0; d < D; ++d) { N[d + 1] = xi[d]; s -= xi[d]; }
    N[0] = s;
  }

  // v[a] as a one-hot weighted sum: a select chain over a local array is turned into a dynamically
  // indexed (scratch) load by the optimiser
  __device__ __forceinline__ R select_a(const R v[K]) const
  {
    R r = 0.;
#pragma unroll
    for(int m = 0; m < K; ++m) r += oh[m] * v[m];
    return r;
  }

  __device__ __forceinline__ void prepare(const AsmArgs& g, uint32_t e, int a_)
  {
    a = a_;
#pragma unroll
    for(int m = 0; m < K; ++m) oh[m] = m == a ? 1. : 0.;
    load_conn<K>(g.conn, e, cn);
    R X[K][D];
    R nus = 0.;
#pragma unroll
    for(int m = 0; m < K; ++m) {
      double xp[4], ad[4];
      unpack(g.xp[cn[m]], xp);
      unpack(g.ad[cn[m]], ad);
#pragma unroll
      for(int d = 0; d < D; ++d) {
        X[m][d] = xp[d];
        ua_n[m][d] = ad[d];
      }
      nu_n[m] = ad[3];
      nus += nu_n[m];
    }
    // J(ksi, x) = x_{ksi+1} - x_0, inverse by the adjugate
    R J[D][D];
#pragma unroll
    for(int i = 0; i < D; ++i)
#pragma unroll
      for(int d = 0; d < D; ++d) J[i][d] = X[i + 1][d] - X[0][d];
    R Ji[D][D], det;
    if constexpr(D == 2) {
      det = J[0][0] * J[1][1] - J[1][0] * J[0][1];
      const R inv = 1. / det;
      Ji[0][0] = J[1][1] * inv; Ji[0][1] = -J[0][1] * inv;
      Ji[1][0] = -J[1][0] * inv; Ji[1][1] = J[0][0] * inv;
    } else {
      const R c00 = J[1][1] * J[2][2] - J[1][2] * J[2][1];
      const R c10 = J[2][1] * J[0][2] - J[2][2] * J[0][1];
      const R c20 = J[0][1] * J[1][2] - J[0][2] * J[1][1];
      det = c00 * J[0][0] + c10 * J[1][0] + c20 * J[2][0];
      const R inv = 1. / det;
      Ji[0][0] = c00 * inv; Ji[0][1] = c10 * inv; Ji[0][2] = c20 * inv;
      Ji[1][0] = (J[1][2] * J[2][0] - J[1][0] * J[2][2]) * inv;
      Ji[1][1] = (J[2][2] * J[0][0] - J[2][0] * J[0][2]) * inv;
      Ji[1][2] = (J[0][2] * J[1][0] - J[0][0] * J[1][2]) * inv;
      Ji[2][0] = (J[1][0] * J[2][1] - J[1][1] * J[2][0]) * inv;
      Ji[2][1] = (J[2][0] * J[0][1] - J[2][1] * J[0][0]) * inv;
      Ji[2][2] = (J[0][0] * J[1][1] - J[0][1] * J[1][0]) * inv;
    }
    if(!(det > 0.)) g.status[0] = 1;
    detw = det;
    // grad N = Jinv * dN/dksi ; dN/dksi of node 0 = -1, node m+1 = e_m
#pragma unroll
    for(int d = 0; d < D; ++d) {
      R s = 0.;
#pragma unroll
      for(int l = 0; l < D; ++l) { G[d][l + 1] = Ji[d][l]; s -= Ji[d][l]; }
      G[d][0] = s;
    }
#pragma unroll
    for(int d = 0; d < D; ++d) Ga[d] = select_a(G[d]);
    // tau from u_adv at the centroid (NavierStokesAssembly.hpp:54, SUPG.hpp:137-219)
    const R nu_e = fabs(nus * (1.0 / K));
    R uc[D];
#pragma unroll
    for(int d = 0; d < D; ++d) {
      R s = 0.;
#pragma unroll
      for(int m = 0; m < K; ++m) s += ua_n[m][d];
      uc[d] = s * (1.0 / K);
    }
    if(g.supg_type == CF3HIP_SUPG_CF2) {
      // volume as the reference's etype::volume: Tetra3D's 24-term expansion, Triag2D's 0.5 det J
      double vol;
      if constexpr(D == 3) {
        double Xv[4][3];
#pragma unroll
        for(int m = 0; m < K; ++m)
#pragma unroll
          for(int d = 0; d < D; ++d) Xv[m][d] = X[m][d];
        vol = tet_volume_ref(Xv);
      } else {
        vol = 0.5 * det;
      }
      R um2 = 0., s = 0.;
#pragma unroll
      for(int d = 0; d < D; ++d) um2 += uc[d] * uc[d];
#pragma unroll
      for(int m = 0; m < K; ++m) {
        R un = 0.;
#pragma unroll
        for(int d = 0; d < D; ++d) un += uc[d] * G[d][m];
        s += un;
      }
      if(!tau_cf2(D, vol, nu_e, sqrt(um2), s, g.dt, g.u_ref, tps, tsu, tbu)) g.status[0] = 2;
    } else if(g.supg_type == CF3HIP_SUPG_METRIC) {
      R gij[D][D];
#pragma unroll
      for(int i = 0; i < D; ++i)
#pragma unroll
        for(int j = 0; j < D; ++j) {
          R s = 0.;
#pragma unroll
          for(int l = 0; l < D; ++l) s += Ji[l][i] * Ji[l][j];
          gij[i][j] = s;
        }
      R ugu = 0., gsq = 0., tr = 0.;
#pragma unroll
      for(int j = 0; j < D; ++j) {
        R s = 0.;
#pragma unroll
        for(int i = 0; i < D; ++i) s += uc[i] * gij[i][j];
        ugu += s * uc[j];
        tr += gij[j][j];
#pragma unroll
        for(int i = 0; i < D; ++i) gsq += gij[i][j] * gij[i][j];
      }
      const R diff = nu_e * nu_e * gsq;
      tsu = 1. / sqrt(g.c1 * g.c1 * g.f4dt2 + fabs(ugu) + g.c2 * diff);
      tps = tsu;
      tbu = sqrt(g.f4dt2 + fabs(ugu) + 16. * diff) / tr;
    } else {
      R h = 1e10;
#pragma unroll
      for(int i = 0; i < K; ++i)
#pragma unroll
        for(int j = i + 1; j < K; ++j) {
          R s = 0.;
#pragma unroll
          for(int d = 0; d < D; ++d) { const R df = X[i][d] - X[j][d]; s += df * df; }
          h = fmin(h, s);
        }
      h = sqrt(h);
      R um = 0.;
#pragma unroll
      for(int d = 0; d < D; ++d) um += uc[d] * uc[d];
      um = sqrt(um);
      tsu = 1. / ((2. * um) / h + 2. / g.dt + (4. * nu_e) / (h * h));
      tps = tsu;
      tbu = tsu * um * um;
    }
    tps *= g.a_ps; tsu *= g.a_su; tbu *= g.a_bu;
  }

  template<int B, bool RHS, typename VR>
  __device__ __forceinline__ void block(const AsmArgs& g, VR* m, R* rhs, const R* xb) const
  {
    R A[NEQ][NEQ];
#pragma unroll
    for(int r = 0; r < NEQ; ++r)
#pragma unroll
      for(int c = 0; c < NEQ; ++c) A[r][c] = 0.;
    R Tuu = 0., Tp[D];   // T is diagonal in the velocity rows; T[p][u_i] in the pressure row
#pragma unroll
    for(int d = 0; d < D; ++d) Tp[d] = 0.;
    R gtg = 0.;
#pragma unroll
    for(int d = 0; d < D; ++d) gtg += Ga[d] * G[d][B];
    const R inv_rho = g.inv_rho;
#pragma unroll
    for(int q = 0; q < NQ; ++q) {
      R xi[D], wq, N[K];
      gauss(q, xi, wq);
      shape(xi, N);
      const R Na = select_a(N);
      const R w = wq * detw;
      R uq[D], nuq = 0.;
#pragma unroll
      for(int d = 0; d < D; ++d) {
        R s = 0.;
#pragma unroll
        for(int mm = 0; mm < K; ++mm) s += N[mm] * ua_n[mm][d];
        uq[d] = s;
      }
#pragma unroll
      for(int mm = 0; mm < K; ++mm) nuq += N[mm] * nu_n[mm];
      R La = 0., Lb = 0.;
#pragma unroll
      for(int d = 0; d < D; ++d) { La += uq[d] * Ga[d]; Lb += uq[d] * G[d][B]; }
      const R SUa = Na + tsu * La;
      const R Lps = 0.5 * tps * La;
#pragma unroll
      for(int i = 0; i < D; ++i) {
        A[D][i] += w * ((Na + Lps) * G[i][B] + (tps * Ga[i]) * Lb);
        A[i][i] += w * (nuq * gtg + SUa * Lb);
        A[i][D] += w * (SUa * G[i][B] * inv_rho);
#pragma unroll
        for(int j = 0; j < D; ++j) A[i][j] += w * ((tbu * Ga[i] + 0.5 * uq[i] * SUa) * G[j][B]);
        Tp[i] += w * (tps * Ga[i] * N[B]);
      }
      Tuu += w * (SUa * N[B]);
      A[D][D] += w * ((tps * gtg) * inv_rho);
    }
    if constexpr(RHS) {
#pragma unroll
      for(int r = 0; r < NEQ; ++r) {
        R s = 0.;
#pragma unroll
        for(int c = 0; c < NEQ; ++c) s += A[r][c] * xb[c];
        rhs[r] -= s;
      }
    }
    const R invdt = g.invdt, th = g.theta, thq = g.thq;
#pragma unroll
    for(int r = 0; r < D; ++r)
#pragma unroll
      for(int c = 0; c < NEQ; ++c)
        m[r * NEQ + c] = (VR)((r == c ? invdt * Tuu : 0.) + th * A[r][c]);
#pragma unroll
    for(int c = 0; c < D; ++c) m[D * NEQ + c] = (VR)(invdt * Tp[c] + thq * A[D][c]);
    m[D * NEQ + D] = (VR)(thq * A[D][D]);
  }

  // _a[u[_i]] += (N + tau_su u_adv grad N)^T g  (NavierStokesAssembly.hpp:65)
  __device__ __forceinline__ void rhs_source(const AsmArgs& g, R* rhs) const
  {
    R g_n[K][D];
#pragma unroll
    for(int m = 0; m < K; ++m)
#pragma unroll
      for(int d = 0; d < D; ++d) g_n[m][d] = g.g[d][cn[m]];
#pragma unroll
    for(int q = 0; q < NQ; ++q) {
      R xi[D], wq, N[K];
      gauss(q, xi, wq);
      shape(xi, N);
      const R Na = select_a(N);
      const R w = wq * detw;
      R uq[D], gq[D];
#pragma unroll
      for(int d = 0; d < D; ++d) {
        R s = 0., sg = 0.;
#pragma unroll
        for(int mm = 0; mm < K; ++mm) { s += N[mm] * ua_n[mm][d]; sg += N[mm] * g_n[mm][d]; }
        uq[d] = s; gq[d] = sg;
      }
      R La = 0.;
#pragma unroll
      for(int d = 0; d < D; ++d) La += uq[d] * Ga[d];
      const R SUa = Na + tsu * La;
#pragma unroll
      for(int i = 0; i < D; ++i) rhs[i] += w * (SUa * gq[i]);
    }
  }
};

// ---------------------------------------------------------------------------------------------
// Row-owner assembly kernel.  RHS = false (FP32 matrix pass of the precision form) skips the
// right-hand side, which is formed by the FP64 pass.
// ---------------------------------------------------------------------------------------------
// the work of one assembly workgroup (row range wg of the system described by g)
template<class Op, typename R, typename VR, bool RHS>
__device__ __forceinline__ void assemble_wg(const AsmArgs& g, uint32_t wg)
{
  constexpr int K = Op::K, NEQ = Op::NEQ, NN = NEQ * NEQ;
  static_assert(K <= 4, "one staging byte per column local node in a 32-bit word");
  constexpr int LDW = lds_row<VR, NN>();
  constexpr size_t kBlkBytes = sizeof(VR) * kThreads * LDW;
  constexpr size_t kRhsBytes = sizeof(R) * kThreads * NEQ;
  __shared__ __align__(16) unsigned char s_raw[kBlkBytes > kRhsBytes ? kBlkBytes : kRhsBytes];
  VR* s_blk = reinterpret_cast<VR*>(s_raw);
  R* s_rhs = reinterpret_cast<R*>(s_raw);   // reused after the values are written
  __shared__ uint32_t s_rowinc[kThreads + 1];
  __shared__ uint16_t s_acc[kThreads];

  const uint32_t r0 = g.wg_rows[wg], r1 = g.wg_rows[wg + 1];
  const uint32_t i0 = g.inc_ptr[r0], ninc = g.inc_ptr[r1] - i0;
  const uint32_t blk0 = g.row_ptr[r0], nblk = g.row_ptr[r1] - blk0;
  const uint32_t nrows = r1 - r0;
  const int t = threadIdx.x;
  if constexpr(RHS)
    for(uint32_t j = t; j <= nrows; j += kThreads) s_rowinc[j] = g.inc_ptr[r0 + j] - i0;
  if((uint32_t)t < nblk) s_acc[t] = g.blk_acc[blk0 + t];

  const bool active = (uint32_t)t < ninc;
  uint32_t posw = 0;
  Op op;
  R rhs[NEQ];
#pragma unroll
  for(int r = 0; r < NEQ; ++r) rhs[r] = R(0);
  if(active) {
    posw = reinterpret_cast<const uint32_t*>(g.inc_pos)[i0 + t];
    const uint32_t ea = g.inc[i0 + t];
    op.prepare(g, ea / K, (int)(ea % K));
  }
  __syncthreads();
  // accumulator thread t: block bs of this workgroup, rank h of c; rows [beg_p + h, end_p) step c
  const uint32_t alast = s_acc[nblk - 1];
  const uint32_t n_acc = (alast & 255u) + (alast >> 8);
  const bool owner = (uint32_t)t < n_acc;
  uint32_t begw = 0, endw = 0, h = 0, c = 1;
  if(owner) {
    uint32_t lo = 0, hi = nblk;
    while(hi - lo > 1) {
      const uint32_t mid = (lo + hi) >> 1;
      if((s_acc[mid] & 255u) <= (uint32_t)t) lo = mid; else hi = mid;
    }
    h = (uint32_t)t - (s_acc[lo] & 255u);
    c = s_acc[lo] >> 8;
    const uint32_t* bb = reinterpret_cast<const uint32_t*>(g.blk_beg);
    begw = bb[blk0 + lo];
    endw = lo + 1 < nblk ? bb[blk0 + lo + 1] : ninc * 0x01010101u;
  }
  R acc[NN];
#pragma unroll
  for(int v = 0; v < NN; ++v) acc[v] = R(0);

  static_for<0, K>([&](auto bc) {
    constexpr int B = decltype(bc)::value;
    if(active) {
      R xb[NEQ];
      if constexpr(RHS) load_state<NEQ, R>(g, op.cn[B], xb);
      op.template block<B, RHS, VR>(g, s_blk + ((posw >> (8 * B)) & 255u) * LDW, rhs, xb);
    }
    __syncthreads();
    if(owner) {
      const uint32_t je = (endw >> (8 * B)) & 255u;
      for(uint32_t j = ((begw >> (8 * B)) & 255u) + h; j < je; j += c) {
        VR v[NN];
        lds_load_row<VR, NN>(s_blk + j * LDW, v);
#pragma unroll
        for(int q = 0; q < NN; ++q) acc[q] += (R)v[q];
      }
    }
    __syncthreads();
  });
  // partial sums to LDS row t, then each block = sum of its accumulator rows in thread order,
  // stored with consecutive lanes on consecutive values
  if(owner) {
    VR* d = s_blk + t * LDW;
#pragma unroll
    for(int q = 0; q < NN; ++q) d[q] = (VR)acc[q];
  }
  __syncthreads();
  {
    VR* dst = static_cast<VR*>(g.values) + (uint64_t)blk0 * NN;
    for(uint32_t o = t; o < nblk * NN; o += kThreads) {
      const uint32_t sb = o / NN, v = o % NN;
      const uint32_t a = s_acc[sb], f = a & 255u, na = a >> 8;
      R sum = (R)s_blk[f * LDW + v];
      for(uint32_t r = 1; r < na; ++r) sum += (R)s_blk[(f + r) * LDW + v];
      dst[o] = (VR)sum;
    }
  }
  if constexpr(RHS) {
    __syncthreads();
    if(active) {
      if(g.body_force) op.rhs_source(g, rhs);
#pragma unroll
      for(int r = 0; r < NEQ; ++r) s_rhs[t * NEQ + r] = rhs[r];
    }
    __syncthreads();
    for(uint32_t o = t; o < nrows * NEQ; o += kThreads) {
      const uint32_t row = o / NEQ, r = o % NEQ;
      const uint32_t qe = s_rowinc[row + 1];
      uint32_t q = s_rowinc[row];
      // four interleaved partial sums (fixed order) shorten the LDS latency chain
      R s0 = R(0), s1 = R(0), s2 = R(0), s3 = R(0);
      for(; q + 4 <= qe; q += 4) {
        s0 += s_rhs[q * NEQ + r];
        s1 += s_rhs[(q + 1) * NEQ + r];
        s2 += s_rhs[(q + 2) * NEQ + r];
        s3 += s_rhs[(q + 3) * NEQ + r];
      }
      for(; q < qe; ++q) s0 += s_rhs[q * NEQ + r];
      g.rhs[(uint64_t)(r0 + row) * NEQ + r] = (double)((s0 + s1) + (s2 + s3));
    }
  }
}

// FP32 kernels: at most 96 VGPRs, so that 5 waves fit per SIMD (104 would allow 4)
template<class Op, typename R, typename VR, bool RHS>
__global__ __launch_bounds__(kThreads, sizeof(R) == sizeof(float) ? 5 : 1) void k_assemble(AsmArgs g)
{
  assemble_wg<Op, R, VR, RHS>(g, xcd_order(blockIdx.x, gridDim.x));
}

// ---------------------------------------------------------------------------------------------
// Specialised simplices by block lists: the work of one plan (sparsity.hip)
//   1. one element per thread: face normals, n . u_avg and six scalars, written to LDS as its record;
//   2. one thread per block list (a CSR block, or plan_list_length of its contributions): the operator sums
//      A and T of the block straight from the records, in registers;
//   3. combine (M = T / dt + theta A) once per list, with its share of the rhs, -A x_b; the lists of a block
//      are added in order through LDS and stored in the order of the values.
// The staged reduction (assemble_wg) instead computes an element once per owned row, forms every element
// block of 16 values, writes it to LDS and reads it back, K passes with two barriers each, and repeats the
// combine and the rhs product for every one.
// Measured (us, staged reduction -> block lists): FP64 tetrahedra 61^3 cells 361 -> 254, 100^3 1535 -> 1080, 128^3 (kernel
// alone) 3147 -> 2189; FP32 215 -> 142, 920 -> 641, 1811 -> 1171; triangles 500^2 63 -> 59 (FP64), 41 -> 36 (FP32).
// At 61^3: 1206 -> 990 VALU instructions per wave and 5/6 of the waves, 25 % fewer LDS instructions; VALU and
// LDS are each busy about 60 % of the time with 5 to 6 workgroups per CU, and neither HBM (1.9 TB/s) nor the
// load chain at the start bounds it: a persistent form that loads the next plan and its nodes during the block
// sums was no faster (its 159 VGPRs cost the waves that hid the same latency).
// dynamic LDS: [nodal states] [other nodal data; then the element records; then the block rows and rhs
// parts], the states kept to the end with RHS.  The nodal data are arrays of 16-byte pairs, (u, v), (w, p),
// (x, y), (z, nu), (u_adv x, y), and u_adv z: whole 32-byte records would put every first half on the same
// half of the banks.
template<int D, typename R>
struct PlanLayout {
  static constexpr int K = D + 1, NEQ = D + 1, NN = NEQ * NEQ;
  static constexpr int COL = D + 1;         // n_b, n_b . u_avg
  static constexpr int ELEM = K * COL;      // tau/(D^2 V), nu/(D^2 V), viscous + bulk, u_avg x, y, V/(12|20 dt)
  static constexpr int WORDS = ELEM + 6;
  // record stride: an odd number of 16-byte pieces, so that the records spread over the banks
  static constexpr int STRIDE = (((WORDS * (int)sizeof(R) + 15) / 16) | 1) * 16 / (int)sizeof(R);
  static constexpr int LDW = D == 3 ? lds_row<R, NN>() : NN;   // 9 values: odd by themselves
  static constexpr size_t lds_bytes(bool rhs, uint32_t nodes, uint32_t elems, uint32_t lists)
  {
    const size_t stage = (size_t)nodes * (rhs ? 56 : 88);
    const size_t rec = sizeof(R) * STRIDE * (elems + 1);
    const size_t row = sizeof(R) * (LDW + (rhs ? NEQ : 0)) * lists;
    return (rhs ? sizeof(double4) * nodes : 0) + std::max(stage, std::max(rec, row));
  }
};

// the fields of a system, and the node records that the packing kernels write from them
struct PackArgs {
  const double* u[3];
  const double* ua[3];
  const double* p;
  const double* nu;
  double4* st;
  double4* ad;
};

template<int D>
__device__ __forceinline__ void read_node(const PackArgs& f, uint64_t i, double4& st, double4& ad)
{
  if constexpr(D == 3) {
    st = make_double4(f.u[0][i], f.u[1][i], f.u[2][i], f.p[i]);
    ad = make_double4(f.ua[0][i], f.ua[1][i], f.ua[2][i], f.nu[i]);
  } else {
    st = make_double4(f.u[0][i], f.u[1][i], f.p[i], 0.);
    ad = make_double4(f.ua[0][i], f.ua[1][i], 0., f.nu[i]);
  }
}

// DIRECT: the nodes' states come from the field arrays, otherwise from the packed records (the batched launch,
// whose pass over all systems packs them).  A plan reads a node once, so the packing pass, a launch of its own,
// costs more than the eight loads per node it saves: linearise + assemble + product, records -> fields, us: 32^2 x 2
// triangles 26.0 -> 23.1; FP32 tetrahedra 23^3 cells 32.7 -> 29.4, 100^3 814 -> 790; FP64 61^3 353 -> 345, 128^3
// 3001 -> 2972.
template<int D, typename R, bool RHS, bool DIRECT>
__device__ __forceinline__ void assemble_lists_wg(const AsmArgs& g, const PackArgs& f, uint32_t wg, unsigned char* smem)
{
  typedef PlanLayout<D, R> Y;
  constexpr int K = Y::K, NEQ = Y::NEQ, NN = Y::NN, LDW = Y::LDW;
  constexpr int LEN = (int)plan_list_length(K);
  __shared__ uint16_t s_first[kThreads + 1];                // first list of each block
  __shared__ uint16_t s_rowfirst[RHS ? kThreads + 1 : 1];   // first list of each row
  __shared__ uint32_t s_wave[2][kThreads / 64];

  const uint32_t t = threadIdx.x, ns = g.plan_nodes;
  const unsigned char* plan = g.plan + (uint64_t)wg * plan_bytes(ns);
  const uint32_t* nodes = reinterpret_cast<const uint32_t*>(plan + kPlanHeadBytes);
  const uint32_t* locs = nodes + ns;
  const uint64_t* los = reinterpret_cast<const uint64_t*>(locs + kThreads);
  const uint32_t loc = locs[t];
  const uint64_t lo = los[t];
  const uint32_t hi = reinterpret_cast<const uint16_t*>(los + kThreads)[t];
  double2* s_uv = reinterpret_cast<double2*>(smem);
  double2* s_wp = s_uv + ns;
  unsigned char* body = smem + (RHS ? 2 * sizeof(double2) * ns : 0);
  double2* s_xy = RHS ? reinterpret_cast<double2*>(body) : s_wp + ns;
  double2* s_zn = s_xy + ns;
  double2* s_ad = s_zn + ns;
  double* s_az = reinterpret_cast<double*>(s_ad + ns);
  R* s_rec = reinterpret_cast<R*>(body);
  R* s_row = reinterpret_cast<R*>(body);
  R* s_rhs = s_row + LDW * g.plan_lists;
  for(uint32_t j = t; j < ns; j += kThreads) {
    const uint32_t nd = nodes[j];
    const double4 xp = g.xp[nd];
    double4 st, ad;
    if constexpr(DIRECT) {
      read_node<D>(f, nd, st, ad);
    } else {
      st = g.st[nd];
      ad = g.ad[nd];
    }
    s_xy[j] = make_double2(xp.x, xp.y);
    s_zn[j] = make_double2(xp.z, ad.w);
    s_uv[j] = make_double2(st.x, st.y);
    s_wp[j] = make_double2(st.z, st.w);
    s_ad[j] = make_double2(ad.x, ad.y);
    if constexpr(D == 3) s_az[j] = ad.z;
  }
  const uint4 h0 = reinterpret_cast<const uint4*>(plan)[0], h1 = reinterpret_cast<const uint4*>(plan)[1];
  const uint32_t r0 = h0.x, nrows = h0.y, ne = h0.z, blk0 = h1.x, nblk = h1.y, nlists = h1.z;
  __syncthreads();
  SpecP1<D, R> op;
  if(t < ne) {
#pragma unroll
    for(int m = 0; m < K; ++m) op.cn[m] = (loc >> (8 * m)) & 255u;
    op.prepare_element(g, [&](uint32_t nd, double* x, double* u, double* w, double& nu) {
      const double2 xy = s_xy[nd], zn = s_zn[nd], uv = s_uv[nd], ad = s_ad[nd];
      x[0] = xy.x; x[1] = xy.y;
      u[0] = uv.x; u[1] = uv.y;
      w[0] = ad.x; w[1] = ad.y;
      if constexpr(D == 3) { x[2] = zn.x; u[2] = s_wp[nd].x; w[2] = s_az[nd]; }
      nu = zn.y;
    });
  }
  const uint64_t bstart = __ballot(lo >> 63), rstart = __ballot(hi >> 15);
  if((t & 63u) == 0) {
    s_wave[0][t >> 6] = (uint32_t)__popcll(bstart);
    s_wave[1][t >> 6] = (uint32_t)__popcll(rstart);
  }
  __syncthreads();   // the element records replace the node records
  if(t < ne) {
    R* rec = s_rec + t * Y::STRIDE;
#pragma unroll
    for(int b = 0; b < K; ++b) {
      R un = R(0);
#pragma unroll
      for(int d = 0; d < D; ++d) {
        rec[b * Y::COL + d] = op.n[b][d];
        un += op.ua[d] * op.n[b][d];
      }
      rec[b * Y::COL + D] = un;
    }
    rec[Y::ELEM] = op.tsdV;
    rec[Y::ELEM + 1] = op.nudV;
    rec[Y::ELEM + 2] = op.visc;
    rec[Y::ELEM + 3] = op.ua[0];
    rec[Y::ELEM + 4] = op.ua[1];
    rec[Y::ELEM + 5] = op.m0dt;
  }
  if(t < (uint32_t)Y::WORDS) s_rec[ne * Y::STRIDE + t] = R(0);   // the record of the unused list entries
  // block of this thread's list; row of the LDS rows: the first list of a block at its block, the others
  // behind the blocks in order
  uint32_t blk = (uint32_t)__popcll(bstart & (~0ull >> (63 - (t & 63u)))) - 1;
  for(uint32_t v = 0; v < (t >> 6); ++v) blk += s_wave[0][v];
  const uint32_t lds_row_t = (lo >> 63) ? blk : nblk + (t - blk - 1);
  if(lo >> 63) s_first[blk] = (uint16_t)t;
  if(RHS && (hi >> 15)) {
    uint32_t row = (uint32_t)__popcll(rstart & ((1ull << (t & 63u)) - 1));
    for(uint32_t v = 0; v < (t >> 6); ++v) row += s_wave[1][v];
    s_rowfirst[row] = (uint16_t)t;
  }
  if(t == 0) {
    s_first[nblk] = (uint16_t)nlists;
    if constexpr(RHS) s_rowfirst[nrows] = (uint16_t)nlists;
  }
  __syncthreads();

  R A[D][D], up[D], pu[D], tp[D], S = R(0), pp = R(0), tu = R(0);
#pragma unroll
  for(int r = 0; r < D; ++r) {
    up[r] = pu[r] = tp[r] = R(0);
#pragma unroll
    for(int c = 0; c < D; ++c) A[r][c] = R(0);
  }
  if(t < nlists) {
    // NavierStokesSpecializations.hpp:66-145 / 196-301, per contribution (element, row node a, column node b)
    const R c0 = R(D == 2 ? 1.0 / 6.0 : 1.0 / 12.0);
    const R ctp = R(D == 2 ? 8.0 : 15.0);   // c0 tau / dt = ctp (tau / (D^2 V)) (V / (12|20 dt))
#pragma unroll
    for(int i = 0; i < LEN; ++i) {
      const uint32_t entry = i < 5 ? (uint32_t)(lo >> (11 * i)) & 2047u : hi & 2047u;
      const R* rec = s_rec + (entry >> 4) * Y::STRIDE;
      const R* ra = rec + ((entry >> 2) & 3u) * Y::COL;
      const R* rb = rec + (entry & 3u) * Y::COL;
      const bool diag = ((entry >> 2) & 3u) == (entry & 3u);
      R na[D], nb[D], nanb = R(0);
#pragma unroll
      for(int d = 0; d < D; ++d) { na[d] = ra[d]; nb[d] = rb[d]; }
      const R una = ra[D], unb = rb[D];
      const R tsdV = rec[Y::ELEM], nudV = rec[Y::ELEM + 1], visc = rec[Y::ELEM + 2];
      const R u0 = rec[Y::ELEM + 3], u1 = rec[Y::ELEM + 4], m0dt = rec[Y::ELEM + 5];
#pragma unroll
      for(int d = 0; d < D; ++d) nanb += na[d] * nb[d];
      const R cc = c0 + tsdV * una;         // convection, standard and SUPG
      const R hc = R(0.5) * cc, h0u = hc * u0, h1u = hc * u1;
      // n_a . u~ with the tetrahedron substitution of vk for wk (lines 236-238)
      R naut = na[0] * u0 + (D == 3 ? na[1] + na[D - 1] : na[1]) * u1;
      const R pn = c0 + (R(0.5) * tsdV) * naut;
      const R tpc = ctp * tsdV * m0dt;
      const R tuo = m0dt + tpc * una;
      S += cc * unb;
      S += nudV * nanb;
      pp += tsdV * nanb;                    // tau_ps = tau_su
      tu += diag ? tuo + m0dt : tuo;
      const R pua = tsdV * unb;
#pragma unroll
      for(int r = 0; r < D; ++r) {
        const R Q = (r == 0 ? h0u : h1u) + visc * na[r];   // W rows use vk (lines 224-226)
#pragma unroll
        for(int c = 0; c < D; ++c) A[r][c] += Q * nb[c];
        up[r] += cc * nb[r];
        pu[r] += pua * na[r];
        pu[r] += pn * nb[r];
        tp[r] += tpc * na[r];
      }
    }
  }
  __syncthreads();   // the block rows replace the records
  if(t < nlists) {
    const R th = (R)g.theta, thq = (R)g.thq, inv_rho = (R)g.inv_rho;
#pragma unroll
    for(int r = 0; r < D; ++r) {
      A[r][r] += S;
      up[r] *= inv_rho;
    }
    pp *= inv_rho;
    if constexpr(RHS) {
      const uint32_t nd = (uint32_t)(lo >> 55) & 255u;
      const double2 uv = s_uv[nd], wp = s_wp[nd];
      const double st[4] = {uv.x, uv.y, wp.x, wp.y};
      R xb[NEQ];
#pragma unroll
      for(int c = 0; c < NEQ; ++c) xb[c] = (R)st[c];
#pragma unroll
      for(int r = 0; r < D; ++r) {
        R s = up[r] * xb[D];
#pragma unroll
        for(int c = 0; c < D; ++c) s += A[r][c] * xb[c];
        s_rhs[t * NEQ + r] = s;
      }
      R s = pp * xb[D];
#pragma unroll
      for(int c = 0; c < D; ++c) s += pu[c] * xb[c];
      s_rhs[t * NEQ + D] = s;
    }
    R m[NN];
#pragma unroll
    for(int r = 0; r < D; ++r) {
#pragma unroll
      for(int c = 0; c < D; ++c) m[r * NEQ + c] = th * A[r][c] + (r == c ? tu : R(0));
      m[r * NEQ + D] = th * up[r];
      m[D * NEQ + r] = tp[r] + thq * pu[r];
    }
    m[NN - 1] = thq * pp;
#pragma unroll
    for(int q = 0; q < NN; ++q) s_row[lds_row_t * LDW + q] = m[q];
  }
  __syncthreads();
  {
    // 16 bytes per lane where a block is a multiple of that (D = 3)
    constexpr int W = (NN * sizeof(R)) % 16 == 0 ? 16 / sizeof(R) : 1;
    constexpr int P = NN / W;   // pieces per block
    struct alignas(W * sizeof(R)) Piece { R v[W]; };
    Piece* dst = reinterpret_cast<Piece*>(static_cast<R*>(g.values) + (uint64_t)blk0 * NN);
    constexpr int U = 4;        // pieces in flight per thread
    for(uint32_t o = t; o < nblk * P; o += U * kThreads) {
      Piece sum[U];
      uint32_t f[U], l[U];
#pragma unroll
      for(int u = 0; u < U; ++u) {
        const uint32_t ou = min(o + u * kThreads, nblk * P - 1), sb = ou / P;
        sum[u] = *reinterpret_cast<const Piece*>(s_row + sb * LDW + (ou % P) * W);
        f[u] = s_first[sb];
        l[u] = s_first[sb + 1];
      }
#pragma unroll
      for(int u = 0; u < U; ++u) {
        const uint32_t ou = o + u * kThreads;
        if(ou >= nblk * P) break;
        const uint32_t sb = ou / P;
        for(uint32_t r = nblk + f[u] - sb; r + sb + 1 < nblk + l[u]; ++r) {   // the other lists of the block
          const Piece add = *reinterpret_cast<const Piece*>(s_row + r * LDW + (ou % P) * W);
#pragma unroll
          for(int q = 0; q < W; ++q) sum[u].v[q] += add.v[q];
        }
        dst[ou] = sum[u];
      }
    }
  }
  if constexpr(RHS) {
    // four lanes per rhs entry, each a quarter of the row's lists (strided), added by shuffles
    const uint32_t h = t & 3u;
    for(uint32_t o = t >> 2; o < (nrows * NEQ + 15) / 16 * 16; o += kThreads / 4) {   // whole waves
      const uint32_t oo = min(o, nrows * NEQ - 1), row = oo / NEQ, r = oo % NEQ;
      const uint32_t qe = s_rowfirst[row + 1];
      R sum = R(0);
      for(uint32_t q = s_rowfirst[row] + h; q < qe; q += 4) sum -= s_rhs[q * NEQ + r];
      sum += __shfl_xor(sum, 1, 64);
      sum += __shfl_xor(sum, 2, 64);
      if(h == 0 && o < nrows * NEQ) g.rhs[(uint64_t)r0 * NEQ + o] = (double)sum;
    }
  }
}

template<int D, typename R, bool RHS>
__global__ __launch_bounds__(kThreads, sizeof(R) == sizeof(float) ? 4 : 3) void k_assemble_lists(AsmArgs g, PackArgs f)
{
  extern __shared__ double4 s_dyn[];
  assemble_lists_wg<D, R, RHS, true>(g, f, xcd_order(blockIdx.x, gridDim.x), reinterpret_cast<unsigned char*>(s_dyn));
}

// ---------------------------------------------------------------------------------------------
// Batched FP32 assembly of many tetrahedral systems (serving): one persistent launch whose
// workgroups walk the concatenated workgroup lists of the systems in a device table.
// ---------------------------------------------------------------------------------------------
struct BatchEntry {
  AsmArgs g;
  PackArgs pk;
  uint32_t wg_begin, node_begin, n_nodes, pad;
};

struct BatchHeader {
  uint32_t n_cases, total_wg, total_nodes, pad;
};

__device__ __forceinline__ uint32_t batch_find(const BatchEntry* e, uint32_t n, uint32_t key, bool by_wg)
{
  uint32_t lo = 0, hi = n;   // last entry with begin <= key
  while(hi - lo > 1) {
    const uint32_t mid = (lo + hi) >> 1;
    if((by_wg ? e[mid].wg_begin : e[mid].node_begin) <= key) lo = mid; else hi = mid;
  }
  return lo;
}

__global__ void k_batch_pack(const BatchHeader* __restrict__ hd, const BatchEntry* __restrict__ e)
{
  const uint32_t total = hd->total_nodes, n = hd->n_cases;
  for(uint32_t j = blockIdx.x * blockDim.x + threadIdx.x; j < total; j += gridDim.x * blockDim.x) {
    const uint32_t c = batch_find(e, n, j, false);
    const uint32_t i = j - e[c].node_begin;
    const PackArgs& a = e[c].pk;
    a.st[i] = make_double4(a.u[0][i], a.u[1][i], a.u[2][i], a.p[i]);
    a.ad[i] = make_double4(a.ua[0][i], a.ua[1][i], a.ua[2][i], a.nu[i]);
  }
}

__global__ __launch_bounds__(kThreads) void k_batch_assemble(const BatchHeader* __restrict__ hd,
                                                              const BatchEntry* __restrict__ e)
{
  extern __shared__ double4 s_dyn[];
  const uint32_t total = hd->total_wg, n = hd->n_cases;
  for(uint32_t task = blockIdx.x; task < total; task += gridDim.x) {
    __syncthreads();   // the previous task's LDS reads are done
    const uint32_t c = batch_find(e, n, task, true);
    assemble_lists_wg<3, float, false, false>(e[c].g, e[c].pk, task - e[c].wg_begin, reinterpret_cast<unsigned char*>(s_dyn));
  }
}

// Matrix-free FP64 residual of the assembled, Dirichlet-constrained system: per node row
// r_i = sum over incident elements of (b_e(a) - M_e(a, :) x~_e), with x~ = x except on constrained dofs
// where it holds the eliminated value (the symmetric elimination moves A[:, c] v_c to the rhs).
// Constrained rows are fixed afterwards (r = v - x).  No matrix is read or written.
template<class Op>
__global__ __launch_bounds__(kThreads) void k_residual(AsmArgs g)
{
  constexpr int K = Op::K, NEQ = Op::NEQ, NN = NEQ * NEQ;
  __shared__ double s_res[kThreads * NEQ];
  __shared__ uint32_t s_rowinc[kThreads + 1];
  const uint32_t wg = xcd_order(blockIdx.x, gridDim.x);
  const uint32_t r0 = g.wg_rows[wg], r1 = g.wg_rows[wg + 1];
  const uint32_t nrows = r1 - r0;
  const uint32_t i0 = g.inc_ptr[r0];
  const uint32_t ninc = g.inc_ptr[r1] - i0;
  const int t = threadIdx.x;
  for(uint32_t j = t; j <= nrows; j += kThreads) s_rowinc[j] = g.inc_ptr[r0 + j] - i0;
  const bool active = (uint32_t)t < ninc;
  Op op;
  double rhs[NEQ], y[NEQ];
#pragma unroll
  for(int r = 0; r < NEQ; ++r) { rhs[r] = 0.; y[r] = 0.; }
  if(active) {
    const uint32_t ea = g.inc[i0 + t];
    op.prepare(g, ea / K, (int)(ea % K));
    static_for<0, K>([&](auto bc) {
      constexpr int B = decltype(bc)::value;
      double xb[NEQ], xt[NEQ], mb[NN];
      load_state<NEQ, double>(g, op.cn[B], xb);
#pragma unroll
      for(int c = 0; c < NEQ; ++c) xt[c] = g.xt[(uint64_t)op.cn[B] * NEQ + c];
      op.template block<B, true, double>(g, mb, rhs, xb);
#pragma unroll
      for(int r = 0; r < NEQ; ++r)
#pragma unroll
        for(int c = 0; c < NEQ; ++c) y[r] += mb[r * NEQ + c] * xt[c];
    });
    if(g.body_force) op.rhs_source(g, rhs);
#pragma unroll
    for(int r = 0; r < NEQ; ++r) s_res[t * NEQ + r] = rhs[r] - y[r];
  }
  __syncthreads();
  for(uint32_t o = t; o < nrows * NEQ; o += kThreads) {
    const uint32_t row = o / NEQ, r = o % NEQ;
    double s = 0.;
    for(uint32_t q = s_rowinc[row]; q < s_rowinc[row + 1]; ++q) s += s_res[q * NEQ + r];
    g.res[(uint64_t)(r0 + row) * NEQ + r] = s;
  }
}

__global__ void k_xtilde(uint64_t dofs, int neq, const uint8_t* __restrict__ mask, const double* __restrict__ vfirst,
                         const double* __restrict__ x, double* __restrict__ xt)
{
  const uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if(i >= dofs) return;
  const uint8_t m = mask ? mask[i / neq] : 0;
  xt[i] = ((m >> (i % neq)) & 1) ? vfirst[i] : x[i];
}

__global__ void k_bc_residual(uint32_t n, const uint32_t* __restrict__ dof, const double* __restrict__ vlast,
                              const double* __restrict__ x, double* __restrict__ r)
{
  const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
  if(i < n) r[dof[i]] = vlast[i] - x[dof[i]];
}

// packed node records
__global__ void k_pack_coords(uint32_t n, int dim, const double* __restrict__ x, const double* __restrict__ y,
                              const double* __restrict__ z, double4* __restrict__ xp)
{
  const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
  if(i >= n) return;
  xp[i] = make_double4(x[i], y[i], dim == 3 ? z[i] : 0., 0.);
}

template<int D>
__global__ void k_pack_fields(uint32_t n, PackArgs a)
{
  const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
  if(i >= n) return;
  double4 st, ad;
  read_node<D>(a, i, st, ad);
  a.st[i] = st;
  a.ad[i] = ad;
}

PackArgs field_args(Fields& F)
{
  PackArgs a = {};
  for(int d = 0; d < F.mesh->dim; ++d) {
    a.u[d] = F.u[d].as<double>();
    a.ua[d] = F.uadv[d].as<double>();
  }
  a.p = F.p.as<double>();
  a.nu = F.nu.as<double>();
  a.st = F.st.as<double4>();
  a.ad = F.ad.as<double4>();
  return a;
}

void pack_fields(Fields& F)
{
  const Mesh& M = *F.mesh;
  Context& c = *M.ctx;
  const PackArgs a = field_args(F);
  if(M.dim == 3) hipLaunchKernelGGL(k_pack_fields<3>, dim3(grid_for(M.n_nodes, 256)), dim3(256), 0, c.stream, M.n_nodes, a);
  else hipLaunchKernelGGL(k_pack_fields<2>, dim3(grid_for(M.n_nodes, 256)), dim3(256), 0, c.stream, M.n_nodes, a);
  HIP_OK(hipGetLastError());
}

template<class Op, typename R, typename VR, bool RHS>
void launch(const AsmArgs& g, const Lss& L)
{
  Context& c = *L.ctx;
  timer_begin(c, CF3HIP_KERNEL_ASSEMBLY);
  hipLaunchKernelGGL((k_assemble<Op, R, VR, RHS>), dim3(L.n_wg), dim3(kThreads), 0, c.stream, g);
  HIP_OK(hipGetLastError());
  timer_end(c, CF3HIP_KERNEL_ASSEMBLY);
}

// specialised simplices: by block lists; a system without plans (a row of more elements or block lists than a
// plan holds) takes the staged reduction
template<int D, typename R, bool RHS>
void launch_spec(const AsmArgs& g, const Lss& L, Fields& F)
{
  if(!g.plan) {
    pack_fields(F);
    launch<SpecP1<D, R>, R, R, RHS>(g, L);
    return;
  }
  Context& c = *L.ctx;
  const size_t lds = PlanLayout<D, R>::lds_bytes(RHS, L.plan_nodes, L.plan_elems, L.plan_lists);
  timer_begin(c, CF3HIP_KERNEL_ASSEMBLY);
  hipLaunchKernelGGL((k_assemble_lists<D, R, RHS>), dim3(L.n_plan), dim3(kThreads), lds, c.stream, g, field_args(F));
  HIP_OK(hipGetLastError());
  timer_end(c, CF3HIP_KERNEL_ASSEMBLY);
}

__global__ void k_clear_flag(int* f) { f[0] = 0; }

AsmArgs make_args(Lss& L, Fields& F, const cf3hip_ns_params& prm, bool pack = true)
{
  if(!L.mesh) CF3_THROW(CF3HIP_ERR_NOT_CREATED, "system was created without a mesh: no element scatter map");
  if(prm.theta < 0. || prm.theta > 1.)
    CF3_THROW(CF3HIP_ERR_NOT_CREATED, "Value for theta option is outside of the valid range from 0 to 1.");
  if(!(prm.dt > 0.)) CF3_THROW(CF3HIP_ERR_INVALID_ARG, "dt must be positive");
  const Mesh& M = *L.mesh;
  if(F.mesh != L.mesh) CF3_THROW(CF3HIP_ERR_INVALID_ARG, "fields belong to another mesh");
  if(L.neq != M.dim + 1) CF3_THROW(CF3HIP_ERR_INVALID_ARG, "the NS system needs neq = dim + 1");
  const bool spec = prm.use_specializations && !is_cell(M.etype);
  if(!spec && prm.supg_type == CF3HIP_SUPG_CF2 && !(prm.u_ref > 0.))
    CF3_THROW(CF3HIP_ERR_INVALID_ARG, "supg_type cf2 needs a positive u_ref (SUPG.hpp:196)");
  AsmArgs g = {};
  g.body_force = F.has_g ? 1 : 0;
  g.xp = M.xp.as<double4>();
  g.st = F.st.as<double4>();
  g.ad = F.ad.as<double4>();
  for(int d = 0; d < 3; ++d) g.g[d] = d < M.dim ? F.g[d].as<double>() : nullptr;
  g.conn = M.conn.as<uint32_t>();
  g.wg_rows = L.wg_rows.as<uint32_t>();
  g.row_ptr = L.row_ptr.as<uint32_t>();
  g.inc_ptr = L.inc_ptr.as<uint32_t>();
  g.inc = L.inc.as<uint32_t>();
  g.inc_pos = L.inc_pos.as<uint8_t>();
  g.blk_beg = L.blk_beg.as<uint8_t>();
  g.blk_acc = L.blk_acc.as<uint16_t>();
  if(L.n_plan) {
    g.plan = L.plan.as<unsigned char>();
    g.plan_nodes = L.plan_nodes; g.plan_elems = L.plan_elems; g.plan_lists = L.plan_lists;
  }
  g.rho = prm.rho; g.inv_rho = 1. / prm.rho;
  g.dt = prm.dt; g.theta = prm.theta; g.thq = prm.theta * (1. / prm.theta);
  g.invdt = 1. / prm.dt; g.f4dt2 = 4. / (prm.dt * prm.dt);
  g.supg_type = prm.supg_type;
  g.c1 = prm.c1; g.c2 = prm.c2; g.a_ps = prm.alpha_ps; g.a_su = prm.alpha_su; g.a_bu = prm.alpha_bu;
  g.u_ref = prm.u_ref;
  g.status = L.ctx->status_flag();
  if(pack) pack_fields(F);
  return g;
}

void check_status(Context& c)
{
  if(c.async_mode) return;
  int st = 0;
  HIP_OK(hipMemcpyAsync(&st, c.status_flag(), sizeof(int), hipMemcpyDeviceToHost, c.stream));
  HIP_OK(hipStreamSynchronize(c.stream));
  if(st == 2) CF3_THROW(CF3HIP_ERR_INVALID_ARG, "ComputeTau cf2: element Reynolds number u_ref he / (2 nu) not positive");
  if(st) CF3_THROW(CF3HIP_ERR_SINGULAR, "non-positive element Jacobian determinant");
}

template<class Op>
void launch_residual(const AsmArgs& g, const Lss& L)
{
  Context& c = *L.ctx;
  timer_begin(c, CF3HIP_KERNEL_RESIDUAL);
  hipLaunchKernelGGL((k_residual<Op>), dim3(L.n_wg), dim3(kThreads), 0, c.stream, g);
  HIP_OK(hipGetLastError());
  timer_end(c, CF3HIP_KERNEL_RESIDUAL);
}

}  // namespace

void mesh_pack_coords(Mesh& M)
{
  Context& c = *M.ctx;
  if(!M.xp.ptr) M.xp.alloc(&c, sizeof(double4) * M.n_nodes);
  hipLaunchKernelGGL(k_pack_coords, dim3(grid_for(M.n_nodes, 256)), dim3(256), 0, c.stream, M.n_nodes, M.dim,
                     M.x[0].as<double>(), M.x[1].as<double>(), M.dim == 3 ? M.x[2].as<double>() : nullptr,
                     M.xp.as<double4>());
  HIP_OK(hipGetLastError());
}

void assemble(Lss& L, Fields& F, const cf3hip_ns_params& prm)
{
  // the specialised kernels read the fields themselves or pack them in launch_spec
  const bool spec = L.mesh && prm.use_specializations && !is_cell(L.mesh->etype);
  AsmArgs g = make_args(L, F, prm, !spec);
  const Mesh& M = *L.mesh;
  if(prm.precision == CF3HIP_FP32 && !L.has_fp32)
    CF3_THROW(CF3HIP_ERR_NOT_CREATED, "FP32 assembly needs cf3hip_lss_enable_fp32");
  Context& c = *L.ctx;
  const bool fp32 = prm.precision == CF3HIP_FP32;
  // ZeroLSS: every value and rhs entry is overwritten by the kernel; the conditions of the previous
  // step are forgotten
  lss_clear_conditions(L);
  // the right-hand side is formed by the FP64 pass only (FP64 outer residual of the precision form)
  g.rhs = fp32 ? nullptr : L.rhs.as<double>();
  // element-validity flag: cleared per call in synchronous mode; in asynchronous mode it accumulates
  // and is reported by cf3hip_context_synchronize
  if(!c.async_mode) hipLaunchKernelGGL(k_clear_flag, dim3(1), dim3(1), 0, c.stream, g.status);
  g.values = fp32 ? L.values32.ptr : L.values.ptr;

  if(is_cell(M.etype)) {
    launch_hex(g, L, fp32 ? 1 : 0);
  } else if(spec && M.etype == CF3HIP_TETRA3D) {
    if(fp32) launch_spec<3, float, false>(g, L, F);
    else launch_spec<3, double, true>(g, L, F);
  } else if(spec && M.etype == CF3HIP_TRIAG2D) {
    if(fp32) launch_spec<2, float, false>(g, L, F);
    else launch_spec<2, double, true>(g, L, F);
  } else if(M.etype == CF3HIP_TETRA3D) {
    if(fp32) launch<GenericP1<3>, double, float, false>(g, L);
    else launch<GenericP1<3>, double, double, true>(g, L);
  } else {
    if(fp32) launch<GenericP1<2>, double, float, false>(g, L);
    else launch<GenericP1<2>, double, double, true>(g, L);
  }
  check_status(c);
}

void ns_residual(Lss& L, Fields& F, const cf3hip_ns_params& prm, const double* x, double* r, bool pack)
{
  if(L.periodic)
    CF3_THROW(CF3HIP_ERR_NOT_IMPLEMENTED, "the matrix-free residual (precision form) takes systems without periodic links");
  AsmArgs g = make_args(L, F, prm, pack);
  const Mesh& M = *L.mesh;
  Context& c = *L.ctx;
  if(L.xtilde.bytes < sizeof(double) * L.dofs) L.xtilde.alloc(&c, sizeof(double) * L.dofs);
  hipLaunchKernelGGL(k_xtilde, dim3(grid_for(L.dofs, 256)), dim3(256), 0, c.stream, L.dofs, L.neq,
                     L.bc_n ? L.bc_mask.as<uint8_t>() : (const uint8_t*)nullptr,
                     L.bc_n ? L.bc_vfirst.as<double>() : (const double*)nullptr, x, L.xtilde.as<double>());
  g.xt = L.xtilde.as<double>();
  g.res = r;
  const bool spec = prm.use_specializations && !is_cell(M.etype);
  if(is_cell(M.etype)) launch_hex(g, L, 2);
  else if(spec && M.etype == CF3HIP_TETRA3D) launch_residual<SpecP1<3, double> >(g, L);
  else if(spec && M.etype == CF3HIP_TRIAG2D) launch_residual<SpecP1<2, double> >(g, L);
  else if(M.etype == CF3HIP_TETRA3D) launch_residual<GenericP1<3> >(g, L);
  else launch_residual<GenericP1<2> >(g, L);
  if(L.bc_n)
    hipLaunchKernelGGL(k_bc_residual, dim3(grid_for(L.bc_n, 256)), dim3(256), 0, c.stream, L.bc_n,
                       L.bc_dof, L.bc_vlast, x, r);
  HIP_OK(hipGetLastError());
}

// ---------------------------------------------------------------------------------------------
// batched FP32 assembly (serving): device table + persistent launch captured once in a hipGraph
// ---------------------------------------------------------------------------------------------
namespace {
constexpr unsigned kBatchPackGrid = 1024;
constexpr unsigned kBatchAsmGrid = 2048;   // persistent workgroups (8 per CU)
constexpr size_t kBatchHeaderBytes = 256;
constexpr size_t kBatchLds = 16384;   // of the captured assembly launch, enough for any plan
static_assert(PlanLayout<3, float>::lds_bytes(false, kPlanNodes, kPlanElems, kAsmThreads) <= kBatchLds);
}  // namespace

size_t batch_table_bytes(uint32_t max_cases) { return kBatchHeaderBytes + sizeof(BatchEntry) * max_cases; }

void batch_assemble(Batch& B, uint32_t n, Lss* const* L, Fields* const* F, const cf3hip_ns_params* prm)
{
  if(n > B.max_cases) CF3_THROW(CF3HIP_ERR_LIMIT, "more systems than the batch was created for");
  BatchHeader* hd = reinterpret_cast<BatchHeader*>(B.host_table);
  BatchEntry* ent = reinterpret_cast<BatchEntry*>(static_cast<char*>(B.host_table) + kBatchHeaderBytes);
  uint32_t wg = 0, nodes = 0;
  for(uint32_t i = 0; i < n; ++i) {
    Lss& Li = *L[i];
    Fields& Fi = *F[i];
    if(!Li.mesh || Li.mesh->etype != CF3HIP_TETRA3D || !prm[i].use_specializations)
      CF3_THROW(CF3HIP_ERR_NOT_IMPLEMENTED, "batched assembly takes tetrahedral systems with the specialised kernel");
    if(!Li.has_fp32) CF3_THROW(CF3HIP_ERR_NOT_CREATED, "batched FP32 assembly needs cf3hip_lss_enable_fp32");
    if(Li.periodic) CF3_THROW(CF3HIP_ERR_NOT_IMPLEMENTED, "batched assembly takes systems without periodic links");
    if((uint64_t)wg + Li.n_plan > 0xffffffffull || (uint64_t)nodes + Li.n_nodes > 0xffffffffull)
      CF3_THROW(CF3HIP_ERR_LIMIT, "batch too large");
    // ZeroLSS: forget the conditions of the previous step (mask cleared on the batch stream)
    lss_forget_conditions(Li);
    HIP_OK(hipStreamSynchronize(Li.ctx->stream));
    if(Li.bc_mask.ptr) HIP_OK(hipMemsetAsync(Li.bc_mask.ptr, 0, Li.n_nodes, B.stream));
    HIP_OK(hipMemsetAsync(Li.ctx->status_flag(), 0, sizeof(int), B.stream));   // element-validity flag
    AsmArgs g = make_args(Li, Fi, prm[i], false);
    g.values = Li.values32.ptr;
    g.rhs = nullptr;
    ent[i].g = g;
    PackArgs& pk = ent[i].pk;
    for(int d = 0; d < 3; ++d) {
      pk.u[d] = Fi.u[d].as<double>();
      pk.ua[d] = Fi.uadv[d].as<double>();
    }
    pk.p = Fi.p.as<double>();
    pk.nu = Fi.nu.as<double>();
    pk.st = Fi.st.as<double4>();
    pk.ad = Fi.ad.as<double4>();
    ent[i].wg_begin = wg;
    ent[i].node_begin = nodes;
    ent[i].n_nodes = Li.n_nodes;
    wg += Li.n_plan;
    nodes += Li.n_nodes;
  }
  hd->n_cases = n;
  hd->total_wg = n ? wg : 0;
  hd->total_nodes = n ? nodes : 0;
  HIP_OK(hipMemcpyAsync(B.table.ptr, B.host_table, kBatchHeaderBytes + sizeof(BatchEntry) * (n ? n : 1),
                        hipMemcpyHostToDevice, B.stream));
  if(!B.exec) {
    // the two launches read the table from device memory, so one capture serves every later batch
    const BatchHeader* dh = B.table.as<BatchHeader>();
    const BatchEntry* de = reinterpret_cast<const BatchEntry*>(B.table.as<char>() + kBatchHeaderBytes);
    hipGraph_t graph = nullptr;
    HIP_OK(hipStreamBeginCapture(B.stream, hipStreamCaptureModeThreadLocal));
    hipLaunchKernelGGL(k_batch_pack, dim3(kBatchPackGrid), dim3(256), 0, B.stream, dh, de);
    hipLaunchKernelGGL(k_batch_assemble, dim3(kBatchAsmGrid), dim3(kThreads), kBatchLds, B.stream, dh, de);
    HIP_OK(hipStreamEndCapture(B.stream, &graph));
    HIP_OK(hipGraphInstantiate(&B.exec, graph, nullptr, nullptr, 0));
    B.graph = graph;
  }
  HIP_OK(hipGraphLaunch(B.exec, B.stream));
  for(uint32_t i = 0; i < n; ++i)   // systems without plans: the staged reduction, after the pack
    if(!L[i]->n_plan)
      hipLaunchKernelGGL((k_assemble<SpecP1<3, float>, float, float, false>), dim3(L[i]->n_wg), dim3(kThreads), 0,
                         B.stream, ent[i].g);
  HIP_OK(hipGetLastError());
  HIP_OK(hipStreamSynchronize(B.stream));
  for(uint32_t i = 0; i < n; ++i) check_status(*L[i]->ctx);
}

}  // namespace cf3hip
