// Inviscid Burgers right-hand side M^-1(-L(u)) (burgers_solver.cc:259-341)
// in the line layout of op_kernel.hpp, for degrees whose over-integration
// tensor fits in LDS and whose rule has at least n = k + 1 points (m =
// k(k+1)/2 >= n: degrees 2 to 4).
//
// The m^dim quadrature values determine the test functions (m >= n), so the
// flux is integrated at the quadrature points as in the advection kernel:
//   sum_d D_d^T (u_c v_d) + sum_faces l_face (x) flux,   v = w adj(J) u,
// with the m-point collocation derivative D, and one contraction R^T per
// direction (R: values at the m Gauss points of the Lagrange basis of the
// n-point rule) leads straight to the n-point Gauss basis of the mass
// matrix, where M^-1 is S^-1 diag(1/JxW).
//
// One thread per (component, line): dim m^(dim-1) threads per cell, every
// 1D product in registers with scalar coefficients in even-odd form; only
// changes of the line direction go through LDS. Faces are element-centric;
// the flux is linear in u- and u+ for given normal speeds, so one task per
// face point (all components) leaves two coefficients.
//
// Measured on one MI355X, before (degree 3 and 4 in 3D: the slab-wise kernel
// of burgers3d_kernel.hpp, which reads both operands of every product from
// LDS; in 2D: one cell per 256-thread workgroup) and now: 3D degree 3, 48^3
// axis-aligned cells 893 -> 421 us; 32^3 perturbed cells 319 -> 207 us;
// degree 2, 32^3 72 -> 32 us; degree 4, 16^3 204 -> 147 us; 2D degree 3,
// 128^2 perturbed cells 201 -> 12 us. Bound by LDS and VALU issue together
// (845 VALU and 84 LDS instructions per wavefront at degree 3). Five waves
// per SIMD fit without spills on axis-aligned cells, three on general ones
// (four spill: 241 us).
#pragma once

#include "burgers_kernel.hpp"

namespace dgops
{
  // out = M in (n -> m)
  template <int n, int m>
  __device__ __forceinline__ void
  eo_rect(const EvenOddRect &M, const double (&in)[n], double (&out)[m])
  {
    constexpr int            h = n / 2, g = m / 2;
    const EoLine<n, double>  v(in);
#pragma unroll
    for (int q = 0; q < g; ++q)
      {
        double se = n % 2 ? M.mc[q] * v.m : M.e[q][0] * v.e[0];
#pragma unroll
        for (int i = n % 2 ? 0 : 1; i < h; ++i)
          se = fma(M.e[q][i], v.e[i], se);
        double so = M.o[q][0] * v.o[0];
#pragma unroll
        for (int i = 1; i < h; ++i)
          so = fma(M.o[q][i], v.o[i], so);
        out[q]         = se + so;
        out[m - 1 - q] = se - so;
      }
    if constexpr (m % 2 == 1)
      {
        double s = n % 2 ? M.mm * v.m : M.mr[0] * v.e[0];
#pragma unroll
        for (int i = n % 2 ? 0 : 1; i < h; ++i)
          s = fma(M.mr[i], v.e[i], s);
        out[g] = s;
      }
  }

  // out = M^T in (m -> n)
  template <int n, int m>
  __device__ __forceinline__ void
  eo_rect_t(const EvenOddRect &M, const double (&in)[m], double (&out)[n])
  {
    constexpr int            h = n / 2, g = m / 2;
    const EoLine<m, double>  v(in);
#pragma unroll
    for (int i = 0; i < h; ++i)
      {
        double se = m % 2 ? M.mr[i] * v.m : M.e[0][i] * v.e[0];
#pragma unroll
        for (int q = m % 2 ? 0 : 1; q < g; ++q)
          se = fma(M.e[q][i], v.e[q], se);
        double so = M.o[0][i] * v.o[0];
#pragma unroll
        for (int q = 1; q < g; ++q)
          so = fma(M.o[q][i], v.o[q], so);
        out[i]         = se + so;
        out[n - 1 - i] = se - so;
      }
    if constexpr (n % 2 == 1)
      {
        double s = m % 2 ? M.mm * v.m : M.mc[0] * v.e[0];
#pragma unroll
        for (int q = m % 2 ? 0 : 1; q < g; ++q)
          s = fma(M.mc[q], v.e[q], s);
        out[h] = s;
      }
  }

  // lines of a cell and component at the m^dim quadrature points
  constexpr int
  burgers_lines(int dim, int m)
  {
    return dim == 3 ? m * m : m;
  }

  // cells per workgroup: about two wavefronts of threads (a barrier every
  // 30 to 60 instructions: with 448 threads degree 3 took 546 us instead of
  // 421, see above; with 256 threads 415 us, but 9% more at 2D degree 4)
  constexpr int
  burgers_line_cells(int dim, int m)
  {
    const int t = dim * burgers_lines(dim, m);
    return t >= 128 ? 1 : 128 / t;
  }

  template <int dim, int n, int m, bool cartesian, int epi, int CPB>
  __global__ void
  __launch_bounds__(CPB *dim *(dim == 3 ? m * m : m))
  __attribute__((amdgpu_waves_per_eu(m <= 6 ? (cartesian ? 5 : 3) : 2)))
  burgers_line_kernel(const OpParams P,
                      const DevBasis<double> *__restrict__   Bd,
                      const BurgersLineTables *__restrict__ BT,
                      const OpBuffers<double> io)
  {
    static_assert(m >= n, "the quadrature values determine the test functions");
    constexpr int L    = burgers_lines(dim, m);
    constexpr int NT   = dim * L; // threads per cell
    constexpr int nn   = dim == 3 ? n * n * n : n * n;
    constexpr int mm   = dim == 3 ? m * m * m : m * m;
    constexpr int nl   = dim == 3 ? n * n : n;
    constexpr int NF   = 2 * dim, LAST = dim - 1, NV = 1 << dim;
    constexpr int XS   = NV * dim | 1;
    constexpr int FS   = NF * L; // one value per face point
    // per component: quadrature values, work space, face values
    constexpr int W1 = mm > FS ? mm : FS;
    constexpr int W2 = FS > n * L ? FS : n * L;
    __shared__ double s_u[CPB * dim * mm];
    __shared__ double s_a[CPB * dim * W1];
    __shared__ double s_f[CPB * dim * W2];
    __shared__ double s_X[cartesian ? 1 : CPB * XS];

    const BurgersLineTables &T   = *BT;
    const DevBasis<double>  &B   = *Bd;
    const int     tid    = threadIdx.x;
    const int     lc     = tid / NT;
    const int     tc     = tid - lc * NT; // thread of the cell
    const int     c      = tc / L;        // component
    const int     r      = tc - c * L;    // line
    const int64_t cell_t = (int64_t)xcd_block(blockIdx.x, gridDim.x) * CPB + lc;
    const bool    active = cell_t < P.n_cells;
    // threads past the last cell repeat it and store nothing
    const int64_t cell = active ? cell_t : P.n_cells - 1;
    double       *Uc = s_u + lc * dim * mm; // [component][point]
    double       *Ac = s_a + lc * dim * W1;
    double       *Fc = s_f + lc * dim * W2;
    double       *U  = Uc + c * mm, *A = Ac + c * W1, *F = Fc + c * W2;
    double       *X  = s_X + (cartesian ? 0 : lc * XS);
    const double *src = io.src + cell * dim * nn + c * nn;
    // (a, b): the line's place in the planes of m points, (i, j) of n points
    const int la = r % m, lb = dim == 3 ? r / m : 0;

    // ---- x sweep of the own values (thread < n^(dim-1)), first tangential
    // sweep of the neighbours' face nodes (line j of face f) ---------------
    if (r < nl)
      {
        double v[n], q[m];
#pragma unroll
        for (int i = 0; i < n; ++i)
          v[i] = src[r * n + i];
        eo_rect<n, m>(T.S, v, q);
        // 3D: U[qx + m (j + n k)], 2D: A[qx + m j]
        double *o = (dim == 3 ? U : A) + r * m;
#pragma unroll
        for (int i = 0; i < m; ++i)
          o[i] = q[i];
      }
    constexpr int NFL = dim == 3 ? NF * n : NF;
#pragma unroll 1
    for (int t = r; t < NFL; t += L)
      {
        const int f = dim == 3 ? t / n : t, j = dim == 3 ? t % n : 0;
        const int d = f / 2, s = f % 2;
        const int sd = d == 0 ? 1 : d == 1 ? n : n * n;
        const int s1 = d == 0 ? n : 1, s2 = d == 2 ? n : n * n;
        const int nb = P.neighbors[cell * NF + f];
        const double *p = io.src + (nb >= 0 ? (int64_t)nb : cell) * dim * nn +
                          c * nn + (s ? 0 : n - 1) * sd +
                          (dim == 3 ? j * s2 : 0);
        double v[n], q[m];
#pragma unroll
        for (int i = 0; i < n; ++i)
          v[i] = p[i * s1];
        eo_rect<n, m>(T.S, v, q);
#pragma unroll
        for (int i = 0; i < m; ++i)
          F[t * m + i] = q[i];
      }
    if constexpr (!cartesian)
      for (int e = tc; e < NV * dim; e += NT)
        X[e] = P.cell_vertices[cell * NV * dim + e];
    __syncthreads();

    // ---- y sweep, second tangential sweep ---------------------------------
    if constexpr (dim == 3)
      {
        if (r < n * m)
          {
            // thread (qx, k): A[qx + m (qy + m k)]
            double v[n], q[m];
#pragma unroll
            for (int j = 0; j < n; ++j)
              v[j] = U[la + m * (j + n * lb)];
            eo_rect<n, m>(T.S, v, q);
#pragma unroll
            for (int j = 0; j < m; ++j)
              A[la + m * (j + m * lb)] = q[j];
          }
        // line aq of face f; held until the first sweep's values are read
        constexpr int NR = (NF * m + L - 1) / L;
        double        tr[NR][m];
#pragma unroll
        for (int k = 0; k < NR; ++k)
          {
            const int t = min(r + k * L, NF * m - 1);
            const int f = t / m, aq = t - f * m;
            double    v[n];
#pragma unroll
            for (int j = 0; j < n; ++j)
              v[j] = F[(f * n + j) * m + aq];
            eo_rect<n, m>(T.S, v, tr[k]);
          }
        __syncthreads();
#pragma unroll
        for (int k = 0; k < NR; ++k)
          {
            const int t = min(r + k * L, NF * m - 1);
            const int f = t / m, aq = t - f * m;
#pragma unroll
            for (int j = 0; j < m; ++j)
              F[f * L + j * m + aq] = tr[k][j];
          }
      }
    // ---- LAST sweep -------------------------------------------------------
    // the point of line r of direction d: offset and stride in the m grid
    auto base = [&](int d) {
      return dim == 3 ? (d == 0 ? m * r : d == 1 ? la + m * m * lb : r) :
                        (d == 0 ? m * r : r);
    };
    auto stride = [&](int d) { return d == 0 ? 1 : d == 1 ? m : m * m; };
    double uz[m];
    {
      double v[n];
#pragma unroll
      for (int k = 0; k < n; ++k)
        v[k] = A[r + L * k];
      eo_rect<n, m>(T.S, v, uz);
#pragma unroll
      for (int k = 0; k < m; ++k)
        U[r + L * k] = uz[k];
    }
    __syncthreads();

    // general cells: row c of w adj(J) times u on the LAST line; adj row c
    // is the cross product of the other two columns of J, which are linear
    // along the line
    double vz[cartesian ? 1 : m];
    if constexpr (!cartesian)
      {
        double xi[3] = {T.x[la], T.x[lb], 0.};
        double x[3], J0[3][3], J1[3][3];
        xi[LAST] = 0.;
        multilinear_map<dim>(X, xi, x, J0);
        xi[LAST] = 1.;
        multilinear_map<dim>(X, xi, x, J1);
        const double w = dim == 3 ? T.w[la] * T.w[lb] : T.w[la];
        if constexpr (dim == 3)
          {
            double a0[3], a1[3], b0[3], b1[3];
#pragma unroll
            for (int e = 0; e < 3; ++e)
              {
                a0[e] = c == 0 ? J0[e][1] : c == 1 ? J0[e][2] : J0[e][0];
                a1[e] = c == 0 ? J1[e][1] : c == 1 ? J1[e][2] : J1[e][0];
                b0[e] = c == 0 ? J0[e][2] : c == 1 ? J0[e][0] : J0[e][1];
                b1[e] = c == 0 ? J1[e][2] : c == 1 ? J1[e][0] : J1[e][1];
                a1[e] -= a0[e];
                b1[e] -= b0[e];
              }
#pragma unroll
            for (int k = 0; k < m; ++k)
              {
                double p[3], q[3];
#pragma unroll
                for (int e = 0; e < 3; ++e)
                  {
                    p[e] = fma(T.x[k], a1[e], a0[e]);
                    q[e] = fma(T.x[k], b1[e], b0[e]);
                  }
                const double *u = Uc + r + L * k;
                double        v = (p[1] * q[2] - p[2] * q[1]) * u[0];
                v = fma(p[2] * q[0] - p[0] * q[2], u[mm], v);
                v = fma(p[0] * q[1] - p[1] * q[0], u[2 * mm], v);
                vz[k] = w * T.w[k] * v;
              }
          }
        else
          {
            // adj = [[J11, -J01], [-J10, J00]]
#pragma unroll
            for (int k = 0; k < m; ++k)
              {
                const double p = c ? -fma(T.x[k], J1[1][0] - J0[1][0], J0[1][0]) :
                                     fma(T.x[k], J1[1][1] - J0[1][1], J0[1][1]);
                const double q = c ? fma(T.x[k], J1[0][0] - J0[0][0], J0[0][0]) :
                                     -fma(T.x[k], J1[0][1] - J0[0][1], J0[0][1]);
                const double *u = Uc + r + L * k;
                vz[k] = w * T.w[k] * fma(p, u[0], q * u[mm]);
              }
          }
      }
    __builtin_amdgcn_sched_barrier(0);

    // ---- lines of the other directions, own end values --------------------
    double ux[m], uy[dim == 3 ? m : 1];
    double um[NF], up[NF];
    auto   ends = [&](const double(&v)[m], int d) {
      double                  e[2];
      const EoLine<m, double> l(v);
      line_ends<m>(T, l, e);
      um[2 * d]     = e[0];
      um[2 * d + 1] = e[1];
    };
#pragma unroll
    for (int i = 0; i < m; ++i)
      ux[i] = U[base(0) + i];
    ends(ux, 0);
    if constexpr (dim == 3)
      {
#pragma unroll
        for (int i = 0; i < m; ++i)
          uy[i] = U[base(1) + i * m];
        ends(uy, 1);
      }
    ends(uz, LAST);
#pragma unroll
    for (int f = 0; f < NF; ++f)
      {
        A[f * L + r] = um[f];
        up[f]        = F[f * L + r];
      }
    __syncthreads();

    // ---- one task per face point: flux_c = ca u-_c + cb u+_c, with the
    // normal speeds of both sides; the coefficients replace the first two
    // components' neighbour values -----------------------------------------
#pragma unroll 1
    for (int t = tc; t < FS; t += NT)
      {
        const int    f = t / L, pt = t - f * L;
        const int    d = f / 2, s = f % 2;
        const int    qa = pt % m, qb = dim == 3 ? pt / m : 0;
        const double w = dim == 3 ? T.w[qa] * T.w[qb] : T.w[qa];
        // normal speeds times the area element
        double unm, unp;
        if constexpr (cartesian)
          {
            // n = -+e_d, area element the product of the other sides
            double len = w * (d == 0 ? P.h[1] : P.h[0]);
            if constexpr (dim == 3)
              len *= d == 2 ? P.h[1] : P.h[2];
            len = s ? len : -len;
            unm = len * Ac[d * W1 + t];
            unp = len * Fc[d * W2 + t];
          }
        else
          {
            // the face's tangents are linear along its edges; corner k of
            // the cell has its coordinates in the bits of k
            const double *Xf = X + ((s ? dim << d : 0));
            const int     t1 = d == 0 ? 1 : 0, t2 = d == 2 ? 1 : 2;
            const int     o1 = dim << t1, o2 = dim << t2;
            const double  a = T.x[qa], b = T.x[qb];
            double        nrm[3];
            if constexpr (dim == 3)
              {
                double c1[3], c2[3];
#pragma unroll
                for (int e = 0; e < 3; ++e)
                  {
                    const double x0 = Xf[e], x1 = Xf[o1 + e], x2 = Xf[o2 + e],
                                 x3 = Xf[o1 + o2 + e];
                    const double p0 = x1 - x0, p1 = x3 - x2;
                    const double q0 = x2 - x0, q1 = x3 - x1;
                    c1[e] = fma(b, p1 - p0, p0);
                    c2[e] = fma(a, q1 - q0, q0);
                  }
                // t1 x t2 points along +xi_d for d = 0, 2 and against it
                // for d = 1
                nrm[0] = c1[1] * c2[2] - c1[2] * c2[1];
                nrm[1] = c1[2] * c2[0] - c1[0] * c2[2];
                nrm[2] = c1[0] * c2[1] - c1[1] * c2[0];
              }
            else
              {
                // the tangent turned to +xi_d
                const double c0 = Xf[o1] - Xf[0], c1 = Xf[o1 + 1] - Xf[1];
                nrm[0] = c1;
                nrm[1] = -c0;
              }
            const double sw = (s != 0) != (d == 1) ? w : -w;
            unm = unp = 0;
#pragma unroll
            for (int e = 0; e < dim; ++e)
              {
                unm = fma(Ac[e * W1 + t], nrm[e], unm);
                unp = fma(Fc[e * W2 + t], nrm[e], unp);
              }
            unm *= sw;
            unp *= sw;
          }
        const double lam = P.alpha * fmax(fabs(unm), fabs(unp));
        Fc[t]            = -0.5 * (unm + lam);
        Fc[W2 + t]       = -0.5 * (unp - lam);
      }
    __syncthreads();
    // general cells: component c of v = w adj(J) u on the LAST lines takes
    // the place of u_c (whose lines are in registers)
    if constexpr (!cartesian)
      {
#pragma unroll
        for (int k = 0; k < m; ++k)
          U[r + L * k] = vz[k];
        __syncthreads();
      }

    // ---- flux and its integration along LAST, (y), x ----------------------
    double f[NF];
#pragma unroll
    for (int k = 0; k < NF; ++k)
      f[k] = fma(Fc[k * L + r], um[k], Fc[W2 + k * L + r] * up[k]);
    double vol = 1;
    if constexpr (cartesian)
      vol = P.h[0] * P.h[1] * (dim == 3 ? P.h[2] : 1.);
    // product of the weights at the line's other coordinates
    const double wl = dim == 3 ? T.w[la] * T.w[lb] : T.w[r];
    double       acc[m];
    auto         direction = [&](const double(&u)[m], int d, bool first) {
      const double *v  = Uc + d * mm + base(d);
      const int     st = stride(d);
      double        g[m];
      const double  cd = cartesian ? wl * vol * P.inv_h[d] : 1.;
#pragma unroll
      for (int i = 0; i < m; ++i)
        g[i] = cartesian ? cd * T.w[i] * v[i * st] * u[i] : v[i * st] * u[i];
      if (first)
        line_integrate<m, false, false>(T, g, f[2 * d], f[2 * d + 1], 0., 0.,
                                        acc);
      else
        line_integrate<m, false, true>(T, g, f[2 * d], f[2 * d + 1], 0., 0.,
                                       acc);
    };
    direction(uz, LAST, true);
#pragma unroll
    for (int i = 0; i < m; ++i)
      A[r + L * i] = acc[i];
    __syncthreads();
    if constexpr (dim == 3)
      {
        double *a = A + base(1);
#pragma unroll
        for (int i = 0; i < m; ++i)
          acc[i] = a[i * m];
        direction(uy, 1, false);
#pragma unroll
        for (int i = 0; i < m; ++i)
          a[i * m] = acc[i];
        __syncthreads();
      }
#pragma unroll
    for (int i = 0; i < m; ++i)
      acc[i] = A[base(0) + i];
    direction(ux, 0, false);

    // ---- to the n-point Gauss basis: x (registers), (y), LAST -------------
    double q[n];
    eo_rect_t<n, m>(T.R, acc, q);
    // F[i + n r] (the face values were last read before the LAST barrier)
#pragma unroll
    for (int i = 0; i < n; ++i)
      F[r * n + i] = q[i];
    __syncthreads();
    if constexpr (dim == 3)
      {
        // thread (i, z): A[i + n (j + n z)]
        if (r < n * m)
          {
            const int i = r % n, z = r / n;
#pragma unroll
            for (int y = 0; y < m; ++y)
              acc[y] = F[i + n * (y + m * z)];
            eo_rect_t<n, m>(T.R, acc, q);
#pragma unroll
            for (int j = 0; j < n; ++j)
              A[i + n * (j + n * z)] = q[j];
          }
        __syncthreads();
      }
    // ---- inverse mass, back to nodal values: LAST, (y), x -----------------
    const bool t_n = r < nl;
    if (t_n)
      {
        const double *a = dim == 3 ? A : F;
#pragma unroll
        for (int z = 0; z < m; ++z)
          acc[z] = a[r + nl * z];
        eo_rect_t<n, m>(T.R, acc, q);
        double ij[n], o[n];
        if constexpr (cartesian)
          {
            double iw = B.winv[r % n] / vol;
            if constexpr (dim == 3)
              iw *= B.winv[r / n];
#pragma unroll
            for (int k = 0; k < n; ++k)
              ij[k] = iw * B.winv[k];
          }
        else
          line_inv_jxw<dim, n, LAST, double, Lay<dim, n>>(X, B.xq, B.w, B.winv,
                                                          r, ij);
#pragma unroll
        for (int k = 0; k < n; ++k)
          q[k] *= ij[k];
        eo_apply<n, false, false, false>(B.eo_Sinv, q, o);
#pragma unroll
        for (int k = 0; k < n; ++k)
          U[r + nl * k] = o[k];
      }
    __syncthreads();
    if constexpr (dim == 3)
      {
        if (t_n)
          {
            double o[n];
            const int a0 = (r % n) + n * n * (r / n);
#pragma unroll
            for (int j = 0; j < n; ++j)
              q[j] = U[a0 + n * j];
            eo_apply<n, false, false, false>(B.eo_Sinv, q, o);
#pragma unroll
            for (int j = 0; j < n; ++j)
              U[a0 + n * j] = o[j];
          }
        __syncthreads();
      }
    if (t_n && active)
      {
        double o[n];
#pragma unroll
        for (int i = 0; i < n; ++i)
          q[i] = U[r * n + i];
        eo_apply<n, false, false, false>(B.eo_Sinv, q, o);
        const int64_t g0 = cell * dim * nn + c * nn + r * n;
#pragma unroll
        for (int i = 0; i < n; ++i)
          {
            const int64_t g = g0 + i;
            if constexpr (epi == epi_store)
              io.dst[g] = io.scale * o[i];
            else
              {
                const double s0 = io.sol_in[g];
                io.sol_out[g]   = fma(io.b_dt, o[i], s0);
                if (!io.last)
                  io.ri_out[g] = fma(io.a_dt, o[i], s0);
              }
          }
      }
  }
} // namespace dgops
