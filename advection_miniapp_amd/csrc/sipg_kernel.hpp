// Advection-diffusion (SIPG, advection_diffusion_solver.cc:469-613) on cells
// of any (multilinear) shape: the whole right-hand side (or implicit
// operator) in one kernel, laid out as the operator kernel (op_kernel.hpp):
// one line of n points per thread, sweeps in registers, LDS between the
// directions. The cell term's geometry (J, adj J, det J) is evaluated point
// by point along the LAST line from the 2^dim corners; the faces' comes from
// a table built once per mesh (sipg_face_table_kernel). Cell term, with the
// explicit sign convention (sign = -1):
//   sign * int grad v . nu grad u = sum_q grad_ref v . (sign nu w_q adj(J)
//   J^-T grad_ref u).
// Faces are element-centric: each cell evaluates its own and the
// neighbour's trace and reference gradient at the face's Gauss points and
// adds its own side of
//   jump = -nu/2 (u- - u+), avg = -nu/2 (d_n u- + d_n u+),
//   value term -sign (jump sigma - avg) JxW, normal-derivative term
//   sign jump JxW (n . J^-T grad_ref v),
// with its own outward normal n; sigma = penalty (|(J-^-1 n)_d| +
// |(J+^-1 n)_d|) / 2 per face point (d the face's reference direction).
// The reference evaluates sigma once per face batch from the exterior cell
// at the first face point (:576-581); on affine meshes the two are equal.
#pragma once

#include "dev_basis.hpp"
#include "dg_common.hpp"
#include "line_geometry.hpp"
#include "op_kernel.hpp"

namespace dgops
{
  // layout of the face table
  template <int dim, int n>
  struct SipgFaces
  {
    static constexpr int nf = dim == 3 ? n * n : n; // points of a face
    static constexpr int nv = 1 << dim;
    // values per face point: J^-1 n of the cell below the face (dim), of
    // the cell above it (dim), JxW
    static constexpr int nt = 2 * dim + 1;
  };

  // Geometry of the face above each cell in each direction d (its face
  // xi_d = 1, the neighbour's xi_d = 0), at the face's Gauss points:
  // T[((cell dim + d) nt + v) nf + pt] = J^-1 n of the cell (v < dim), of
  // the neighbour (dim <= v < 2 dim), JxW (v = 2 dim), with the cell's unit
  // outward normal n. Seen from the neighbour the two J^-1 n exchange and
  // change sign, which gives every cell the face below it. Only interior
  // vertices are perturbed, so faces across periodic boundaries match.
  template <int dim, int n, int d>
  __device__ __forceinline__ void
  sipg_face_entry(const OpParams &P, const DevBasis<double> &B, int64_t cell,
                  int pt, double *__restrict__ T)
  {
    using L          = SipgFaces<dim, n>;
    constexpr int nf = L::nf, NV = L::nv;
    constexpr int t1 = d == 0 ? 1 : 0, t2 = d == 2 ? 1 : 2;
    const int     a = pt % n, b = dim == 3 ? pt / n : 0;
    double        xi[3] = {0, 0, 0};
    xi[t1] = B.xq[a];
    if constexpr (dim == 3)
      xi[t2] = B.xq[b];
    double x[3], J[3][3], adj[3][3], Jn[3][3], adjn[3][3];
    xi[d] = 1;
    multilinear_map<dim>(P.cell_vertices + cell * NV * dim, xi, x, J);
    const double det = adjugate<dim>(J, adj);
    const int    nb  = P.neighbors[cell * 2 * dim + 2 * d + 1];
    xi[d] = 0;
    multilinear_map<dim>(P.cell_vertices + (int64_t)(nb >= 0 ? nb : cell) *
                                             NV * dim,
                         xi, x, Jn);
    const double detn = adjugate<dim>(Jn, adjn);
    // area vector of the face (row d of adj J, along +xi_d)
    double len = 0;
#pragma unroll
    for (int e = 0; e < dim; ++e)
      len = fma(adj[d][e], adj[d][e], len);
    len = sqrt(len);
    double nrm[3] = {0, 0, 0};
#pragma unroll
    for (int e = 0; e < dim; ++e)
      nrm[e] = adj[d][e] / len;
    double JxW = len * B.w[a];
    if constexpr (dim == 3)
      JxW *= B.w[b];
    double *t = T + ((cell * dim + d) * L::nt) * nf + pt;
#pragma unroll
    for (int k = 0; k < dim; ++k)
      {
        double jn = 0, jnn = 0;
#pragma unroll
        for (int e = 0; e < dim; ++e)
          {
            jn  = fma(adj[k][e], nrm[e], jn);
            jnn = fma(adjn[k][e], nrm[e], jnn);
          }
        t[k * nf]         = jn / det;
        t[(dim + k) * nf] = jnn / detn;
      }
    t[2 * dim * nf] = JxW;
  }

  template <int dim, int n>
  __global__ void __launch_bounds__(256)
  sipg_face_table_kernel(const OpParams                       P,
                         const DevBasis<double> *__restrict__ Bp,
                         double *__restrict__                 T)
  {
    constexpr int nf = SipgFaces<dim, n>::nf;
    const int64_t e  = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (e >= P.n_cells * dim * nf)
      return;
    const int     pt   = (int)(e % nf);
    const int64_t cd   = e / nf;
    const int     d    = (int)(cd % dim);
    const int64_t cell = cd / dim;
    if (d == 0)
      sipg_face_entry<dim, n, 0>(P, *Bp, cell, pt, T);
    else if (d == 1)
      sipg_face_entry<dim, n, 1>(P, *Bp, cell, pt, T);
    else if constexpr (dim == 3)
      sipg_face_entry<dim, n, 2>(P, *Bp, cell, pt, T);
  }

  // The operator on the cells of one workgroup, in the line layout of the
  // operator kernel (op_kernel.hpp): every thread owns a line of n points.
  // Phases: values and neighbour traces at the Gauss points; derivatives and
  // end values of the y and x lines; the fluxes at the points of the LAST
  // line (all three derivatives meet there) and at the face points; the
  // integration along x, y and LAST; back to nodal values. Tangential
  // derivatives at a face come from the traces of all its points (LDS), and
  // their share of the test functions' normal derivative is integrated over
  // the face the same way.
  // Bound by LDS and memory latency at two wavefronts per SIMD: degree 3 in
  // 3D, 32^3 cells, takes 53 us on one MI355X in a kernel trace (three
  // wavefronts at 168 registers spill and take 120 us). Before, the
  // advection kernel in integrate form, a diffusion kernel with one point
  // per task and all operands in LDS, and the inverse mass took 25 + 129 +
  // 16 us: three passes over the vector, and 2 to 3 LDS reads per product.
  template <int dim, int n, bool skew, int fin, int epi>
  __global__ void __launch_bounds__(block_cells(dim == 3 ? n * n : n) *
                                    (dim == 3 ? n * n : n))
  __attribute__((amdgpu_waves_per_eu(2)))
  sipg_operator_kernel(const OpParams                       P,
                       const DevBasis<double> *__restrict__ Bp,
                       const double *__restrict__           faces,
                       const OpBuffers<double>              io)
  {
    using L            = Lay<dim, n>;
    using FT           = SipgFaces<dim, n>;
    constexpr int nl   = L::nl, nd = L::nd, STR = L::stride;
    constexpr int NF   = 2 * dim, NV = 1 << dim, LAST = dim - 1;
    constexpr int CPB  = cells_per_block<dim, n>();
    constexpr int XS   = NV * dim | 1; // LDS stride of the corners
    constexpr int nt   = FT::nt;
    __shared__ double s_u[CPB * STR];
    __shared__ double s_gx[CPB * STR];
    __shared__ double s_gy[dim == 3 ? CPB * STR : 1];
    __shared__ double s_f[CPB * 2 * NF * nl];
    __shared__ double s_X[CPB * XS];
    // rows of S and D that a thread picks by its place in the face: from LDS
    // (a row stride of n | 1 spreads the banks)
    constexpr int     RS = n | 1;
    __shared__ double s_S[n * RS], s_D[n * RS];

    const DevBasis<double> &B   = *Bp;
    const double           *src = io.src;
    const int     tid    = threadIdx.x;
    const int     lc     = tid / nl;
    const int     p      = tid - lc * nl;
    const int64_t cell_t = (int64_t)xcd_block(blockIdx.x, gridDim.x) * CPB + lc;
    const bool    active = cell_t < P.n_cells;
    // threads past the last cell repeat it and store nothing
    const int64_t cell = active ? cell_t : P.n_cells - 1;
    double       *u_l = s_u + lc * STR, *gx_l = s_gx + lc * STR;
    double       *gy_l = s_gy + (dim == 3 ? lc * STR : 0);
    double       *f_l  = s_f + lc * 2 * NF * nl;
    double       *X    = s_X + lc * XS;
    const int     ia   = p % n, ib = dim == 3 ? p / n : 0;

    // ---- values and traces at the Gauss points --------------------------
    __builtin_amdgcn_s_setprio(3);
    double r[n], t[n];
#pragma unroll
    for (int i = 0; i < n; ++i)
      r[i] = src[cell * nd + L::template off<0>(p, i)];
    for (int e = tid; e < n * n; e += CPB * nl)
      {
        s_S[(e / n) * RS + e % n] = B.S[e / n][e % n];
        s_D[(e / n) * RS + e % n] = B.D[e / n][e % n];
      }
    int64_t nb[NF]; // SIPG meshes are periodic: every neighbour exists
#pragma unroll
    for (int f = 0; f < NF; ++f)
      nb[f] = P.neighbors[cell * NF + f];
    for (int e = p; e < NV * dim; e += nl)
      X[e] = P.cell_vertices[cell * NV * dim + e];
    double up[NF], dp[NF];
#pragma unroll
    for (int f = 0; f < NF; ++f)
      {
        constexpr int n2 = n * n;
        const int     d = f / 2, s = f % 2;
        const int     st = d == 0 ? 1 : d == 1 ? n : n2;
        const int     s1 = d == 0 ? n : 1, s2 = d == 2 ? n : n2;
        const double *q = src + nb[f] * nd + ia * s1 + (dim == 3 ? ib * s2 : 0);
        const double(&dphi)[max_n] = s ? B.dphi0 : B.dphi1;
        double nv[n], dv = 0;
#pragma unroll
        for (int l = 0; l < n; ++l)
          nv[l] = q[l * st];
#pragma unroll
        for (int l = 0; l < n; ++l)
          dv = fma(dphi[l], nv[l], dv);
        up[f] = nv[s ? 0 : n - 1];
        dp[f] = dv;
      }
    __builtin_amdgcn_s_setprio(0);
    eo_apply<n, false, false, false>(B.eo_S, r, t);
    lds_write_line<dim, n, 0>(u_l, p, t);
    auto put_traces = [&](const double(&a)[NF], const double(&b)[NF]) {
#pragma unroll
      for (int f = 0; f < NF; ++f)
        {
          f_l[f * nl + p]        = a[f];
          f_l[(NF + f) * nl + p] = b[f];
        }
    };
    put_traces(up, dp);
    __syncthreads();
#pragma unroll
    for (int f = 0; f < NF; ++f)
      {
        double v = 0, w = 0;
#pragma unroll
        for (int i = 0; i < n; ++i)
          {
            v = fma(s_S[ia * RS + i], f_l[f * nl + ib * n + i], v);
            w = fma(s_S[ia * RS + i], f_l[(NF + f) * nl + ib * n + i], w);
          }
        up[f] = v;
        dp[f] = w;
      }
    lds_read_line<dim, n, 1>(u_l, p, t);
    eo_apply<n, false, false, false>(B.eo_S, t, r);
    if constexpr (dim == 3)
      {
        __syncthreads();
        put_traces(up, dp);
        lds_write_line<dim, n, 1>(u_l, p, r);
        __syncthreads();
#pragma unroll
        for (int f = 0; f < NF; ++f)
          {
            double v = 0, w = 0;
#pragma unroll
            for (int j = 0; j < n; ++j)
              {
                v = fma(s_S[ib * RS + j], f_l[f * nl + j * n + ia], v);
                w = fma(s_S[ib * RS + j], f_l[(NF + f) * nl + j * n + ia], w);
              }
            up[f] = v;
            dp[f] = w;
          }
        lds_read_line<dim, n, 2>(u_l, p, t);
        eo_apply<n, false, false, false>(B.eo_S, t, r);
      }
    __syncthreads();

    // ---- derivatives and end values along every direction ----------------
    // r: values on the LAST line; dm: own end derivatives; the own and the
    // neighbours' end values go to LDS (face slots f and NF + f)
    double           dm[NF];
    EoSum<n, double> dl; // derivative along the LAST line
    auto ends = [&](const EoLine<n, double> &v, int d) {
      double a[2], b[2];
      line_ends<n>(B, v, a);
      line_end_derivatives<n>(B, v, b);
#pragma unroll
      for (int s = 0; s < 2; ++s)
        {
          f_l[(2 * d + s) * nl + p] = a[s];
          dm[2 * d + s]             = b[s];
        }
    };
#pragma unroll
    for (int f = 0; f < NF; ++f)
      f_l[(NF + f) * nl + p] = up[f];
    auto expand = [](const EoSum<n, double> &e, double(&o)[n]) {
      constexpr int h = n / 2;
#pragma unroll
      for (int q = 0; q < h; ++q)
        {
          o[q]         = e.e[q] + e.o[q];
          o[n - 1 - q] = e.e[q] - e.o[q];
        }
      if constexpr (n % 2 == 1)
        o[h] = e.m;
    };
    lds_write_line<dim, n, LAST>(u_l, p, r);
    {
      const EoLine<n, double> v(r);
      ends(v, LAST);
      eo_derivative<n, false>(B.eo_D, v, dl);
    }
    __syncthreads();
    {
      double            q[n];
      EoSum<n, double> e;
      lds_read_line<dim, n, 0>(u_l, p, q);
      const EoLine<n, double> v(q);
      ends(v, 0);
      eo_derivative<n, false>(B.eo_D, v, e);
      expand(e, q);
      lds_write_line<dim, n, 0>(gx_l, p, q);
    }
    if constexpr (dim == 3)
      {
        double            q[n];
        EoSum<n, double> e;
        lds_read_line<dim, n, 1>(u_l, p, q);
        const EoLine<n, double> v(q);
        ends(v, 1);
        eo_derivative<n, false>(B.eo_D, v, e);
        expand(e, q);
        lds_write_line<dim, n, 1>(gy_l, p, q);
      }
    __syncthreads();

    // ---- fluxes at the points of the LAST line ---------------------------
    const double              vf = P.vel_factor[0];
    const FluxFactors<double> F(P, vf);
    const double              fcell = -(1. - P.skew) * P.sign * vf;
    const double              fs    = P.skew * P.sign * vf;
    double fl[n];  // flux along LAST
    double acc[n]; // terms tested with the values (mass, skew form)
    double ij[n];  // 1/JxW
    {
      const double *tab = static_cast<const double *>(P.tab_cell);
      double        g0[n];
      expand(dl, g0);
      int q[3];
      L::template idx<LAST>(p, 0, q);
      double xi[3] = {B.xq[q[0]], B.xq[q[1]], dim == 3 ? B.xq[q[2]] : 0.};
      double wl    = B.w[q[0]];
      double rwl   = B.winv[q[0]];
      if constexpr (dim == 3)
        {
          wl *= B.w[q[1]];
          rwl *= B.winv[q[1]];
        }
      double x[3], J0[3][3], J1[3][3];
      xi[LAST] = 0.;
      multilinear_map<dim>(X, xi, x, J0);
      xi[LAST] = 1.;
      multilinear_map<dim>(X, xi, x, J1);
      const double nu = P.sign * P.viscosity;
#pragma unroll
      for (int i = 0; i < n; ++i)
        {
          // the Jacobian is linear along the line
          double J[3][3], adj[3][3];
#pragma unroll
          for (int a = 0; a < dim; ++a)
#pragma unroll
            for (int b = 0; b < dim; ++b)
              J[a][b] = b == LAST ?
                          J0[a][b] :
                          fma(B.xq[i], J1[a][b] - J0[a][b], J0[a][b]);
          const double det = adjugate<dim>(J, adj);
          // 1/det: hardware estimate and two Newton steps
          double rd = __builtin_amdgcn_rcp(det);
          rd        = fma(rd, fma(-det, rd, 1.), rd);
          rd        = fma(rd, fma(-det, rd, 1.), rd);
          const double w = wl * B.w[i];
          ij[i]          = rwl * B.winv[i] * rd;
          const int    o = L::template loff<LAST>(p, i);
          double       g[3], gu[3], h[3], cv[3];
          g[LAST] = g0[i];
          g[0]    = gx_l[o];
          if constexpr (dim == 3)
            g[1] = gy_l[o];
          // diffusion: nu w / det adj(J) adj(J)^T grad_ref u
#pragma unroll
          for (int e = 0; e < dim; ++e)
            {
              gu[e] = adj[0][e] * g[0];
#pragma unroll
              for (int d = 1; d < dim; ++d)
                gu[e] = fma(adj[d][e], g[d], gu[e]);
            }
          const double cd = nu * w * rd;
#pragma unroll
          for (int d = 0; d < dim; ++d)
            {
              h[d] = adj[d][0] * gu[0];
#pragma unroll
              for (int e = 1; e < dim; ++e)
                h[d] = fma(adj[d][e], gu[e], h[d]);
            }
          // advection: w adj(J) a, from the corners for a constant speed,
          // else from the geometry table (row d in the order of direction d)
          if (P.vel_kind == vel_constant)
            {
#pragma unroll
              for (int d = 0; d < dim; ++d)
                {
                  double s = adj[d][0] * P.vel_const[0];
#pragma unroll
                  for (int e = 1; e < dim; ++e)
                    s = fma(adj[d][e], P.vel_const[e], s);
                  cv[d] = w * s;
                }
            }
          else
            {
              const double *row = tab + cell * TableLay<dim, n, double>::stride;
              if constexpr (dim == 3)
                {
                  cv[0] = row[ia * nl + ib + n * i];
                  cv[1] = row[nd + ib * nl + ia + n * i];
                }
              else
                cv[0] = row[ia * nl + i];
              cv[LAST] = row[LAST * nd + i * nl + p];
            }
          const double uc = r[i];
          double       v  = 0;
          if constexpr (fin == fin_integrate)
            if (P.has_mass)
              v = P.mass[0][0] * w * det * uc;
          if constexpr (skew)
            {
              double s = cv[0] * g[0];
#pragma unroll
              for (int d = 1; d < dim; ++d)
                s = fma(cv[d], g[d], s);
              v = fma(fs, s, v);
            }
          acc[i]        = v;
          const double fu = fcell * uc;
          gx_l[o]       = fma(cd, h[0], fu * cv[0]);
          if constexpr (dim == 3)
            gy_l[o] = fma(cd, h[1], fu * cv[1]);
          fl[i] = fma(cd, h[LAST], fu * cv[LAST]);
          __builtin_amdgcn_sched_barrier(0);
        }
    }

    // ---- fluxes at the face points ---------------------------------------
    // f, fd: coefficients of the test function and of its reference
    // derivative normal to the face; c1, c2: of its tangential derivatives
    double f[NF], fd[NF], c1[NF], c2[NF];
    {
      const double *tab_f = static_cast<const double *>(P.tab_face);
      double        D1[n], D2[n];
#pragma unroll
      for (int i = 0; i < n; ++i)
        {
          D1[i] = s_D[ia * RS + i];
          if constexpr (dim == 3)
            D2[i] = s_D[ib * RS + i];
        }
#pragma unroll
      for (int k = 0; k < NF; ++k)
        {
          const int d = k / 2, s = k % 2;
          const int t1 = d == 0 ? 1 : 0, t2 = d == 2 ? 1 : 2;
          // geometry of this face: face 1 is the entry of this cell, face 0
          // the entry of the neighbour below, with the two J^-1 n exchanged
          // and negated
          const int64_t own = s ? cell : nb[k];
          const double *T   = faces + (own * dim + d) * nt * nl + p;
          double        jm[3] = {0, 0, 0}, jp[3] = {0, 0, 0};
#pragma unroll
          for (int e = 0; e < dim; ++e)
            {
              const double a = T[e * nl], b = T[(dim + e) * nl];
              jm[e] = s ? a : -b;
              jp[e] = s ? b : -a;
            }
          const double JxW = T[2 * dim * nl];
          const double an  = s ? tab_f[(nb[k] * dim + d) * nl + p] :
                                 -tab_f[(cell * dim + d) * nl + p];
          // tangential derivatives of both traces
          double g1m = 0, g1p = 0, g2m = 0, g2p = 0;
#pragma unroll
          for (int i = 0; i < n; ++i)
            {
              g1m = fma(D1[i], f_l[k * nl + ib * n + i], g1m);
              g1p = fma(D1[i], f_l[(NF + k) * nl + ib * n + i], g1p);
              if constexpr (dim == 3)
                {
                  g2m = fma(D2[i], f_l[k * nl + i * n + ia], g2m);
                  g2p = fma(D2[i], f_l[(NF + k) * nl + i * n + ia], g2p);
                }
            }
          double dn = fma(jm[d], dm[k], jp[d] * dp[k]);
          dn        = fma(jm[t1], g1m, fma(jp[t1], g1p, dn));
          if constexpr (dim == 3)
            dn = fma(jm[t2], g2m, fma(jp[t2], g2p, dn));
          const double um = f_l[k * nl + p], un = f_l[(NF + k) * nl + p];
          const double j  = um - un;
          const double si = 0.5 * P.penalty * (fabs(jm[d]) + fabs(jp[d]));
          const double W  = 0.5 * P.sign * P.viscosity * JxW;
          f[k]            = fma(an, fma(F.c_own, um, F.c_nb * un),
                     F.c_abs * fabs(an) * j);
          f[k]            = fma(W, fma(si, j, -dn), f[k]);
          const double cd = -W * j;
          fd[k]           = cd * jm[d];
          c1[k]           = cd * jm[t1];
          c2[k]           = dim == 3 ? cd * jm[t2] : 0.;
          // one face's table entries in flight at a time: hoisting those of
          // all faces costs an occupancy step
          __builtin_amdgcn_sched_barrier(0);
        }
    }
    __syncthreads();
    put_traces(c1, c2);
    __syncthreads();
    {
      double D1[n], D2[n];
#pragma unroll
      for (int i = 0; i < n; ++i)
        {
          D1[i] = s_D[i * RS + ia];
          if constexpr (dim == 3)
            D2[i] = s_D[i * RS + ib];
        }
#pragma unroll
      for (int k = 0; k < NF; ++k)
#pragma unroll
        for (int i = 0; i < n; ++i)
          {
            f[k] = fma(D1[i], f_l[k * nl + ib * n + i], f[k]);
            if constexpr (dim == 3)
              f[k] = fma(D2[i], f_l[(NF + k) * nl + i * n + ia], f[k]);
          }
    }

    // ---- integration along x, y and LAST ---------------------------------
    lds_read_line<dim, n, 0>(gx_l, p, t);
    line_integrate<n, true, false>(B, t, f[0], f[1], fd[0], fd[1], r);
    lds_write_line<dim, n, 0>(u_l, p, r);
    __syncthreads();
    if constexpr (dim == 3)
      {
        lds_read_line<dim, n, 1>(gy_l, p, t);
        lds_read_line<dim, n, 1>(u_l, p, r);
        line_integrate<n, true, true>(B, t, f[2], f[3], fd[2], fd[3], r);
        lds_write_line<dim, n, 1>(u_l, p, r);
        __syncthreads();
      }
    lds_read_line<dim, n, LAST>(u_l, p, r);
    line_integrate<n, true, true>(B, fl, f[2 * LAST], f[2 * LAST + 1],
                                  fd[2 * LAST], fd[2 * LAST + 1], r);
#pragma unroll
    for (int i = 0; i < n; ++i)
      {
        if constexpr (skew || fin == fin_integrate)
          r[i] += acc[i];
        if constexpr (fin == fin_inverse_mass)
          r[i] *= ij[i];
      }

    // ---- back to nodal values: LAST (registers), x, y --------------------
    auto back = [&](const double(&a)[n], double(&b)[n]) {
      if constexpr (fin == fin_inverse_mass)
        eo_apply<n, false, false, false>(B.eo_Sinv, a, b);
      else
        eo_apply<n, false, true, false>(B.eo_S, a, b);
    };
    back(r, t);
    lds_write_line<dim, n, LAST>(u_l, p, t);
    __syncthreads();
    lds_read_line<dim, n, 0>(u_l, p, r);
    back(r, t);
    constexpr int OUT = dim == 3 ? 1 : 0;
    if constexpr (dim == 3)
      {
        __syncthreads();
        lds_write_line<dim, n, 0>(u_l, p, t);
        __syncthreads();
        lds_read_line<dim, n, 1>(u_l, p, r);
        back(r, t);
      }
    __builtin_amdgcn_s_setprio(3);
    if (active)
      {
#pragma unroll
        for (int i = 0; i < n; ++i)
          {
            const int64_t k = cell * nd + L::template off<OUT>(p, i);
            if constexpr (epi == epi_store)
              io.dst[k] = io.scale * t[i];
            else
              {
                const double s0 = io.sol_in[k];
                io.sol_out[k]   = fma(io.b_dt, t[i], s0);
                if (!io.last)
                  io.ri_out[k] = fma(io.a_dt, t[i], s0);
              }
          }
      }
  }
} // namespace dgops
