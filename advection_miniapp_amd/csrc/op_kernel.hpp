// Fused matrix-free DG advection operator for gfx950.
//
// One workgroup handles a batch of cells; inside a cell every thread owns
// one 1D line of (k+1) points (n^(dim-1) threads per cell) and keeps it in
// registers. Contractions along the owned line run in registers; changing
// the line direction goes through LDS (write the line, barrier, read the
// line of the new direction).
//
// The operator is evaluated in quadrature space: with S the nodal-to-Gauss
// interpolation matrix, D the collocation derivative at the Gauss points
// and l0/l1 the Gauss-Lagrange values at the faces,
//   integrate(values v, gradients g, face values f) =
//        S^T (v + sum_d D_d^T g_d + sum_faces l_face (x) f)
// so the inverse mass matrix M^-1 = S^-1 diag(1/JxW) S^-T collapses to
//   M^-1 integrate(...) = S^-1 diag(1/JxW) (v + sum_d D_d^T g_d + ...).
// This is the same operator as deal.II's FEEvaluation::integrate followed
// by CellwiseInverseMassMatrix::apply (advection_solver.cc:495-513 and
// :635-657), computed with 9 one-dimensional sweeps per cell instead of
// 12 + 6 in two passes.
//
// Faces are processed element-centric: every cell computes the numerical
// flux on its 2*dim faces with its own outward normal, reading the
// neighbour's face nodes (Gauss-Lobatto nodes make the trace a plain
// subset of the neighbour's values). The flux for the plus side of a
// reference face equals the minus-side flux with the normal reversed
// (advection_solver.cc:560-575), so the result matches the face-centric
// loop of the reference and every dof is written exactly once.
#pragma once

#include <hip/hip_runtime.h>

#include "analytic.hpp"
#include "dev_basis.hpp"
#include "dg_common.hpp"
#include "line_geometry.hpp"

namespace dgops
{
  // Strides of the y and z coordinates and of the cell in LDS. An even
  // number of points gets one element of padding per x row: with rows of
  // 8 (4) values the lanes of a wavefront that read the i-th element of
  // their x lines share 4 (8) of the 32 double-wide banks, with 9 (5) they
  // spread over all. Counted over the lanes of a workgroup in all three
  // directions, the bank cycles per access (1 = no conflict) drop from
  // 8, 4, 1 to 1, 1, 2 for n = 8 and from 2, 4, 2 to 1, 1, 2 for n = 4
  // (x, y, z lines, doubles); odd n are conflict free along x already.
  struct LdsStrides
  {
    int x, y, cell;
  };

  constexpr LdsStrides
  lds_strides(int dim, int n)
  {
    const int x = n % 2 == 1 || (dim == 3 && n == 2) ? n : n + 1;
    const int y = dim == 3 && n == 2 ? 5 : n * x;
    return {x, y, dim == 2 ? y : n == 2 ? 12 : n * y};
  }

  template <int dim, int n>
  struct Lay
  {
    static constexpr int nl = dim == 3 ? n * n : n; // lines per cell
    static constexpr int nd = nl * n;               // dofs per cell

    static constexpr int sx     = lds_strides(dim, n).x;
    static constexpr int sy     = lds_strides(dim, n).y;
    static constexpr int stride = lds_strides(dim, n).cell;

    // LDS offset of point i on line p of direction dir
    template <int dir>
    __device__ static __forceinline__ int
    loff(int p, int i)
    {
      if constexpr (dim == 3)
        {
          if constexpr (dir == 0)
            return i + sx * (p % n) + sy * (p / n);
          else if constexpr (dir == 1)
            return (p % n) + sx * i + sy * (p / n);
          else
            return (p % n) + sx * (p / n) + sy * i;
        }
      else
        {
          if constexpr (dir == 0)
            return i + sx * p;
          else
            return p + sx * i;
        }
    }

    // storage offset of point i on line p of direction dir
    template <int dir>
    __device__ static __forceinline__ int
    off(int p, int i)
    {
      if constexpr (dim == 3)
        {
          if constexpr (dir == 0)
            return i + n * p;
          else if constexpr (dir == 1)
            return (p % n) + n * i + n * n * (p / n);
          else
            return p + n * n * i;
        }
      else
        {
          if constexpr (dir == 0)
            return i + n * p;
          else
            return p + n * i;
        }
    }

    template <int dir>
    __device__ static __forceinline__ void
    idx(int p, int i, int (&q)[3])
    {
      if constexpr (dim == 3)
        {
          if constexpr (dir == 0)
            {
              q[0] = i;
              q[1] = p % n;
              q[2] = p / n;
            }
          else if constexpr (dir == 1)
            {
              q[0] = p % n;
              q[1] = i;
              q[2] = p / n;
            }
          else
            {
              q[0] = p % n;
              q[1] = p / n;
              q[2] = i;
            }
        }
      else
        {
          if constexpr (dir == 0)
            {
              q[0] = i;
              q[1] = p;
            }
          else
            {
              q[0] = p;
              q[1] = i;
            }
          q[2] = 0;
        }
    }
  };

  // Workgroups are handed round-robin to the 8 XCDs of the chip, each with
  // its own L2. This bijection of [0, nb) gives every XCD one contiguous
  // range of blocks, so the neighbour cells of a Morton-ordered mesh (and
  // their face traces and tables) are read through the same L2.
  __device__ __forceinline__ unsigned
  xcd_block(unsigned b, unsigned nb)
  {
    constexpr unsigned nx   = 8;
    const unsigned     full = nb / nx, rem = nb % nx;
    const unsigned     x = b % nx, i = b / nx;
    return x < rem ? x * (full + 1) + i : rem * (full + 1) + (x - rem) * full + i;
  }

  // how a kernel obtains the geometry and transport speed at its points
  enum Geometry : int
  {
    geo_table    = 0, // precomputed w adj(J) a, 1/JxW and face tables
    geo_analytic = 1, // axis-aligned cells, speed evaluated per point
    geo_uniform  = 2  // axis-aligned cells, constant speed: products of
                      // 1D weights and per-mesh constants
  };

  // cells per workgroup: two wavefronts' worth of lines, so that every
  // barrier holds back two waves only and more workgroups share a CU
  // (3D degree 4: 5 cells, 125 of 128 lanes busy)
  constexpr int
  block_cells(int lines_per_cell)
  {
    return lines_per_cell >= 128 ? 1 : 128 / lines_per_cell;
  }

  template <int dim, int n>
  constexpr int
  cells_per_block()
  {
    return block_cells(Lay<dim, n>::nl);
  }

  // Tile shapes of the operator kernels, chosen per kernel variant by the
  // autotuner: shape 0 = the default above (two wavefronts), 1 = at most
  // one wavefront of lines, 2 = at most four wavefronts.
  constexpr int n_tile_shapes = 3;

  constexpr int
  shape_cells(int lines_per_cell, int shape)
  {
    return shape == 1 ? (lines_per_cell >= 64 ? 1 : 64 / lines_per_cell) :
           shape == 2 ? (lines_per_cell >= 256 ? 1 : 256 / lines_per_cell) :
                        block_cells(lines_per_cell);
  }

  // ---- small register contractions ---------------------------------------

  // Even-odd products with a centrosymmetric (skew = false) or
  // skew-centrosymmetric (skew = true) matrix M (EvenOdd in dev_basis.hpp):
  // out = M in, or M^T in (transpose), added to out (add). With
  // e_i = in_i + in_{n-1-i}, o_i = in_i - in_{n-1-i}, rows q and n-1-q share
  //   se = sum_i E[q][i] e_i + M[q][m] in_m,   so = sum_i O[q][i] o_i
  // as out_q = se + so and out_{n-1-q} = se - so (so - se when skew); the
  // middle row is sum_i M[m][i] e_i + M[m][m] in_m (sum_i M[m][i] o_i when
  // skew). M^T has the same form with E, O transposed (and exchanged when
  // skew) and the middle row and column exchanged.
  template <int n, bool skew, bool transpose, bool add, typename T>
  __device__ __forceinline__ void
  eo_apply(const EvenOdd<T> &M, const T (&in)[n], T (&out)[n])
  {
    constexpr int  h   = n / 2;
    constexpr int  m   = h;
    constexpr bool odd = n % 2 == 1;
    T              e[h > 0 ? h : 1], o[h > 0 ? h : 1];
#pragma unroll
    for (int i = 0; i < h; ++i)
      {
        e[i] = in[i] + in[n - 1 - i];
        o[i] = in[i] - in[n - 1 - i];
      }
    auto E = [&](int q, int i) -> T {
      if constexpr (!transpose)
        return M.e[q][i];
      else if constexpr (!skew)
        return M.e[i][q];
      else
        return M.o[i][q];
    };
    auto O = [&](int q, int i) -> T {
      if constexpr (!transpose)
        return M.o[q][i];
      else if constexpr (!skew)
        return M.o[i][q];
      else
        return M.e[i][q];
    };
    auto col = [&](int q) -> T { return transpose ? M.mr[q] : M.mc[q]; };
    auto row = [&](int i) -> T { return transpose ? M.mc[i] : M.mr[i]; };
#pragma unroll
    for (int q = 0; q < h; ++q)
      {
        T se = odd ? col(q) * in[m] : E(q, 0) * e[0];
#pragma unroll
        for (int i = odd ? 0 : 1; i < h; ++i)
          se = fma(E(q, i), e[i], se);
        T so = O(q, 0) * o[0];
#pragma unroll
        for (int i = 1; i < h; ++i)
          so = fma(O(q, i), o[i], so);
        const T lo = se + so, hi = skew ? so - se : se - so;
        out[q]         = add ? out[q] + lo : lo;
        out[n - 1 - q] = add ? out[n - 1 - q] + hi : hi;
      }
    if constexpr (odd)
      {
        T s;
        if constexpr (skew)
          {
            s = h > 0 ? row(0) * o[0] : (T)0;
#pragma unroll
            for (int i = 1; i < h; ++i)
              s = fma(row(i), o[i], s);
          }
        else
          {
            s = M.mm * in[m];
#pragma unroll
            for (int i = 0; i < h; ++i)
              s = fma(row(i), e[i], s);
          }
        out[m] = add ? out[m] + s : s;
      }
  }

  template <int dim, int n, int dir, typename T>
  __device__ __forceinline__ void
  lds_write_line(T *buf, int p, const T (&v)[n])
  {
#pragma unroll
    for (int i = 0; i < n; ++i)
      buf[Lay<dim, n>::template loff<dir>(p, i)] = v[i];
  }

  template <int dim, int n, int dir, typename T>
  __device__ __forceinline__ void
  lds_read_line(const T *buf, int p, T (&v)[n])
  {
#pragma unroll
    for (int i = 0; i < n; ++i)
      v[i] = buf[Lay<dim, n>::template loff<dir>(p, i)];
  }

  // Geometry table of a cell: dim rows of nd speeds and the row of 1/JxW of
  // the inverse mass. The determinant of a trilinear map is quadratic along
  // a line, so FP64 rows of more than three points hold its coefficients in
  // the line coordinate times the weight product of the line's other
  // coordinates instead: 3 values of n, for two multiplications, an estimate
  // and two Newton steps per point in kernels that are bound by the table's
  // bytes (MI355X, perturbed cells, before and after: degree 4, 64^3 cells 362
  // -> 347 us, 32^3 cells degree 5 74 -> 68, 6 122 -> 114, 7 172 -> 158 us;
  // degree 3, 64^3 cells 175 -> 172). Tables that stay in the caches do not
  // gain by it: up to 8^3 cells degrees 3 to 6 are even, and degree 7 takes 2
  // to 4% more (a second set of kernels would give 0.3 of 8 us back). FP32
  // keeps the values themselves (the sum of three rounded coefficients would
  // add to their error), and so does 2D (rows of 2n values, small meshes).
  template <int dim, int n, typename T>
  struct TableLay
  {
    static constexpr bool coef   = dim == 3 && n > 3 && sizeof(T) == 8;
    static constexpr int  nij    = coef ? 3 : n;
    static constexpr int  stride =
      dim * Lay<dim, n>::nd + nij * Lay<dim, n>::nl;
  };

  // NV values of row `row` of a cell's geometry table along line p of the
  // direction the row is stored in (the direction it is read along: row d
  // along d, row dim along x), value i at i * nl + p, so that the lanes of
  // a cell read contiguous memory
  template <int dim, int n, typename T, int NV>
  __device__ __forceinline__ void
  table_line(const T *tab, int64_t cell, int row, int p, T (&v)[NV])
  {
    constexpr int nd   = Lay<dim, n>::nd;
    constexpr int nl   = Lay<dim, n>::nl;
    const T      *base = tab + cell * TableLay<dim, n, T>::stride + row * nd;
#pragma unroll
    for (int i = 0; i < NV; ++i)
      v[i] = base[i * nl + p];
  }

  // ---- geometry ------------------------------------------------------------

  // Per quadrature point data of the cell term: cv[d] = w * (adj(J) a)_d
  // (the reference-space transport speed times JxW, which is what
  // advection_solver_implicit_real.cc:1126-1128 and :998-1007 fold
  // together) and JxW = w det(J), on a multilinear cell (the geometry
  // table builder).
  template <int dim>
  __device__ __forceinline__ void
  cell_point_data(const OpParams &P,
                  const double   *X,
                  const double   *xq,
                  const double   *wq,
                  const int (&q)[3],
                  double (&cv)[3],
                  double &JxW)
  {
    double w = wq[q[0]] * wq[q[1]];
    if (dim == 3)
      w *= wq[q[2]];
    double       x[3], a[3] = {0, 0, 0};
    const double xi[3] = {xq[q[0]], xq[q[1]], dim == 3 ? xq[q[2]] : 0.};
    double       J[3][3], adj[3][3];
    multilinear_map<dim>(X, xi, x, J);
    velocity_field<dim>(P.vel_kind, P.vel_const, x, a);
    const double det = adjugate<dim>(J, adj);
    for (int d = 0; d < dim; ++d)
      {
        double s = 0;
        for (int e = 0; e < dim; ++e)
          s += adj[d][e] * a[e];
        cv[d] = w * s;
      }
    JxW = w * det;
  }

  // Face point data: an = a . n dA (outward normal of this cell, including
  // the face quadrature weight) and the physical point x, on a multilinear
  // cell (the face and boundary table builders).
  template <int dim>
  __device__ __forceinline__ void
  face_point_data(const OpParams &P,
                  const double   *X,
                  const double   *xq,
                  const double   *wq,
                  int             dir,
                  int             side,
                  const int (&q)[3],
                  double &an,
                  double (&x)[3])
  {
    double w = 1.;
    for (int e = 0; e < dim; ++e)
      if (e != dir)
        w *= wq[q[e]];
    double xi[3];
    for (int e = 0; e < 3; ++e)
      xi[e] = (e < dim) ? xq[q[e]] : 0.;
    xi[dir] = side ? 1. : 0.;
    double a[3] = {0, 0, 0};
    double J[3][3], adj[3][3];
    multilinear_map<dim>(X, xi, x, J);
    velocity_field<dim>(P.vel_kind, P.vel_const, x, a);
    adjugate<dim>(J, adj);
    double s = 0;
    for (int e = 0; e < dim; ++e)
      s += adj[dir][e] * a[e];
    an = (side ? 1. : -1.) * w * s;
  }


  // The value is needed here, by all lanes: without this the compiler moves
  // a load whose value a select takes or leaves into a branch under the
  // lanes that take it.
  template <typename T>
  __device__ __forceinline__ void
  needed(T &v)
  {
    asm volatile("" : "+v"(v));
  }

  // ---- one direction of the operator -----------------------------------------

  // A line of n values in even-odd form: e_i = v_i + v_{n-1-i}, o_i = v_i -
  // v_{n-1-i} for i < n/2 and the middle value m of odd n.
  template <int n, typename T>
  struct EoLine
  {
    static constexpr int h = n / 2;
    T                    e[h > 0 ? h : 1], o[h > 0 ? h : 1], m;

    __device__ __forceinline__
    EoLine(const T (&v)[n])
    {
#pragma unroll
      for (int i = 0; i < h; ++i)
        {
          e[i] = v[i] + v[n - 1 - i];
          o[i] = v[i] - v[n - 1 - i];
        }
      m = v[h];
    }
  };

  // Symmetric part e, antisymmetric part o and middle value m of a line:
  // v_q = e_q + o_q, v_{n-1-q} = e_q - o_q, v_{n/2} = m.
  template <int n, typename T>
  struct EoSum
  {
    static constexpr int h = n / 2;
    T                    e[h > 0 ? h : 1], o[h > 0 ? h : 1], m;
  };

  // D (transpose: D^T) times the line v; D is skew-centrosymmetric, so the
  // products with v.e are antisymmetric and those with v.o symmetric (see
  // eo_apply, which this equals)
  template <int n, bool transpose, typename Table, typename T>
  __device__ __forceinline__ void
  eo_derivative(const Table &M, const EoLine<n, T> &v, EoSum<n, T> &r)
  {
    constexpr int  h   = n / 2;
    constexpr bool odd = n % 2 == 1;
#pragma unroll
    for (int q = 0; q < h; ++q)
      {
        T se = odd ? (transpose ? M.mr[q] : M.mc[q]) * v.m :
                     (transpose ? M.o[0][q] : M.e[q][0]) * v.e[0];
#pragma unroll
        for (int i = odd ? 0 : 1; i < h; ++i)
          se = fma(transpose ? M.o[i][q] : M.e[q][i], v.e[i], se);
        T so = (transpose ? M.e[0][q] : M.o[q][0]) * v.o[0];
#pragma unroll
        for (int i = 1; i < h; ++i)
          so = fma(transpose ? M.e[i][q] : M.o[q][i], v.o[i], so);
        r.e[q] = so;
        r.o[q] = se;
      }
    r.m = 0;
    if constexpr (odd)
      {
        r.m = (transpose ? M.mc[0] : M.mr[0]) * v.o[0];
#pragma unroll
        for (int i = 1; i < h; ++i)
          r.m = fma(transpose ? M.mc[i] : M.mr[i], v.o[i], r.m);
      }
  }

  // values of the line v at its two ends
  template <int n, typename Basis, typename T>
  __device__ __forceinline__ void
  line_ends(const Basis &B, const EoLine<n, T> &v, T (&um)[2])
  {
    constexpr int  h   = n / 2;
    constexpr bool odd = n % 2 == 1;
    T ve = odd ? B.lm * v.m : B.le[0] * v.e[0], vo = B.lo[0] * v.o[0];
#pragma unroll
    for (int i = odd ? 0 : 1; i < h; ++i)
      ve = fma(B.le[i], v.e[i], ve);
#pragma unroll
    for (int i = 1; i < h; ++i)
      vo = fma(B.lo[i], v.o[i], vo);
    um[0] = ve + vo;
    um[1] = ve - vo;
  }

  // reference derivatives of the line v at its two ends
  template <int n, typename T>
  __device__ __forceinline__ void
  line_end_derivatives(const DevBasis<T> &B, const EoLine<n, T> &v,
                       T (&dm)[2])
  {
    constexpr int  h   = n / 2;
    constexpr bool odd = n % 2 == 1;
    T de = odd ? B.dm * v.m : B.de[0] * v.e[0], d_o = B.dd[0] * v.o[0];
#pragma unroll
    for (int i = odd ? 0 : 1; i < h; ++i)
      de = fma(B.de[i], v.e[i], de);
#pragma unroll
    for (int i = 1; i < h; ++i)
      d_o = fma(B.dd[i], v.o[i], d_o);
    dm[0] = de + d_o;
    dm[1] = d_o - de;
  }

  // acc (+)= D^T g + sum_s l_s f[s] (+ sum_s l_s' fd[s] with `diff`)
  template <int n, bool diff, bool add, typename Basis, typename T>
  __device__ __forceinline__ void
  line_integrate(const Basis &B, const T (&g)[n], T f0, T f1, T fd0,
                 T fd1, T (&acc)[n])
  {
    constexpr int      h   = n / 2;
    constexpr bool     odd = n % 2 == 1;
    const EoLine<n, T> ge(g);
    EoSum<n, T>        r;
    eo_derivative<n, true>(B.eo_D, ge, r);
    const T fs = f0 + f1, fm = f0 - f1;
    const T ds = fd0 + fd1, dd = fd0 - fd1;
#pragma unroll
    for (int q = 0; q < h; ++q)
      {
        T se = fma(B.le[q], fs, r.e[q]), so = fma(B.lo[q], fm, r.o[q]);
        if constexpr (diff)
          {
            se = fma(B.de[q], dd, se);
            so = fma(B.dd[q], ds, so);
          }
        acc[q]         = add ? acc[q] + (se + so) : se + so;
        acc[n - 1 - q] = add ? acc[n - 1 - q] + (se - so) : se - so;
      }
    if constexpr (odd)
      {
        T sm = fma(B.lm, fs, r.m);
        if constexpr (diff)
          sm = fma(B.dm, dd, sm);
        acc[h] = add ? acc[h] + sm : sm;
      }
  }

  // Per-launch factors of one component's terms, uniform over the grid:
  // flux = an (c_own u- + c_nb u+) + c_abs |an| (u- - u+) is sign times the
  // numerical flux 1/2 [(u- + u+) an + alpha |an| (u- - u+)] - skew an u-
  // (advection_solver_implicit_real.cc:1032-1058, an = a . n dA on the
  // cell's outward normal) at the speed factor vf.
  template <typename T>
  struct FluxFactors
  {
    T c_own, c_nb, c_abs;

    __device__ __forceinline__
    FluxFactors(const OpParams &P, double vf)
      : c_own((T)(P.sign * vf * (0.5 - P.skew)))
      , c_nb((T)(P.sign * vf * 0.5))
      , c_abs((T)(P.sign * fabs(vf) * 0.5 * P.alpha))
    {}
  };

  // Cell and face terms of direction `dir` on the line owned by this
  // thread: acc (+)= D^T g + s D u + sum_sides l_side (x) flux, with
  //   g: the cell flux at the line's points (the caller's, plus the
  //      diffusion flux cd w_i (D u)_i with `diff`),
  //   s (skew): the factor of the values' derivative,
  // and the faces at the line's two ends (fan: a . n dA, up / dp: the
  // neighbours' traces and reference derivatives normal to the face).
  // Everything works on even and odd parts: the two end values share their
  // products (l1 is l0 reversed, the end derivatives change sign), D u and
  // the end values share the split of u, and the lift of the end values
  // joins D^T g before the parts are put together. Per line of n points
  // the faces then cost 2 n products instead of 4 n (4 n instead of 10 n
  // with diffusion, whose cell flux shares the D^T product of the advective
  // one), and the reciprocals 1/h come from the launch: these kernels are
  // bound by VALU issue with diffusion. One MI355X, before and after,
  // together with the staging of the normal derivatives in the value phase
  // (FP64 degree 7: 3203 -> 1647 VALU instructions per wave, 236 -> 160
  // registers): SIPG on 32^3 cells, degree 5 FP64 131 -> 81 us, degree 7
  // FP32 144 -> 84 us; without diffusion, degree 4 on 64^3 perturbed cells
  // FP64 375 -> 366 us, degree 6 FP32 on 24^3 cells 32.2 -> 28.0 us.
  // SIPG (advection_diffusion_solver.cc:569-613) on axis-aligned cells: with
  // jump = -nu/2 (u- - u+), avg = -nu/2 (d_n u- + d_n u+) the value term is
  // -(jump sigma - avg) and the normal derivative of the test function is
  // weighted with jump; wd is the product of the weights of the line's other
  // coordinates. bmask: bit f is set where a lane of the wavefront has its
  // face f on the boundary.
  template <int dim, int n, int dir, typename T, bool skew, bool diff,
            bool boundary, bool add>
  __device__ __forceinline__ void
  line_operator(const OpParams       &P,
                const DevBasis<T>    &B,
                const FluxFactors<T> &F,
                int64_t               cell,
                int                   p,
                unsigned              bmask,
                const T (&uplus)[2 * dim],
                const T (&dplus)[2 * dim],
                const T (&fan)[2 * dim],
                const T (&uq)[n],
                T (&g)[n],
                const T (&sk)[n],
                T wd,
                T (&acc)[n])
  {
    constexpr int      h   = n / 2;
    constexpr bool     odd = n % 2 == 1;
    const EoLine<n, T> u(uq);
    T um[2];
    line_ends<n>(B, u, um);
    T       f[2], fd[2];
    T       ub[2] = {uplus[2 * dir], uplus[2 * dir + 1]};
    if (boundary && (bmask >> (2 * dir) & 3))
      {
        // Dirichlet data, evaluated before the launch
        // (boundary_value_kernel)
        int    nb[2];
        double bv[2];
#pragma unroll
        for (int s = 0; s < 2; ++s)
          {
            nb[s] = P.neighbors[cell * 2 * dim + 2 * dir + s];
            bv[s] = P.bnd_value[(int64_t)max(~nb[s], 0) * Lay<dim, n>::nl + p];
          }
#pragma unroll
        for (int s = 0; s < 2; ++s)
          {
            needed(bv[s]);
            ub[s] = nb[s] < 0 ? (T)bv[s] : ub[s];
          }
      }
#pragma unroll
    for (int s = 0; s < 2; ++s)
      {
        const int fc = 2 * dir + s;
        const T   up = ub[s];
        const T an = fan[fc], j = um[s] - up;
        f[s] = fma(an, fma(F.c_own, um[s], F.c_nb * up),
                   F.c_abs * fabs(an) * j);
        fd[s] = j;
      }
    EoSum<n, T> du;
    if constexpr (skew || diff)
      eo_derivative<n, false>(B.eo_D, u, du);
    if constexpr (diff)
      {
        T dm[2];
        line_end_derivatives<n>(B, u, dm);
        double  vol   = P.h[0] * P.h[1];
        if (dim == 3)
          vol *= P.h[2];
        const double ih = P.inv_h[dir];
        // W = sign nu/2 times the face weight
        const T W  = wd * (T)(0.5 * P.sign * P.viscosity * vol * ih);
        const T si = (T)(P.penalty * ih), tih = (T)ih;
        const T cd = (T)2 * tih * W;
#pragma unroll
        for (int s = 0; s < 2; ++s)
          {
            const T gs = s ? tih : -tih;
            const T j  = fd[s];
            f[s] = fma(W, fma(si, j, -gs * (dm[s] + dplus[2 * dir + s])),
                       f[s]);
            fd[s] = -gs * W * j;
          }
        // cell diffusion flux sign nu |K| / h^2 w D u
#pragma unroll
        for (int i = 0; i < h; ++i)
          {
            g[i] = fma(cd * B.w[i], du.e[i] + du.o[i], g[i]);
            g[n - 1 - i] =
              fma(cd * B.w[n - 1 - i], du.e[i] - du.o[i], g[n - 1 - i]);
          }
        if constexpr (odd)
          g[h] = fma(cd * B.w[h], du.m, g[h]);
      }
    line_integrate<n, diff, add>(B, g, f[0], f[1], fd[0], fd[1], acc);
    if constexpr (skew)
      {
#pragma unroll
        for (int q = 0; q < h; ++q)
          {
            acc[q] = fma(sk[q], du.e[q] + du.o[q], acc[q]);
            acc[n - 1 - q] =
              fma(sk[n - 1 - q], du.e[q] - du.o[q], acc[n - 1 - q]);
          }
        if constexpr (odd)
          acc[h] = fma(sk[h], du.m, acc[h]);
      }
  }

  // ---- the kernel ------------------------------------------------------------

  enum Finalize : int
  {
    fin_inverse_mass = 0, // S^-1 diag(1/JxW): explicit right-hand side
    fin_integrate    = 1, // S^T: operator action (implicit vmult)
    fin_local        = 2  // cell-local operator in the Gauss-point
                          // collocation basis: input and output at the
                          // Gauss points, neighbour traces zero
                          // (CellwiseOperator::vmult,
                          // advection_solver_irk_real.cc:545-711)
  };

  enum Epilogue : int
  {
    epi_store = 0, // dst = scale * y
    epi_lsrk  = 1  // k = y; sol_out = sol_in + b k; ri_out = sol_in + a k
  };

  template <typename T>
  struct OpBuffers
  {
    const T *src; // [NC][comp_stride]
    T       *dst; // [NC][comp_stride]
    int64_t  comp_stride;
    T        scale;
    // LSRK epilogue (NC == 1)
    const T *sol_in;
    T       *sol_out;
    T       *ri_out;
    T        b_dt, a_dt;
    int      last;
  };

  // y_c = fin( sign * L_c u_c + sum_b mass[c][b] M u_b ), c < NC, with
  // L_c the advection operator at velocity vel_factor[c] * a(x).
  // With `diff` (axis-aligned cells) L also contains the SIPG diffusion
  // operator of advection_diffusion_solver.cc:531-613.
  // The operator on the cells of workgroup `block` (one batch of CPB
  // cells); P and io live in kernel arguments or, for the
  // batched launch, in global memory (uniform per workgroup either way).
  template <int dim, int n, int NC, typename T, int geo, bool skew,
            bool diff, int fin, int epi, int CPB>
  __device__ __forceinline__ void
  operator_body(const OpParams                       &P,
                const DevBasis<T> *__restrict__      Bp,
                const DevBasis<double> *__restrict__ Bd,
                const OpBuffers<T>                   &io,
                unsigned                              block)
  {
    static_assert(!diff || geo != geo_table, "SIPG needs axis-aligned cells");
    static_assert(fin != fin_local || (!diff && epi == epi_store),
                  "the cell-local operator is built for advection");
    using L            = Lay<dim, n>;
    constexpr int nl   = L::nl;
    constexpr int nd   = L::nd;
    constexpr int STR  = L::stride;
    constexpr int FSTR = (diff ? 2 : 1) * 2 * dim * nl;
    constexpr int NV   = 1 << dim;
    constexpr int LAST = dim - 1;
    constexpr int NX   = geo == geo_table ? NV * dim : dim;

    // analytic (axis-aligned) geometry evaluates the transport speed at
    // LAST-line points and hands the other directions over through LDS;
    // tabulated and uniform geometry produce every direction in its own
    // line layout
    constexpr bool AN  = geo == geo_analytic;
    constexpr bool UNI = geo == geo_uniform;
    __shared__ T      s_u[CPB * STR];
    __shared__ T      s_acc[CPB * STR];
    __shared__ T      s_g0[AN ? CPB * STR : 1];
    __shared__ T      s_g1[(AN && dim == 3) ? CPB * STR : 1];
    __shared__ T      s_sk0[(AN && skew) ? CPB * STR : 1];
    __shared__ T      s_sk1[(AN && skew && dim == 3) ? CPB * STR : 1];
    __shared__ T      s_face[CPB * FSTR];
    __shared__ T      s_fan[AN ? CPB * 2 * (dim - 1) * nl : 1];
    __shared__ double s_X[CPB * NX];
    // several components (IRK stages): their values at the quadrature
    // points wait in LDS between the value phase and the operator phase
    // instead of holding NC lines in registers through the operator phase.
    // Every thread writes and reads its own LAST line only, so the points
    // lie thread by thread: no bank conflicts and no padding, and degree 5
    // with four stages keeps to four FP64 workgroups per CU
    // (32^3 cells 353 -> 292 us on one MI355X, 297 -> 238 with uniform
    // geometry)
    constexpr bool STAGE_LDS = NC > 1;
    __shared__ T   s_stage[STAGE_LDS ? NC * CPB * nd : 1];
    // several components, advection: the neighbour traces of component
    // c are interpolated at the start of its operator phase instead of in
    // the value phase, so that one component's traces are live at a time
    // (NC sets of traces held through the operator phase cost one
    // occupancy step)
    constexpr bool TRACE_LATE = STAGE_LDS && !diff && fin != fin_local;
    const T *tab_c = static_cast<const T *>(P.tab_cell);
    const T *tab_f = static_cast<const T *>(P.tab_face);

    const DevBasis<T> &B    = *Bp;
    const int          tid  = threadIdx.x;
    const int          lc   = tid / nl;
    const int          p    = tid - lc * nl;
    // threads past the last cell repeat it and store nothing: no load below
    // is in a branch of the source's under a part of the lanes (a neighbour
    // across a boundary face is read from the cell itself and replaced by a
    // select). Such branches cost moves and split the load batches, and at
    // 250 and more registers the compiler has placed live-range copies
    // before the mask is restored. It still makes branches of the selects of
    // one component's boundary data: with the loads forced out of them (see
    // needed()) the boundary meshes lost 4 to 9%, the implicit operator up
    // to 40% by spills.
    const int64_t      cell_t = (int64_t)block * CPB + lc;
    const bool         active = cell_t < P.n_cells;
    const int64_t      cell   = active ? cell_t : P.n_cells - 1;

    T      *u_l   = s_u + lc * STR;
    T      *acc_l = s_acc + lc * STR;
    T      *g0_l  = AN ? s_g0 + lc * STR : s_g0;
    T      *g1_l  = (AN && dim == 3) ? s_g1 + lc * STR : s_g1;
    T      *sk0_l = (AN && skew) ? s_sk0 + lc * STR : s_sk0;
    T      *sk1_l = (AN && skew && dim == 3) ? s_sk1 + lc * STR : s_sk1;
    T      *f_l   = s_face + lc * FSTR;
    T      *fan_l = AN ? s_fan + lc * 2 * (dim - 1) * nl : s_fan;
    double *X     = s_X + lc * NX;
    auto    stage_l = [&](int c) -> T * {
      return s_stage + (STAGE_LDS ? c * CPB * nd + tid : 0);
    };

    // the cell's own values of the first component are requested first:
    // the x sweep then overlaps the neighbour-index -> trace load chain
    // (values at the Gauss points of the collocation basis are read along
    // LAST-direction lines, where the operator starts)
    constexpr int in_dir = fin == fin_local ? LAST : 0;
    auto          load_own = [&](const T *src, T(&r)[n]) {
#pragma unroll
      for (int i = 0; i < n; ++i)
        r[i] = src[cell * nd + L::template off<in_dir>(p, i)];
    };
    // waves that are issuing global loads (the cell's values and traces,
    // the tables) or stores get issue priority, so that requests leave
    // early while other waves compute
    __builtin_amdgcn_s_setprio(3);
    T r0[n];
    load_own(io.src, r0);
    // cell vertices: analytic geometry, and JxW of the mass term with
    // tabulated geometry
    constexpr bool needX = AN || (geo == geo_table && fin != fin_inverse_mass);
    if constexpr (needX)
      {
        for (int e = p; e < NX; e += nl)
          X[e] = P.cell_vertices[cell * NV * dim + e];
      }
    int nb[2 * dim];
    if (dim == 3 && P.morton_bits >= 0)
      {
        // one periodic coarse cell: the neighbours are Morton increments
        // of the cell index (dilated integers, carries confined to one
        // coordinate's bits), so the trace loads below need no index load
        // first
        const unsigned full = (1u << (3 * P.morton_bits)) - 1u;
        const unsigned m    = (unsigned)cell;
#pragma unroll
        for (int d = 0; d < dim; ++d)
          {
            const unsigned M = (0x09249249u << d) & full;
            nb[2 * d]     = (int)((((m & M) - 1u) & M) | (m & ~M));
            nb[2 * d + 1] = (int)((((m | ~M) + 1u) & M) | (m & ~M));
          }
      }
    else
      {
#pragma unroll
        for (int f = 0; f < 2 * dim; ++f)
          nb[f] = P.neighbors[cell * 2 * dim + f];
        // wait for them here (vmcnt 0, the others untouched): a wait after
        // the branches join would hold back the trace loads of the Morton
        // case behind the cell's own values
        __builtin_amdgcn_s_waitcnt(0x0F70);
      }
    // several components: bit f is set where a lane of the wavefront has its
    // face f on the boundary. In a scalar register: the wavefronts inside
    // the mesh skip the boundary faces' data by a scalar branch. Three
    // components with inflow data on two sides on one MI355X, when every
    // wavefront loaded them and now: degree 4, 32^3 cells FP64 145 -> 117 us,
    // FP32 81 -> 66; degree 1, 64^3 cells FP64 113 -> 79. (One component
    // holds its neighbours and loads once: there the six comparisons cost as
    // much as they save.)
    unsigned bmask = 0;
    if (TRACE_LATE && P.has_boundary)
      {
#pragma unroll
        for (int f = 0; f < 2 * dim; ++f)
          bmask |= __builtin_amdgcn_ballot_w64(nb[f] < 0) != 0 ? 1u << f : 0u;
      }
    // the cell a face's neighbour data are read from
    auto nb_cell = [&](int f) -> int64_t {
      return nb[f] >= 0 ? (int64_t)nb[f] : cell;
    };
    if constexpr (needX)
      __syncthreads();

    // tabulated geometry: LAST-direction speed on this thread's line, the
    // y and x speed rows, and a . n dA on the faces its lines end on (lower
    // face of this cell, upper face = lower face of the upper neighbour,
    // boundary faces apart). Requested after the value phase: holding them
    // across its barriers costs an occupancy step, which loses more than
    // the overlap gains, with one component and with several.
    T cv[3][n], jxw[n], cvy[n], cvx[n];
    T fan[2 * dim];
    auto load_tables = [&]() {
        table_line<dim, n>(tab_c, cell, LAST, p, cv[LAST]);
#pragma unroll
        for (int d = 0; d < dim; ++d)
          {
            fan[2 * d]     = -tab_f[(cell * dim + d) * nl + p];
            fan[2 * d + 1] = tab_f[(nb_cell(2 * d + 1) * dim + d) * nl + p];
          }
        if (NC > 1 ? bmask != 0 : P.has_boundary)
          {
#pragma unroll
            for (int f = 0; f < 2 * dim; ++f)
              {
                const int b = NC > 1 ? P.neighbors[cell * 2 * dim + f] : nb[f];
                const T   an =
                  (T)P.tab_bnd[((int64_t)max(~b, 0) * nl + p) * (1 + dim)];
                fan[f] = b < 0 ? an : fan[f];
              }
          }
    };
    auto load_speed_rows = [&]() {
      if constexpr (dim == 3)
        table_line<dim, n>(tab_c, cell, 1, p, cvy);
      table_line<dim, n>(tab_c, cell, 0, p, cvx);
    };

    // ---- per component: neighbour traces and values at quadrature points
    constexpr int NUP = TRACE_LATE ? 1 : NC;
    T             uplus[NUP][2 * dim];
    T             dplus[NUP][2 * dim];
    // values at the quadrature points on this thread's LAST line: in
    // registers for one component, in s_stage for several
    T    uqs[STAGE_LDS ? 1 : NC][n];
    auto keep_uq = [&](int c, const T(&v)[n]) {
      if constexpr (STAGE_LDS)
#pragma unroll
        for (int i = 0; i < n; ++i)
          stage_l(c)[i * CPB * nl] = v[i];
      else
#pragma unroll
        for (int i = 0; i < n; ++i)
          uqs[0][i] = v[i];
    };
    auto get_uq = [&](int c, T(&v)[n]) {
      if constexpr (STAGE_LDS)
#pragma unroll
        for (int i = 0; i < n; ++i)
          v[i] = stage_l(c)[i * CPB * nl];
      else
#pragma unroll
        for (int i = 0; i < n; ++i)
          v[i] = uqs[0][i];
    };
#pragma unroll
    for (int c = 0; c < NC; ++c)
      {
        const T *src = io.src + c * io.comp_stride;
        T        r[n], t[n];
        if (c == 0)
#pragma unroll
          for (int i = 0; i < n; ++i)
            r[i] = r0[i];
        else
          load_own(src, r);
        if constexpr (fin == fin_local)
          {
            // already at the Gauss points; the neighbours do not couple
            keep_uq(c, r);
#pragma unroll
            for (int f = 0; f < 2 * dim; ++f)
              uplus[c][f] = dplus[c][f] = 0;
            continue;
          }
        // neighbours' face nodes for LDS staging (thread (i, j) loads node
        // (t1 = i, t2 = j) of every face, one load per face; with diffusion
        // also the nodal derivative normal to the face, from the n values
        // of the neighbour's line through that node: n loads and n products
        // per face and thread, where forming it inside the tangential
        // interpolation takes n^2 of both); stored after the x sweep so
        // that the sweep does not wait for them
        constexpr int NTR = diff ? 2 : 1; // trace kinds per face
        T             tv[NTR][2 * dim];
        if constexpr (!TRACE_LATE)
          {
            const int i0 = p % n, j0 = dim == 3 ? p / n : 0;
#pragma unroll
            for (int f = 0; f < 2 * dim; ++f)
              {
                constexpr int n2 = n * n;
                const int     d = f / 2, s = f % 2;
                const int     st = d == 0 ? 1 : d == 1 ? n : n2;
                const int     s1 = d == 0 ? n : 1;
                const int     s2 = d == 2 ? n : n2;
                const int     lay = s ? 0 : n - 1;
                const T      *nsrc = src + nb_cell(f) * nd + i0 * s1 +
                                (dim == 3 ? j0 * s2 : 0);
                if constexpr (diff)
                  {
                    const T(&dp)[max_n] = s ? B.dphi0 : B.dphi1;
                    T nv[n], dv = 0;
#pragma unroll
                    for (int l = 0; l < n; ++l)
                      nv[l] = nsrc[l * st];
#pragma unroll
                    for (int l = 0; l < n; ++l)
                      dv = fma(dp[l], nv[l], dv);
                    tv[0][f] = nv[lay];
                    tv[1][f] = dv;
                  }
                else
                  tv[0][f] = nsrc[lay * st];
              }
          }
        // own values, sweep along x
        __builtin_amdgcn_s_setprio(0);
        eo_apply<n, false, false, false>(B.eo_S, r, t);
        lds_write_line<dim, n, 0>(acc_l, p, t);
        if constexpr (!TRACE_LATE)
          {
#pragma unroll
            for (int k = 0; k < NTR; ++k)
#pragma unroll
              for (int f = 0; f < 2 * dim; ++f)
                f_l[(k * 2 * dim + f) * nl + p] = tv[k][f];
          }
        __syncthreads();
        if constexpr (!TRACE_LATE)
          {
            // first tangential interpolation of the staged nodes: thread
            // (aq, j); in 3D written back after the next barrier
            const int aq = p % n, j = dim == 3 ? p / n : 0;
#pragma unroll
            for (int k = 0; k < NTR; ++k)
#pragma unroll
              for (int f = 0; f < 2 * dim; ++f)
                {
                  T v = 0;
#pragma unroll
                  for (int i = 0; i < n; ++i)
                    v = fma(B.S[aq][i],
                            f_l[(k * 2 * dim + f) * nl + j * n + i], v);
                  if constexpr (dim == 3)
                    tv[k][f] = v;
                  else
                    (k ? dplus : uplus)[c][f] = v;
                }
          }
        lds_read_line<dim, n, 1>(acc_l, p, t);
        eo_apply<n, false, false, false>(B.eo_S, t, r);
        if constexpr (dim == 3)
          {
            __syncthreads();
            if constexpr (!TRACE_LATE)
              {
#pragma unroll
                for (int k = 0; k < NTR; ++k)
#pragma unroll
                  for (int f = 0; f < 6; ++f)
                    f_l[(k * 6 + f) * nl + p] = tv[k][f];
              }
            lds_write_line<dim, n, 1>(acc_l, p, r);
            __syncthreads();
            if constexpr (!TRACE_LATE)
              {
                // second tangential interpolation: thread (aq, bq)
                const int aq = p % n, bq = p / n;
#pragma unroll
                for (int k = 0; k < NTR; ++k)
#pragma unroll
                  for (int f = 0; f < 6; ++f)
                    {
                      T v = 0;
#pragma unroll
                      for (int jj = 0; jj < n; ++jj)
                        v = fma(B.S[bq][jj],
                                f_l[(k * 6 + f) * nl + jj * n + aq], v);
                      (k ? dplus : uplus)[c][f] = v;
                    }
              }
            lds_read_line<dim, n, 2>(acc_l, p, t);
            eo_apply<n, false, false, false>(B.eo_S, t, r);
          }
        keep_uq(c, r);
        __syncthreads();
      }

    // ---- geometry and velocity: this thread's LAST-line points and the
    // faces its line ends on; faces normal to the other directions are
    // evaluated along LAST-direction lines by up to one task per thread and
    // handed over through LDS
    // uniform geometry: w adj(J) a at point (i, line p of direction d) is
    // w_i wl_d(p) |K| / h_d a_d, with wl_d(p) the product of the 1D
    // weights at the line's other coordinates; a . n dA on the faces of
    // that line is -+ wl_d(p) |K| / h_d a_d
    double vol = 0, cdir[3] = {0, 0, 0}, wl[3] = {1, 1, 1};
    if constexpr (UNI || diff)
      {
        vol = P.h[0] * P.h[1] * (dim == 3 ? P.h[2] : 1.);
#pragma unroll
        for (int d = 0; d < dim; ++d)
          cdir[d] = vol * P.inv_h[d] * P.vel_const[d];
        int q[3];
#pragma unroll
        for (int d = 0; d < dim; ++d)
          {
            if (d == 0)
              L::template idx<0>(p, 0, q);
            else if (d == 1)
              L::template idx<(dim > 1 ? 1 : 0)>(p, 0, q);
            else
              L::template idx<LAST>(p, 0, q);
#pragma unroll
            for (int e = 0; e < dim; ++e)
              if (e != d)
                wl[d] *= Bd->w[q[e]];
          }
      }
    if constexpr (UNI)
      {
        const double cl = wl[LAST] * cdir[LAST];
#pragma unroll
        for (int i = 0; i < n; ++i)
          {
            cv[LAST][i] = (T)(Bd->w[i] * cl);
            jxw[i] = fin != fin_inverse_mass ? (T)(Bd->w[i] * wl[LAST] * vol)
                                          : (T)1;
          }
#pragma unroll
        for (int d = 0; d < dim; ++d)
          {
            fan[2 * d]     = (T)(-wl[d] * cdir[d]);
            fan[2 * d + 1] = (T)(wl[d] * cdir[d]);
          }
      }
    else if constexpr (!AN)
      {
        __builtin_amdgcn_s_setprio(3);
        load_tables();
        __builtin_amdgcn_s_setprio(0);
        // JxW of the mass term on this thread's line
        if (fin != fin_inverse_mass && P.has_mass)
          line_jxw<dim, n, LAST, T, L>(X, Bd->xq, Bd->w, p, jxw);
        else
#pragma unroll
          for (int i = 0; i < n; ++i)
            jxw[i] = 1;
      }
    else
    {
      int q[3];
      L::template idx<LAST>(p, 0, q);
      T fl[2] = {0, 0};
      line_cell_data<dim, n, LAST, true, T>(P, X, Bd, q, cv, jxw, fl);
      fan[2 * LAST]     = fl[0];
      fan[2 * LAST + 1] = fl[1];
      constexpr int ntask = dim == 3 ? 4 * n : 2;
      // threads without a task of their own repeat the last one (the same
      // values to the same place) instead of leaving the wavefront
#pragma unroll 1
      for (int k = 0; k < (ntask + nl - 1) / nl; ++k)
        {
          const int task = min(p + k * nl, ntask - 1);
          const int d    = dim == 3 ? task / (2 * n) : 0;
          const int s    = dim == 3 ? (task / n) % 2 : task;
          const int j    = dim == 3 ? task % n : 0;
          face_line_data<dim, n, LAST, true, T>(
            P, X, Bd, d, s, j, fan_l + (2 * d + s) * nl + j * n);
        }
      __syncthreads();
      const int fidx = dim == 3 ? (p % n) * n + p / n : p;
#pragma unroll
      for (int f = 0; f < 2 * LAST; ++f)
        fan[f] = fan_l[f * nl + fidx];
    }

    // speed rows of the y and x phases, read once for all components
    if constexpr (geo == geo_table)
      load_speed_rows();
    // tabulated inverse mass: the 1/JxW row is requested after the LAST
    // phase (one component; several components read it per component
    // after their x phase)
    constexpr bool early_ij = geo == geo_table && fin == fin_inverse_mass;
    using TL = TableLay<dim, n, T>;
    T ij_row[early_ij ? TL::nij : 1];
    if constexpr (UNI)
      {
#pragma unroll
        for (int i = 0; i < n; ++i)
          {
            cvy[i] = (T)(Bd->w[i] * wl[dim == 3 ? 1 : 0] * cdir[1]);
            cvx[i] = (T)(Bd->w[i] * wl[0] * cdir[0]);
          }
      }
#pragma unroll
    for (int c = 0; c < NC; ++c)
      {
        if constexpr (TRACE_LATE)
          {
            // neighbour traces of component c: thread (i0, j0) stages node
            // (t1 = i0, t2 = j0) of each face, then interpolates along t1
            // (thread (aq = i0, j0)) and along t2 (thread (aq = i0, bq = j0))
            const T  *src = io.src + c * io.comp_stride;
            const int i0 = p % n, j0 = dim == 3 ? p / n : 0;
            T         tv[2 * dim];
            __builtin_amdgcn_s_setprio(3);
#pragma unroll
            for (int f = 0; f < 2 * dim; ++f)
              {
                constexpr int n2 = n * n;
                const int     d = f / 2, s = f % 2;
                const int     st = d == 0 ? 1 : d == 1 ? n : n2;
                const int     s1 = d == 0 ? n : 1;
                const int     s2 = d == 2 ? n : n2;
                tv[f] = src[nb_cell(f) * nd + i0 * s1 +
                            (dim == 3 ? j0 * s2 : 0) + (s ? 0 : n - 1) * st];
              }
            __builtin_amdgcn_s_setprio(0);
#pragma unroll
            for (int f = 0; f < 2 * dim; ++f)
              f_l[f * nl + p] = tv[f];
            __syncthreads();
#pragma unroll
            for (int f = 0; f < 2 * dim; ++f)
              {
                T v = 0;
#pragma unroll
                for (int i = 0; i < n; ++i)
                  v = fma(B.S[i0][i], f_l[f * nl + j0 * n + i], v);
                (dim == 3 ? tv : uplus[0])[f] = v;
              }
            if constexpr (dim == 3)
              {
                __syncthreads();
#pragma unroll
                for (int f = 0; f < 6; ++f)
                  f_l[f * nl + p] = tv[f];
                __syncthreads();
#pragma unroll
                for (int f = 0; f < 6; ++f)
                  {
                    T v = 0;
#pragma unroll
                    for (int jj = 0; jj < n; ++jj)
                      v = fma(B.S[j0][jj], f_l[f * nl + jj * n + i0], v);
                    uplus[0][f] = v;
                  }
              }
          }
        // Dirichlet data of the boundary faces: one component reads those
        // of all faces here, in one round of loads; direction by direction
        // a small mesh waited for three (and as many for the face numbers,
        // before they came with the neighbours; degree 2, 24x16x8 cells:
        // 6.07 -> 4.96 us). Several components keep to that and read the
        // neighbours again: the registers cost them more (degree 4, 32^3
        // cells, three components: operator and FDM 206 -> 212 us; degree 2
        // 50 -> 54 us).
        constexpr bool BND  = !diff && fin != fin_local;
        constexpr bool LATE = BND && NC > 1;
        if constexpr (BND && !LATE)
          if (P.has_boundary)
            {
              T bv[2 * dim];
#pragma unroll
              for (int f = 0; f < 2 * dim; ++f)
                bv[f] = (T)P.bnd_value[(int64_t)max(~nb[f], 0) * nl + p];
#pragma unroll
              for (int f = 0; f < 2 * dim; ++f)
                {
                  T &u = uplus[0][f];
                  u    = nb[f] < 0 ? bv[f] : u;
                }
            }
        const T vf    = (T)P.vel_factor[c];
        const T fcell = (T)(-(1. - P.skew) * P.sign) * vf;
        const T fs    = (T)(P.skew * P.sign) * vf;
        const FluxFactors<T> F(P, P.vel_factor[c]);
        constexpr bool       MASS = fin != fin_inverse_mass;
        const T (&up)[2 * dim] = uplus[NUP > 1 ? c : 0];
        const T (&dp)[2 * dim] = dplus[NUP > 1 ? c : 0];
        T acc[n];
        // ---- LAST direction (z in 3D, y in 2D) ----
        {
          if constexpr (MASS)
#pragma unroll
            for (int i = 0; i < n; ++i)
              acc[i] = 0;
          if (MASS && P.has_mass)
            {
#pragma unroll
              for (int b = 0; b < NC; ++b)
                {
                  const T m = (T)P.mass[c][b];
                  T       ub[n];
                  get_uq(b, ub);
#pragma unroll
                  for (int i = 0; i < n; ++i)
                    acc[i] = fma(m * jxw[i], ub[i], acc[i]);
                }
            }
          T uc[n];
          get_uq(c, uc);
          T g[n], sk[n];
#pragma unroll
          for (int i = 0; i < n; ++i)
            {
              g[i] = fcell * cv[LAST][i] * uc[i];
              if constexpr (skew)
                sk[i] = fs * cv[LAST][i];
            }
          line_operator<dim, n, LAST, T, skew, diff, LATE, MASS>(
            P, B, F, cell, p, bmask, up, dp, fan, uc, g, sk,
            (T)wl[LAST], acc);
          if constexpr (early_ij)
            {
              // the row of the inverse mass, requested here (the LAST speed
              // row is dead) so that it arrives during the y and x phases
              // instead of after them, without registers at the kernel's
              // peak
              __builtin_amdgcn_s_setprio(3);
              table_line<dim, n>(tab_c, cell, dim, p, ij_row);
              __builtin_amdgcn_s_setprio(0);
            }
          lds_write_line<dim, n, LAST>(u_l, p, uc);
          lds_write_line<dim, n, LAST>(acc_l, p, acc);
          if constexpr (AN)
            {
#pragma unroll
              for (int i = 0; i < n; ++i)
                g[i] = fcell * cv[0][i] * uc[i];
              lds_write_line<dim, n, LAST>(g0_l, p, g);
              if constexpr (dim == 3)
                {
#pragma unroll
                  for (int i = 0; i < n; ++i)
                    g[i] = fcell * cv[1][i] * uc[i];
                  lds_write_line<dim, n, LAST>(g1_l, p, g);
                }
              if constexpr (skew)
                {
#pragma unroll
                  for (int i = 0; i < n; ++i)
                    g[i] = fs * cv[0][i];
                  lds_write_line<dim, n, LAST>(sk0_l, p, g);
                  if constexpr (dim == 3)
                    {
#pragma unroll
                      for (int i = 0; i < n; ++i)
                        g[i] = fs * cv[1][i];
                      lds_write_line<dim, n, LAST>(sk1_l, p, g);
                    }
                }
            }
          __syncthreads();
        }

        // ---- y direction in 3D ----
        if constexpr (dim == 3)
          {
            T        uq[n], g[n], sk[n];
            const T(&cvd)[n] = cvy;
            lds_read_line<dim, n, 1>(u_l, p, uq);
            if constexpr (AN)
              lds_read_line<dim, n, 1>(g1_l, p, g);
            else
              {
#pragma unroll
                for (int i = 0; i < n; ++i)
                  g[i] = fcell * cvd[i] * uq[i];
              }
            lds_read_line<dim, n, 1>(acc_l, p, acc);
            if constexpr (skew && AN)
              lds_read_line<dim, n, 1>(sk1_l, p, sk);
            else if constexpr (skew)
              {
#pragma unroll
                for (int i = 0; i < n; ++i)
                  sk[i] = fs * cvd[i];
              }
            line_operator<dim, n, 1, T, skew, diff, LATE, true>(
              P, B, F, cell, p, bmask, up, dp, fan, uq, g, sk, (T)wl[1],
              acc);
            lds_write_line<dim, n, 1>(acc_l, p, acc);
            __syncthreads();
          }

        // ---- x direction ----
        {
          T        uq[n], g[n], sk[n];
          const T(&cvd)[n] = cvx;
          lds_read_line<dim, n, 0>(u_l, p, uq);
          if constexpr (AN)
            lds_read_line<dim, n, 0>(g0_l, p, g);
          else
            {
#pragma unroll
              for (int i = 0; i < n; ++i)
                g[i] = fcell * cvd[i] * uq[i];
            }
          lds_read_line<dim, n, 0>(acc_l, p, acc);
          if constexpr (skew && AN)
            lds_read_line<dim, n, 0>(sk0_l, p, sk);
          else if constexpr (skew)
            {
#pragma unroll
              for (int i = 0; i < n; ++i)
                sk[i] = fs * cvd[i];
            }
          line_operator<dim, n, 0, T, skew, diff, LATE, true>(
            P, B, F, cell, p, bmask, up, dp, fan, uq, g, sk, (T)wl[0],
            acc);
        }
        __syncthreads();
        if constexpr (fin == fin_local)
          {
            // the result stays at the Gauss points, stored from x-lines
            __builtin_amdgcn_s_setprio(3);
            if (active)
              {
                const int64_t base = c * io.comp_stride + cell * nd;
#pragma unroll
                for (int i = 0; i < n; ++i)
                  io.dst[base + L::template off<0>(p, i)] = io.scale * acc[i];
              }
            __builtin_amdgcn_s_setprio(0);
            continue;
          }
        if constexpr (fin == fin_inverse_mass)
          {
            T ij[n];
            if constexpr (AN)
              {
                // 1/JxW sits at LAST-line points; move it to x-lines
#pragma unroll
                for (int i = 0; i < n; ++i)
                  ij[i] = (T)1 / jxw[i];
                lds_write_line<dim, n, LAST>(g0_l, p, ij);
                __syncthreads();
                lds_read_line<dim, n, 0>(g0_l, p, ij);
              }
            else if constexpr (UNI)
              {
                const T r = (T)(1. / (wl[0] * vol));
#pragma unroll
                for (int i = 0; i < n; ++i)
                  ij[i] = B.winv[i] * r;
              }
            else if constexpr (TL::coef)
              {
                // 1 / (w_i det): the hardware's estimate of the reciprocal
                // and two Newton steps (~1 ulp, det > 0)
#pragma unroll
                for (int i = 0; i < n; ++i)
                  {
                    const T x = B.xq[i];
                    const T d = fma(fma(ij_row[2], x, ij_row[1]), x, ij_row[0]);
                    T       r = __builtin_amdgcn_rcp(d);
                    r         = fma(r, fma(-d, r, (T)1), r);
                    r         = fma(r, fma(-d, r, (T)1), r);
                    ij[i]     = B.winv[i] * r;
                  }
              }
            else
#pragma unroll
              for (int i = 0; i < n; ++i)
                ij[i] = ij_row[i];
#pragma unroll
            for (int i = 0; i < n; ++i)
              acc[i] *= ij[i];
          }

        // ---- back to nodal values: x (registers), y, (z) ----
        {
          T t[n];
          if constexpr (fin == fin_inverse_mass)
            eo_apply<n, false, false, false>(B.eo_Sinv, acc, t);
          else
            eo_apply<n, false, true, false>(B.eo_S, acc, t);
          lds_write_line<dim, n, 0>(acc_l, p, t);
          __syncthreads();
          lds_read_line<dim, n, 1>(acc_l, p, t);
          if constexpr (fin == fin_inverse_mass)
            eo_apply<n, false, false, false>(B.eo_Sinv, t, acc);
          else
            eo_apply<n, false, true, false>(B.eo_S, t, acc);
          if constexpr (dim == 3)
            {
              __syncthreads();
              lds_write_line<dim, n, 1>(acc_l, p, acc);
              __syncthreads();
              lds_read_line<dim, n, 2>(acc_l, p, t);
              if constexpr (fin == fin_inverse_mass)
                eo_apply<n, false, false, false>(B.eo_Sinv, t, acc);
              else
                eo_apply<n, false, true, false>(B.eo_S, t, acc);
            }
        }

        // ---- epilogue on LAST-direction lines (coalesced) ----
        __builtin_amdgcn_s_setprio(3);
        if (active)
          {
            const int64_t base = c * io.comp_stride + cell * nd;
            if constexpr (epi == epi_store)
              {
#pragma unroll
                for (int i = 0; i < n; ++i)
                  __builtin_nontemporal_store(
                    io.scale * acc[i],
                    &io.dst[base + L::template off<LAST>(p, i)]);
              }
            else
              {
#pragma unroll
                for (int i = 0; i < n; ++i)
                  {
                    const int64_t k  = base + L::template off<LAST>(p, i);
                    const T       s0 = io.sol_in[k];
                    __builtin_nontemporal_store(fma(io.b_dt, acc[i], s0),
                                                &io.sol_out[k]);
                    if (!io.last)
                      __builtin_nontemporal_store(fma(io.a_dt, acc[i], s0),
                                                  &io.ri_out[k]);
                  }
              }
          }
        if (NC > 1)
          {
            __builtin_amdgcn_s_setprio(0);
            __syncthreads();
          }
      }
  }

  // Wavefronts per SIMD the compiler has to leave room for. Left alone its
  // scheduler hoists the loads of a whole phase (there is no branch to stop
  // at) and takes one or two occupancy steps more than the values need; the
  // figures are the steps that cost at most a few spilled registers. In 2D
  // they show in the FP32 implicit operator alone (against no figure, 256^2
  // cells: degree 4 12.7 -> 11.0 us, degrees 1, 2, 5, 7 up to 14% less or
  // even, degree 6 19.4 -> 21.2); all others, also small meshes, are even.
  template <int dim, int n, int NC, typename T, int geo, bool skew, bool diff,
            int fin>
  constexpr int
  operator_waves()
  {
    constexpr bool f64 = sizeof(T) == 8;
    if (geo == geo_analytic)
      // FP32 takes 135 registers in 2D at degree 3 and 278 in 3D at degree
      // 7 on its own: 20.7 -> 17.5 us (256^2 cells) and 50 -> 38 us (16^3)
      // with one wavefront more; FP64 and the implicit operator at degree 7
      // spill too much for it
      return !f64 && dim == 2 && n <= 4                            ? 4 :
             !f64 && dim == 3 && n == 8 && fin == fin_inverse_mass ? 2 :
                                                                     1;
    if (diff)
      return 2;
    if (NC > 1 && fin == fin_integrate)
      // uniform degree 1 in FP64: 128 registers instead of 130, two stages
      // on 64^3 cells 40.9 -> 37.8 us
      return dim == 3 ? (f64 ? (n <= 2 ? (geo == geo_uniform ? 4 : 3) : 2) :
                               (n <= 5 ? (geo == geo_table ? 4 : 3) : 2)) :
                        (f64 ? (n <= 4 ? 3 : 2) : (n <= 5 ? 4 : 3));
    if (dim == 2)
      return f64 ? (n <= 6 ? 4 : 3) : (n <= 6 ? 6 : 5);
    if (fin == fin_inverse_mass)
      return f64 ? (n <= 5 || !skew ? 4 : 2) : (n <= 5 ? 6 : 2);
    if (fin == fin_integrate)
      // 3D degree 4: 126-128 VGPRs with at most 8 spilled, instead of
      // 132-146 at three; FP32 degree 5: 128 instead of 132, 32^3 cells
      // with boundary faces 54 -> 51 us
      return n <= 5 || (!f64 && n == 6) ? 4 : 2;
    return 2;
  }

  // One batch of CPB cells per workgroup: workgroup b of n_blocks covers
  // the cells of block xcd_block(b, n_blocks). (A grid-stride loop over
  // several batches per workgroup was measured and rejected: the loop lets
  // the compiler keep loop-invariant loads live across iterations, 107 ->
  // 149 VGPRs at 3D degree 4, one occupancy step lost.)
  template <int dim, int n, int NC, typename T, int geo, bool skew,
            bool diff, int fin, int epi, int CPB>
  __global__ void __launch_bounds__(CPB * (dim == 3 ? n * n : n))
  __attribute__((amdgpu_waves_per_eu(
    operator_waves<dim, n, NC, T, geo, skew, diff, fin>())))
  dg_operator_kernel(const OpParams                       P,
                     const DevBasis<T> *__restrict__      Bp,
                     const DevBasis<double> *__restrict__ Bd,
                     const OpBuffers<T>                   io)
  {
    operator_body<dim, n, NC, T, geo, skew, diff, fin, epi, CPB>(
      P, Bp, Bd, io, xcd_block(blockIdx.x, gridDim.x));
  }

  // one member of a batched launch: an independent operator (its own mesh,
  // speed and vectors) of the same variant, owning the workgroups
  // [first_block, first_block + blocks)
  template <typename T>
  struct BatchItem
  {
    OpParams     P;
    OpBuffers<T> io;
    unsigned     first_block;
  };

  // Several operators of one variant in a single launch (the serving loop
  // advances all active solves of one degree by one LSRK stage with it).
  // Items are sorted by first_block; the lookup is uniform per workgroup.
  template <int dim, int n, int NC, typename T, int geo, bool skew,
            bool diff, int fin, int epi, int CPB>
  __global__ void __launch_bounds__(CPB * (dim == 3 ? n * n : n))
  __attribute__((amdgpu_waves_per_eu(
    operator_waves<dim, n, NC, T, geo, skew, diff, fin>())))
  dg_operator_batch_kernel(const BatchItem<T> *__restrict__      items,
                           int                                  n_items,
                           const DevBasis<T> *__restrict__      Bp,
                           const DevBasis<double> *__restrict__ Bd)
  {
    const unsigned b = xcd_block(blockIdx.x, gridDim.x);
    int            r = 0;
    for (int k = 1; k < n_items; ++k)
      if (items[k].first_block <= b)
        r = k;
    const BatchItem<T> &it = items[r];
    operator_body<dim, n, NC, T, geo, skew, diff, fin, epi, CPB>(
      it.P, Bp, Bd, it.io, b - it.first_block);
  }
} // namespace dgops
