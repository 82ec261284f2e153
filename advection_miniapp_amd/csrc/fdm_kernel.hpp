// Cellwise fast-diagonalization (FDM) preconditioner for gfx950: the exact
// inverse of the separable part of the cell operator
//   detJ [ (Lambda_stage / dt) (x) M(x)M(x)M + I (x) sum_d a_d M..K_d..M ]
// (block Jacobi: the inflow neighbour coupling is dropped), as in
// CellwisePreconditionerFDM (advection_solver_irk_real.cc:807-1199; single
// stage advection_solver_implicit_real.cc:539-813):
//   1. stage transform T^-1 (IRK)                          :950-985
//   2. d sweeps with V^-1 M^-1                             :997-1009
//   3. pointwise inverse on the real-pair blocks           :1019-1052
//   4. d sweeps with V                                     :1055-1065
//   5. stage transform T                                   :1068-1110
// The reference keeps one 1D eigenbasis per velocity sign and picks the one
// of the sign of the cell's mean reference-space velocity (:838-844). The
// upwind matrices of the two signs are mirror images,
//   M^-1 K(-) = -R M^-1 K(+) R,   R M R = M,   R = line reversal,
// so a direction with a < 0 uses the eigenbasis of the + sign on the
// reversed line and the eigenvalues of a M^-1 K(-) are |a| lambda(+). The
// reversal is a permutation of the line's points: it is folded into the
// per-lane addresses of the loads, LDS accesses and stores, and the 1D
// tables stay uniform across the wavefront.
//
// Step 3 diagonalizes every 2x2 real-pair block [[a, b], [-b, a]] with
// U = [[1, 1], [i, -i]] (eigenvalues lambda, conj(lambda)) and divides by
// sigma + sum_d |a_d| lambda_d in complex arithmetic; the same holds for
// the stage pairs of A^-1. Lines are owned by threads as in op_kernel.hpp.
//
// Bound by vector instructions and latency (at degree 4 with three stages
// the products need 540 fused multiply-adds of a thread; the dofs in and out
// 39 us at 5 TB/s in FP64). Step 3 works on conjugate halves, reads task
// records with ready LDS offsets and spreads over both wavefronts, and the
// sweeps share each table row between the stages: 1410 instead of 2280 vector
// instructions at degree 4, 2750 instead of 5690 at degree 7, and 126 (FP64)
// and 72 (FP32) instead of 139 and 109 registers. Degree 4, three stages,
// 32768 cells on MI355X: FP32 59 -> 43 us, FP64 operator and FDM together
// 225 -> 206 us.
#pragma once

#include "op_kernel.hpp"

namespace dgops
{
  // step-3 tasks per cell: at most 2 stage blocks (s <= 4) times 4^3
  // direction blocks (n <= 8)
  constexpr int max_fdm_tasks = 128;

  // one step-3 task: a block of real-pair-coupled points of one cell. The
  // factors are 0 = stage, 1 + d = direction d; the paired ones are listed
  // first, with the LDS distance of the partner points and the imaginary
  // part of the eigenvalue.
  template <typename T>
  struct alignas(16) FdmTask
  {
    int16_t base;      // LDS offset of the first point in the cell's blocks
    int16_t delta[4];  // of paired factor b
    uint8_t factor[4]; // of paired factor b
    T       re[4];     // real parts, factor f times |a_d| or 1/dt
    T       im[4];     // imaginary parts, of paired factor b
  };

  template <typename T>
  struct FdmDev
  {
    // 1D eigenbasis of M^-1 K(+) (velocity sign +)
    T   VinvMinv[max_n][max_n]; // [i][j]
    T   V[max_n][max_n];
    T   lre[max_n], lim[max_n];
    int kind[max_n];               // 0 real, 1 first of pair, 2 second
    int n_blocks;                  // blocks per direction
    int block_col[max_n];          // first column of block b
    int block_size[max_n];         // 1 or 2
    // stages (Radau IIA A^-1 = T Lambda T^-1), s <= 5
    T   Tinv[5][5], Tm[5][5];
    T   mre[5], mim[5];
    int n_stage_blocks;
    int stage_block_col[5];
    int stage_block_size[5];
    // step-3 tasks of one cell sorted by their number of paired factors
    // NB: tasks[task_start[NB] .. task_start[NB + 1])
    int        task_start[6];
    FdmTask<T> tasks[max_fdm_tasks];
  };

  struct FdmParams
  {
    int64_t       n_cells;
    const double *cell_velocity; // [cell][dim], reference space, t = 0
    const double *cell_invdet;   // [cell]
    double        vel_scale;     // time factor
    double        inv_dt;
    int64_t       block;         // stage block size (dofs)
  };

  // LDS stride from cell to cell. Step 3 has the cells of a task on
  // successive lanes; with an even number of stages an even stride leaves
  // them few banks (degree 3, four stages: 80 values in 2D, 320 in 3D, two
  // banks of 32), an odd one all. Four stages on one MI355X, before and
  // after: 3D degree 1, 64^3 cells 65 -> 40 us in FP64 and 39 -> 24 in FP32;
  // 2D degree 3, 256^2 cells, FP64 34 -> 26 us. Odd stage counts keep the
  // stride: their sweeps lose as much as step 3 gains.
  template <int dim, int n, int NS>
  constexpr int
  fdm_cell_stride()
  {
    const int s = NS * Lay<dim, n>::stride;
    return NS % 2 == 0 ? s | 1 : s;
  }

  // offsets of the points of LDS line p of direction dir, in reverse order
  // when `rev`: one start and one step per line
  template <int dim, int n, int dir>
  __device__ __forceinline__ void
  lds_line_m(int p, bool rev, int (&a)[n])
  {
    using L        = Lay<dim, n>;
    constexpr int s = dir == 0 ? 1 : dir == 1 ? L::sx : L::sy;
    const int  step = rev ? -s : s;
    a[0]            = L::template loff<dir>(p, 0) + (rev ? (n - 1) * s : 0);
#pragma unroll
    for (int i = 1; i < n; ++i)
      a[i] = a[i - 1] + step;
  }

  // inverse of one block of 2^NB real-pair-coupled points (NB paired
  // factors among stage, x, y, z): load, U^-1 on every paired factor,
  // complex division by the eigenvalue sum, U, store. `delta[b]` is the
  // storage distance to the partner along paired factor b, lr the real
  // part of the eigenvalue sum and li[b] the imaginary part of paired
  // factor b (conjugated when the point's bit b is set).
  //
  // The values are real, so after U^-1 the point with all bits flipped holds
  // the conjugate value, before and after the division. Only the 2^(NB-1)
  // points with bit 0 clear are computed: the transform of bit 0 pairs two
  // real values to one complex one on the load and splits it on the store.
  // The factors 1/2 of U^-1 (and 2 of Re, Im at the end) are in `invdet`.
  template <int NB, typename T>
  __device__ __forceinline__ void
  fdm_block(T *data, int base, const int (&delta)[4], T lr,
            const T (&li)[4], T invdet)
  {
    if constexpr (NB == 0)
      {
        data[base] *= lr * (invdet / (lr * lr));
        return;
      }
    // point h: bit b - 1 of h is the bit of paired factor b
    constexpr int NH = NB == 0 ? 1 : 1 << (NB - 1);
    int           a[NH];
    T             re[NH], im[NH];
#pragma unroll
    for (int h = 0; h < NH; ++h)
      {
        a[h] = base;
#pragma unroll
        for (int b = 1; b < NB; ++b)
          if ((h >> (b - 1)) & 1)
            a[h] += delta[b];
        // (x0, x1) -> x0 - i x1
        re[h] = data[a[h]];
        im[h] = -data[a[h] + delta[0]];
      }
    // U^-1: (z0, z1) -> (z0 - i z1, z0 + i z1)
#pragma unroll
    for (int b = 1; b < NB; ++b)
#pragma unroll
      for (int h = 0; h < NH; ++h)
        if (!((h >> (b - 1)) & 1))
          {
            const int h1 = h | (1 << (b - 1));
            const T   r0 = re[h], i0 = im[h], r1 = re[h1], i1 = im[h1];
            re[h]        = r0 + i1;
            im[h]        = i0 - r1;
            re[h1]       = r0 - i1;
            im[h1]       = i0 + r1;
          }
    // times invdet / (lr + i lim_h), lim_h = sum_b +-li[b]
    const T scale = invdet * (T)(1. / (1 << (NB == 0 ? 0 : NB - 1)));
#pragma unroll
    for (int h = 0; h < NH; ++h)
      {
        // four divisions at a time (registers for four wavefronts per SIMD instead of three)
        if constexpr (NB == 4)
          if (h == 4)
            asm volatile(""
                         : "+v"(lr), "+v"(re[0]), "+v"(re[1]), "+v"(re[2]),
                           "+v"(re[3]));
        T lim = li[0];
#pragma unroll
        for (int b = 1; b < NB; ++b)
          lim += ((h >> (b - 1)) & 1) ? -li[b] : li[b];
        const T q  = scale / (lr * lr + lim * lim);
        const T sr = lr * q, si = -lim * q;
        const T r = re[h], i = im[h];
        re[h]     = r * sr - i * si;
        im[h]     = r * si + i * sr;
      }
    // U: (y+, y-) -> (y+ + y-, i (y+ - y-))
#pragma unroll
    for (int b = 1; b < NB; ++b)
#pragma unroll
      for (int h = 0; h < NH; ++h)
        if (!((h >> (b - 1)) & 1))
          {
            const int h1 = h | (1 << (b - 1));
            const T   r0 = re[h], i0 = im[h], r1 = re[h1], i1 = im[h1];
            re[h]        = r0 + r1;
            im[h]        = i0 + i1;
            re[h1]       = i1 - i0;
            im[h1]       = r0 - r1;
          }
    // y- = conj(y+): (2 Re y+, -2 Im y+)
#pragma unroll
    for (int h = 0; h < NH; ++h)
      {
        data[a[h]]            = re[h];
        data[a[h] + delta[0]] = -im[h];
      }
  }

  // step 3 for the tasks with NB paired factors of the CPB cells of a
  // workgroup (task k of cell lc on thread k * CPB + lc after thread
  // `first`, strided by the workgroup size); s_cell[lc] = (1/dt,
  // |a_0|, |a_1|, |a_2|, det J^-1)
  template <int NB, int dim, int n, int NS, int CPB, typename Tc>
  __device__ __forceinline__ void
  fdm_pointwise_group(const FdmDev<Tc> &F, Tc *s_data,
                      const Tc (*s_cell)[5], int64_t cell0, int64_t n_cells,
                      int first)
  {
    const int tid =
      (int)threadIdx.x - first + ((int)threadIdx.x < first ? blockDim.x : 0);
    const int     t0  = F.task_start[NB];
    const int     nt  = (F.task_start[NB + 1] - t0) * CPB;
    for (int t = tid; t < nt; t += blockDim.x)
      {
        const int k  = t / CPB;
        const int lc = t - k * CPB;
        if (cell0 + lc >= n_cells)
          continue;
        const FdmTask<Tc> &tk = F.tasks[t0 + k];
        const Tc          *m  = s_cell[lc];
        Tc                 lr = tk.re[0] * m[0];
#pragma unroll
        for (int d = 0; d < dim; ++d)
          lr += tk.re[1 + d] * m[1 + d];
        int delta[4];
        Tc  li[4];
#pragma unroll
        for (int b = 0; b < NB; ++b)
          {
            delta[b] = tk.delta[b];
            li[b]    = tk.im[b] * m[tk.factor[b]];
          }
        fdm_block<NB, Tc>(s_data + lc * fdm_cell_stride<dim, n, NS>(), tk.base,
                          delta, lr, li, m[4]);
      }
  }

  // A 1D matrix product on the thread's lines of all NS stages, row by row:
  // out(q, v) gets the values v[j] = sum_i M[q][i] in[j][i] of the stages.
  // One row of the table is in scalar registers at a time and used for all
  // stages. The pointer is opaque for every sweep, so that the compiler
  // loads the rows again (from the scalar cache) instead of keeping a whole
  // table over the sweeps: n = 8 has 64 doubles, more than there are scalar
  // registers, and spent 3200 of 6300 vector instructions on spilling them.
  template <int n, int NS, typename T, typename F>
  __device__ __forceinline__ void
  fdm_sweep(const T (&table)[max_n][max_n], const T (&in)[NS][n], F &&out)
  {
    using CT = const __attribute__((address_space(4))) T;
    CT *M    = (CT *)(uintptr_t)&table[0][0];
    asm volatile("" : "+s"(M));
#pragma unroll
    for (int q = 0; q < n; ++q)
      {
        T v[NS];
#pragma unroll
        for (int j = 0; j < NS; ++j)
          v[j] = M[q * max_n] * in[j][0];
#pragma unroll
        for (int i = 1; i < n; ++i)
#pragma unroll
          for (int j = 0; j < NS; ++j)
            v[j] = fma(M[q * max_n + i], in[j][i], v[j]);
        out(q, v);
      }
  }

  template <int dim, int n, int NS, typename Tc, typename Tin, typename Tout>
  __global__ void __launch_bounds__(128)
  fdm_kernel(const FdmParams P, const FdmDev<Tc> *__restrict__ Fp,
             const Tin *__restrict__ src, Tout *__restrict__ dst)
  {
    using L           = Lay<dim, n>;
    constexpr int nl  = L::nl;
    constexpr int nd  = L::nd;
    constexpr int CPB = cells_per_block<dim, n>();
    constexpr int STR = L::stride;
    constexpr int CS  = fdm_cell_stride<dim, n, NS>();
    constexpr int LAST = dim - 1;

    __shared__ Tc s_data[CPB * CS];

    const FdmDev<Tc> &F    = *Fp;
    const int         tid  = threadIdx.x;
    const int         lc   = tid / nl;
    const int         p    = tid - lc * nl;
    const int64_t     cell0 = (int64_t)xcd_block(blockIdx.x, gridDim.x) * CPB;
    const bool        active = cell0 + lc < P.n_cells;
    Tc               *data   = s_data + lc * CS;
    // threads past the last cell load it and store nothing
    const int64_t     cell   = active ? cell0 + lc : P.n_cells - 1;

    // 1/dt, |speed| per direction and det J^-1 of the workgroup's cells,
    // read by any thread in step 3
    __shared__ Tc s_cell[CPB][5];
    bool rv[3] = {false, false, false};
#pragma unroll
    for (int d = 0; d < dim; ++d)
      {
        const double a = P.cell_velocity[cell * dim + d] * P.vel_scale;
        rv[d]          = a < 0.;
        if (active && p == 0)
          s_cell[lc][1 + d] = (Tc)fabs(a);
      }
    if (active && p == 0)
      {
        s_cell[lc][0] = (Tc)P.inv_dt;
        s_cell[lc][4] = (Tc)P.cell_invdet[cell];
      }
    // x-line in the vectors, mirrored
    const int64_t x0 = cell * nd + L::template off<0>(p, 0) +
                       (rv[0] ? n - 1 : 0);
    const int     xs = rv[0] ? -1 : 1;
    Tc            r[NS][n];
    int           al[n];

    // 1-2: load (x mirrored), stage transform, V^-1 M^-1 sweeps x, y, (z)
    // with the y and z mirrors on the LDS reads. Every stage has its own
    // LDS block; a thread rewrites exactly the positions of its own line
    // (the mirrors permute within a line), so all stages share one barrier
    // per direction change.
#pragma unroll
    for (int t = 0; t < NS; ++t)
#pragma unroll
      for (int i = 0; i < n; ++i)
        r[t][i] = (Tc)src[t * P.block + x0 + i * xs];
    if constexpr (NS > 1)
#pragma unroll
      for (int i = 0; i < n; ++i)
        {
          Tc w[NS];
#pragma unroll
          for (int j = 0; j < NS; ++j)
            {
              w[j] = 0;
#pragma unroll
              for (int k = 0; k < NS; ++k)
                w[j] = fma(F.Tinv[j][k], r[k][i], w[j]);
            }
#pragma unroll
          for (int j = 0; j < NS; ++j)
            r[j][i] = w[j];
        }
    fdm_sweep<n, NS>(F.VinvMinv, r, [&](int q, const Tc(&v)[NS]) {
#pragma unroll
      for (int j = 0; j < NS; ++j)
        data[j * STR + L::template loff<0>(p, q)] = v[j];
    });
    __syncthreads();
    lds_line_m<dim, n, 1>(p, rv[1], al);
#pragma unroll
    for (int j = 0; j < NS; ++j)
#pragma unroll
      for (int i = 0; i < n; ++i)
        r[j][i] = data[j * STR + al[i]];
    fdm_sweep<n, NS>(F.VinvMinv, r, [&](int q, const Tc(&v)[NS]) {
#pragma unroll
      for (int j = 0; j < NS; ++j)
        data[j * STR + L::template loff<1>(p, q)] = v[j];
    });
    if constexpr (dim == 3)
      {
        __syncthreads();
        lds_line_m<dim, n, 2>(p, rv[2], al);
#pragma unroll
        for (int j = 0; j < NS; ++j)
#pragma unroll
          for (int i = 0; i < n; ++i)
            r[j][i] = data[j * STR + al[i]];
        fdm_sweep<n, NS>(F.VinvMinv, r, [&](int q, const Tc(&v)[NS]) {
#pragma unroll
          for (int j = 0; j < NS; ++j)
            data[j * STR + L::template loff<2>(p, q)] = v[j];
        });
      }
    __syncthreads();

    // 3: pointwise inverse on the blocks of the workgroup's cells, one
    // group of block shapes (number of paired factors NB) after the other:
    // the threads of a wave run one shape at a time. The last and costliest
    // group starts on the second wavefront, the others on the first: with
    // all of them on the first (five groups of 5 to 100 tasks for n = 5 and
    // three stages) the second waits for it.
    {
      constexpr int TOP = dim + (NS > 1 ? 1 : 0);
      fdm_pointwise_group<0, dim, n, NS, CPB>(F, s_data, s_cell, cell0,
                                              P.n_cells, 0);
      fdm_pointwise_group<1, dim, n, NS, CPB>(F, s_data, s_cell, cell0,
                                              P.n_cells, 0);
      fdm_pointwise_group<2, dim, n, NS, CPB>(F, s_data, s_cell, cell0,
                                              P.n_cells, TOP == 2 ? 64 : 0);
      if constexpr (TOP >= 3)
        fdm_pointwise_group<3, dim, n, NS, CPB>(F, s_data, s_cell, cell0,
                                                P.n_cells,
                                                TOP == 3 ? 64 : 0);
      if constexpr (TOP >= 4)
        fdm_pointwise_group<4, dim, n, NS, CPB>(F, s_data, s_cell, cell0,
                                                P.n_cells, 64);
      __syncthreads();
    }

    // the line's offsets again, instead of kept in registers over step 3
    int pv = p;
    asm volatile("" : "+v"(pv));

    // 4: V sweeps LAST, ..., x with the mirrors on the writes; the x
    // mirror goes into the store
    lds_line_m<dim, n, LAST>(pv, rv[LAST], al);
#pragma unroll
    for (int j = 0; j < NS; ++j)
      lds_read_line<dim, n, LAST>(data + j * STR, pv, r[j]);
    fdm_sweep<n, NS>(F.V, r, [&](int q, const Tc(&v)[NS]) {
#pragma unroll
      for (int j = 0; j < NS; ++j)
        data[j * STR + al[q]] = v[j];
    });
    __syncthreads();
    if constexpr (dim == 3)
      {
        lds_line_m<dim, n, 1>(pv, rv[1], al);
#pragma unroll
        for (int j = 0; j < NS; ++j)
          lds_read_line<dim, n, 1>(data + j * STR, pv, r[j]);
        fdm_sweep<n, NS>(F.V, r, [&](int q, const Tc(&v)[NS]) {
#pragma unroll
          for (int j = 0; j < NS; ++j)
            data[j * STR + al[q]] = v[j];
        });
        __syncthreads();
      }
#pragma unroll
    for (int j = 0; j < NS; ++j)
      lds_read_line<dim, n, 0>(data + j * STR, pv, r[j]);

    // 5: x sweep, back stage transform and store (x-lines, mirrored in x)
    if (active)
      fdm_sweep<n, NS>(F.V, r, [&](int q, const Tc(&v)[NS]) {
#pragma unroll
        for (int t = 0; t < NS; ++t)
          {
            Tc s = v[0];
            if constexpr (NS > 1)
              {
                s = 0;
#pragma unroll
                for (int j = 0; j < NS; ++j)
                  s = fma(F.Tm[t][j], v[j], s);
              }
            dst[t * P.block + x0 + q * xs] = (Tout)s;
          }
      });
  }
} // namespace dgops
