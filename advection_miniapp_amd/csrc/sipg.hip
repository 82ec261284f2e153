// Launcher of the SIPG operator kernel for cells of any shape
// (sipg_kernel.hpp): instances per dimension, degree and form; the face
// geometry table is built on the first call of an operator handle.
#include "aux.hpp"
#include "internal.hpp"
#include "sipg_kernel.hpp"

namespace dgops
{
  namespace
  {
    struct Launch
    {
      Operator                &op;
      const OpParams          &P;
      int                      fin, epi;
      const OpBuffers<double> &io;
    };

    template <int dim, int n, bool skew, int fin, int epi>
    void
    launch_form(const Launch &a)
    {
      constexpr int CPB    = cells_per_block<dim, n>();
      const int64_t blocks = (a.P.n_cells + CPB - 1) / CPB;
      hipLaunchKernelGGL((sipg_operator_kernel<dim, n, skew, fin, epi>),
                         dim3((unsigned)blocks),
                         dim3(CPB * Lay<dim, n>::nl), 0, a.op.stream, a.P,
                         a.op.d_basis_d.as<const DevBasis<double>>(),
                         a.op.d_sipg_faces.as<const double>(), a.io);
    }

    template <int dim, int n>
    bool
    launch(int want, const Launch &a)
    {
      if (want != n)
        return false;
      using FT = SipgFaces<dim, n>;
      if (!a.op.sipg_faces_ready)
        {
          const int64_t entries = a.P.n_cells * dim * FT::nf;
          a.op.d_sipg_faces.alloc(sizeof(double) * entries * FT::nt);
          hipLaunchKernelGGL((sipg_face_table_kernel<dim, n>),
                             dim3((entries + 255) / 256), dim3(256), 0,
                             a.op.stream, a.P,
                             a.op.d_basis_d.as<const DevBasis<double>>(),
                             a.op.d_sipg_faces.as<double>());
          hip_check(hipGetLastError(), "SIPG face table kernel");
          a.op.sipg_faces_ready = true;
        }
      if (a.fin == fin_integrate)
        launch_form<dim, n, true, fin_integrate, epi_store>(a);
      else if (a.epi == epi_store)
        launch_form<dim, n, false, fin_inverse_mass, epi_store>(a);
      else
        launch_form<dim, n, false, fin_inverse_mass, epi_lsrk>(a);
      return true;
    }

    template <int dim, int... ns>
    bool
    launch_any(int n, const Launch &a)
    {
      return (launch<dim, ns>(n, a) || ...);
    }
  } // namespace

  void
  aux_sipg_general(Operator &op, const OpParams &P_in, int fin, int epi,
                   const void *io)
  {
    if (op.mesh.n_cells == 0)
      return;
    aux_geometry_tables(op, DG_FP64);
    OpParams P = P_in;
    P.tab_cell = op.d_tab_cell[0].ptr;
    P.tab_face = op.d_tab_face[0].ptr;
    const Launch a{op, P, fin, epi,
                   *static_cast<const OpBuffers<double> *>(io)};
    const bool   ok = op.cfg.dim == 3 ?
                        launch_any<3, 2, 3, 4, 5, 6, 7, 8>(op.n, a) :
                        launch_any<2, 2, 3, 4, 5, 6, 7, 8>(op.n, a);
    if (!ok)
      throw Error(DG_ERR_UNSUPPORTED, "SIPG on general cells: degree 1..7");
    hip_check(hipGetLastError(), "SIPG operator kernel");
  }
} // namespace dgops
