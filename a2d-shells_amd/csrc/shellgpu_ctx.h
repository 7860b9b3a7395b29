// shellgpu_ctx.h -- the context and matrix objects behind the C ABI
// (host-side state shared by the translation units of the library).
#pragma once

#include <algorithm>
#include <memory>
#include <string>
#include <utility>
#include <vector>

#include "shellgpu_internal.h"

namespace shellgpu {
struct NdLayout;
}

struct shellgpu_ctx {
  int device = 0;
  hipStream_t stream = nullptr;
  std::string err;

  int nnodes = 0, nelems = 0, nnzb = 0, ncolors = 0, nbatch = 0;
  std::vector<int> h_conn, h_rowp, h_cols, h_color, h_color_ptr, h_color_elems, h_blk;
  int *d_conn = nullptr, *d_rowp = nullptr, *d_cols = nullptr, *d_blk = nullptr;
  // per node the block index of its diagonal block; per block the index of
  // the transposed block (the pattern is structurally symmetric)
  int *d_diag = nullptr, *d_tpos = nullptr;
  int *d_color_elems = nullptr;
  // per element, bit 4 i + j: this element is the first, in colour launch
  // order, to reach BSR block (node i, node j), so a matrix assembly can
  // write that block instead of adding to a zeroed one; null when an element
  // repeats a node (two of its blocks coincide)
  int *d_first = nullptr;
  double *d_X = nullptr;
  // per node n the places 4 element + corner where it stands, in element
  // order: d_corner[d_nptr[n]..d_nptr[n + 1]) (one allocation)
  int *d_nptr = nullptr;
  const int *d_corner = nullptr;

  // element colouring: 0 greedy first fit in element order, 1 greedy first
  // fit with the elements of most neighbours first (shellgpu_tune chooses)
  int coloring = 0;
  // compiled schedule of each element-kernel mode (launch_elem_kernel's
  // variant); shellgpu_tune and shellgpu_set_elem_schedule choose another, and
  // the tuner's report.  The default, four elements per workgroup, is the
  // fastest for every size measured (us, schedules 0 / 1 / 4 / 5):
  //   K        200 x 400 285 / 308 / 257 / 292, 20 x 40 48 / 50 / 46 / 48
  //   tangent  150 x 301 378 / 390 / 341 / 352, 20 x 40 77 / 79 / 73 / 75
  //   G        200 x 400 743 / 755 / 690 / 703, 20 x 40 88 / 90 / 85 / 87
  //   tangent with residual
  //            150 x 301 369 / 382 / 335 / 343, 20 x 40 81 / 82 / 78 / 78
  int elem_variant[32];
  shellgpu_ctx() { std::fill(elem_variant, elem_variant + 32, 4); }
  std::string schedule;

  shellgpu::Material mat = shellgpu::make_material(70e9, 0.3, 2700.0, 0.0, 10.0);

  int nbc = 0;
  std::vector<int> h_bc_nodes, h_bc_mask;
  int *d_bc_nodes = nullptr, *d_bc_mask = nullptr;
  double *d_bc_vals = nullptr;
  int *d_bc_rows = nullptr;  // the masks per node, for a mesh of bc_rows nodes
  int bc_rows = 0;

  double *d_thick = nullptr, *d_temp = nullptr;
  bool same_designs = false;  // every design has the same thickness and temperature
  double *d_coef = nullptr;  // 4 * nbatch per-design kernel coefficients
  // element gradients of run_xpt and run_dv, 24 doubles per element for as
  // many designs as xpt_designs() allows at a time
  double *d_xg = nullptr;
  size_t xg_doubles = 0;
  // timing
  bool timing = false;
  std::vector<std::pair<hipEvent_t, hipEvent_t>> elem_ev, spmv_ev;
  int elem_launches = 0;  // element-kernel launches inside the elem_ev pairs
  hipEvent_t t0 = nullptr, t1 = nullptr;

  // the device's copy of the library's static scratch array (mapped at
  // shellgpu_create; shared by every context on the device) and its size
  double *scratch = nullptr;
  size_t scratch_doubles = 0;

  // solver state
  std::vector<int> order_seed;  // BFS seed nodes of the level ordering
  // nested-dissection order and front layout of the mesh, made by the first
  // factor and shared by the later ones (an analysis has two); dropped with
  // the mesh or the coordinates it was made from
  std::shared_ptr<const shellgpu::NdLayout> nd_layout;
  void *blas = nullptr;         // rocblas_handle bound to `stream`
};

struct shellgpu_mat {
  shellgpu_ctx *ctx = nullptr;
  int nbatch = 0;
  double *vals = nullptr;
  // every design's values are equal (zeroed, or assembled from identical
  // designs without a per-design state, and changed only uniformly since):
  // a product then reads one copy for all designs' vectors
  bool same = false;
};

namespace shellgpu {
// element-kernel arguments for the context's mesh, material and designs
// with state u (NULL = zero)
ElemArgs base_args(shellgpu_ctx *ctx, const double *u);
// launch one element-kernel mode colour by colour (no two elements of a
// launch share a node, so scatters need no atomics)
int run_colored(shellgpu_ctx *ctx, int mode, ElemArgs a);
// coordinate-derivative kernel over all elements; coef (device, 4 per
// design), vectors with stride 6*nnodes, dfdX with stride 3*nnodes
int run_xpt(shellgpu_ctx *ctx, const double *phi, const double *u, const double *psi, const double *coef,
            int nonlin, int terms, double *dfdX);
// the thickness derivatives of the same scalars, and d(phi^T G(u) phi)/du
// (dfdt, stride nelems, and dfdu, stride 6*nnodes, may be null)
int run_dv(shellgpu_ctx *ctx, const double *phi, const double *u, const double *psi, const double *coef, int nonlin,
           int terms, double *dfdt, double *dfdu);
}  // namespace shellgpu
