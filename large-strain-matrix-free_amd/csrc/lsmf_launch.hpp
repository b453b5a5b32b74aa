// lsmf_launch.hpp -- host launchers for one (dim, N) instantiation; included
// by the lsmf_inst_*.hip units, each of which instantiates one LaunchTable.
#pragma once

#include "lsmf_error.hpp"
#include "lsmf_kernels.hpp"
#include "lsmf_op.hpp"

namespace lsmf {

template <int DIM, int N> struct Launch {
  using CS = CellShape<DIM, N>;

  // products of the compact forms on wide Q2 tiles that run the plane kernel: K
  // from the displacement, or cached in FP32.  With 17 cached FP64 values per point
  // (bilinear cells) the line kernel is the faster one, the values of a plane
  // lane's column do not fit its registers: 64^3 311 us against 410, 32^3 41.1
  // against 48, on another stream 69.7 against 79.
  template <typename T, int VAR> static constexpr bool planes_ok() {
    return DIM == 3 && N == 3 &&
           (VAR == V_COMPACT_U || (sizeof(T) == 4 && (VAR == V_COMPACT || VAR == V_COMPACT_AFFINE)));
  }
  // wide tiles with the line kernel: 3D Q4 and Q2, the other variants that run on
  // tensor2 / tensor4 operators (their products, residual and residual VJP)
  template <typename T, int VAR> static constexpr bool wide_ok() {
    return DIM == 3 && (N == 5 || N == 3) && !planes_ok<T, VAR>() &&
           !(N == 3 && sizeof(T) == 8 && VAR == V_COMPACT_AFFINE) &&
           (VAR == V_TENSOR2 || VAR == V_TENSOR4 || VAR == V_COMPACT || VAR == V_COMPACT_AFFINE ||
            VAR == V_RESIDUAL || VAR == V_ADJOINT);
  }
  template <typename T, int VAR> static constexpr bool kinematic_planes() {
    return DIM == 3 && N == 3 && sizeof(T) == 8 && (VAR == V_RESIDUAL || VAR == V_ADJOINT);
  }
  // K from the displacement: that kernel only (cache_variant)
  static constexpr bool recompute_ok() { return DIM == 3 && N == 3; }

  // one colour's fused cell kernel, or with LM_ONE all tiles': n tiles (tiled
  // layouts) or n cells, nv vectors (grid y)
  template <typename T, int VAR, bool ADD, bool CONSTR, unsigned PH, int MODE = LM_COLOUR>
  static int launch_vmult(const lsmf_op *op, const VmultParams<T> &P, int n, unsigned nv, hipStream_t s) {
    if (op->tile_kind == kTileWide) {
      if constexpr (planes_ok<T, VAR>() || kinematic_planes<T, VAR>()) {
        // residual and VJP: formulation 1 on affine cells
        if (planes_ok<T, VAR>() || (op->d_cgeo && op->formulation == 1)) {
          hipLaunchKernelGGL((k_vmult_planes<N, T, VAR, ADD, CONSTR, PH, kTileWide, MODE>), dim3(n, nv),
                             dim3((PlaneShape<N, T, kTileWide>::WG)), 0, s, P);
          return 0;
        }
      }
      if constexpr (wide_ok<T, VAR>())
        hipLaunchKernelGGL((k_vmult<DIM, N, T, VAR, ADD, CONSTR, PH, kTileWide, MODE>), dim3(n, nv),
                           dim3(tile_threads<kTileWide>()), 0, s, P);
      else
        return LSMF_ERR_UNSUPPORTED;
    } else if constexpr (VAR == V_COMPACT_U) {
      return LSMF_ERR_UNSUPPORTED;
    } else if (op->tile_kind == 1) {
      if constexpr (DIM == 3 && N == 3 && VAR == V_SCALAR) {
        // formulation 1 on affine cells with the Q1 metric
        if (op->d_cgeo && op->formulation == 1) {
          hipLaunchKernelGGL((k_vmult_planes<N, T, VAR, ADD, CONSTR, PH, 1, MODE>), dim3(n, nv),
                             dim3((PlaneShape<N, T, 1>::WG)), 0, s, P);
          return 0;
        }
      }
      hipLaunchKernelGGL((k_vmult<DIM, N, T, VAR, ADD, CONSTR, PH, 1, MODE>), dim3(n, nv), dim3(kWG), 0, s, P);
    } else if constexpr (MODE == LM_ONE) {
      return LSMF_ERR_UNSUPPORTED;
    } else {
      hipLaunchKernelGGL((k_vmult<DIM, N, T, VAR, ADD, CONSTR, PH, 0, MODE>), dim3(grid_for(n), nv), dim3(kWG), 0, s, P);
    }
    return 0;
  }

  // even-odd forms of S (rows r < R) and D, from the plain tables
  template <typename T> static void pack_sf(const lsmf_op *op, T *sf) {
    using EO = EvenOdd<N, T>;
    for (int m = 0; m < 2; ++m) {
      const double *M = op->h_sf + m * N * N;
      T *pk = sf + m * EO::PK;
      for (int r = 0; r < EO::R; ++r) {
        for (int k = 0; k < EO::H; ++k) {
          pk[r * EO::H + k] = T(0.5 * (M[r * N + k] + M[r * N + N - 1 - k]));
          pk[EO::R * EO::H + r * EO::H + k] = T(0.5 * (M[r * N + k] - M[r * N + N - 1 - k]));
        }
        pk[2 * EO::R * EO::H + r] = EO::ODD ? T(M[r * N + EO::H]) : T(0);
      }
    }
  }

  template <typename T, int VAR> static VmultParams<T> params(const lsmf_op *op, int k) {
    VmultParams<T> P{};
    P.idx = op->d_idx;
    P.cache = static_cast<const T *>(op->d_cache);
    P.fs = op->field_stride;
    P.tab = static_cast<const T *>(op->d_tab);
    P.u = static_cast<const T *>(VAR == V_COMPACT_U ? op->d_uc : op->d_u);
    P.coords = op->d_coords;
    P.mu = static_cast<const T *>(op->d_mu);
    P.lambda = static_cast<const T *>(op->d_lambda);
    const std::vector<int> &ptr = op->tiled ? op->tile_ptr : op->colour_ptr;
    P.cell_begin = ptr[k];
    P.cell_end = ptr[k + 1];
    P.formulation = op->formulation;
    P.curved = op->curved;
    P.tnodes = op->d_ctile_nodes;
    P.tinfo = op->d_ctile_info;
    P.hang = op->d_hang;
    P.hcons = op->d_hcons;
    P.hbuf = static_cast<T *>(op->d_hbuf);
    P.hstride = (size_t)op->n_hang_inst * DIM;
    P.hptr = op->d_hptr;
    P.dcell = op->d_dcell;
    P.deptr = op->d_deptr;
    P.dtptr = op->d_dtptr;
    P.dta = op->d_dta;
    P.dtw = static_cast<const T *>(op->d_dtw);
    P.dbuf = static_cast<T *>(op->d_dbuf);
    P.hmaster = op->d_hmaster;
    P.hw = static_cast<const T *>(op->d_hw);
    P.dmu = op->adj_dmu;
    P.dlambda = op->adj_dlambda;
    P.perm = op->d_perm;
    P.caff = op->d_caff;
    P.cgeo = op->d_cgeo;
    for (int k = 0; k < 3; ++k) P.qw[k] = op->h_qw[k];
    static_assert(sizeof(P.sf) / sizeof(P.sf[0]) >= 2 * EvenOdd<N, T>::PK, "1D matrices do not fit the kernel arguments");
    pack_sf<T>(op, P.sf);
    return P;
  }

  static int grid_for(int n) { return (n + CS::CPW - 1) / CS::CPW; }
  // with node constraints every write adds (no first-touch stores): zero first
  template <typename T> static void zero_if_constrained(const lsmf_op *op, T *dst, bool add, hipStream_t s) {
    if (op->n_node_cons > 0 && !add)
      hipLaunchKernelGGL(k_zero<T>, dim3((unsigned)((op->n_dofs + 255) / 256)), dim3(256), 0, s, dst, op->n_dofs);
  }
  // DoFs that no cell touches keep whatever dst held: zero them (set mode)
  template <typename T> static void zero_orphans(const lsmf_op *op, T *dst, hipStream_t s) {
    if (op->n_orphan > 0)
      hipLaunchKernelGGL(k_zero_list<T>, dim3((op->n_orphan + 255) / 256), dim3(256), 0, s, op->d_orphan,
                         op->n_orphan, dst);
  }
  static int n_colours(const lsmf_op *op) {
    return (int)(op->tiled ? op->tile_ptr.size() : op->colour_ptr.size()) - 1;
  }

  // the masters' share of the constrained nodes' results, after the colours
  // (nv vectors at dst + b * vstride)
  template <typename T, bool CONSTR> static void hang_gather(const lsmf_op *op, T *dst, size_t vstride, unsigned nv,
                                                              hipStream_t s) {
    if (op->n_hang_masters == 0) return;
    hipLaunchKernelGGL((k_hang_gather<DIM, T, CONSTR>), dim3((op->n_hang_masters + 255) / 256, nv), dim3(256), 0, s,
                       dst, vstride, static_cast<const T *>(op->d_hbuf), (size_t)op->n_hang_inst * DIM,
                       op->d_hg_node, op->d_hg_ptr, op->d_hg_inst, static_cast<const T *>(op->d_hg_w),
                       op->n_hang_masters);
  }

  // parameters of one launch over all tiles
  template <typename T, int VAR> static VmultParams<T> tile_params(const lsmf_op *op) {
    VmultParams<T> P = params<T, VAR>(op, 0);
    P.tnodes = op->d_tile_nodes;
    P.tinfo = op->d_tile_info;
    P.cell_begin = 0;
    P.cell_end = op->tile_ptr.back();
    P.tpriv = op->d_tile_priv;
    P.tbuf = static_cast<T *>(op->d_tile_buf);
    return P;
  }

  // the sums of the nodes that several tiles share, after such a launch
  template <typename T, bool ADD, bool CONSTR>
  static void tile_sum(const lsmf_op *op, T *dst, const T *src, int identity, hipStream_t s,
                       const Epilogue<T> &ep = Epilogue<T>()) {
    const int n = op->sum_begin[op->n_sum_groups];
    if (n == 0) return;
    TileSumParams<T> S{};
    S.node = op->d_sum_node;
    S.slot = op->d_sum_slot;
    S.buf = static_cast<const T *>(op->d_tile_buf);
    S.src = src;
    S.dst = dst;
    S.identity = identity;
    S.ep = ep;
    S.n_groups = op->n_sum_groups;
    for (int g = 0; g < S.n_groups; ++g) {
      S.begin[g] = op->sum_begin[g];
      S.mult[g] = op->sum_mult[g];
      S.first_slot[g] = op->sum_first_slot[g];
    }
    S.begin[S.n_groups] = n;
    hipLaunchKernelGGL((k_tile_sum<DIM, T, ADD, CONSTR>), dim3((n + kWG - 1) / kWG), dim3(kWG), 0, s, S);
  }

  // all tiles in one launch, then the sums of the nodes they share (with
  // CONSTR and identity also the constrained rows)
  template <typename T, int VAR, bool ADD, bool CONSTR, unsigned PH>
  static int run_tiles(const lsmf_op *op, T *dst, const T *src, int identity, hipStream_t s,
                       const Epilogue<T> &ep = Epilogue<T>()) {
    if (op->ws_capture) (void)both_formulations(op, s);  // its owner's graph
    VmultParams<T> P = tile_params<T, VAR>(op);
    P.ep = ep;
    P.src = src;
    P.dst = dst;
    P.identity = identity;
    if (op->prof) op->prof->before(s);
    const int rc = launch_vmult<T, VAR, ADD, CONSTR, PH, LM_ONE>(op, P, P.cell_end, 1, s);
    if (rc) return rc;
    tile_sum<T, ADD, CONSTR>(op, dst, src, identity, s, ep);
    if (op->prof) op->prof->after(s);
    return 0;
  }

  // the cell kernels of one product: one launch over all tiles where the
  // stream may use the tile buffer, else one launch per colour.  *identity:
  // in, the constrained rows are wanted; out, they are still to be done
  // (rows of DoFs that no cell touches are done by the list either way)
  template <typename T, int VAR, bool ADD, bool CONSTR, unsigned PH>
  static int run_cells(const lsmf_op *op, T *dst, const T *src, bool *identity, hipStream_t s) {
    if (op->d_tile_buf) {
      const TileBufferLock lock(op, s);
      if (lock) {
        const int fold = identity && *identity && op->n_orphan == 0;
        if (fold) *identity = false;
        return run_tiles<T, VAR, ADD, CONSTR, PH>(op, dst, src, fold, s);
      }
    }
    return run_colours<T, VAR, ADD, CONSTR, PH>(op, dst, src, s);
  }

  // A product recorded in a caller's graph: the caller may switch the
  // formulation, cache and replay, so where the formulations take other kernels
  // both are recorded, in one launch or two, and on a replay the one whose values
  // are cached runs (*P.form).  The owner of a bound operator records its graphs anew instead.
  static constexpr size_t kRecordedBlocks = 256;  // one workgroup per CU: one launch for both (k_vmult_recorded)
  static bool both_formulations(const lsmf_op *op, hipStream_t s) {
    if (!op->d_form || !capturing(s)) return false;
    op->recorded = true;
    return !(op->ws_capture && s == op->ws_stream);
  }
  template <typename T, int VAR, bool ADD, bool CONSTR, unsigned PH>
  static int launch_recorded(const lsmf_op *op, VmultParams<T> P, int n, unsigned nv, hipStream_t s) {
    P.form = op->d_form;
    P.u = static_cast<const T *>(VAR == V_COMPACT_U ? op->d_uc : op->d_u);
    const unsigned blocks = op->tile_kind ? (unsigned)n : grid_for(n);
    if ((size_t)blocks * nv > kRecordedBlocks) {
      const int rc = launch_vmult<T, V_TENSOR4, ADD, CONSTR, PH, LM_RECORDED>(op, P, n, nv, s);
      return rc ? rc : launch_vmult<T, VAR, ADD, CONSTR, PH, LM_RECORDED>(op, P, n, nv, s);
    }
    if (op->tile_kind == kTileWide) {
      if constexpr (planes_ok<T, VAR>() || wide_ok<T, VAR>()) {
        hipLaunchKernelGGL((k_vmult_recorded<DIM, N, T, VAR, ADD, CONSTR, PH, kTileWide, planes_ok<T, VAR>()>),
                           dim3(blocks, nv), dim3(tile_threads<kTileWide>()), 0, s, P);
        return 0;
      }
    } else if constexpr (VAR != V_COMPACT_U) {
      if (op->tile_kind == 1) {
        if constexpr (!(DIM == 3 && (N == 5 || N == 3))) {  // tensor4 has wide tiles there
          hipLaunchKernelGGL((k_vmult_recorded<DIM, N, T, VAR, ADD, CONSTR, PH, 1, false>), dim3(blocks, nv), dim3(kWG),
                             0, s, P);
          return 0;
        }
      } else {
        hipLaunchKernelGGL((k_vmult_recorded<DIM, N, T, VAR, ADD, CONSTR, PH, 0, false>), dim3(blocks, nv), dim3(kWG), 0,
                           s, P);
        return 0;
      }
    }
    return LSMF_ERR_UNSUPPORTED;
  }
  // one colour's cell kernel, or with both the kernels of both formulations
  template <typename T, int VAR, bool ADD, bool CONSTR, unsigned PH>
  static int launch_colour(const lsmf_op *op, const VmultParams<T> &P, int n, unsigned nv, bool both, hipStream_t s) {
    if (!both) return launch_vmult<T, VAR, ADD, CONSTR, PH>(op, P, n, nv, s);
    if constexpr (VAR == V_TENSOR4 || VAR == V_COMPACT || VAR == V_COMPACT_AFFINE || VAR == V_COMPACT_U) {
      switch (compact_variant(op)) {
        case V_COMPACT: return launch_recorded<T, V_COMPACT, ADD, CONSTR, PH>(op, P, n, nv, s);
        case V_COMPACT_AFFINE: return launch_recorded<T, V_COMPACT_AFFINE, ADD, CONSTR, PH>(op, P, n, nv, s);
        default:
          if constexpr (recompute_ok() && sizeof(T) == 8)
            return launch_recorded<T, V_COMPACT_U, ADD, CONSTR, PH>(op, P, n, nv, s);
      }
    }
    return LSMF_ERR_UNSUPPORTED;
  }

  // one launch per colour; the tiled layout launches one workgroup per tile
  template <typename T, int VAR, bool ADD, bool CONSTR, unsigned PH>
  static int run_colours(const lsmf_op *op, T *dst, const T *src, hipStream_t s) {
    const int nc = n_colours(op);
    const bool both = both_formulations(op, s);
    for (int k = 0; k < nc; ++k) {
      VmultParams<T> P = params<T, VAR>(op, k);
      P.src = src;
      P.dst = dst;
      const int n = P.cell_end - P.cell_begin;
      if (n <= 0) continue;
      if (op->prof) op->prof->before(s);
      const int rc = launch_colour<T, VAR, ADD, CONSTR, PH>(op, P, n, 1, both, s);
      if (op->prof) op->prof->after(s);
      if (rc) return rc;
    }
    if (op->n_node_cons > 0) hang_gather<T, CONSTR>(op, dst, 0, 1, s);
    return 0;
  }

  template <typename T, int VAR>
  static int vmult_t(const lsmf_op *op, void *dst_, const void *src_, bool add, bool constr, unsigned ph,
                     hipStream_t s) {
    T *dst = static_cast<T *>(dst_);
    const T *src = static_cast<const T *>(src_);
    constexpr unsigned FULL = PH_SF | PH_QD;
    zero_if_constrained(op, dst, add, s);
    if (!add) zero_orphans(op, dst, s);
    int rc;
    if (constr) {
      bool identity = op->n_cons > 0;
      if (ph == FULL) {
        if (add) rc = run_cells<T, VAR, true, true, FULL>(op, dst, src, &identity, s);
        else rc = run_cells<T, VAR, false, true, FULL>(op, dst, src, &identity, s);
      } else if (ph == PH_SF) {
        rc = run_cells<T, VAR, false, true, PH_SF>(op, dst, src, &identity, s);
      } else {
        rc = run_cells<T, VAR, false, true, 0u>(op, dst, src, &identity, s);
      }
      if (identity)
        hipLaunchKernelGGL(k_constrained_identity<T>, dim3((op->n_cons + 255) / 256), dim3(256), 0, s, op->d_cons,
                           op->n_cons, src, dst, add ? 1 : 0);
    } else {
      if (add) rc = run_cells<T, VAR, true, false, FULL>(op, dst, src, nullptr, s);
      else rc = run_cells<T, VAR, false, false, FULL>(op, dst, src, nullptr, s);
    }
    if (rc) return rc;
    return hipGetLastError() == hipSuccess ? 0 : LSMF_ERR_HIP;
  }

  // a product with an epilogue, where it can run in one launch over all tiles
  // (*done; else nothing was launched)
  template <typename T, int VAR>
  static int smooth_t(const lsmf_op *op, const SmoothArgs &a, bool *done, hipStream_t s) {
    *done = false;
    if (op->n_orphan > 0) return 0;
    const TileBufferLock lock(op, s);
    if (!lock) return 0;
    *done = true;
    T *x = static_cast<T *>(a.x);
    const Epilogue<T> ep{a.kind, static_cast<const T *>(a.b), static_cast<const T *>(a.invd), static_cast<T *>(a.d), x,
                         T(a.f1), T(a.f2)};
    T *dst = a.kind == EP_RESIDUAL ? static_cast<T *>(a.dst) : x;
    const int rc = run_tiles<T, VAR, false, true, PH_SF | PH_QD>(op, dst, x, 1, s, ep);
    if (rc) return rc;
    return hipGetLastError() == hipSuccess ? 0 : LSMF_ERR_HIP;
  }
  static int smooth(const lsmf_op *op, const SmoothArgs &a, bool *done, hipStream_t s) {
    const bool f64 = op->precision == LSMF_FP64;
    *done = false;
    switch (cache_variant(op)) {
      case V_COMPACT_U:
        if constexpr (recompute_ok()) return smooth_t<double, V_COMPACT_U>(op, a, done, s);
        return 0;
      case V_COMPACT_AFFINE:
        return f64 ? smooth_t<double, V_COMPACT_AFFINE>(op, a, done, s)
                   : smooth_t<float, V_COMPACT_AFFINE>(op, a, done, s);
      case V_COMPACT:
        return f64 ? smooth_t<double, V_COMPACT>(op, a, done, s) : smooth_t<float, V_COMPACT>(op, a, done, s);
      case V_TENSOR4:
        return f64 ? smooth_t<double, V_TENSOR4>(op, a, done, s) : smooth_t<float, V_TENSOR4>(op, a, done, s);
      case V_TENSOR2:
        return f64 ? smooth_t<double, V_TENSOR2>(op, a, done, s) : smooth_t<float, V_TENSOR2>(op, a, done, s);
      case V_SCALAR:
        return f64 ? smooth_t<double, V_SCALAR>(op, a, done, s) : smooth_t<float, V_SCALAR>(op, a, done, s);
      default: return 0;
    }
  }

  // nvec products in set mode with constraints, vector b at b * n_dofs:
  // one launch per colour for all vectors (grid y = vector), the same code
  // path per vector as vmult_t
  template <typename T, int VAR> static int vmult_batched_t(const lsmf_op *op, T *dst, const T *src, int nvec,
                                                            hipStream_t s) {
    constexpr unsigned FULL = PH_SF | PH_QD;
    // grid y holds the vectors; with node constraints, as many as d_hbuf holds
    const int kMaxY = op->n_node_cons > 0 ? kHangBatch : 65535;
    const size_t n = op->n_dofs;
    const int nc = n_colours(op);
    const bool both = both_formulations(op, s);
    for (int v0 = 0; v0 < nvec; v0 += kMaxY) {
      const unsigned nv = (unsigned)std::min(nvec - v0, kMaxY);
      T *d = dst + (size_t)v0 * n;
      const T *x = src + (size_t)v0 * n;
      if (op->n_node_cons > 0)
        hipLaunchKernelGGL(k_zero<T>, dim3((unsigned)((nv * n + 255) / 256)), dim3(256), 0, s, d, nv * n);
      if (op->n_orphan > 0)
        hipLaunchKernelGGL(k_zero_list_batch<T>, dim3((op->n_orphan + 255) / 256, nv), dim3(256), 0, s,
                           op->d_orphan, op->n_orphan, d, n);
      for (int k = 0; k < nc; ++k) {
        VmultParams<T> P = params<T, VAR>(op, k);
        P.src = x;
        P.dst = d;
        P.vstride = n;
        const int nb = P.cell_end - P.cell_begin;
        if (nb <= 0) continue;
        const int rc = launch_colour<T, VAR, false, true, FULL>(op, P, nb, nv, both, s);
        if (rc) return rc;
      }
      if (op->n_node_cons > 0) hang_gather<T, true>(op, d, n, nv, s);
      if (op->n_cons > 0)
        hipLaunchKernelGGL(k_constrained_identity_batch<T>, dim3((op->n_cons + 255) / 256, nv), dim3(256), 0, s,
                           op->d_cons, op->n_cons, x, d, n);
    }
    return hipGetLastError() == hipSuccess ? 0 : LSMF_ERR_HIP;
  }

  static int vmult_batched(const lsmf_op *op, void *dst, const void *src, int nvec, hipStream_t s) {
    const bool f64 = op->precision == LSMF_FP64;
#define LSMF_BATCH(V)                                                                          \
  return f64 ? vmult_batched_t<double, V>(op, (double *)dst, (const double *)src, nvec, s) \
             : vmult_batched_t<float, V>(op, (float *)dst, (const float *)src, nvec, s)
    switch (cache_variant(op)) {
      case V_COMPACT: LSMF_BATCH(V_COMPACT);
      case V_COMPACT_AFFINE: LSMF_BATCH(V_COMPACT_AFFINE);
      case V_COMPACT_U:
        if constexpr (recompute_ok()) return vmult_batched_t<double, V_COMPACT_U>(op, (double *)dst, (const double *)src, nvec, s);
        return LSMF_ERR_UNSUPPORTED;
      case V_TENSOR4: LSMF_BATCH(V_TENSOR4);
      case V_TENSOR2: LSMF_BATCH(V_TENSOR2);
      case V_SCALAR: LSMF_BATCH(V_SCALAR);
      case V_TENSOR4_NS: LSMF_BATCH(V_TENSOR4_NS);
      case V_SCALAR_REF: LSMF_BATCH(V_SCALAR_REF);
      default:
        return fail(LSMF_ERR_UNKNOWN_CACHING, "vmult_batched: caching variant not available on the GPU");
    }
#undef LSMF_BATCH
  }

  static int vmult(const lsmf_op *op, void *dst, const void *src, bool add, bool constr, unsigned ph,
                   hipStream_t s) {
    const bool f64 = op->precision == LSMF_FP64;
    switch (cache_variant(op)) {
      case V_COMPACT:
        return f64 ? vmult_t<double, V_COMPACT>(op, dst, src, add, constr, ph, s)
                   : vmult_t<float, V_COMPACT>(op, dst, src, add, constr, ph, s);
      case V_COMPACT_U:
        if constexpr (recompute_ok()) return vmult_t<double, V_COMPACT_U>(op, dst, src, add, constr, ph, s);
        return LSMF_ERR_UNSUPPORTED;
      case V_COMPACT_AFFINE:
        return f64 ? vmult_t<double, V_COMPACT_AFFINE>(op, dst, src, add, constr, ph, s)
                   : vmult_t<float, V_COMPACT_AFFINE>(op, dst, src, add, constr, ph, s);
      case V_TENSOR4:
        return f64 ? vmult_t<double, V_TENSOR4>(op, dst, src, add, constr, ph, s)
                   : vmult_t<float, V_TENSOR4>(op, dst, src, add, constr, ph, s);
      case V_TENSOR2:
        return f64 ? vmult_t<double, V_TENSOR2>(op, dst, src, add, constr, ph, s)
                   : vmult_t<float, V_TENSOR2>(op, dst, src, add, constr, ph, s);
      case V_SCALAR:
        return f64 ? vmult_t<double, V_SCALAR>(op, dst, src, add, constr, ph, s)
                   : vmult_t<float, V_SCALAR>(op, dst, src, add, constr, ph, s);
      case V_TENSOR4_NS:
        return f64 ? vmult_t<double, V_TENSOR4_NS>(op, dst, src, add, constr, ph, s)
                   : vmult_t<float, V_TENSOR4_NS>(op, dst, src, add, constr, ph, s);
      case V_SCALAR_REF:
        return f64 ? vmult_t<double, V_SCALAR_REF>(op, dst, src, add, constr, ph, s)
                   : vmult_t<float, V_SCALAR_REF>(op, dst, src, add, constr, ph, s);
      default:
        return fail(LSMF_ERR_UNKNOWN_CACHING, "vmult: caching variant not available on the GPU");
    }
  }

  template <typename T, int VAR> static int cache_t(const lsmf_op *op, int *bad, hipStream_t s) {
    CacheParams P{};
    P.idx = op->d_idx;
    P.tab = op->d_tab64;
    P.u = op->d_u64;
    P.coords = op->d_coords;
    P.mu = op->d_mu64;
    P.lambda = op->d_lambda64;
    P.cache = op->d_cache;
    P.caff = op->d_caff;
    P.fs = op->field_stride;
    P.n_cells = op->n_cells;
    P.formulation = op->formulation;
    P.curved = op->curved;
    P.affine = op->affine;
    P.bad = bad;
    pack_sf<double>(op, P.sf);
    hipLaunchKernelGGL((k_cache<DIM, N, T, VAR>), dim3(grid_for(op->n_cells)), dim3(kWG), 0, s, P);
    return hipGetLastError() == hipSuccess ? 0 : LSMF_ERR_HIP;
  }

  static int cache(const lsmf_op *op, int *bad, hipStream_t s) {
    const bool f64 = op->precision == LSMF_FP64;
    switch (cache_variant(op)) {
      case V_COMPACT:
        return f64 ? cache_t<double, V_COMPACT>(op, bad, s) : cache_t<float, V_COMPACT>(op, bad, s);
      case V_COMPACT_U:
        if constexpr (recompute_ok()) {
          // the products read this copy: the next linearisation state may be
          // set while they run
          if (hipMemcpyAsync(op->d_uc, op->d_u64, op->n_dofs * sizeof(double), hipMemcpyDeviceToDevice, s) != hipSuccess)
            return LSMF_ERR_HIP;
          return cache_t<double, V_COMPACT_U>(op, bad, s);
        }
        return LSMF_ERR_UNSUPPORTED;
      case V_COMPACT_AFFINE:
        return f64 ? cache_t<double, V_COMPACT_AFFINE>(op, bad, s) : cache_t<float, V_COMPACT_AFFINE>(op, bad, s);
      case V_TENSOR4:
        return f64 ? cache_t<double, V_TENSOR4>(op, bad, s) : cache_t<float, V_TENSOR4>(op, bad, s);
      case V_TENSOR2:
        return f64 ? cache_t<double, V_TENSOR2>(op, bad, s) : cache_t<float, V_TENSOR2>(op, bad, s);
      case V_SCALAR:
        return f64 ? cache_t<double, V_SCALAR>(op, bad, s) : cache_t<float, V_SCALAR>(op, bad, s);
      case V_TENSOR4_NS:
        return f64 ? cache_t<double, V_TENSOR4_NS>(op, bad, s) : cache_t<float, V_TENSOR4_NS>(op, bad, s);
      case V_SCALAR_REF:
        return f64 ? cache_t<double, V_SCALAR_REF>(op, bad, s) : cache_t<float, V_SCALAR_REF>(op, bad, s);
      default:
        return fail(LSMF_ERR_UNKNOWN_CACHING, "cache: caching variant not available on the GPU");
    }
  }

  template <typename T, int VAR> static int diagonal_t(const lsmf_op *op, hipStream_t s) {
    // with node constraints every cell adds (no first-touch bits): start
    // from zero; cells with constrained nodes leave per-entry results that
    // the gather below adds per node
    if (op->n_node_cons > 0)
      hipLaunchKernelGGL(k_zero<T>, dim3((unsigned)((op->n_dofs + 255) / 256)), dim3(256), 0, s,
                         static_cast<T *>(op->d_diag), op->n_dofs);
    auto cells = [&](VmultParams<T> P, int n) {
      P.dst = static_cast<T *>(op->d_diag);
      // scalar_referential shares the scalar kernel but integrates on the Q1
      // vertex map on any mesh (include/mf_nh_operator.h:1255-1400)
      if (op->caching == LSMF_CACHING_SCALAR_REFERENTIAL) P.curved = 0;
      if (n <= 0) return 0;
      if (op->tile_kind == kTileWide) {
        if constexpr (wide_ok<T, VAR>() || planes_ok<T, VAR>())
          hipLaunchKernelGGL((k_diagonal_tiles<DIM, N, T, VAR, kTileWide>), dim3(n),
                             dim3(tile_threads<kTileWide>()), 0, s, P);
        else
          return (int)LSMF_ERR_UNSUPPORTED;
      } else if constexpr (VAR == V_COMPACT_U) {
        return (int)LSMF_ERR_UNSUPPORTED;
      } else if (op->tile_kind == 1) {
        hipLaunchKernelGGL((k_diagonal_tiles<DIM, N, T, VAR, 1>), dim3(n), dim3(kWG), 0, s, P);
      } else {
        hipLaunchKernelGGL((k_diagonal<DIM, N, T, VAR>), dim3(grid_for(n)), dim3(kWG), 0, s, P);
      }
      return 0;
    };
    int rc = 0;
    const TileBufferLock lock(op, s);
    if (lock) {
      const VmultParams<T> P = tile_params<T, VAR>(op);
      rc = cells(P, P.cell_end);
      if (!rc) tile_sum<T, false, true>(op, static_cast<T *>(op->d_diag), nullptr, 0, s);
    } else {
      for (int k = 0; k < n_colours(op) && !rc; ++k) {
        const VmultParams<T> P = params<T, VAR>(op, k);
        rc = cells(P, P.cell_end - P.cell_begin);
      }
    }
    if (rc) return rc;
    T *diag = static_cast<T *>(op->d_diag);
    if (op->n_diag_nodes > 0)
      hipLaunchKernelGGL((k_hang_gather<DIM, T, true>), dim3((op->n_diag_nodes + 255) / 256), dim3(256), 0, s, diag,
                         (size_t)0, static_cast<const T *>(op->d_dbuf), (size_t)0, op->d_dg_node, op->d_dg_ptr,
                         op->d_dg_ent, static_cast<const T *>(nullptr), op->n_diag_nodes);
    zero_orphans(op, diag, s);
    if (op->n_cons > 0)
      hipLaunchKernelGGL(k_set_one<T>, dim3((op->n_cons + 255) / 256), dim3(256), 0, s, op->d_cons, op->n_cons, diag);
    const size_t n = op->n_dofs;
    hipLaunchKernelGGL(k_zero<int>, dim3(1), dim3(64), 0, s, op->d_bad, (size_t)1);
    hipLaunchKernelGGL(k_invert<T>, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, diag,
                       static_cast<T *>(op->d_inv_diag), n, op->d_bad);
    return hipGetLastError() == hipSuccess ? 0 : LSMF_ERR_HIP;
  }


  static int diagonal(const lsmf_op *op, hipStream_t s) {
    const bool f64 = op->precision == LSMF_FP64;
    switch (cache_variant(op)) {
      case V_COMPACT:
        return f64 ? diagonal_t<double, V_COMPACT>(op, s) : diagonal_t<float, V_COMPACT>(op, s);
      case V_COMPACT_U:
        if constexpr (recompute_ok()) return diagonal_t<double, V_COMPACT_U>(op, s);
        return LSMF_ERR_UNSUPPORTED;
      case V_COMPACT_AFFINE:
        return f64 ? diagonal_t<double, V_COMPACT_AFFINE>(op, s) : diagonal_t<float, V_COMPACT_AFFINE>(op, s);
      case V_TENSOR4:
        return f64 ? diagonal_t<double, V_TENSOR4>(op, s) : diagonal_t<float, V_TENSOR4>(op, s);
      case V_TENSOR2:
        return f64 ? diagonal_t<double, V_TENSOR2>(op, s) : diagonal_t<float, V_TENSOR2>(op, s);
      case V_SCALAR:
      case V_SCALAR_REF:  // c is field 0 of both caches; F from u
        return f64 ? diagonal_t<double, V_SCALAR>(op, s) : diagonal_t<float, V_SCALAR>(op, s);
      case V_TENSOR4_NS:
        return f64 ? diagonal_t<double, V_TENSOR4_NS>(op, s) : diagonal_t<float, V_TENSOR4_NS>(op, s);
      default:
        return fail(LSMF_ERR_UNKNOWN_CACHING, "diagonal: caching variant not available on the GPU");
    }
  }

  static int residual(const lsmf_op *op, double *rhs, hipStream_t s) {
    if (op->precision != LSMF_FP64) return fail(LSMF_ERR_INVALID_ARGUMENT, "residual needs an FP64 operator");
    constexpr unsigned FULL = PH_SF | PH_QD;
    zero_if_constrained(op, rhs, false, s);
    zero_orphans(op, rhs, s);
    const int rc = run_cells<double, V_RESIDUAL, false, false, FULL>(op, rhs, nullptr, nullptr, s);
    if (rc) return rc;
    return hipGetLastError() == hipSuccess ? 0 : LSMF_ERR_HIP;
  }

  static int residual_vjp(const lsmf_op *op, double *du, const double *w, hipStream_t s) {
    if (op->precision != LSMF_FP64) return fail(LSMF_ERR_INVALID_ARGUMENT, "residual VJP needs an FP64 operator");
    constexpr unsigned FULL = PH_SF | PH_QD;
    zero_if_constrained(op, du, false, s);
    zero_orphans(op, du, s);
    const int rc = run_cells<double, V_ADJOINT, false, false, FULL>(op, du, w, nullptr, s);
    if (rc) return rc;
    return hipGetLastError() == hipSuccess ? 0 : LSMF_ERR_HIP;
  }

  static const LaunchTable *table() {
    static const LaunchTable t{&vmult, &vmult_batched, &smooth, &cache, &diagonal, &residual, &residual_vjp};
    return &t;
  }
};

}  // namespace lsmf

#define LSMF_INSTANTIATE(D, NN)                                                          \
  namespace lsmf {                                                                       \
  const LaunchTable *launch_table_##D##_##NN() { return Launch<D, NN>::table(); }        \
  }
