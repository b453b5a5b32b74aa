// lsmf_op.hpp -- the operator object behind the opaque lsmf_op handle, and
// the per-(dim, N) launch table the instantiation units fill in.
#pragma once

#include <hip/hip_runtime.h>

#include <atomic>
#include <cstdint>
#include <mutex>
#include <string>
#include <vector>

#include "lsmf.h"

namespace lsmf {
// per-launch event timing of the operator's cell kernels (the reference's
// TimerOutput / LIKWID regions around vmult, include/mf_nh_operator.h:108-119)
struct Profiler {
  bool on = false;
  std::vector<hipEvent_t> start, stop;
  size_t used = 0;
  void before(hipStream_t s) {
    if (!on) return;
    if (used == start.size()) {
      hipEvent_t a, b;
      if (hipEventCreate(&a) != hipSuccess) return;
      if (hipEventCreate(&b) != hipSuccess) {
        (void)hipEventDestroy(a);
        return;
      }
      start.push_back(a);
      stop.push_back(b);
    }
    (void)hipEventRecord(start[used], s);
  }
  void after(hipStream_t s) {
    if (!on || used >= start.size()) return;
    (void)hipEventRecord(stop[used], s);
    ++used;
  }
  ~Profiler() {
    for (auto e : start) (void)hipEventDestroy(e);
    for (auto e : stop) (void)hipEventDestroy(e);
  }
};
}  // namespace lsmf

// vectors per k_hang_gather pass of a batched product (the size of d_hbuf)
constexpr int kHangBatch = 8;

namespace lsmf {
struct FormState;  // lsmf_kernels.hpp
}

struct lsmf_op {
  lsmf::Profiler *prof = nullptr;
  // shape
  int dim = 0, degree = 0, nq = 0, N = 0, nqp = 0;
  int precision = LSMF_FP64, caching = LSMF_CACHING_TENSOR4;
  int formulation = 1;  // material formulation (include/material.h:82-94)
  bool curved = false;  // some support point off its cell's Q1 map: Eulerian Q_p current metric
  bool affine = false;  // every cell's Q1 map is affine: one J_ref per cell
  int n_cells = 0, n_nodes = 0;
  size_t n_dofs = 0;
  int n_fields = 0;
  size_t field_stride = 0;
  // colouring (host): sorted cells [colour_ptr[k], colour_ptr[k+1])
  std::vector<int> colour_ptr;
  std::vector<int> perm;      // sorted position -> mesh cell
  std::vector<int> inv_perm;  // mesh cell -> sorted position
  // device data
  uint32_t *d_idx = nullptr;        // [n_cells][nqp] node | constraint bits | first-touch bit
  double *d_coords = nullptr;       // [n_nodes][dim]
  void *d_tab = nullptr;            // S, D, St, Dt, qp, qw in operator precision
  double *d_tab64 = nullptr;        // same tables in FP64 (cache kernel)
  double h_sf[2 * 25] = {};         // S[q][k] then D[q][k] (N x N each), kernel-argument copy
  double h_qw[3] = {};              // 1D quadrature weights, the first half
  double *d_mu64 = nullptr, *d_lambda64 = nullptr;  // per sorted cell
  void *d_mu = nullptr, *d_lambda = nullptr;        // operator precision
  double *d_u64 = nullptr;          // linearisation state copy
  void *d_u = nullptr;              // operator precision copy (scalar variant)
  void *d_cache = nullptr;
  // tensor4 operators whose formulations keep different cached values: a product
  // recorded in a caller's graph launches the kernels of both, and a replay runs
  // the one that d_form names.  From the first recorded product on, each
  // formulation keeps its own memory (d_cache_other: the one not in use)
  lsmf::FormState *d_form = nullptr;
  void *d_cache_other = nullptr;
  const void *form_cache = nullptr;  // *d_form as last written (nullptr: never)
  int form_changes = 0;
  mutable std::atomic<bool> recorded{false};
  double *d_caff = nullptr;         // affine compact form: [sorted cell][kAffineStride]
  void *d_uc = nullptr;             // u of the last cache() where the products recompute K from it
  double *d_cgeo = nullptr;         // affine cells' geometry (VmultParams::cgeo), where the residual uses it
  void *d_diag = nullptr, *d_inv_diag = nullptr;
  int32_t *d_cons = nullptr;        // constrained DoF list
  int n_cons = 0;
  int32_t *d_orphan = nullptr;      // DoFs of nodes that no cell references (zero rows)
  int n_orphan = 0;
  int *d_bad = nullptr;
  int32_t *d_perm = nullptr;        // sorted position -> mesh cell
  double *adj_dmu = nullptr, *adj_dlambda = nullptr;  // outputs of the running residual VJP
  // tiled layout (structured meshes): each tile's cells are consecutive sorted
  // cells.  Operators whose products run in one launch over all tiles order
  // them by the grid (x fastest), and coloured launches have their own tables,
  // by colour: a list of tiles to look up would put one more load at the head
  // of every launch (0.3 us of 6 to 8).  The others have the order by colour
  // alone.  Tiles of colour k are entries [tile_ptr[k], tile_ptr[k+1])
  bool tiled = false;
  int tile_kind = 0;  // TILE argument of the cell kernels: 0 cells, 1 tiles, 2 wide tiles
  bool few_tiles = false;  // 3D Q2, kFewTiles + 1 to kLineTiles wide tiles (lsmf_op.hip)
  std::vector<int> tile_ptr;
  uint32_t *d_tile_nodes = nullptr;  // [n_tiles][TN] node | constraint bits | first-touch bit, or kNoNode
  int32_t *d_tile_info = nullptr;    // [n_tiles][2] first sorted cell, extents ex | ey << 8 | ez << 16
  uint32_t *d_tile_tables = nullptr;  // the memory of the tables below
  uint32_t *d_ctile_copy = nullptr;         // memory of d_ctile_nodes where it is not d_tile_nodes
  const uint32_t *d_ctile_nodes = nullptr;  // the same two by colour
  const int32_t *d_ctile_info = nullptr;
  // products in one launch over all tiles (k_vmult, k_tile_sum):
  // private-node bits, the shared nodes and their slots, and the tiles' shares
  // of them (d_tile_buf: nullptr when its memory could not be had)
  const uint32_t *d_tile_priv = nullptr, *d_sum_node = nullptr, *d_sum_slot = nullptr;
  void *d_tile_buf = nullptr;
  int n_sum_groups = 0;
  int sum_begin[9] = {}, sum_mult[8] = {};
  size_t sum_first_slot[8] = {};
  size_t bytes_sum = 0;
  // d_tile_buf serves one stream: the first that asks for it, or the one the
  // operator's owner binds (bind_stream); calls on any other stream, and
  // captured ones unless the owner allows them, take the coloured launches,
  // which share nothing.  The mutex keeps the two launches of a product
  // together when threads share the stream.
  mutable std::mutex ws_mu;
  mutable bool ws_bound = false;
  mutable hipStream_t ws_stream = nullptr;
  bool ws_capture = false;
  // node (hanging) constraints: cells layout, all-add scatter after a zero
  // pass.  Instances
  // (cell, constrained node) leave their results in d_hbuf; the masters
  // gather them after the colours (d_hg_*: per master its instances and
  // weights, in instance order), so masters do not enter the cell colouring.
  int n_node_cons = 0;
  int32_t *d_hang = nullptr, *d_hptr = nullptr, *d_hcons = nullptr;
  uint32_t *d_hmaster = nullptr;
  void *d_hw = nullptr;
  int n_hang_inst = 0, n_hang_masters = 0;
  uint32_t *d_hg_node = nullptr;  // master node | its Dirichlet bits
  int32_t *d_hg_ptr = nullptr, *d_hg_inst = nullptr;
  void *d_hg_w = nullptr;
  void *d_hbuf = nullptr;  // kHangBatch vectors of n_hang_inst * dim values
  // closed-form diagonal with node constraints (VmultParams::dcell ...):
  // cells with constrained nodes evaluate one entry per node they couple;
  // d_dg_*: per node its entries, in entry order, for the gather
  int32_t *d_dcell = nullptr, *d_deptr = nullptr, *d_dtptr = nullptr, *d_dta = nullptr;
  void *d_dtw = nullptr, *d_dbuf = nullptr;
  int n_diag_nodes = 0;
  uint32_t *d_dg_node = nullptr;
  int32_t *d_dg_ptr = nullptr, *d_dg_ent = nullptr;
  bool material_set = false, linearization_set = false, cached = false, diag_ok = false;
  size_t bytes_idx = 0, bytes_cache = 0;
};

namespace lsmf {

size_t elem_size(const lsmf_op *op);

// The owner of an operator that runs it on one stream only, its graphs
// included, gives it d_tile_buf on that stream, captured or not.
void bind_stream(lsmf_op *op, hipStream_t s);

// Holds d_tile_buf for the launches of one call on stream s, if it may.
class TileBufferLock {
 public:
  TileBufferLock(const lsmf_op *op, hipStream_t s);
  explicit operator bool() const { return lock_.owns_lock(); }

 private:
  std::unique_lock<std::mutex> lock_;
};

// A product A x with a vector update in the operator's precision (EpilogueKind
// of lsmf_kernels.hpp): kind 1: dst = b - A x; kinds 2, 3: the Chebyshev step on
// x and d.  *done false: not available for this operator (too large, another
// stream's), nothing was launched.
struct SmoothArgs {
  int kind;
  void *dst, *x;
  const void *b, *invd;
  void *d;
  double f1, f2;
};
int smooth(lsmf_op *op, const SmoothArgs &a, bool *done, hipStream_t s);

// launch entry points of one (dim, N) instantiation unit
struct LaunchTable {
  int (*vmult)(const lsmf_op *, void *dst, const void *src, bool add, bool constr, unsigned ph, hipStream_t);
  int (*vmult_batched)(const lsmf_op *, void *dst, const void *src, int nvec, hipStream_t);
  int (*smooth)(const lsmf_op *, const SmoothArgs &, bool *done, hipStream_t);
  int (*cache)(const lsmf_op *, int *bad, hipStream_t);  // bad: det F <= 0 counter (zeroed by the caller)
  int (*diagonal)(const lsmf_op *, hipStream_t);
  int (*residual)(const lsmf_op *, double *rhs, hipStream_t);
  int (*residual_vjp)(const lsmf_op *, double *du, const double *w, hipStream_t);
};

const LaunchTable *launch_table(int dim, int N);
// the Variant whose cached values the operator's products read
int cache_variant(const lsmf_op *op);
// the same for tensor2 / tensor4 operators with the Q1 metric in formulation 1
int compact_variant(const lsmf_op *op);
// work submitted to s now goes into a graph
bool capturing(hipStream_t s);

}  // namespace lsmf
