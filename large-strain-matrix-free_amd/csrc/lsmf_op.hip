// lsmf_op.hip -- C ABI of the operator (include/lsmf.h): creation,
// colouring, index tables, material, linearisation, cache, diagonal, vmult,
// residual.  Host logic only; kernels live in lsmf_kernels.hpp and are
// instantiated per (dim, N) in lsmf_inst_*.hip.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <array>
#include <cstring>
#include <limits>
#include <mutex>
#include <new>
#include <string>
#include <vector>

#include "lsmf.h"
#include "lsmf_error.hpp"
#include "lsmf_fe.hpp"
#include "lsmf_kernels.hpp"
#include "lsmf_op.hpp"

namespace lsmf {

std::string &last_error_string() {
  static thread_local std::string s;
  return s;
}

const LaunchTable *launch_table_2_2();
const LaunchTable *launch_table_2_3();
const LaunchTable *launch_table_2_5();
const LaunchTable *launch_table_3_2();
const LaunchTable *launch_table_3_3();
const LaunchTable *launch_table_3_5();

const LaunchTable *launch_table(int dim, int N) {
  if (dim == 2 && N == 2) return launch_table_2_2();
  if (dim == 2 && N == 3) return launch_table_2_3();
  if (dim == 2 && N == 5) return launch_table_2_5();
  if (dim == 3 && N == 2) return launch_table_3_2();
  if (dim == 3 && N == 3) return launch_table_3_3();
  if (dim == 3 && N == 5) return launch_table_3_5();
  return nullptr;
}

size_t elem_size(const lsmf_op *op) { return op->precision == LSMF_FP64 ? sizeof(double) : sizeof(float); }

// Tensor2 and tensor4 operators run the compact form of the same tangent
// where it exists: formulation 1 with the Q1 metric.  Curved meshes (Eulerian
// Q_p metric: K F is no longer J_ref^-1) and formulation 0 keep the stored
// tensors.
// K from the displacement instead of from memory (one cached value per point
// instead of ten), by the plane kernel: FP64 operators on wide Q2 tiles of affine
// cells, but for kFewTiles + 1 to kLineTiles of them.  Against the line kernel
// with K cached, us: 128^3 1500 / 1820, 64^3 249 / 282, 32^3 39.7 / 41.1.  FP32
// operators keep K, which is rounded once from FP64; from an FP32 displacement
// it would lose the digits of |u| / h.
static bool recompute_k(const lsmf_op *op) {
  return op->affine && op->precision == LSMF_FP64 && op->dim == 3 && op->N == 3 && op->tile_kind == kTileWide &&
         !op->few_tiles;
}
// Wide-tile operators of up to kFewPoints points keep all values of the compact
// form per point on affine cells too: their caches stay on the chip, and a load
// of the cell's constants more is what such short launches wait for.  Per point /
// per cell, us: 16^3 Q2 FP32 11.1 / 11.7 in one launch, 49.7 / 54 in coloured
// ones, 16^3 Q4 (512 k points) FP64 30.0 / 30.0 and 68.4 / 72.9, FP32 20.4 / 20.3
// and 53.5 / 59.7; 28^3 Q2 FP32 (593 k) 21.0 / 20.8, 32^3 Q4 FP64 216 / 200.
constexpr size_t kFewPoints = (size_t)1 << 19;
int compact_variant(const lsmf_op *op) {
  if (recompute_k(op)) return V_COMPACT_U;
  const bool few = op->tile_kind == kTileWide && op->field_stride <= kFewPoints;
  return op->affine && !few ? V_COMPACT_AFFINE : V_COMPACT;
}
int cache_variant(const lsmf_op *op) {
  switch (op->caching) {
    case LSMF_CACHING_TENSOR4:
    case LSMF_CACHING_TENSOR2:
      if (op->formulation == 1 && !op->curved) return compact_variant(op);
      return op->caching == LSMF_CACHING_TENSOR4 ? V_TENSOR4 : V_TENSOR2;
    case LSMF_CACHING_TENSOR4_NS: return V_TENSOR4_NS;
    case LSMF_CACHING_SCALAR: return V_SCALAR;
    case LSMF_CACHING_SCALAR_REFERENTIAL: return V_SCALAR_REF;
    default: return -1;
  }
}

int smooth(lsmf_op *op, const SmoothArgs &a, bool *done, hipStream_t s) {
  *done = false;
  if (!op->cached) return fail(LSMF_ERR_NOT_CACHED, "smooth: call cache() first");
  const int rc = launch_table(op->dim, op->N)->smooth(op, a, done, s);
  return rc ? fail(rc, "smooth: kernel launch failed") : LSMF_OK;
}

void bind_stream(lsmf_op *op, hipStream_t s) {
  op->ws_bound = true;
  op->ws_stream = s;
  op->ws_capture = true;
}

bool capturing(hipStream_t s) {
  hipStreamCaptureStatus st = hipStreamCaptureStatusNone;
  if (hipStreamIsCapturing(s, &st) == hipSuccess) return st != hipStreamCaptureStatusNone;
  (void)hipGetLastError();
  return true;  // the legacy stream while another one captures: launches fail too
}

TileBufferLock::TileBufferLock(const lsmf_op *op, hipStream_t s) {
  if (!op->d_tile_buf || s == hipStreamPerThread) return;  // that handle is a stream per thread
  if (!op->ws_capture && capturing(s)) return;  // a captured product may be replayed on any stream
  std::unique_lock<std::mutex> lock(op->ws_mu);
  if (!op->ws_bound) {
    op->ws_bound = true;
    op->ws_stream = s;
  }
  if (op->ws_stream == s) lock_ = std::move(lock);
}

namespace {
template <int DIM> int fields_of(int variant) {
  switch (variant) {
    case V_COMPACT: return CacheFields<DIM, V_COMPACT>::value;
    case V_COMPACT_AFFINE: return CacheFields<DIM, V_COMPACT_AFFINE>::value;
    case V_COMPACT_U: return CacheFields<DIM, V_COMPACT_U>::value;
    case V_TENSOR4: return CacheFields<DIM, V_TENSOR4>::value;
    case V_TENSOR2: return CacheFields<DIM, V_TENSOR2>::value;
    case V_TENSOR4_NS: return CacheFields<DIM, V_TENSOR4_NS>::value;
    case V_SCALAR: return CacheFields<DIM, V_SCALAR>::value;
    case V_SCALAR_REF: return CacheFields<DIM, V_SCALAR_REF>::value;
    default: return -1;
  }
}
int n_cache_fields(const lsmf_op *op) {
  return op->dim == 3 ? fields_of<3>(cache_variant(op)) : fields_of<2>(cache_variant(op));
}
}  // namespace

namespace {

#define LSMF_HIP_TRY(expr, what)                                                                   \
  do {                                                                                             \
    hipError_t e_ = (expr);                                                                        \
    if (e_ != hipSuccess)                                                                          \
      return fail(e_ == hipErrorOutOfMemory ? LSMF_ERR_OUT_OF_MEMORY : LSMF_ERR_HIP,               \
                  std::string(what) + ": " + hipGetErrorString(e_));                               \
  } while (0)

template <typename T> int dalloc(T **p, size_t n, const char *what) {
  *p = nullptr;
  if (n == 0) n = 1;
  hipError_t e = hipMalloc((void **)p, n * sizeof(T));
  if (e != hipSuccess) {
    *p = nullptr;
    return fail(e == hipErrorOutOfMemory ? LSMF_ERR_OUT_OF_MEMORY : LSMF_ERR_HIP,
                std::string("hipMalloc(") + what + "): " + hipGetErrorString(e));
  }
  return 0;
}

void free_op(lsmf_op *op) {
  void *ptrs[] = {op->d_form, op->d_cache_other, op->d_cgeo, op->d_uc,   op->d_idx,  op->d_coords,    op->d_tab,  op->d_tab64, op->d_mu64,     op->d_lambda64,
                  op->d_mu,   op->d_lambda,    op->d_cache, op->d_caff, op->d_diag, op->d_inv_diag, op->d_cons,
                  op->d_bad,  op->d_perm,      op->d_tile_nodes, op->d_tile_info, op->d_tile_tables,
                  op->d_tile_buf, op->d_ctile_copy, op->d_orphan, op->d_hang, op->d_hptr,
                  op->d_hmaster, op->d_hw, op->d_hcons, op->d_hg_node, op->d_hg_ptr, op->d_hg_inst, op->d_hg_w,
                  op->d_hbuf, op->d_dcell, op->d_deptr, op->d_dtptr, op->d_dta, op->d_dtw, op->d_dbuf,
                  op->d_dg_node, op->d_dg_ptr, op->d_dg_ent};
  for (void *p : ptrs)
    if (p) (void)hipFree(p);
  if (op->d_u64) (void)hipFree(op->d_u64);
  if (op->d_u && op->d_u != op->d_u64) (void)hipFree(op->d_u);
}

__global__ void k_zero_int(int *p) { *p = 0; }

// The lexicographic structured numbering of lsmf_mesh_create:
// node(ix, iy, iz) = ix + Nx (iy + Ny iz), cell (cx, cy, cz) = cx + nx (cy + ny cz),
// local node a = a0 + N (a1 + N a2) at (cx p + a0, cy p + a1, cz p + a2).
// Returns the cells per direction when cell_nodes is exactly that.
bool structured_dims(const lsmf_mesh_desc *m, int dim, int p, int nqp, long long n[3]) {
  const int N = p + 1;
  const int32_t *c0 = m->cell_nodes;
  if (c0[0] != 0 || c0[1] != 1) return false;
  const long long Nx = c0[N];
  if (Nx < N || (Nx - 1) % p) return false;
  long long Ny, Nz = 1;
  if (dim == 3) {
    const long long NxNy = c0[N * N];
    if (NxNy % Nx) return false;
    Ny = NxNy / Nx;
    if (m->n_nodes % (Nx * Ny)) return false;
    Nz = m->n_nodes / (Nx * Ny);
  } else {
    if (m->n_nodes % Nx) return false;
    Ny = m->n_nodes / Nx;
  }
  if ((Ny - 1) % p || (Nz - 1) % p || Ny < N || (dim == 3 && Nz < N)) return false;
  n[0] = (Nx - 1) / p;
  n[1] = (Ny - 1) / p;
  n[2] = dim == 3 ? (Nz - 1) / p : 1;
  if (n[0] * n[1] * n[2] != m->n_cells) return false;
  for (long long cz = 0; cz < n[2]; ++cz)
    for (long long cy = 0; cy < n[1]; ++cy)
      for (long long cx = 0; cx < n[0]; ++cx) {
        const int32_t *cn = c0 + (size_t)(cx + n[0] * (cy + n[1] * cz)) * nqp;
        for (int a = 0; a < nqp; ++a) {
          const int a0 = a % N, a1 = (a / N) % N, a2 = dim == 3 ? a / (N * N) : 0;
          if (cn[a] != (cx * p + a0) + Nx * ((cy * p + a1) + Ny * (cz * p + a2))) return false;
        }
      }
  return true;
}

// Cell grid of a logically structured mesh: cell_at[cx + n0 (cy + n1 cz)]
// is the mesh cell at grid position (cx, cy, cz), recovered from the cells'
// shared faces whatever the node and cell numbering (a box renumbered by
// deal.II's Cuthill-McKee, include/mf_elasticity.h:1610-1708, tiles like
// one in lsmf_mesh_create's lexicographic numbering, which is checked
// first without any search).  Every cell must be in standard orientation:
// the neighbour across local face +d has this cell across its local face
// -d.  Returns false for anything else (the cells layout then serves it).
bool cell_grid(const lsmf_mesh_desc *m, int dim, int p, int nqp, long long n[3], std::vector<int32_t> &cell_at) {
  const int nc = m->n_cells;
  if (structured_dims(m, dim, p, nqp, n)) {
    cell_at.resize(nc);
    for (int c = 0; c < nc; ++c) cell_at[c] = c;
    return true;
  }
  const int N = p + 1, nf = 2 * dim, ncorner = 1 << (dim - 1);
  // local index of corner k of face f = 2 d + s
  auto corner = [&](int f, int k) {
    const int d = f / 2, s = f % 2;
    int bits[3] = {0, 0, 0}, b = 0;
    for (int e = 0; e < dim; ++e) bits[e] = e == d ? s : (k >> b++) & 1;
    int a = 0, stride = 1;
    for (int e = 0; e < dim; ++e, stride *= N) a += bits[e] * p * stride;
    return a;
  };
  struct Face {
    int32_t v[4];
    int64_t id;  // cell * nf + face
  };
  std::vector<Face> faces((size_t)nc * nf);
  for (int c = 0; c < nc; ++c)
    for (int f = 0; f < nf; ++f) {
      Face &F = faces[(size_t)c * nf + f];
      F.v[2] = F.v[3] = -1;
      for (int k = 0; k < ncorner; ++k) F.v[k] = m->cell_nodes[(size_t)c * nqp + corner(f, k)];
      std::sort(F.v, F.v + ncorner);
      F.id = (int64_t)c * nf + f;
    }
  std::sort(faces.begin(), faces.end(), [](const Face &a, const Face &b) {
    return std::lexicographical_compare(a.v, a.v + 4, b.v, b.v + 4);
  });
  std::vector<int32_t> nbr((size_t)nc * nf, -1);
  for (size_t i = 0; i < faces.size();) {
    size_t j = i + 1;
    while (j < faces.size() && std::equal(faces[i].v, faces[i].v + 4, faces[j].v)) ++j;
    if (j - i > 2) return false;
    if (j - i == 2) {
      const int64_t a = faces[i].id, b = faces[i + 1].id;
      const int fa = (int)(a % nf), fb = (int)(b % nf);
      if ((fa ^ 1) != fb) return false;  // not face +d against face -d
      nbr[a] = (int32_t)(b / nf);
      nbr[b] = (int32_t)(a / nf);
    }
    i = j;
  }
  // the one cell without -x, -y, -z neighbours is the grid's origin
  int origin = -1;
  for (int c = 0; c < nc; ++c) {
    bool o = true;
    for (int d = 0; d < dim; ++d) o = o && nbr[(size_t)c * nf + 2 * d] < 0;
    if (o) {
      if (origin >= 0) return false;
      origin = c;
    }
  }
  if (origin < 0) return false;
  n[0] = n[1] = n[2] = 1;
  for (int d = 0; d < dim; ++d) {
    long long len = 1;
    for (int c = origin; nbr[(size_t)c * nf + 2 * d + 1] >= 0; c = nbr[(size_t)c * nf + 2 * d + 1])
      if (++len > nc) return false;
    n[d] = len;
  }
  if (n[0] * n[1] * n[2] != nc) return false;
  cell_at.assign(nc, -1);
  std::vector<uint8_t> seen(nc, 0);
  auto at = [&](long long x, long long y, long long z) -> int32_t & { return cell_at[x + n[0] * (y + n[1] * z)]; };
  for (long long z = 0; z < n[2]; ++z)
    for (long long y = 0; y < n[1]; ++y)
      for (long long x = 0; x < n[0]; ++x) {
        int32_t c = x > 0   ? nbr[(size_t)at(x - 1, y, z) * nf + 1]
                    : y > 0 ? nbr[(size_t)at(x, y - 1, z) * nf + 3]
                    : z > 0 ? nbr[(size_t)at(x, y, z - 1) * nf + 5]
                            : origin;
        if (c < 0 || seen[c]) return false;
        seen[c] = 1;
        at(x, y, z) = c;
      }
  // every face link agrees with the grid
  for (long long z = 0; z < n[2]; ++z)
    for (long long y = 0; y < n[1]; ++y)
      for (long long x = 0; x < n[0]; ++x) {
        const long long g[3] = {x, y, z};
        const int32_t c = at(x, y, z);
        for (int d = 0; d < dim; ++d)
          for (int s = 0; s < 2; ++s) {
            long long h[3] = {g[0], g[1], g[2]};
            h[d] += s ? 1 : -1;
            const int32_t expect = (h[d] < 0 || h[d] >= n[d]) ? -1 : at(h[0], h[1], h[2]);
            if (nbr[(size_t)c * nf + 2 * d + s] != expect) return false;
          }
      }
  return true;
}

// Some support point lies off its cell's Q1 (multi)linear map of the
// vertices (beyond round-off relative to the cell size): the current
// configuration then needs the Eulerian Q_p metric of all support points.
bool support_points_curved(const lsmf_mesh_desc *m, int dim, int p, int nqp) {
  const int N = p + 1, NV = 1 << dim;
  const std::vector<double> g = lobatto_points(p);
  std::vector<double> wq1((size_t)nqp * NV);  // Q1 weight of vertex v at support point a
  std::vector<int> corner(NV);
  for (int v = 0; v < NV; ++v) {
    int a = 0, stride = 1;
    for (int d = 0; d < dim; ++d) {
      a += ((v >> d) & 1) * p * stride;
      stride *= N;
    }
    corner[v] = a;
  }
  for (int a = 0; a < nqp; ++a) {
    int rem = a;
    double xi[3] = {0, 0, 0};
    for (int d = 0; d < dim; ++d) {
      xi[d] = g[rem % N];
      rem /= N;
    }
    for (int v = 0; v < NV; ++v) {
      double w = 1.0;
      for (int d = 0; d < dim; ++d) w *= ((v >> d) & 1) ? xi[d] : 1.0 - xi[d];
      wq1[(size_t)a * NV + v] = w;
    }
  }
  for (int c = 0; c < m->n_cells; ++c) {
    const int32_t *cn = m->cell_nodes + (size_t)c * nqp;
    double X[8][3], h = 0.0;
    for (int v = 0; v < NV; ++v)
      for (int i = 0; i < dim; ++i) {
        X[v][i] = m->coords[(size_t)cn[corner[v]] * dim + i];
        h = std::max(h, std::fabs(X[v][i] - X[0][i]));
      }
    for (int a = 0; a < nqp; ++a)
      for (int i = 0; i < dim; ++i) {
        double x = 0.0;
        for (int v = 0; v < NV; ++v) x += wq1[(size_t)a * NV + v] * X[v][i];
        if (std::fabs(x - m->coords[(size_t)cn[a] * dim + i]) > 1e-10 * h) return true;
      }
  }
  return false;
}

// Every cell's Q1 vertex map is affine to the rounding of its coordinates: the
// mixed differences of its vertices (xy, yz, zx, xyz) vanish, so J_ref is one
// matrix per cell.  The bound is a few units in the last place of the cell's
// own largest coordinate, what representing its vertices costs and what the
// weighted sums of q1_jacobian lose in any case; the extent of the mesh, or a
// node that no cell has, says nothing about a cell.
bool cells_affine(const lsmf_mesh_desc *m, int dim, int p, int nqp) {
  const int N = p + 1, NV = 1 << dim;
  int corner[8];
  for (int v = 0; v < NV; ++v) {
    int a = 0, stride = 1;
    for (int d = 0; d < dim; ++d, stride *= N) a += ((v >> d) & 1) * p * stride;
    corner[v] = a;
  }
  for (int c = 0; c < m->n_cells; ++c) {
    const int32_t *cn = m->cell_nodes + (size_t)c * nqp;
    const double *X[8];
    for (int v = 0; v < NV; ++v) X[v] = m->coords + (size_t)cn[corner[v]] * dim;
    // largest difference of a vertex from the affine map of vertex 0 and its
    // neighbours; NaN counts as one
    double off = 0.0;
    for (int i = 0; i < dim; ++i)
      for (int v = 3; v < NV; ++v) {
        double x = X[0][i];
        for (int d = 0; d < dim; ++d)
          if ((v >> d) & 1) x += X[1 << d][i] - X[0][i];
        const double e = std::fabs(x - X[v][i]);
        if (!(e <= off) && !std::isnan(off)) off = e;
      }
    if (off == 0.0) continue;
    double top = 0.0;
    for (int v = 0; v < NV; ++v)
      for (int i = 0; i < dim; ++i) top = std::max(top, std::fabs(X[v][i]));
    if (!(off <= 8.0 * std::numeric_limits<double>::epsilon() * top)) return false;
  }
  return true;
}

struct TileDims {
  int tx, ty, tz, nx, ny, nz, tn;
};
template <int D, int NN, int WG> TileDims tile_dims_of() {
  using TS = TileShape<D, NN, WG>;
  return {TS::TX, TS::TY, TS::TZ, TS::NX, TS::NY, TS::NZ, TS::TN};
}
bool tile_dims(int dim, int N, int kind, TileDims &t) {
  if (dim == 2 && N == 2) t = tile_dims_of<2, 2, kWG>();
  else if (dim == 2 && N == 3) t = tile_dims_of<2, 3, kWG>();
  else if (dim == 2 && N == 5) t = tile_dims_of<2, 5, kWG>();
  else if (dim == 3 && N == 2) t = tile_dims_of<3, 2, kWG>();
  else if (dim == 3 && N == 3 && kind == kTileWide) t = tile_dims_of<3, 3, 2 * kWG>();
  else if (dim == 3 && N == 3) t = tile_dims_of<3, 3, kWG>();
  else if (dim == 3 && N == 5 && kind == kTileWide) t = tile_dims_of<3, 5, 2 * kWG>();
  else if (dim == 3 && N == 5) t = tile_dims_of<3, 5, kWG>();
  else return false;
  return true;
}

// Tiles of a logically structured mesh (cell grid cell_at, n cells per
// direction), coloured by the parity of their position so that no two tiles of
// one colour share a node, in the order of the grid where products run in one
// launch and by colour elsewhere.  Fills perm (tile order, the cells of a tile
// consecutive in slot order), the tile node table (node ids from the cells'
// own node lists; first-touch bit: the node's first tile in colour order),
// tile info, and for products in one launch the tables by colour, the
// private-node bits and the shared nodes with their slots.  Returns
// kNotTileable when cells that share a tile node position disagree about its
// node (the cells layout then serves the mesh).
constexpr int kNotTileable = 1;
// Largest operator whose products run in one launch: above it the tiles'
// shares of common nodes travel to HBM and back and cost more than the
// coloured launches' starts and tails save.  One launch against 8 coloured
// ones, us: 3D Q2 tensor4 FP64 40 / 68 (32^3), 110 / 138 (48^3, 2.7 M DoF), 165 /
// 189 (56^3, 4.3 M), 250 / 246 (64^3, 6.4 M), 443 / 402 (80^3), 1889 / 1491
// (128^3); FP32 145 / 155 (64^3), 251 / 234 (80^3); scalar 128 / 154 (48^3), 301 /
// 285 (64^3); Q4 tensor4 FP32 51 / 75 (24^3, 2.7 M), 119 / 116 (32^3, 6.4 M), 222 /
// 204 (40^3), tensor2 FP64 77 / 107 and 180 / 197; 2D Q2 FP64 (4 colours) 52 / 60
// (2.1 M), 191 / 173 (8.4 M).
constexpr size_t kOneLaunchDofs = 4000000;
// FP64 products on affine Q2 cells of kFewTiles + 1 to kLineTiles wide tiles cache
// K and run the line kernel: there a launch lasts as long as one tile, and the
// plane kernel's tile (two evaluations, one wave per six cells) takes longer.
// Line / planes, us: 16^3 (256 tiles) 13.4 / 14.0 in one launch, 62 / 69 in
// coloured ones (64 with the stored tensors), 8^3 (32) 12.0 / 12.4 and 32.7 / 34.9;
// 20^3 (600) 20.8 / 19.8 and 62 / 68, 32^3 41.1 / 39.7.  Below, batches of unit
// vectors (coarse matrices) count: 4^3 (8 tiles), 2187 vectors, 253 / 211.
// FP32: the plane kernel at every size (16^3 11.8 / 11.7, 32^3 28 / 24.7).
constexpr int kFewTiles = 16, kLineTiles = 512;
struct TileTables {
  std::vector<uint32_t> nodes, priv, sum_node, sum_slot;
  std::vector<int32_t> info, cinfo, by_colour;  // the last two: products in one launch
};
int build_tiles(lsmf_op *op, const lsmf_mesh_desc *mesh, const long long n[3], const std::vector<int32_t> &cell_at,
                TileTables &tt) {
  const int dim = op->dim, p = op->degree, N = p + 1, nqp = op->nqp;
  TileDims td;
  if (!tile_dims(dim, op->N, op->tile_kind, td)) return fail(LSMF_ERR_UNSUPPORTED, "tiles: no tile shape");
  const long long TXn = (n[0] + td.tx - 1) / td.tx, TYn = (n[1] + td.ty - 1) / td.ty,
                  TZn = (n[2] + td.tz - 1) / td.tz;
  const long long n_tiles = TXn * TYn * TZn;
  const int n_col = 1 << dim, tw = (td.tn + 31) / 32;
  std::vector<uint8_t> tcol(n_tiles);
  for (long long b = 0; b < n_tiles; ++b)
    tcol[b] = (uint8_t)((b % TXn & 1) | ((b / TXn % TYn & 1) << 1) | ((b / (TXn * TYn) & 1) << 2));
  const bool one = op->n_dofs <= kOneLaunchDofs;
  std::vector<int32_t> by_colour;
  by_colour.reserve(n_tiles);
  op->tile_ptr.assign(n_col + 1, 0);
  for (int col = 0; col < n_col; ++col) {
    for (long long b = 0; b < n_tiles; ++b)
      if (tcol[b] == col) by_colour.push_back((int32_t)b);
    op->tile_ptr[col + 1] = (int)by_colour.size();
  }
  op->perm.assign(op->n_cells, 0);
  op->inv_perm.assign(op->n_cells, 0);
  tt.info.assign((size_t)n_tiles * 2, 0);
  tt.nodes.assign((size_t)n_tiles * td.tn, kNoNode);
  std::vector<uint8_t> cols(mesh->n_nodes, 0);  // colours of the tiles that touch a node
  // tile position l: (slot, local node) of the tile's cells that hold it
  std::vector<std::pair<int, int>> at;
  std::vector<int> at_ptr(1, 0);
  for (int l = 0; l < td.tn; ++l) {
    const int X = l % td.nx, Y = (l / td.nx) % td.ny, Z = l / (td.nx * td.ny);
    for (int sz = 0; sz < td.tz; ++sz)
      for (int sy = 0; sy < td.ty; ++sy)
        for (int sx = 0; sx < td.tx; ++sx) {
          const int x = X - sx * p, y = Y - sy * p, z = Z - sz * p;
          if (x >= 0 && x <= p && y >= 0 && y <= p && z >= 0 && z <= p)
            at.push_back({sx + td.tx * (sy + td.ty * sz), x + N * (y + N * z)});
        }
    at_ptr.push_back((int)at.size());
  }
  std::vector<const int32_t *> cell_nodes(td.tx * td.ty * td.tz);
  auto extents = [&](long long b, int e[3]) {
    e[0] = (int)std::min<long long>(td.tx, n[0] - b % TXn * td.tx);
    e[1] = (int)std::min<long long>(td.ty, n[1] - b / TXn % TYn * td.ty);
    e[2] = (int)std::min<long long>(td.tz, n[2] - b / (TXn * TYn) * td.tz);
  };
  // place of each tile in the tables, and its first cell in tile order; the walk
  // below is in the order of the grid, as the mesh lies in memory
  std::vector<int32_t> place(n_tiles);
  int pos = 0;
  for (long long i = 0; i < n_tiles; ++i) {
    const long long b = one ? i : by_colour[i];
    int e[3];
    extents(b, e);
    place[b] = (int32_t)i;
    tt.info[(size_t)i * 2] = pos;
    tt.info[(size_t)i * 2 + 1] = e[0] | (e[1] << 8) | (e[2] << 16);
    pos += e[0] * e[1] * e[2];
  }
  if (pos != op->n_cells) return fail(LSMF_ERR_INVALID_ARGUMENT, "tiles: cell count mismatch");
  for (long long b = 0; b < n_tiles; ++b) {
    const long long bx = b % TXn, by = (b / TXn) % TYn, bz = b / (TXn * TYn);
    int e[3];
    extents(b, e);
    const int ex = e[0], ey = e[1], ez = e[2];
    const size_t i = (size_t)place[b];
    pos = tt.info[i * 2];
    auto tile_cell = [&](int sx, int sy, int sz) {
      return cell_at[(bx * td.tx + sx) + n[0] * ((by * td.ty + sy) + n[1] * (bz * td.tz + sz))];
    };
    std::fill(cell_nodes.begin(), cell_nodes.end(), nullptr);
    for (int sz = 0; sz < ez; ++sz)
      for (int sy = 0; sy < ey; ++sy)
        for (int sx = 0; sx < ex; ++sx) {
          const int cell = tile_cell(sx, sy, sz);
          cell_nodes[sx + td.tx * (sy + td.ty * sz)] = mesh->cell_nodes + (size_t)cell * nqp;
          op->perm[pos] = cell;
          op->inv_perm[cell] = pos;
          ++pos;
        }
    for (int l = 0; l < td.tn; ++l) {
      // the node from every cell of the tile that holds this position (the
      // kernels sum those cells' contributions into it); none: beyond a
      // ragged tile
      long long node = -1;
      for (int k = at_ptr[l]; k < at_ptr[l + 1]; ++k) {
        const int32_t *cn = cell_nodes[at[k].first];
        if (!cn) continue;
        const long long nd = cn[at[k].second];
        if (node >= 0 && nd != node) return kNotTileable;
        node = nd;
      }
      if (node < 0) continue;
      if ((cols[node] >> tcol[b]) & 1u) return kNotTileable;  // two tiles of one colour share a node
      cols[node] |= (uint8_t)(1u << tcol[b]);
      tt.nodes[i * td.tn + l] = (uint32_t)node;
    }
  }
  auto cons_bits = [&](size_t node) {
    uint32_t bits = 0;
    if (mesh->constrained)
      for (int comp = 0; comp < dim; ++comp)
        if (mesh->constrained[node * dim + comp]) bits |= 1u << (kConsShift + comp);
    return bits;
  };
  if (!one) {
    for (long long b = 0; b < n_tiles; ++b)
      for (int l = 0; l < td.tn; ++l) {
        uint32_t &code = tt.nodes[(size_t)place[b] * td.tn + l];
        if (code == kNoNode) continue;
        const uint32_t node = code;
        code |= cons_bits(node);
        if (!(cols[node] & ((1u << tcol[b]) - 1u))) code |= kFirstBit;
      }
    return LSMF_OK;
  }
  // shared nodes by the number of tiles that touch them, in node order
  std::vector<uint32_t> where(mesh->n_nodes, 0);  // position within its group
  size_t count[9] = {};
  for (int node = 0; node < mesh->n_nodes; ++node) {
    const int m = __builtin_popcount(cols[node]);
    where[node] = (uint32_t)count[m]++;
  }
  int group[9] = {};
  size_t n_shared = 0, n_slots = 0;
  op->n_sum_groups = 0;
  for (int m = 2; m <= n_col; ++m) {
    if (count[m] == 0) continue;
    const int g = group[m] = op->n_sum_groups++;
    op->sum_begin[g] = (int)n_shared;
    op->sum_mult[g] = m;
    op->sum_first_slot[g] = n_slots;
    n_shared += count[m];
    n_slots += (size_t)m * count[m];
  }
  op->sum_begin[op->n_sum_groups] = (int)n_shared;
  tt.sum_node.resize(n_shared);
  tt.sum_slot.resize(n_slots);
  tt.priv.assign((size_t)n_tiles * tw, 0);
  for (long long b = 0; b < n_tiles; ++b)
    for (int l = 0; l < td.tn; ++l) {
      uint32_t &code = tt.nodes[(size_t)b * td.tn + l];
      if (code == kNoNode) continue;
      const uint32_t node = code, c = cols[node], below = c & ((1u << tcol[b]) - 1u);
      code |= cons_bits(node);
      const int m = __builtin_popcount(c);
      if (m == 1) {
        tt.priv[(size_t)b * tw + l / 32] |= 1u << (l % 32);
      } else {
        // this tile's place among the node's tiles, in colour order
        const int g = group[m], k = __builtin_popcount(below);
        if (k == 0) tt.sum_node[op->sum_begin[g] + where[node]] = code;
        tt.sum_slot[op->sum_first_slot[g] + (size_t)k * count[m] + where[node]] = (uint32_t)(b * td.tn + l);
      }
      if (!below) code |= kFirstBit;
    }
  tt.cinfo.reserve(tt.info.size());
  for (const int32_t b : by_colour) tt.cinfo.insert(tt.cinfo.end(), {tt.info[(size_t)b * 2], tt.info[(size_t)b * 2 + 1]});
  tt.by_colour = std::move(by_colour);
  return LSMF_OK;
}

__global__ void k_tiles_by_colour(uint32_t *__restrict__ out, const uint32_t *__restrict__ nodes,
                                  const uint32_t *__restrict__ tiles, int tn) {
  for (int l = threadIdx.x; l < tn; l += blockDim.x)
    out[(size_t)blockIdx.x * tn + l] = nodes[(size_t)tiles[blockIdx.x] * tn + l];
}
__global__ void k_set_form(lsmf::FormState *f, int formulation, const void *cache) {
  f->formulation = formulation;
  f->cache = (const __attribute__((address_space(1))) void *)cache;
}
__global__ void k_convert_f64_f32(const double *__restrict__ a, float *__restrict__ b, size_t n) {
  const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) b[i] = float(a[i]);
}

}  // namespace
}  // namespace lsmf

namespace lsmf {
namespace {
bool cell_constants(const lsmf_op *op) {
  return cache_variant(op) == V_COMPACT_AFFINE || cache_variant(op) == V_COMPACT_U;
}
// bytes of the cached values a product reads
size_t cache_bytes(const lsmf_op *op) {
  const size_t es = elem_size(op);
  return (size_t)op->n_fields * op->field_stride * es +
         (cell_constants(op) ? (size_t)op->n_cells * kAffineStride * sizeof(double) : 0) +
         (cache_variant(op) == V_COMPACT_U ? op->n_dofs * es : 0);
}

// cache(): zero the det F <= 0 counter bad_dev, run the cache kernel, read
// the count back (synchronising the stream)
lsmf_status cache_with_counter(lsmf_op *op, int *bad_dev, hipStream_t s, const char *what) {
  if (!op) return fail(LSMF_ERR_INVALID_ARGUMENT, std::string(what) + ": null operator");
  if (!op->material_set) return fail(LSMF_ERR_INVALID_ARGUMENT, std::string(what) + ": set_material was not called");
  if (!op->linearization_set)
    return fail(LSMF_ERR_INVALID_ARGUMENT, std::string(what) + ": set_linearization was not called");
  hipLaunchKernelGGL(k_zero_int, dim3(1), dim3(1), 0, s, bad_dev);
  int rc = launch_table(op->dim, op->N)->cache(op, bad_dev, s);
  if (rc) return fail(rc, std::string(what) + ": kernel launch failed");
  if (op->d_form && op->form_cache != op->d_cache) {
    hipLaunchKernelGGL(k_set_form, dim3(1), dim3(1), 0, s, op->d_form, op->formulation, (const void *)op->d_cache);
    LSMF_HIP_TRY(hipGetLastError(), "cache: formulation");
    op->form_cache = op->d_cache;
  }
  int bad = 0;
  LSMF_HIP_TRY(hipMemcpyAsync(&bad, bad_dev, sizeof(int), hipMemcpyDeviceToHost, s), "cache: read det F count");
  LSMF_HIP_TRY(hipStreamSynchronize(s), "cache: synchronize");
  if (bad > 0) {
    op->cached = false;
    return fail(LSMF_ERR_NONPOSITIVE_DET_F,
                "det_F is not positive at " + std::to_string(bad) + " quadrature points");
  }
  op->cached = true;
  op->diag_ok = false;
  return LSMF_OK;
}

// Scratch of lsmf_cache_noalloc: a file-scope device array (each GPU holds
// its own copy for the life of the process), reached through the device
// address hipGetSymbolAddress returns for the current device -- in host
// code the array's name is only a stand-in symbol.  kNoAllocScratchInts
// ints: [0] counts the quadrature points with det F <= 0.
constexpr int kNoAllocScratchInts = 64;
__device__ __align__(256) int scratch[kNoAllocScratchInts];

std::mutex g_scratch_mu;
std::vector<int *> g_scratch_ptr;  // per device ordinal, nullptr until looked up

lsmf_status scratch_for_current_device(int **out) {
  int dev = -1;
  LSMF_HIP_TRY(hipGetDevice(&dev), "cache_noalloc: current device");
  std::lock_guard<std::mutex> lock(g_scratch_mu);
  if ((int)g_scratch_ptr.size() <= dev) g_scratch_ptr.resize(dev + 1, nullptr);
  if (!g_scratch_ptr[dev]) {
    void *p = nullptr;
    LSMF_HIP_TRY(hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)), "cache_noalloc: scratch address");
    if (!p) return fail(LSMF_ERR_HIP, "cache_noalloc: null scratch address");
    g_scratch_ptr[dev] = static_cast<int *>(p);
  }
  *out = g_scratch_ptr[dev];
  return LSMF_OK;
}
}  // namespace
}  // namespace lsmf

using namespace lsmf;

extern "C" {

const char *lsmf_last_error(void) { return last_error_string().c_str(); }

lsmf_status lsmf_op_create(const lsmf_mesh_desc *mesh, const lsmf_op_options *opt, lsmf_op **out) {
  if (!mesh || !opt || !out) return fail(LSMF_ERR_INVALID_ARGUMENT, "lsmf_op_create: null argument");
  *out = nullptr;
  const int dim = mesh->dim, p = mesh->degree, nq = opt->n_q_1d;
  if (dim != 2 && dim != 3) return fail(LSMF_ERR_INVALID_ARGUMENT, "lsmf_op_create: dim must be 2 or 3");
  if (opt->precision != LSMF_FP64 && opt->precision != LSMF_FP32)
    return fail(LSMF_ERR_INVALID_ARGUMENT, "lsmf_op_create: unknown precision");
  if (opt->caching < LSMF_CACHING_SCALAR || opt->caching > LSMF_CACHING_SCALAR_REFERENTIAL)
    return fail(LSMF_ERR_UNKNOWN_CACHING, "Unknown caching");
  if (nq != p + 1 || !launch_table(dim, nq))
    return fail(LSMF_ERR_UNSUPPORTED, "lsmf_op_create: (dim, degree, n_q_1d) = (" + std::to_string(dim) + ", " +
                                          std::to_string(p) + ", " + std::to_string(nq) + ") is not instantiated");
  if (mesh->n_cells <= 0 || mesh->n_nodes <= 0 || !mesh->cell_nodes || !mesh->coords)
    return fail(LSMF_ERR_INVALID_ARGUMENT, "lsmf_op_create: empty mesh");
  if (mesh->n_nodes >= (1 << 28)) return fail(LSMF_ERR_INVALID_ARGUMENT, "lsmf_op_create: more than 2^28 nodes");
  const int N = nq;
  int nqp = 1;
  for (int d = 0; d < dim; ++d) nqp *= N;
  const int nc = mesh->n_cells;
  for (long long i = 0; i < (long long)nc * nqp; ++i)
    if (mesh->cell_nodes[i] < 0 || mesh->cell_nodes[i] >= mesh->n_nodes)
      return fail(LSMF_ERR_INVALID_ARGUMENT, "lsmf_op_create: cell_nodes entry out of range");

  lsmf_op *op = new (std::nothrow) lsmf_op;
  if (!op) return fail(LSMF_ERR_OUT_OF_MEMORY, "lsmf_op_create: host allocation");
  op->dim = dim;
  op->degree = p;
  op->nq = nq;
  op->N = N;
  op->nqp = nqp;
  op->precision = opt->precision;
  op->caching = opt->caching;
  op->n_cells = nc;
  op->n_nodes = mesh->n_nodes;
  op->n_dofs = (size_t)mesh->n_nodes * dim;
  op->field_stride = (size_t)nc * nqp;

  // --- node (hanging) constraints: validated, closed (masters are free)
  const int nnc = mesh->n_node_constraints;
  std::vector<int> hang_of;
  if (nnc < 0 || (nnc > 0 && (!mesh->nc_nodes || !mesh->nc_ptr || !mesh->nc_masters || !mesh->nc_weights))) {
    delete op;
    return fail(LSMF_ERR_INVALID_ARGUMENT, "lsmf_op_create: bad node constraint arrays");
  }
  if (nnc > 0) {
    hang_of.assign(mesh->n_nodes, -1);
    if (mesh->nc_ptr[0] != 0) {
      delete op;
      return fail(LSMF_ERR_INVALID_ARGUMENT, "lsmf_op_create: nc_ptr[0] must be 0");
    }
    for (int k = 0; k < nnc; ++k) {
      const int n = mesh->nc_nodes[k];
      if (n < 0 || n >= mesh->n_nodes || hang_of[n] >= 0 || mesh->nc_ptr[k + 1] < mesh->nc_ptr[k]) {
        delete op;
        return fail(LSMF_ERR_INVALID_ARGUMENT, "lsmf_op_create: bad constrained node or nc_ptr");
      }
      hang_of[n] = k;
      if (mesh->constrained)
        for (int c = 0; c < dim; ++c)
          if (mesh->constrained[(size_t)n * dim + c]) {
            delete op;
            return fail(LSMF_ERR_INVALID_ARGUMENT, "lsmf_op_create: a node is both constrained and Dirichlet");
          }
    }
    for (int j = 0; j < mesh->nc_ptr[nnc]; ++j) {
      const int m = mesh->nc_masters[j];
      if (m < 0 || m >= mesh->n_nodes || hang_of[m] >= 0) {
        delete op;
        return fail(LSMF_ERR_INVALID_ARGUMENT, "lsmf_op_create: masters must be unconstrained nodes");
      }
    }
  }
  op->n_node_cons = nnc;
  // nodes cell c writes in its colour: its own nodes (the masters of its
  // constrained ones receive their share after the colours)
  auto write_nodes = [&](int c, std::vector<int> &w) {
    w.clear();
    for (int a = 0; a < nqp; ++a) w.push_back(mesh->cell_nodes[(size_t)c * nqp + a]);
  };
  std::vector<int> wbuf;

  op->curved = p > 1 && support_points_curved(mesh, dim, p, nqp);
  op->affine = cells_affine(mesh, dim, p, nqp);
  // --- cell order of the tiled layout (structured meshes), else by colour;
  // the per-cell index table of tiles carries no first-touch bits
  TileTables tt;
  long long sn[3] = {1, 1, 1};
  std::vector<int32_t> cell_at;
  op->tiled = opt->layout == LSMF_LAYOUT_AUTO && nnc == 0 && cell_grid(mesh, dim, p, nqp, sn, cell_at);
  // wide (512-thread) tiles for 3D Q2 / Q4 tensor2 and tensor4 products
  op->tile_kind = !op->tiled ? 0
                  : (dim == 3 && (op->N == 5 || op->N == 3) &&
                     (op->caching == LSMF_CACHING_TENSOR2 || op->caching == LSMF_CACHING_TENSOR4))
                      ? kTileWide
                      : 1;
  if (op->tiled) {
    const int rc = build_tiles(op, mesh, sn, cell_at, tt);
    if (rc == kNotTileable) {  // the cells layout
      op->tiled = false;
      op->tile_kind = 0;
      op->tile_ptr.clear();
      op->n_sum_groups = 0;
      tt = TileTables();
    } else if (rc) {
      delete op;
      return rc;
    }
  }
  if (op->tiled && dim == 3 && N == 3 && op->tile_kind == kTileWide)
    op->few_tiles = op->tile_ptr.back() > kFewTiles && op->tile_ptr.back() <= kLineTiles;
  op->n_fields = n_cache_fields(op);
  // --- colouring (given and checked, or greedy first fit): no node is written
  // by two cells of one colour; used[n] = colours of the cells that write n.
  // Tiles need none, but a given one is checked for them too.
  const bool colouring = !op->tiled || mesh->cell_colour;
  std::vector<int> colour(colouring ? nc : 0, 0);
  std::vector<uint64_t> used(mesh->n_nodes, 0);
  for (int c = 0; c < nc; ++c) {
    write_nodes(c, wbuf);
    if (!colouring) {
      for (int n : wbuf) used[n] = 1;
      continue;
    }
    uint64_t m = 0;
    for (int n : wbuf) m |= used[n];
    int col = 0;
    if (mesh->cell_colour) {
      col = mesh->cell_colour[c];
      if (col < 0 || col > 63) {
        delete op;
        return fail(LSMF_ERR_INVALID_ARGUMENT, "lsmf_op_create: colour out of [0, 63]");
      }
      if ((m >> col) & 1ull) {
        delete op;
        return fail(LSMF_ERR_INVALID_ARGUMENT, "lsmf_op_create: two cells of one colour share a node");
      }
    } else {
      while (col < 64 && (m >> col) & 1ull) ++col;
      if (col == 64) {
        delete op;
        return fail(LSMF_ERR_INVALID_ARGUMENT, "lsmf_op_create: greedy colouring needs more than 64 colours");
      }
    }
    colour[c] = col;
    for (int n : wbuf) used[n] |= (1ull << col);
  }
  std::vector<int> min_col;
  if (!op->tiled) {
    min_col.assign(mesh->n_nodes, 1 << 30);
    for (int n = 0; n < mesh->n_nodes; ++n)
      if (used[n]) min_col[n] = __builtin_ctzll(used[n]);
    int n_col = 0;
    for (int c = 0; c < nc; ++c) n_col = std::max(n_col, colour[c] + 1);
    op->colour_ptr.assign(n_col + 1, 0);
    for (int c = 0; c < nc; ++c) op->colour_ptr[colour[c] + 1]++;
    for (int k = 0; k < n_col; ++k) op->colour_ptr[k + 1] += op->colour_ptr[k];
    op->perm.assign(nc, 0);
    op->inv_perm.assign(nc, 0);
    {
      std::vector<int> fill(op->colour_ptr.begin(), op->colour_ptr.end() - 1);
      for (int c = 0; c < nc; ++c) {
        const int pos = fill[colour[c]]++;
        op->perm[pos] = c;
        op->inv_perm[c] = pos;
      }
    }
  }
  // --- index table (sorted cells): node | constraint bits | first-touch bit
  std::vector<uint32_t> idx((size_t)nc * nqp);
  for (int c = 0; c < nc; ++c) {
    const int pos = op->inv_perm[c];
    for (int a = 0; a < nqp; ++a) {
      const int nd = mesh->cell_nodes[(size_t)c * nqp + a];
      uint32_t code = (uint32_t)nd;
      if (mesh->constrained)
        for (int comp = 0; comp < dim; ++comp)
          if (mesh->constrained[(size_t)nd * dim + comp]) code |= 1u << (kConsShift + comp);
      if (!op->tiled && nnc == 0 && colour[c] == min_col[nd]) code |= kFirstBit;
      idx[(size_t)pos * nqp + a] = code;
    }
  }
  std::vector<int32_t> cons;
  if (mesh->constrained)
    for (size_t i = 0; i < op->n_dofs; ++i)
      if (mesh->constrained[i]) cons.push_back((int32_t)i);
  // constrained nodes' rows act as identity, like Dirichlet rows
  for (int k = 0; k < nnc; ++k)
    for (int c = 0; c < dim; ++c) cons.push_back(mesh->nc_nodes[k] * dim + c);
  op->n_cons = (int)cons.size();
  // DoFs of nodes that no cell references: their rows are zero, and the
  // first-touch stores never write them
  std::vector<int32_t> orphan;
  for (int nd = 0; nd < mesh->n_nodes; ++nd)
    if (!used[nd])
      for (int c = 0; c < dim; ++c) orphan.push_back(nd * dim + c);
  op->n_orphan = (int)orphan.size();

  // --- node-constraint tables: instances and their masters (products), and
  // the per-entry tables of the closed-form diagonal
  std::vector<int32_t> hang_tab, hptr;
  std::vector<uint32_t> hmaster;
  std::vector<double> hw;
  std::vector<int32_t> dcell, deptr, dtptr, dta, dg_ptr, dg_ent, dent_node;
  std::vector<double> dtw;
  std::vector<uint32_t> dg_node;
  std::vector<int32_t> hcons, hg_ptr, hg_inst;
  std::vector<uint32_t> hg_node;
  std::vector<double> hg_w;
  if (nnc > 0) {
    // instances in sorted-cell order
    hang_tab.assign((size_t)nc * nqp, -1);
    for (int pos = 0; pos < nc; ++pos)
      for (int a = 0; a < nqp; ++a) {
        const int k = hang_of[mesh->cell_nodes[(size_t)op->perm[pos] * nqp + a]];
        if (k < 0) continue;
        hang_tab[(size_t)pos * nqp + a] = (int32_t)hcons.size();
        hcons.push_back(k);
      }
    hptr.assign(mesh->nc_ptr, mesh->nc_ptr + nnc + 1);
    for (int j = 0; j < mesh->nc_ptr[nnc]; ++j) {
      const int m = mesh->nc_masters[j];
      uint32_t code = (uint32_t)m;
      if (mesh->constrained)
        for (int c = 0; c < dim; ++c)
          if (mesh->constrained[(size_t)m * dim + c]) code |= 1u << (kConsShift + c);
      hmaster.push_back(code);
      hw.push_back(mesh->nc_weights[j]);
    }
    // per master: (instance, weight) in instance order
    std::vector<std::array<int64_t, 3>> ent;  // master, instance, constraint entry
    for (int i = 0; i < (int)hcons.size(); ++i)
      for (int j = mesh->nc_ptr[hcons[i]]; j < mesh->nc_ptr[hcons[i] + 1]; ++j)
        ent.push_back({mesh->nc_masters[j], i, j});
    std::sort(ent.begin(), ent.end());
    for (size_t e = 0; e < ent.size(); ++e) {
      if (e == 0 || ent[e][0] != ent[e - 1][0]) {
        hg_ptr.push_back((int32_t)e);
        hg_node.push_back(hmaster[ent[e][2]]);
      }
      hg_inst.push_back((int32_t)ent[e][1]);
      hg_w.push_back(hw[ent[e][2]]);
    }
    hg_ptr.push_back((int32_t)ent.size());
    op->n_hang_inst = (int)hcons.size();
    op->n_hang_masters = (int)hg_node.size();
    // closed-form diagonal: per cell with constrained nodes, one entry per
    // node it couples (first appearance over the local nodes), each the
    // weighted sum of local basis functions that is that node's constrained
    // basis function on the cell; then per node its entries
    dcell.assign(nc, -1);
    deptr.push_back(0);
    dtptr.push_back(0);
    std::vector<int> eg;                               // entry -> node
    std::vector<std::vector<std::pair<int, double>>> et;  // entry -> (local node, weight)
    for (int pos = 0; pos < nc; ++pos) {
      const int c = op->perm[pos];
      bool any = false;
      for (int a = 0; a < nqp && !any; ++a) any = hang_of[mesh->cell_nodes[(size_t)c * nqp + a]] >= 0;
      if (!any) continue;
      dcell[pos] = (int32_t)(deptr.size() - 1);
      eg.clear();
      et.clear();
      auto add = [&](int g, int a, double w) {
        size_t k = 0;
        while (k < eg.size() && eg[k] != g) ++k;
        if (k == eg.size()) {
          eg.push_back(g);
          et.emplace_back();
        }
        et[k].push_back({a, w});
      };
      for (int a = 0; a < nqp; ++a) {
        const int n = mesh->cell_nodes[(size_t)c * nqp + a];
        const int k = hang_of[n];
        if (k < 0) add(n, a, 1.0);
        else
          for (int j = mesh->nc_ptr[k]; j < mesh->nc_ptr[k + 1]; ++j) add(mesh->nc_masters[j], a, mesh->nc_weights[j]);
      }
      for (size_t k = 0; k < eg.size(); ++k) {
        dent_node.push_back(eg[k]);
        for (const auto &tw : et[k]) {
          dta.push_back(tw.first);
          dtw.push_back(tw.second);
        }
        dtptr.push_back((int32_t)dta.size());
      }
      deptr.push_back((int32_t)dent_node.size());
    }
    std::vector<std::pair<int, int>> ne;  // (node, entry)
    for (int e = 0; e < (int)dent_node.size(); ++e) ne.push_back({dent_node[e], e});
    std::sort(ne.begin(), ne.end());
    for (size_t k = 0; k < ne.size(); ++k) {
      if (k == 0 || ne[k].first != ne[k - 1].first) {
        const int m = ne[k].first;
        uint32_t code = (uint32_t)m;
        if (mesh->constrained)
          for (int c = 0; c < dim; ++c)
            if (mesh->constrained[(size_t)m * dim + c]) code |= 1u << (kConsShift + c);
        dg_ptr.push_back((int32_t)k);
        dg_node.push_back(code);
      }
      dg_ent.push_back(ne[k].second);
    }
    dg_ptr.push_back((int32_t)ne.size());
    op->n_diag_nodes = (int)dg_node.size();
  }

  // --- 1D tables: S, D, St, Dt, qp, qw, and the collocation derivative on
  // the Gauss points Dc[q][k] = l_k'(x_q) (l_k: Lagrange basis on the Gauss
  // points; scalar_referential)
  Tables1D t1;
  t1.init(p, nq);
  std::vector<double> tab(5 * N * N + 2 * N);
  for (int q = 0; q < N; ++q)
    for (int k = 0; k < N; ++k) tab[4 * N * N + 2 * N + q * N + k] = lagrange_derivative(t1.qpts, k, t1.qpts[q]);
  for (int q = 0; q < N; ++q)
    for (int a = 0; a < N; ++a) {
      tab[q * N + a] = t1.S[q * N + a];
      tab[N * N + q * N + a] = t1.D[q * N + a];
      tab[2 * N * N + a * N + q] = t1.S[q * N + a];
      tab[3 * N * N + a * N + q] = t1.D[q * N + a];
    }
  for (int q = 0; q < N; ++q) {
    tab[4 * N * N + q] = t1.qpts[q];
    tab[4 * N * N + N + q] = t1.qw[q];
  }
  for (int i = 0; i < 2 * N * N; ++i) op->h_sf[i] = tab[i];
  for (int k = 0; k < (N + 1) / 2; ++k) op->h_qw[k] = t1.qw[k];

  // affine cells' geometry: residual and VJP on wide Q2 tiles, scalar products
  // on the others
  std::vector<double> cgeo;
  const bool kin_geo = op->affine && op->precision == LSMF_FP64 && dim == 3 && N == 3 && op->tile_kind == kTileWide;
  if (kin_geo || (op->caching == LSMF_CACHING_SCALAR && op->tile_kind == 1 && dim == 3 && N == 3 && op->affine &&
                  !op->curved)) {
    cgeo.resize((size_t)nc * kAffineStride);
    int corner[8];
    for (int v = 0; v < 8; ++v) corner[v] = p * ((v & 1) + N * ((v >> 1 & 1) + N * (v >> 2 & 1)));
    for (int c = 0; c < nc; ++c) {
      const int pos = op->inv_perm[c];
      const int32_t *cn = mesh->cell_nodes + (size_t)c * nqp;
      double X[24], J[3][3], R[3][3];
      for (int v = 0; v < 8; ++v)
        for (int i = 0; i < 3; ++i) X[v * 3 + i] = mesh->coords[(size_t)cn[corner[v]] * 3 + i];
      affine_jacobian<3>(X, J);
      double *g = &cgeo[(size_t)pos * kAffineStride];
      g[0] = inverse<3>(J, R);
      for (int v = 0; v < 6; ++v) {
        const int i = voigt_first<3>(v), j = voigt_second<3>(v);
        g[1 + v] = g[0] * (R[i][0] * R[j][0] + R[i][1] * R[j][1] + R[i][2] * R[j][2]);
      }
      for (int i = 0; i < 3; ++i)
        for (int d = 0; d < 3; ++d) g[7 + 3 * i + d] = kin_geo ? R[i][d] : J[i][d];
    }
  }
  // the tables of products in one launch in one piece: info by colour, tiles by
  // colour, private bits, shared nodes, slots
  std::vector<uint32_t> tile_tables(tt.cinfo.begin(), tt.cinfo.end());
  tile_tables.insert(tile_tables.end(), tt.by_colour.begin(), tt.by_colour.end());
  for (const auto *v : {&tt.priv, &tt.sum_node, &tt.sum_slot}) tile_tables.insert(tile_tables.end(), v->begin(), v->end());

  const size_t es = elem_size(op);
  int rc = 0;
  if ((rc = dalloc(&op->d_idx, idx.size(), "index table")) ||
      (rc = dalloc(&op->d_coords, (size_t)mesh->n_nodes * dim, "coordinates")) ||
      (rc = dalloc(&op->d_tab64, tab.size(), "tables")) ||
      (rc = dalloc((char **)&op->d_tab, tab.size() * es, "tables")) ||
      (rc = dalloc(&op->d_mu64, (size_t)nc, "mu")) || (rc = dalloc(&op->d_lambda64, (size_t)nc, "lambda")) ||
      (rc = dalloc((char **)&op->d_mu, (size_t)nc * es, "mu")) ||
      (rc = dalloc((char **)&op->d_lambda, (size_t)nc * es, "lambda")) ||
      (rc = dalloc(&op->d_u64, op->n_dofs, "displacement")) ||
      (rc = dalloc((char **)&op->d_cache, (size_t)op->n_fields * op->field_stride * es, "cache")) ||
      (cache_variant(op) == V_COMPACT_U && (rc = dalloc((char **)&op->d_uc, op->n_dofs * es, "cached displacement"))) ||
      (!cgeo.empty() && (rc = dalloc(&op->d_cgeo, cgeo.size(), "cell geometry"))) ||
      (cell_constants(op) &&
       (rc = dalloc(&op->d_caff, (size_t)nc * kAffineStride, "cell constants"))) ||
      (op->caching == LSMF_CACHING_TENSOR4 && !op->curved && (rc = dalloc(&op->d_form, 1, "formulation"))) ||
      (rc = dalloc((char **)&op->d_diag, op->n_dofs * es, "diagonal")) ||
      (rc = dalloc((char **)&op->d_inv_diag, op->n_dofs * es, "inverse diagonal")) ||
      (rc = dalloc(&op->d_cons, cons.size(), "constrained list")) || (rc = dalloc(&op->d_bad, 1, "counter")) ||
      (rc = dalloc(&op->d_orphan, orphan.size(), "unreferenced DoFs")) ||
      (rc = dalloc(&op->d_perm, (size_t)nc, "cell permutation")) ||
      (rc = dalloc(&op->d_tile_nodes, tt.nodes.size(), "tile nodes")) ||
      (rc = dalloc(&op->d_tile_info, tt.info.size(), "tile info")) ||
      (rc = dalloc(&op->d_tile_tables, tile_tables.size(), "tile tables")) ||
      (!tt.by_colour.empty() && (rc = dalloc(&op->d_ctile_copy, tt.nodes.size(), "tile nodes by colour"))) ||
      (nnc > 0 && ((rc = dalloc(&op->d_hang, hang_tab.size(), "constraint table")) ||
                   (rc = dalloc(&op->d_hptr, hptr.size(), "constraint offsets")) ||
                   (rc = dalloc(&op->d_hmaster, hmaster.size(), "constraint masters")) ||
                   (rc = dalloc((char **)&op->d_hw, hw.size() * es, "constraint weights")) ||
                   (rc = dalloc(&op->d_hcons, hcons.size(), "constraint instances")) ||
                   (rc = dalloc(&op->d_hg_node, hg_node.size(), "master nodes")) ||
                   (rc = dalloc(&op->d_hg_ptr, hg_ptr.size(), "master offsets")) ||
                   (rc = dalloc(&op->d_hg_inst, hg_inst.size(), "master instances")) ||
                   (rc = dalloc((char **)&op->d_hg_w, hg_w.size() * es, "master weights")) ||
                   (rc = dalloc((char **)&op->d_hbuf, (size_t)kHangBatch * hcons.size() * dim * es,
                                "constrained-node results")) ||
                   (rc = dalloc(&op->d_dcell, dcell.size(), "diagonal cells")) ||
                   (rc = dalloc(&op->d_deptr, deptr.size(), "diagonal entries")) ||
                   (rc = dalloc(&op->d_dtptr, dtptr.size(), "diagonal terms")) ||
                   (rc = dalloc(&op->d_dta, dta.size(), "diagonal local nodes")) ||
                   (rc = dalloc((char **)&op->d_dtw, dtw.size() * es, "diagonal weights")) ||
                   (rc = dalloc((char **)&op->d_dbuf, dent_node.size() * dim * es, "diagonal entry results")) ||
                   (rc = dalloc(&op->d_dg_node, dg_node.size(), "diagonal nodes")) ||
                   (rc = dalloc(&op->d_dg_ptr, dg_ptr.size(), "diagonal node offsets")) ||
                   (rc = dalloc(&op->d_dg_ent, dg_ent.size(), "diagonal node entries"))))) {
    free_op(op);
    delete op;
    return rc;
  }
  if (op->precision == LSMF_FP64) op->d_u = op->d_u64;
  else if ((rc = dalloc((char **)&op->d_u, op->n_dofs * es, "displacement (fp32)"))) {
    free_op(op);
    delete op;
    return rc;
  }
  if (!tt.priv.empty()) {
    // without this memory the coloured launches serve every product
    const size_t bytes = tt.nodes.size() * dim * es;
    if (hipMalloc(&op->d_tile_buf, bytes) != hipSuccess) {
      (void)hipGetLastError();
      op->d_tile_buf = nullptr;
    } else {
      op->bytes_sum = bytes;
    }
  }
  op->bytes_sum += tile_tables.size() * sizeof(uint32_t);
  op->bytes_idx = idx.size() * sizeof(uint32_t);
  op->bytes_cache = cache_bytes(op);
  hipError_t e = hipSuccess;
  e = hipMemcpy(op->d_idx, idx.data(), idx.size() * sizeof(uint32_t), hipMemcpyHostToDevice);
  if (e == hipSuccess)
    e = hipMemcpy(op->d_coords, mesh->coords, (size_t)mesh->n_nodes * dim * sizeof(double), hipMemcpyHostToDevice);
  if (e == hipSuccess) e = hipMemcpy(op->d_tab64, tab.data(), tab.size() * sizeof(double), hipMemcpyHostToDevice);
  if (e == hipSuccess) {
    if (op->precision == LSMF_FP64) {
      e = hipMemcpy(op->d_tab, tab.data(), tab.size() * sizeof(double), hipMemcpyHostToDevice);
    } else {
      std::vector<float> tf(tab.begin(), tab.end());
      e = hipMemcpy(op->d_tab, tf.data(), tf.size() * sizeof(float), hipMemcpyHostToDevice);
    }
  }
  if (e == hipSuccess && !cons.empty())
    e = hipMemcpy(op->d_cons, cons.data(), cons.size() * sizeof(int32_t), hipMemcpyHostToDevice);
  if (e == hipSuccess && !orphan.empty())
    e = hipMemcpy(op->d_orphan, orphan.data(), orphan.size() * sizeof(int32_t), hipMemcpyHostToDevice);
  if (e == hipSuccess) e = hipMemcpy(op->d_perm, op->perm.data(), (size_t)nc * sizeof(int32_t), hipMemcpyHostToDevice);
  if (e == hipSuccess && !tt.nodes.empty())
    e = hipMemcpy(op->d_tile_nodes, tt.nodes.data(), tt.nodes.size() * sizeof(uint32_t), hipMemcpyHostToDevice);
  if (e == hipSuccess && !tt.info.empty())
    e = hipMemcpy(op->d_tile_info, tt.info.data(), tt.info.size() * sizeof(int32_t), hipMemcpyHostToDevice);
  if (e == hipSuccess && !cgeo.empty())
    e = hipMemcpy(op->d_cgeo, cgeo.data(), cgeo.size() * sizeof(double), hipMemcpyHostToDevice);
  op->bytes_idx += cgeo.size() * sizeof(double);
  op->d_ctile_nodes = op->d_tile_nodes;
  op->d_ctile_info = op->d_tile_info;
  if (e == hipSuccess && !tile_tables.empty()) {
    e = hipMemcpy(op->d_tile_tables, tile_tables.data(), tile_tables.size() * sizeof(uint32_t), hipMemcpyHostToDevice);
    op->d_ctile_info = reinterpret_cast<const int32_t *>(op->d_tile_tables);
    op->d_ctile_nodes = op->d_ctile_copy;
    const uint32_t *by_colour = op->d_tile_tables + tt.cinfo.size();
    op->d_tile_priv = by_colour + tt.by_colour.size();
    const size_t n_tiles = tt.by_colour.size(), tn = tt.nodes.size() / n_tiles;
    hipLaunchKernelGGL(k_tiles_by_colour, dim3((unsigned)n_tiles), dim3(256), 0, nullptr, op->d_ctile_copy,
                       op->d_tile_nodes, by_colour, (int)tn);
    if (e == hipSuccess) e = hipGetLastError();
    if (e == hipSuccess) e = hipStreamSynchronize(nullptr);  // products may start on any stream
    op->d_sum_node = op->d_tile_priv + tt.priv.size();
    op->d_sum_slot = op->d_sum_node + tt.sum_node.size();
  }
  if (e == hipSuccess && nnc > 0) {
    e = hipMemcpy(op->d_hang, hang_tab.data(), hang_tab.size() * sizeof(int32_t), hipMemcpyHostToDevice);
    if (e == hipSuccess) e = hipMemcpy(op->d_hptr, hptr.data(), hptr.size() * sizeof(int32_t), hipMemcpyHostToDevice);
    if (e == hipSuccess)
      e = hipMemcpy(op->d_hmaster, hmaster.data(), hmaster.size() * sizeof(uint32_t), hipMemcpyHostToDevice);
    if (e == hipSuccess) {
      if (op->precision == LSMF_FP64) {
        e = hipMemcpy(op->d_hw, hw.data(), hw.size() * sizeof(double), hipMemcpyHostToDevice);
      } else {
        std::vector<float> hf(hw.begin(), hw.end());
        e = hipMemcpy(op->d_hw, hf.data(), hf.size() * sizeof(float), hipMemcpyHostToDevice);
      }
    }
    if (e == hipSuccess && !hcons.empty())
      e = hipMemcpy(op->d_hcons, hcons.data(), hcons.size() * sizeof(int32_t), hipMemcpyHostToDevice);
    if (e == hipSuccess && !hg_node.empty())
      e = hipMemcpy(op->d_hg_node, hg_node.data(), hg_node.size() * sizeof(uint32_t), hipMemcpyHostToDevice);
    if (e == hipSuccess)
      e = hipMemcpy(op->d_hg_ptr, hg_ptr.data(), hg_ptr.size() * sizeof(int32_t), hipMemcpyHostToDevice);
    if (e == hipSuccess && !hg_inst.empty())
      e = hipMemcpy(op->d_hg_inst, hg_inst.data(), hg_inst.size() * sizeof(int32_t), hipMemcpyHostToDevice);
    if (e == hipSuccess && !hg_w.empty()) {
      if (op->precision == LSMF_FP64) {
        e = hipMemcpy(op->d_hg_w, hg_w.data(), hg_w.size() * sizeof(double), hipMemcpyHostToDevice);
      } else {
        std::vector<float> wf(hg_w.begin(), hg_w.end());
        e = hipMemcpy(op->d_hg_w, wf.data(), wf.size() * sizeof(float), hipMemcpyHostToDevice);
      }
    }
    auto up = [&](void *dst, const void *src, size_t bytes) {
      if (e == hipSuccess && bytes > 0) e = hipMemcpy(dst, src, bytes, hipMemcpyHostToDevice);
    };
    up(op->d_dcell, dcell.data(), dcell.size() * sizeof(int32_t));
    up(op->d_deptr, deptr.data(), deptr.size() * sizeof(int32_t));
    up(op->d_dtptr, dtptr.data(), dtptr.size() * sizeof(int32_t));
    up(op->d_dta, dta.data(), dta.size() * sizeof(int32_t));
    up(op->d_dg_node, dg_node.data(), dg_node.size() * sizeof(uint32_t));
    up(op->d_dg_ptr, dg_ptr.data(), dg_ptr.size() * sizeof(int32_t));
    up(op->d_dg_ent, dg_ent.data(), dg_ent.size() * sizeof(int32_t));
    if (op->precision == LSMF_FP64) {
      up(op->d_dtw, dtw.data(), dtw.size() * sizeof(double));
    } else {
      std::vector<float> wf(dtw.begin(), dtw.end());
      up(op->d_dtw, wf.data(), wf.size() * sizeof(float));
    }
  }
  op->bytes_idx += tt.nodes.size() * sizeof(uint32_t) + tt.info.size() * sizeof(int32_t);
  if (op->d_ctile_copy) op->bytes_sum += tt.nodes.size() * sizeof(uint32_t);
  if (e != hipSuccess) {
    free_op(op);
    delete op;
    return fail(LSMF_ERR_HIP, std::string("lsmf_op_create upload: ") + hipGetErrorString(e));
  }
  *out = op;
  return LSMF_OK;
}

lsmf_status lsmf_op_destroy(lsmf_op *op) {
  if (!op) return LSMF_OK;
  delete op->prof;
  free_op(op);
  delete op;
  return LSMF_OK;
}

lsmf_status lsmf_set_material_per_cell(lsmf_op *op, const double *mu, const double *lambda) {
  if (!op || !mu || !lambda) return fail(LSMF_ERR_INVALID_ARGUMENT, "set_material: null argument");
  const int nc = op->n_cells;
  std::vector<double> m(nc), l(nc);
  for (int c = 0; c < nc; ++c) {
    m[op->inv_perm[c]] = mu[c];
    l[op->inv_perm[c]] = lambda[c];
  }
  LSMF_HIP_TRY(hipMemcpy(op->d_mu64, m.data(), nc * sizeof(double), hipMemcpyHostToDevice), "set_material");
  LSMF_HIP_TRY(hipMemcpy(op->d_lambda64, l.data(), nc * sizeof(double), hipMemcpyHostToDevice), "set_material");
  if (op->precision == LSMF_FP64) {
    LSMF_HIP_TRY(hipMemcpy(op->d_mu, m.data(), nc * sizeof(double), hipMemcpyHostToDevice), "set_material");
    LSMF_HIP_TRY(hipMemcpy(op->d_lambda, l.data(), nc * sizeof(double), hipMemcpyHostToDevice), "set_material");
  } else {
    std::vector<float> mf(m.begin(), m.end()), lf(l.begin(), l.end());
    LSMF_HIP_TRY(hipMemcpy(op->d_mu, mf.data(), nc * sizeof(float), hipMemcpyHostToDevice), "set_material");
    LSMF_HIP_TRY(hipMemcpy(op->d_lambda, lf.data(), nc * sizeof(float), hipMemcpyHostToDevice), "set_material");
  }
  op->material_set = true;
  op->cached = false;
  op->diag_ok = false;
  return LSMF_OK;
}

lsmf_status lsmf_set_material_two(lsmf_op *op, const uint8_t *material_id, double mu0, double lambda0, double mu1,
                                  double lambda1) {
  if (!op || !material_id) return fail(LSMF_ERR_INVALID_ARGUMENT, "set_material: null argument");
  std::vector<double> m(op->n_cells), l(op->n_cells);
  for (int c = 0; c < op->n_cells; ++c) {
    m[c] = material_id[c] ? mu1 : mu0;
    l[c] = material_id[c] ? lambda1 : lambda0;
  }
  return lsmf_set_material_per_cell(op, m.data(), l.data());
}

lsmf_status lsmf_set_formulation(lsmf_op *op, int formulation) {
  if (!op) return fail(LSMF_ERR_INVALID_ARGUMENT, "set_formulation: null operator");
  if (formulation != 0 && formulation != 1)
    return fail(LSMF_ERR_INVALID_ARGUMENT, "set_formulation: Unknown material formulation");
  if (formulation == 0 && op->caching != LSMF_CACHING_SCALAR && op->caching != LSMF_CACHING_TENSOR4)
    return fail(LSMF_ERR_UNSUPPORTED, "set_formulation: formulation 0 needs scalar or tensor4 caching");
  op->cached = false;
  op->diag_ok = false;
  if (formulation == op->formulation) return LSMF_OK;
  // the cached values of the other formulation take another amount of memory;
  // the ones that a recorded product may still read stay
  const int before = op->formulation;
  op->formulation = formulation;
  const int nf = n_cache_fields(op);
  if (nf != op->n_fields) {
    const size_t es = elem_size(op);
    void *p = op->d_cache_other;
    op->d_cache_other = nullptr;
    const int rc = p ? 0 : dalloc((char **)&p, (size_t)nf * op->field_stride * es, "cache");
    if (rc) {
      op->formulation = before;
      return rc;
    }
    if (op->recorded) {
      op->d_cache_other = op->d_cache;
    } else {
      (void)hipFree(op->d_cache);
      op->form_cache = nullptr;  // its address may come back
    }
    op->d_cache = p;
    op->n_fields = nf;
  }
  ++op->form_changes;
  op->bytes_cache = cache_bytes(op);
  return LSMF_OK;
}

lsmf_status lsmf_set_linearization(lsmf_op *op, const double *u_dev, lsmf_stream stream) {
  if (!op || !u_dev) return fail(LSMF_ERR_INVALID_ARGUMENT, "set_linearization: null argument");
  hipStream_t s = (hipStream_t)stream;
  LSMF_HIP_TRY(hipMemcpyAsync(op->d_u64, u_dev, op->n_dofs * sizeof(double), hipMemcpyDeviceToDevice, s),
               "set_linearization");
  if (op->precision == LSMF_FP32) {
    hipLaunchKernelGGL(k_convert_f64_f32, dim3((unsigned)((op->n_dofs + 255) / 256)), dim3(256), 0, s, op->d_u64,
                       (float *)op->d_u, op->n_dofs);
    LSMF_HIP_TRY(hipGetLastError(), "set_linearization convert");
  }
  op->linearization_set = true;
  op->cached = false;
  op->diag_ok = false;
  return LSMF_OK;
}

lsmf_status lsmf_cache(lsmf_op *op, lsmf_stream stream) {
  if (!op) return fail(LSMF_ERR_INVALID_ARGUMENT, "cache: null operator");
  return cache_with_counter(op, op->d_bad, (hipStream_t)stream, "cache");
}

lsmf_status lsmf_cache_noalloc(lsmf_op *op, lsmf_stream stream) {
  int *scr = nullptr;
  const lsmf_status st = scratch_for_current_device(&scr);
  if (st != LSMF_OK) return st;
  return cache_with_counter(op, scr, (hipStream_t)stream, "cache_noalloc");
}

lsmf_status lsmf_compute_diagonal(lsmf_op *op, lsmf_stream stream) {
  if (!op) return fail(LSMF_ERR_INVALID_ARGUMENT, "compute_diagonal: null operator");
  if (!op->cached) return fail(LSMF_ERR_NOT_CACHED, "compute_diagonal: call cache() first");
  hipStream_t s = (hipStream_t)stream;
  int rc = launch_table(op->dim, op->N)->diagonal(op, s);
  if (rc) return fail(rc, "compute_diagonal: kernel launch failed");
  // entries <= 0 other than the zero rows of unreferenced DoFs
  int bad = 0;
  LSMF_HIP_TRY(hipMemcpyAsync(&bad, op->d_bad, sizeof(int), hipMemcpyDeviceToHost, s),
               "compute_diagonal: read the non-positive count");
  LSMF_HIP_TRY(hipStreamSynchronize(s), "compute_diagonal: synchronize");
  bad -= op->n_orphan;
  if (bad > 0) {
    op->diag_ok = false;
    return fail(LSMF_ERR_NONPOSITIVE_DIAGONAL, "No diagonal entry in a positive definite operator should be zero or "
                                               "negative: " + std::to_string(bad) + " entries");
  }
  op->diag_ok = true;
  return LSMF_OK;
}

lsmf_status lsmf_vmult(lsmf_op *op, void *dst, const void *src, int add, unsigned mask, lsmf_stream stream) {
  if (!op || !dst || !src) return fail(LSMF_ERR_INVALID_ARGUMENT, "vmult: null argument");
  if (dst == src) return fail(LSMF_ERR_INVALID_ARGUMENT, "vmult: dst and src alias");
  if (!op->cached) return fail(LSMF_ERR_NOT_CACHED, "vmult: call cache() first");
  const bool plain = (mask & LSMF_MASK_PLAIN) != 0;
  if (!plain && !(mask & LSMF_MASK_RW)) {
    // no read/write phase: the reference's cell loop neither reads src nor
    // writes dst, and the constrained rows get nothing (:703-705 is under RW)
    if (!add) {
      const size_t bytes = op->n_dofs * elem_size(op);
      hipLaunchKernelGGL(k_zero<unsigned char>, dim3((unsigned)((bytes + 255) / 256)), dim3(256), 0,
                         (hipStream_t)stream, static_cast<unsigned char *>(dst), bytes);
      LSMF_HIP_TRY(hipGetLastError(), "vmult: zero");
    }
    return LSMF_OK;
  }
  unsigned ph = mask & (LSMF_MASK_SF | LSMF_MASK_QD);
  if (!(ph & LSMF_MASK_SF)) ph = 0;  // no sum factorization: gather/scatter only
  if (plain || add) ph = LSMF_MASK_SF | LSMF_MASK_QD;
  const int rc = launch_table(op->dim, op->N)->vmult(op, dst, src, add != 0, !plain, ph, (hipStream_t)stream);
  if (rc) return fail(rc, "vmult: kernel launch failed");
  return LSMF_OK;
}

lsmf_status lsmf_vmult_batched(lsmf_op *op, void *dst, const void *src, int n_vectors, lsmf_stream stream) {
  if (!op || !dst || !src) return fail(LSMF_ERR_INVALID_ARGUMENT, "vmult_batched: null argument");
  if (n_vectors <= 0) return fail(LSMF_ERR_INVALID_ARGUMENT, "vmult_batched: n_vectors must be positive");
  const size_t bytes = (size_t)n_vectors * op->n_dofs * (op->precision == LSMF_FP64 ? 8 : 4);
  const char *d = static_cast<const char *>(dst), *x = static_cast<const char *>(src);
  if (d < x + bytes && x < d + bytes) return fail(LSMF_ERR_INVALID_ARGUMENT, "vmult_batched: dst and src overlap");
  if (!op->cached) return fail(LSMF_ERR_NOT_CACHED, "vmult_batched: call cache() first");
  const int rc = launch_table(op->dim, op->N)->vmult_batched(op, dst, src, n_vectors, (hipStream_t)stream);
  if (rc) return fail(rc, "vmult_batched: kernel launch failed");
  return LSMF_OK;
}

lsmf_status lsmf_get_diagonal(lsmf_op *op, const void **diag_dev, const void **inv_diag_dev) {
  if (!op) return fail(LSMF_ERR_INVALID_ARGUMENT, "get_diagonal: null operator");
  if (!op->diag_ok) return fail(LSMF_ERR_NOT_CACHED, "get_diagonal: call compute_diagonal() first");
  if (diag_dev) *diag_dev = op->d_diag;
  if (inv_diag_dev) *inv_diag_dev = op->d_inv_diag;
  return LSMF_OK;
}

lsmf_status lsmf_precondition_jacobi(lsmf_op *op, void *dst, const void *src, double omega, lsmf_stream stream) {
  if (!op || !dst || !src) return fail(LSMF_ERR_INVALID_ARGUMENT, "precondition_Jacobi: null argument");
  if (!op->diag_ok) return fail(LSMF_ERR_NOT_CACHED, "precondition_Jacobi: call compute_diagonal() first");
  hipStream_t s = (hipStream_t)stream;
  const unsigned g = (unsigned)((op->n_dofs + 255) / 256);
  if (op->precision == LSMF_FP64)
    hipLaunchKernelGGL(k_scale_mul<double>, dim3(g), dim3(256), 0, s, (double *)dst, (const double *)src,
                       (const double *)op->d_inv_diag, omega, op->n_dofs);
  else
    hipLaunchKernelGGL(k_scale_mul<float>, dim3(g), dim3(256), 0, s, (float *)dst, (const float *)src,
                       (const float *)op->d_inv_diag, (float)omega, op->n_dofs);
  LSMF_HIP_TRY(hipGetLastError(), "precondition_Jacobi");
  return LSMF_OK;
}

size_t lsmf_op_size(const lsmf_op *op) { return op ? op->n_dofs : 0; }

size_t lsmf_memory_consumption(const lsmf_op *op) {
  if (!op) return 0;
  const size_t es = elem_size(op);
  size_t b = op->bytes_cache + op->bytes_idx + op->bytes_sum + 2 * (size_t)op->n_cells * es;
  if (op->caching == LSMF_CACHING_SCALAR || op->caching == LSMF_CACHING_SCALAR_REFERENTIAL)
    b += op->n_dofs * es + (size_t)op->n_nodes * op->dim * sizeof(double);
  return b;
}

lsmf_status lsmf_profile_enable(lsmf_op *op, int enable) {
  if (!op) return fail(LSMF_ERR_INVALID_ARGUMENT, "profile_enable: null operator");
  if (!op->prof) op->prof = new (std::nothrow) Profiler;
  if (!op->prof) return fail(LSMF_ERR_OUT_OF_MEMORY, "profile_enable: host allocation");
  op->prof->on = enable != 0;
  op->prof->used = 0;
  return LSMF_OK;
}

lsmf_status lsmf_profile_read(lsmf_op *op, double *total_ms, int *n_launches) {
  if (!op || !total_ms || !n_launches) return fail(LSMF_ERR_INVALID_ARGUMENT, "profile_read: null argument");
  *total_ms = 0.0;
  *n_launches = 0;
  if (!op->prof) return LSMF_OK;
  LSMF_HIP_TRY(hipDeviceSynchronize(), "profile_read: synchronize");
  double sum = 0.0;
  for (size_t i = 0; i < op->prof->used; ++i) {
    float ms = 0.f;
    LSMF_HIP_TRY(hipEventElapsedTime(&ms, op->prof->start[i], op->prof->stop[i]), "profile_read: elapsed");
    sum += ms;
  }
  *total_ms = sum;
  *n_launches = (int)op->prof->used;
  op->prof->used = 0;
  return LSMF_OK;
}

lsmf_status lsmf_residual_vjp(lsmf_op *op, const double *w_dev, double *du_dev, double *dmu, double *dlambda,
                              lsmf_stream stream) {
  if (!op || !w_dev || !du_dev || !dmu || !dlambda) return fail(LSMF_ERR_INVALID_ARGUMENT, "residual_vjp: null argument");
  if (op->precision != LSMF_FP64) return fail(LSMF_ERR_INVALID_ARGUMENT, "residual_vjp: operator must be FP64");
  if ((const void *)w_dev == (const void *)du_dev) return fail(LSMF_ERR_INVALID_ARGUMENT, "residual_vjp: w and du alias");
  if (!op->material_set || !op->linearization_set)
    return fail(LSMF_ERR_INVALID_ARGUMENT, "residual_vjp: material and linearisation must be set");
  if (op->formulation != 1) return fail(LSMF_ERR_UNSUPPORTED, "residual_vjp: formulation 1 only");
  op->adj_dmu = dmu;
  op->adj_dlambda = dlambda;
  const int rc = launch_table(op->dim, op->N)->residual_vjp(op, du_dev, w_dev, (hipStream_t)stream);
  op->adj_dmu = op->adj_dlambda = nullptr;
  if (rc) return fail(rc, "residual_vjp: kernel launch failed");
  return LSMF_OK;
}

lsmf_status lsmf_residual(lsmf_op *op, double *rhs_dev, lsmf_stream stream) {
  if (!op || !rhs_dev) return fail(LSMF_ERR_INVALID_ARGUMENT, "residual: null argument");
  if (op->precision != LSMF_FP64) return fail(LSMF_ERR_INVALID_ARGUMENT, "residual: operator must be FP64");
  if (!op->material_set || !op->linearization_set)
    return fail(LSMF_ERR_INVALID_ARGUMENT, "residual: material and linearisation must be set");
  const int rc = launch_table(op->dim, op->N)->residual(op, rhs_dev, (hipStream_t)stream);
  if (rc) return fail(rc, "residual: kernel launch failed");
  return LSMF_OK;
}

}  // extern "C"
