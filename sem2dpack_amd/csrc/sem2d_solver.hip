// sem2d_solver.hip -- C ABI (include/sem2d.h) of the MI355X explicit SEM time step.
//
// Host side: owns the device buffers of one problem and one HIP stream, builds
// the element colour schedule, and launches the per-step kernel sequence of
// solve_Newmark (SRC/solver.f90:42-84):
//   predictor -> element forces (one launch per colour) -> sources -> absorbing
//   boundaries (in BC order) -> fault -> a = f*rmass + corrector -> receiver and
//   fault records.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstdarg>
#include <cstdio>
#include <cstring>
#include <cstdlib>
#include <map>
#include <mutex>
#include <unordered_map>
#include <string>
#include <vector>

#include "sem2d.h"
#include "sem2d_fault.hpp"
#include "sem2d_kernels.hpp"
#include "sem2d_tile.hpp"

using namespace sem2d;

namespace {

struct DevBuf {
  void* p = nullptr;
  size_t bytes = 0;
};

struct AbsoDev {
  int n;
  int* node;
  double* C;
  // Stacey (P-SV): boundary elements, their edge points' global nodes [nbe][NG] and K
  // [nbe][NG][2]; per boundary node the contributions e*NG+k (element order) soff/sidx
  int nbe = 0;
  int *enode = nullptr, *soff = nullptr, *sidx = nullptr;
  bool ends = false;  // the end nodes take both ends' contributions (sem2d_set_abso_periodic)
  double* K = nullptr;
  double* nrm = nullptr;  // [2][n] node normals of a boundary that is not flat (general path)
  // incident plane wave (general path): node coordinates [2][n], unit-amplitude Vin and
  // Tin [ndof][n], weights B [n]
  double *wxz = nullptr, *wV = nullptr, *wT = nullptr, *wB = nullptr;
  WavePar wp = {};
};

struct AbsoHost {
  std::vector<int> node;   // 0-based reference nodes
  std::vector<double> C;   // [ndof][n]
  std::vector<int> senode;  // Stacey: [nbe][NG] boundary-local node of each edge point
  std::vector<double> sK;   // [nbe][NG][2]
  std::vector<double> nrm;  // [2][n] node normals of a boundary that is not flat
};

// Structured-mesh fast path (node-grid field order, fused tile kernel)
struct StructState {
  bool on = false;
  int ready = 0;  // 1: the tables of the step kernels are there; -1: the general path has none
  int nx = 0, nz = 0, ezflt = 0, NX1 = 0, NZ1 = 0;
  int ROW = 0;                    // storage slots per node row (4*TX per tile column)
  std::vector<int> gmap;          // reference node (0-based) -> storage index
  std::vector<int> gridx;         // reference node (0-based) -> grid index Z*NX1 + X
  int nvl = 0;                    // vertical tile-edge lines (stored column-contiguous)
  size_t NS = 0;                  // field component stride: ROW*NZ1 + nvl*NZ1
  std::vector<int4> tiles;
  int ntiles = 0;
  int pipe_wgs = 0;  // persistent workgroups of the tile kernel (0: one per tile)
  // Kelvin-Voigt eta and 2.5D coefficient per element point, cell order [cell][25] (bulk
  // type), or null; either makes the tile kernel form d + eta v at the element points
  void *eta = nullptr, *b25 = nullptr;
  int4* tiles_dev = nullptr;
  int4* grids_dev = nullptr;
  bool w32 = false;  // field, partial-force and per-cell arrays below 4 GiB per component
  // Stacey terms: boundary elements (storage-index edge nodes, K), per absorbing entry
  // of the deferred nodes the element points it subtracts, and their values per step
  int s_nbe = 0;
  int *s_enode = nullptr, *ak_off = nullptr, *ak_idx = nullptr;
  double *s_K = nullptr, *kxd = nullptr;
  int* spec_cnt = nullptr;
  int* spec_idx = nullptr;
  int* mark_of = nullptr;  // recorded nodes inside tiles (TileArgs)
  uint32_t* marks = nullptr;
  RecOut rec;   // receivers at nodes, recorded by k_deferred
  FaultOut fo;  // fault outputs, made by k_deferred
  void* fpart = nullptr;
  size_t FPS = 0;
  DefTable defs;
  const DefDev* fdef = nullptr;  // entries of the fault pairs' nodes, [side][pair]
  DefDev* gen_def = nullptr;  // general path: the records of defs
  int ndef = 0;
  int* part_off = nullptr;
  SrcEntry* dsrc = nullptr;
  double *dabso = nullptr, *dabson = nullptr;
  void* rmdef = nullptr;
  void* rmass0 = nullptr;
  void *coefs = nullptr, *geom = nullptr;  // cell-ordered per-element arrays
  // compact moduli once per node in the field layout ([ndof][NS], bulk type), when every
  // element sharing a node holds the same values there (COEF_NODE tile kernel)
  void* nodemod = nullptr;
  // ... once per element in cell order ([cell][ndof]), when all its points hold the same
  // (COEF_ELEM)
  void* elemmod = nullptr;
  // k_run_steps: neighbours of the tiles, deferred node of each partial force, the second
  // array of partial forces, flags and count, whether a launch has given up; run_ok: 0 not
  // asked yet, 1 the grid's tiles are resident together, -1 not so or not a run's grid;
  // launches kept and given up so far
  int *nbr = nullptr, *slot_def = nullptr, *run_fail = nullptr;
  unsigned *run_flag = nullptr, *run_count = nullptr;
  void* fpart2 = nullptr;
  unsigned epoch = 0;
  int run_ok = -1, runs_taken = 0, runs_given_up = 0;
  std::vector<void*> prep_allocs;  // freed when the deferred tables are rebuilt
  std::vector<int> cell_elem;      // cell (iz*nx + ix) -> element (0-based)
  std::vector<int> def_ref;        // deferred node -> reference node (0-based)
};

struct FaultHost {
  bool on = false;
  FaultDev dev;
  std::vector<void*> allocs;
  int oit, oitd, oix1, oixn, oixd, nout, nsamp, taken;
  double* rec;  // device [nsamp][6][nout]
  double* srec = nullptr;  // osides: device [nsamp][4*ndof][nout] (d, v of each side)
  double* pot = nullptr;  // device [pot_cap][2*(ndof+1)] potency rows, one per step from it = 0
  int pot_rows = 0, pot_cap = 0;
};

}  // namespace

struct AdjState;
void adj_free(AdjState* A);

struct sem2d_solver {
  int ndof, nelem, npoin, nelast, coef_mode, fp32;
  size_t fstride = 0;  // component stride of the device field arrays
  double dt, beta, gamma;
  int leapfrog = 0;  // 1: central-difference scheme (SRC/solver.f90:140-160)
  int hht = 0;       // 1: HHT-alpha (SRC/solver.f90:89-131): forces at d, v of n + alpha
  double alpha = 1.0;
  void *da = nullptr, *va = nullptr;  // the fields at n + alpha (bulk type)
  int ng = NG, np = NP;     // NGLL and GLL points per element
  double* hg = nullptr;     // h'_i(x_j) at hg[i*ng+j] (general element kernel, Stacey)
  hipStream_t stream = nullptr;
  hipEvent_t ev0 = nullptr, ev1 = nullptr;
  // bulk arrays (type R = double or float, stored as raw bytes)
  void *d = nullptr, *v = nullptr, *a = nullptr, *rmass = nullptr, *coefs = nullptr, *geom = nullptr;
  int* ibool = nullptr;  // colour-sorted, 0-based
  std::vector<int> colour_start;  // ncolour+1 offsets into the sorted order
  std::vector<int> elem_order;    // sorted position -> original element (0-based)
  // Dirichlet boundaries (BC_DIRNEU 'D' components), in registration order
  struct DirBC {
    std::vector<int> node;  // 0-based reference nodes
    int comp = 0;           // bit c: component c set to zero
    bool after_fault = false;
    int* node_dev = nullptr;
  };
  std::vector<DirBC> dirs;
  // boundaries and sources
  std::vector<AbsoDev> abso;
  std::vector<AbsoHost> abso_host;
  std::vector<double> rmass_host;          // [ndof][npoin], reference order
  std::vector<int> fault_n1, fault_n2;     // 0-based reference nodes
  StructState st;
  std::vector<SrcEntry> src_host;
  std::vector<std::vector<double>> stf;
  int nsrc = 0;
  SrcEntry* src_dev = nullptr;
  double* ampl_dev = nullptr;
  int ampl_nt = 0;
  bool src_dirty = false;
  // receivers
  int nrec = 0, isamp = 1, field = 1, nsamp = 0, taken = 0;
  std::vector<int> rec_ref;      // reference nodes that are recorded (0-based)
  int* rec_node = nullptr;       // [nrec] node, or [nrec][25] element nodes when interpolated
  double* rec_w = nullptr;       // [nrec][25] interpolation weights (nullptr: receivers at nodes)
  double* seis = nullptr;
  FaultHost flt;
  int* flags = nullptr;  // [0] Newton failure
  int it = 0;
  double last_ms = 0.0;
  std::string err;
  std::vector<void*> allocs;
  AdjState* adj = nullptr;
  std::vector<int> elem_ibool;  // [nelem][25] 0-based reference nodes (interpolated receivers)
  // linear slip fault (BC_LSF): node pairs, side-1 normals [2][n], B, W1, W2 [ndof][n]
  int nlsf = 0;
  int *lsf_n1 = nullptr, *lsf_n2 = nullptr;
  double *lsf_nrm = nullptr, *lsf_B = nullptr, *lsf_W1 = nullptr, *lsf_W2 = nullptr;
  double lsf_kt = 0, lsf_kn = 0;
  int nper = 0;                 // periodic node pairs (master, slave; 0-based)
  int *per_m = nullptr, *per_s = nullptr;
  void* kv_eta = nullptr;       // Kelvin-Voigt viscosity [element in colour order][25] (bulk type)
  void* beta25 = nullptr;       // 2.5D coefficients [element in colour order][25] (bulk type)
  // progress rows (it, time, max |v|, max |d|) every itinfo steps, and the non-finite
  // watchdog (k_field_max, k_info_row)
  int itinfo = 0, info_rows = 0, info_cap = 0;
  double* info = nullptr;                 // device [info_cap][4]
  unsigned long long* info_acc = nullptr;  // device [2]
  int* info_cnt = nullptr;                 // device [2]
};

namespace {

int set_err(sem2d_solver* h, int code, const char* fmt, ...) {
  char buf[512];
  va_list ap;
  va_start(ap, fmt);
  vsnprintf(buf, sizeof buf, fmt, ap);
  va_end(ap);
  if (h) h->err = buf;
  return code;
}

#define HIPCHK(h, call)                                                                   \
  do {                                                                                    \
    hipError_t e_ = (call);                                                               \
    if (e_ != hipSuccess)                                                                 \
      return set_err(h, 10, "%s failed: %s (%s:%d)", #call, hipGetErrorString(e_), __FILE__, __LINE__); \
  } while (0)

template <typename T>
int dev_alloc(sem2d_solver* h, T** p, size_t n) {
  void* q = nullptr;
  hipError_t e = hipMalloc(&q, std::max<size_t>(n, 1) * sizeof(T));
  if (e != hipSuccess) return set_err(h, 11, "hipMalloc(%zu bytes): %s", n * sizeof(T), hipGetErrorString(e));
  h->allocs.push_back(q);
  *p = (T*)q;
  return 0;
}

template <typename T>
int upload(sem2d_solver* h, T** p, const T* src, size_t n) {
  int rc = dev_alloc(h, p, n);
  if (rc) return rc;
  if (n) HIPCHK(h, hipMemcpyAsync(*p, src, n * sizeof(T), hipMemcpyHostToDevice, h->stream));
  HIPCHK(h, hipStreamSynchronize(h->stream));
  return 0;
}

size_t rsize(const sem2d_solver* h) { return h->fp32 ? sizeof(float) : sizeof(double); }

// copy a double host array into a bulk (R) device array
int upload_bulk(sem2d_solver* h, void** p, const double* src, size_t n) {
  if (!h->fp32) return upload(h, (double**)p, src, n);
  std::vector<float> tmp(n);
  for (size_t k = 0; k < n; ++k) tmp[k] = (float)src[k];
  return upload(h, (float**)p, tmp.data(), n);
}

// rows of `per` values, row e of src to row to[e] of dst, in the bulk type
template <typename R>
__global__ void k_scatter_rows(size_t n, int per, const double* __restrict__ src, const int* __restrict__ to,
                               R* __restrict__ dst) {
  const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const size_t e = i / per;
  dst[(size_t)to[e] * per + (i - e * per)] = (R)src[i];
}
// Uploads the rows of a per-element array into one or two other orders of the elements:
// copied once as they are, in pieces, and put in their places on the device (the ten
// coefficients of 24,120 elements: a new solver 16 ms where the host ordered them first, 6 ms
// so).
struct RowOrder {
  void** p;
  const std::vector<int>* to;
};
int upload_rows(sem2d_solver* h, const double* src, int nelem, int per, std::initializer_list<RowOrder> orders) {
  int rc;
  for (const RowOrder& o : orders)
    if ((rc = dev_alloc(h, (char**)o.p, (size_t)nelem * per * rsize(h)))) return rc;
  const int piece = std::min<int>(nelem, std::max<size_t>(1, ((size_t)64 << 20) / (per * sizeof(double))));
  const size_t bytes = (size_t)piece * per * sizeof(double);
  char* tmp = nullptr;
  HIPCHK(h, hipMalloc((void**)&tmp, bytes + orders.size() * nelem * sizeof(int)));
  int* const pos = (int*)(tmp + bytes);
  hipError_t e = hipSuccess;
  int k = 0;
  for (const RowOrder& o : orders)
    if (e == hipSuccess)
      e = hipMemcpyAsync(pos + (size_t)nelem * k++, o.to->data(), (size_t)nelem * sizeof(int),
                         hipMemcpyHostToDevice, h->stream);
  for (int e0 = 0; e0 < nelem && e == hipSuccess; e0 += piece) {
    const size_t n = (size_t)std::min(piece, nelem - e0) * per;
    e = hipMemcpyAsync(tmp, src + (size_t)e0 * per, n * sizeof(double), hipMemcpyHostToDevice, h->stream);
    const unsigned blocks = (unsigned)((n + 255) / 256);
    k = 0;
    for (const RowOrder& o : orders) {
      const int* to = pos + (size_t)nelem * k++ + e0;
      if (h->fp32) k_scatter_rows<float><<<blocks, 256, 0, h->stream>>>(n, per, (double*)tmp, to, (float*)*o.p);
      else k_scatter_rows<double><<<blocks, 256, 0, h->stream>>>(n, per, (double*)tmp, to, (double*)*o.p);
    }
  }
  if (e == hipSuccess) e = hipStreamSynchronize(h->stream);
  hipFree(tmp);
  HIPCHK(h, e);
  return 0;
}

int write_bulk(sem2d_solver* h, void* dst, const double* src, size_t n) {
  if (!h->fp32) {
    HIPCHK(h, hipMemcpyAsync(dst, src, n * sizeof(double), hipMemcpyHostToDevice, h->stream));
    HIPCHK(h, hipStreamSynchronize(h->stream));
    return 0;
  }
  std::vector<float> tmp(n);
  for (size_t k = 0; k < n; ++k) tmp[k] = (float)src[k];
  HIPCHK(h, hipMemcpyAsync(dst, tmp.data(), n * sizeof(float), hipMemcpyHostToDevice, h->stream));
  HIPCHK(h, hipStreamSynchronize(h->stream));
  return 0;
}

int read_bulk(sem2d_solver* h, double* dst, const void* src, size_t n) {
  if (!h->fp32) {
    HIPCHK(h, hipMemcpyAsync(dst, src, n * sizeof(double), hipMemcpyDeviceToHost, h->stream));
    HIPCHK(h, hipStreamSynchronize(h->stream));
    return 0;
  }
  std::vector<float> tmp(n);
  HIPCHK(h, hipMemcpyAsync(tmp.data(), src, n * sizeof(float), hipMemcpyDeviceToHost, h->stream));
  HIPCHK(h, hipStreamSynchronize(h->stream));
  for (size_t k = 0; k < n; ++k) dst[k] = tmp[k];
  return 0;
}

// Scratch memory of sem2d_compute_fint_noalloc: a file-scope device array, one copy per
// GPU, held until the process ends.  Host code never passes the array's name to a kernel
// or a copy (on the host it names a stand-in, not device memory); it uses the device
// address taken once per device with hipGetSymbolAddress (scratch_on_device).
constexpr size_t NOALLOC_SCRATCH_BYTES = (size_t)64 << 20;
__device__ __align__(256) unsigned char scratch[NOALLOC_SCRATCH_BYTES];
constexpr int MAX_DEVICES = 64;
std::mutex g_scratch_mu;
void* g_scratch_ptr[MAX_DEVICES] = {};

// device address of this device's scratch array (taken at set-up, once per device, with
// the device current); nullptr with an error message on failure
void* scratch_on_device(sem2d_solver* h) {
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= MAX_DEVICES) {
    set_err(h, 10, "scratch: no current device");
    return nullptr;
  }
  std::lock_guard<std::mutex> lock(g_scratch_mu);
  if (!g_scratch_ptr[dev]) {
    void* p = nullptr;
    const hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
    if (e != hipSuccess || !p) {
      set_err(h, 10, "hipGetSymbolAddress(scratch): %s", hipGetErrorString(e));
      return nullptr;
    }
    g_scratch_ptr[dev] = p;
  }
  return g_scratch_ptr[dev];
}

// staging kernels of sem2d_compute_fint_noalloc (grid-stride)
template <typename T>
__global__ void k_fill(T* __restrict__ x, T val, size_t n) {
  for (size_t k = (size_t)blockIdx.x * blockDim.x + threadIdx.x; k < n; k += (size_t)gridDim.x * blockDim.x)
    x[k] = val;
}
__global__ void k_to_float(const double* __restrict__ x, float* __restrict__ y, size_t n) {
  for (size_t k = (size_t)blockIdx.x * blockDim.x + threadIdx.x; k < n; k += (size_t)gridDim.x * blockDim.x)
    y[k] = (float)x[k];
}
__global__ void k_to_double(const float* __restrict__ x, double* __restrict__ y, size_t n) {
  for (size_t k = (size_t)blockIdx.x * blockDim.x + threadIdx.x; k < n; k += (size_t)gridDim.x * blockDim.x)
    y[k] = (double)x[k];
}

// Element colouring: no two elements of one colour share a node.
// Structured boxes use the 2x2 checkerboard of cells; otherwise greedy first-fit
// in element order.
int build_colours(sem2d_solver* h, const sem2d_desc* s, std::vector<int>& colour, int& ncol) {
  const int ne = s->nelem;
  const int NP = s->ngll * s->ngll;  // points per element
  colour.assign(ne, -1);
  if (s->nx > 0 && s->elem_of_cell) {
    if ((long)s->nx * s->nz != ne) return set_err(h, 3, "nx*nz (%d*%d) != nelem (%d)", s->nx, s->nz, ne);
    for (int iz = 0; iz < s->nz; ++iz)
      for (int ix = 0; ix < s->nx; ++ix) {
        int e = s->elem_of_cell[(size_t)iz * s->nx + ix] - 1;
        if (e < 0 || e >= ne || colour[e] != -1) return set_err(h, 3, "elem_of_cell is not a permutation");
        colour[e] = (ix & 1) + 2 * (iz & 1);
      }
    ncol = 4;
  } else {
    std::vector<std::vector<int>> node_elems(s->npoin);
    for (int e = 0; e < ne; ++e)
      for (int p = 0; p < NP; ++p) node_elems[s->ibool[(size_t)e * NP + p] - 1].push_back(e);
    ncol = 0;
    std::vector<int> used;
    for (int e = 0; e < ne; ++e) {
      used.assign(ncol + 1, 0);
      for (int p = 0; p < NP; ++p)
        for (int o : node_elems[s->ibool[(size_t)e * NP + p] - 1])
          if (colour[o] >= 0) used[colour[o]] = 1;
      int c = 0;
      while (c < ncol && used[c]) ++c;
      colour[e] = c;
      if (c == ncol) ++ncol;
    }
  }
  // verify: each node is touched at most once per colour
  std::vector<int> stamp((size_t)s->npoin, -1);
  for (int c = 0; c < ncol; ++c)
    for (int e = 0; e < ne; ++e) {
      if (colour[e] != c) continue;
      for (int p = 0; p < NP; ++p) {
        int g = s->ibool[(size_t)e * NP + p] - 1;
        if (stamp[g] == c) {
          // repeated node inside one element is legal only for the element itself
          bool same = false;
          for (int q = 0; q < p; ++q)
            if (s->ibool[(size_t)e * NP + q] - 1 == g) same = true;
          if (!same) return set_err(h, 3, "colouring conflict at node %d colour %d", g + 1, c);
        }
        stamp[g] = c;
      }
    }
  return 0;
}

template <typename R, int NDOF, int NELAST, int MODE, int NGL>
void launch_force_t(sem2d_solver* h, const R* d, R* f, const R* v, const ElemStep<R>& E) {
  const R* kv = v ? (const R*)h->kv_eta : nullptr;
  constexpr int EPB = fe_epb(NGL);
  if (E.fe) {
    k_force_colour<R, NDOF, NELAST, MODE, NGL, true><<<(h->nelem + EPB - 1) / EPB, 256, 0, h->stream>>>(
        0, h->nelem, h->ibool, (const R*)h->coefs, (const R*)h->geom, d, f, h->npoin, v, kv, (const R*)h->beta25,
        h->hg, E);
    return;
  }
  for (size_t c = 0; c + 1 < h->colour_start.size(); ++c) {
    const int e0 = h->colour_start[c], ne = h->colour_start[c + 1] - e0;
    if (ne <= 0) continue;
    k_force_colour<R, NDOF, NELAST, MODE, NGL><<<(ne + EPB - 1) / EPB, 256, 0, h->stream>>>(
        e0, ne, h->ibool, (const R*)h->coefs, (const R*)h->geom, d, f, h->npoin, v, kv, (const R*)h->beta25,
        h->hg);
  }
}

template <typename R, int NDOF, int NELAST, int NGL>
void launch_force_m(sem2d_solver* h, const R* d, R* f, const R* v, const ElemStep<R>& E) {
  switch (h->coef_mode) {
    case COEF_SHARED: launch_force_t<R, NDOF, NELAST, COEF_SHARED, NGL>(h, d, f, v, E); break;
    case COEF_COMPACT:  // built for NGLL = 5 only (checked at creation)
      if constexpr ((NELAST == 2 || NELAST == 6) && NGL == NG)
        launch_force_t<R, NDOF, NELAST, COEF_COMPACT, NGL>(h, d, f, v, E);
      break;
    default: launch_force_t<R, NDOF, NELAST, COEF_PER_ELEM, NGL>(h, d, f, v, E);
  }
}

template <typename R, int NGL>
void launch_force_n(sem2d_solver* h, const R* d, R* f, const R* v, const ElemStep<R>& E) {
  if (h->ndof == 2) {
    if (h->nelast == 6) launch_force_m<R, 2, 6, NGL>(h, d, f, v, E);
    else launch_force_m<R, 2, 10, NGL>(h, d, f, v, E);
  } else {
    if (h->nelast == 2) launch_force_m<R, 1, 2, NGL>(h, d, f, v, E);
    else launch_force_m<R, 1, 3, NGL>(h, d, f, v, E);
  }
}

// f = -K d, or -K (d + eta v) in Kelvin-Voigt elements when v is given; with E.fe the
// element forces of a step instead (ElemStep)
template <typename R>
void launch_force(sem2d_solver* h, const R* d, R* f, const R* v = nullptr, const ElemStep<R>& E = {}) {
  switch (h->ng) {
    case 3: launch_force_n<R, 3>(h, d, f, v, E); break;
    case 4: launch_force_n<R, 4>(h, d, f, v, E); break;
    case 6: launch_force_n<R, 6>(h, d, f, v, E); break;
    case 7: launch_force_n<R, 7>(h, d, f, v, E); break;
    case 8: launch_force_n<R, 8>(h, d, f, v, E); break;
    case 9: launch_force_n<R, 9>(h, d, f, v, E); break;
    case 10: launch_force_n<R, 10>(h, d, f, v, E); break;
    default: launch_force_n<R, NG>(h, d, f, v, E);
  }
}

int grid_for(size_t n, int block) {
  size_t g = (n + block - 1) / block;
  return (int)std::min<size_t>(std::max<size_t>(g, 1), 65536);
}

int sync_sources(sem2d_solver* h) {
  if (!h->src_dirty) return 0;
  h->src_dirty = false;
  int nt = 0;
  for (auto& t : h->stf) nt = std::max<int>(nt, (int)t.size());
  std::vector<double> tab((size_t)std::max(h->nsrc, 1) * std::max(nt, 1), 0.0);
  for (int s = 0; s < h->nsrc; ++s)
    for (size_t k = 0; k < h->stf[s].size(); ++k) tab[(size_t)s * nt + k] = h->stf[s][k];
  if (h->src_dev) hipFree(h->src_dev);
  if (h->ampl_dev) hipFree(h->ampl_dev);
  h->src_dev = nullptr;
  h->ampl_dev = nullptr;
  HIPCHK(h, hipMalloc(&h->src_dev, std::max<size_t>(h->src_host.size(), 1) * sizeof(SrcEntry)));
  HIPCHK(h, hipMalloc(&h->ampl_dev, tab.size() * sizeof(double)));
  if (!h->src_host.empty())
    HIPCHK(h, hipMemcpyAsync(h->src_dev, h->src_host.data(), h->src_host.size() * sizeof(SrcEntry),
                             hipMemcpyHostToDevice, h->stream));
  HIPCHK(h, hipMemcpyAsync(h->ampl_dev, tab.data(), tab.size() * sizeof(double), hipMemcpyHostToDevice, h->stream));
  HIPCHK(h, hipStreamSynchronize(h->stream));
  h->ampl_nt = nt;
  return 0;
}

// whether the state after step it is a receiver sample
bool sampled(const sem2d_solver* h, int it) { return h->nrec && it % h->isamp == 0 && it / h->isamp < h->nsamp; }

// marked: the recorded field is in the a array at the recorded nodes (StepOut::rec)
template <typename R>
int record_receivers(sem2d_solver* h, bool marked = false) {
  if (!sampled(h, h->it)) return 0;
  const int s = h->it / h->isamp;
  const R* fld = (const R*)(marked || h->field == 2 ? h->a : (h->field == 0 ? h->d : h->v));
  if (h->rec_w)
    k_receivers_interp<R><<<grid_for(h->nrec, 64), 64, 0, h->stream>>>(
        h->nrec, h->ndof, h->rec_node, h->rec_w, fld, h->fstride, h->seis + (size_t)s * h->ndof * h->nrec, h->np);
  else
    k_receivers<R><<<grid_for(h->nrec, 64), 64, 0, h->stream>>>(h->nrec, h->ndof, h->rec_node, fld, h->fstride,
                                                                h->seis + (size_t)s * h->ndof * h->nrec);
  h->taken = std::max(h->taken, s + 1);
  return 0;
}

// room for `rows` potency rows (grown outside any step loop)
int info_reserve(sem2d_solver* h, int rows) {
  if (rows <= h->info_cap) return 0;
  const int cap = std::max(rows, std::max(64, 2 * h->info_cap));
  double* p = nullptr;
  HIPCHK(h, hipMalloc(&p, (size_t)cap * 4 * sizeof(double)));
  if (h->info && h->info_rows)
    HIPCHK(h, hipMemcpyAsync(p, h->info, (size_t)h->info_rows * 4 * sizeof(double), hipMemcpyDeviceToDevice,
                             h->stream));
  HIPCHK(h, hipStreamSynchronize(h->stream));
  if (h->info) hipFree(h->info);
  h->info = p;
  h->info_cap = cap;
  return 0;
}

// the progress row of step it (after that step's kernels)
template <typename R>
void record_info(sem2d_solver* h, int it) {
  if (h->itinfo <= 0 || it % h->itinfo != 0) return;
  const size_t n = (size_t)h->ndof * h->fstride;
  k_field_max<R><<<std::min<size_t>((n + 255) / 256, 4096), 256, 0, h->stream>>>(
      n, (const R*)h->d, (const R*)h->v, (const R*)h->a, h->info_acc, h->info_cnt);
  k_info_row<<<1, 64, 0, h->stream>>>(it, it * h->dt, h->info_acc, h->info_cnt, h->info + 4 * (size_t)h->info_rows);
  ++h->info_rows;
}

int potency_reserve(sem2d_solver* h, int rows) {
  FaultHost& F = h->flt;
  if (rows <= F.pot_cap) return 0;
  const int cap = std::max(rows, 2 * F.pot_cap);
  const size_t nc = 2 * (h->ndof + 1);
  double* p = nullptr;
  HIPCHK(h, hipMalloc(&p, (size_t)cap * nc * sizeof(double)));
  if (F.pot && F.pot_rows)
    HIPCHK(h, hipMemcpyAsync(p, F.pot, (size_t)F.pot_rows * nc * sizeof(double), hipMemcpyDeviceToDevice, h->stream));
  HIPCHK(h, hipStreamSynchronize(h->stream));
  if (F.pot) hipFree(F.pot);
  F.pot = p;
  F.pot_cap = cap;
  return 0;
}

template <typename R>
void record_potency(sem2d_solver* h) {
  FaultHost& F = h->flt;
  if (F.pot_rows >= F.pot_cap) return;  // reserved by the caller
  k_fault_potency<R><<<1, 256, 0, h->stream>>>(F.dev, (const R*)h->d, (const R*)h->v, h->fstride,
                                               F.pot + (size_t)F.pot_rows * 2 * (h->ndof + 1));
  F.pot_rows++;
}

// per-side record (osides) of sample slot s from the current fields, or from
// FaultDev::side (sides: the steps of a structured grid)
void record_sides(sem2d_solver* h, int s, int sides) {
  FaultHost& F = h->flt;
  double* out = F.srec + (size_t)s * 4 * h->ndof * F.nout;
  if (h->fp32)
    k_fault_sides<float><<<grid_for(F.nout, 64), 64, 0, h->stream>>>(F.dev, (const float*)h->d, (const float*)h->v,
                                                                      h->fstride, F.oix1, F.oixd, F.nout, out, sides);
  else
    k_fault_sides<double><<<grid_for(F.nout, 64), 64, 0, h->stream>>>(
        F.dev, (const double*)h->d, (const double*)h->v, h->fstride, F.oix1, F.oixd, F.nout, out, sides);
}

int record_fault(sem2d_solver* h) {
  FaultHost& F = h->flt;
  if (!F.on) return 0;
  if (h->fp32) record_potency<float>(h);
  else record_potency<double>(h);
  if (h->it < F.oit) return 0;
  if (F.taken < F.nsamp) {
    k_fault_record<<<grid_for(F.nout, 64), 64, 0, h->stream>>>(F.dev, F.oix1, F.oixd, F.nout,
                                                               F.rec + (size_t)F.taken * 6 * F.nout);
    if (F.srec) record_sides(h, F.taken, 0);
    F.taken++;
  }
  F.oit += F.oitd;
  return 0;
}

// structured grids: the fault outputs that k_deferred makes at step it ...
void fault_out_step(sem2d_solver* h, int it, FaultOut& O) {
  FaultHost& F = h->flt;
  O.pot = F.pot;
  O.pot_cap = F.pot_cap;
  O.pot_row = F.pot_rows;
  O.rec_slot = it >= F.oit && F.taken < F.nsamp ? F.taken : -1;
}
// ... and the bookkeeping after it, with the per-side record
void fault_out_done(sem2d_solver* h, int it) {
  FaultHost& F = h->flt;
  if (F.pot_rows < F.pot_cap) F.pot_rows++;
  if (it < F.oit) return;
  if (F.taken < F.nsamp) {
    if (F.srec) record_sides(h, F.taken, 1);
    F.taken++;
  }
  F.oit += F.oitd;
}

// ---------------------------------------------------------------------------
// structured path set-up
// ---------------------------------------------------------------------------
// Grid map from ibool and the cell -> element table; returns false if ibool does not
// number a MESH_CART box the way the node grid does (the general path is used then).
// Storage index of grid node (X, Z): nodes on vertical tile-edge lines (X a multiple
// of 4*TX, or the right domain edge) live column-contiguous after the grid block, so
// that the column edges of the tiles are read and written with unit stride.
// The other nodes are stored row by row, each tile column's 4*TX-1 nodes in a segment
// of 4*TX slots (ROW = 4*TX * tile columns slots per row), so every segment starts on
// a cache-line boundary.
static size_t storage_index(const StructState& S, int X, int Z) {
  const int W = 4 * TX;
  int k = -1;
  if (X % W == 0) k = X / W;
  else if (X == S.NX1 - 1) k = S.nvl - 1;
  if (k >= 0) return (size_t)S.ROW * S.NZ1 + (size_t)k * S.NZ1 + Z;
  return (size_t)Z * S.ROW + (size_t)(X / W) * W + (X % W) - 1;
}

// Workgroups of the tile kernel per CU.  Two by default: with six wavefronts each they keep
// to 128 registers where the dispatcher packs four on a SIMD (P-SV, 1000 x 500 elements,
// us per step with 1 / 2 / 3 / 4: FP64 225 / 182 / 198 / 210, FP32 176 / 117 / 137 / 118;
// SH FP64, 600 x 300: 58 / 45 / 48 / 53).  The SH kernel with FP32 fields needs 62
// registers and 25 KB of LDS at most: four (333 x 251: 30 / 24 / 22 / 21).
static int tile_wgs_per_cu(bool fp32, int ndof) { return fp32 && ndof == 1 ? 4 : 2; }

bool structured_map(sem2d_solver* h, const sem2d_desc* s) {
  StructState& S = h->st;
  const int nx = s->nx, nz = s->nz, ez = s->ezflt;
  if (nx <= 0 || nz <= 0 || !s->elem_of_cell || (long)nx * nz != s->nelem) return false;
  if (nx > 0x7fff || ez < 0 || ez >= nz) return false;
  S.nx = nx; S.nz = nz; S.ezflt = ez;
  S.NX1 = 4 * nx + 1;
  S.NZ1 = 4 * nz + 1 + (ez > 0 ? 1 : 0);
  if ((long)S.NX1 * S.NZ1 != s->npoin) return false;
  S.nvl = (nx + TX - 1) / TX + 1;
  S.ROW = 4 * TX * (S.nvl - 1);
  // component stride rounded to 4*TX slots so that every component (and every batch
  // member placed at a multiple of it) keeps the segments line-aligned
  S.NS = (size_t)S.ROW * S.NZ1 + (size_t)S.nvl * S.NZ1;
  S.NS = (S.NS + 4 * TX - 1) / (4 * TX) * (4 * TX);
  S.gmap.assign(s->npoin, -1);
  std::vector<char> used((size_t)s->npoin, 0);
  for (int iz = 0; iz < nz; ++iz) {
    const int sh = (ez > 0 && iz >= ez) ? 1 : 0;
    for (int ix = 0; ix < nx; ++ix) {
      const int e = s->elem_of_cell[(size_t)iz * nx + ix] - 1;
      if (e < 0 || e >= s->nelem) return false;
      for (int j = 0; j < NG; ++j)
        for (int i = 0; i < NG; ++i) {
          const int ref = s->ibool[(size_t)e * NP + j * NG + i] - 1;
          const int g = (4 * iz + j + sh) * S.NX1 + 4 * ix + i;
          if (S.gmap[ref] == -1) {
            if (used[g]) return false;
            S.gmap[ref] = g;
            used[g] = 1;
          } else if (S.gmap[ref] != g) {
            return false;
          }
        }
    }
  }
  for (int k = 0; k < s->npoin; ++k)
    if (S.gmap[k] < 0) return false;
  S.gridx = S.gmap;
  for (int k = 0; k < s->npoin; ++k) S.gmap[k] = (int)storage_index(S, S.gridx[k] % S.NX1, S.gridx[k] / S.NX1);
  // tiles: element-row bands split at the fault, TX x TZ tiles in each band
  S.tiles.clear();
  const int nb = ez > 0 ? 2 : 1;
  for (int b = 0; b < nb; ++b) {
    const int r0 = (b == 0) ? 0 : ez, r1 = (nb == 1) ? nz : (b == 0 ? ez : nz);
    const int sh = b;
    for (int tz0 = r0; tz0 < r1; tz0 += TZ)
      for (int tx0 = 0; tx0 < nx; tx0 += TX) {
        const int nxe = std::min(TX, nx - tx0), nze = std::min(TZ, r1 - tz0);
        S.tiles.push_back(make_int4(tx0, tz0, nxe | (nze << 8) | (nx << 16), 4 * tz0 + sh));
      }
  }
  S.ntiles = (int)S.tiles.size();
  {
    int dev = 0, ncu = 256;
    if (hipGetDevice(&dev) == hipSuccess) hipDeviceGetAttribute(&ncu, hipDeviceAttributeMultiprocessorCount, dev);
    int per_cu = tile_wgs_per_cu(h->fp32, h->ndof);
    const char* env = getenv("SEM2D_TILE_WG_PER_CU");
    if (env) per_cu = atoi(env);
    S.pipe_wgs = std::max(0, (ncu * per_cu + 7) / 8 * 8);
  }
  return true;
}

// f(t) for every tile t whose patch holds grid node (X, Z).  The tiles of a split grid are two
// bands, each cut from its own first element row, the upper one a node row further up.
template <typename F>
static void tiles_at(const StructState& S, int X, int Z, F f) {
  const int W = 4 * TX, ncx = (S.nx + TX - 1) / TX;
  int t0 = 0;
  for (int b = 0; b < (S.ezflt > 0 ? 2 : 1); ++b) {
    const int r0 = b ? S.ezflt : 0, r1 = S.ezflt > 0 && !b ? S.ezflt : S.nz;
    const int nrow = (r1 - r0 + TZ - 1) / TZ, z = Z - (4 * r0 + b);
    if (z >= 0 && z <= 4 * (r1 - r0))
      for (int tz = std::max(z - 1, 0) / (4 * TZ); tz <= z / (4 * TZ) && tz < nrow; ++tz)
        for (int tx = std::max(X - 1, 0) / W; tx <= X / W && tx < ncx; ++tx) f(t0 + tz * ncx + tx);
    t0 += nrow * ncx;
  }
}

// ngp, fps: field and partial-force component strides; ncoef: entries of the per-cell
// coefficient array
static bool fits32(size_t ngp, size_t fps, size_t ncoef, size_t rs) {
  return std::max(std::max(ngp, fps), ncoef) * rs < (size_t(1) << 32);
}

// device form of a deferred-node list (DefDev records and their side table); false when
// a count does not fit its 8 bits
bool pack_defs(const std::vector<DefNode>& in, const std::vector<int>& part_off, std::vector<DefDev>& node,
               std::vector<int4>& ext) {
  node.resize(in.size());
  ext.clear();
  for (size_t q = 0; q < in.size(); ++q) {
    const DefNode& n = in[q];
    if (n.pcnt < 0 || n.pcnt > 255 || n.scnt < 0 || n.scnt > 255 || n.acnt < 0 || n.acnt > 255) return false;
    DefDev e;
    e.g = n.g;
    e.pstart = n.pstart;
    e.cnt = n.pcnt | (n.scnt << 8) | (n.acnt << 16) | ((n.fault ? 1 : 0) << 24) | ((n.dmask & 3) << 26) |
            ((n.rec ? 1 : 0) << 28);
    e.x = -1;
    if (n.scnt > 0 || n.acnt > 0 || n.rec_at >= 0) {
      e.x = (int)ext.size();
      ext.push_back(make_int4(n.sstart, n.astart, n.rec_at, 0));
    } else if (!part_off.empty() && (n.pcnt == 1 || n.pcnt == 2)) {  // offsets inline
      e.cnt |= 1 << 25;
      e.pstart = part_off[n.pstart];
      e.x = n.pcnt == 2 ? part_off[n.pstart + 1] : -1;
    }
    node[q] = e;
  }
  return true;
}

template <typename T>
int prep_upload(sem2d_solver* h, T** p, const T* src, size_t n) {
  void* q = nullptr;
  HIPCHK(h, hipMalloc(&q, std::max<size_t>(n, 1) * sizeof(T)));
  h->st.prep_allocs.push_back(q);
  *p = (T*)q;
  if (n) HIPCHK(h, hipMemcpyAsync(q, src, n * sizeof(T), hipMemcpyHostToDevice, h->stream));
  return 0;
}

int prep_upload_bulk(sem2d_solver* h, void** p, const std::vector<double>& src) {
  if (!h->fp32) return prep_upload(h, (double**)p, src.data(), src.size());
  std::vector<float> tmp(src.begin(), src.end());
  int rc = prep_upload(h, (float**)p, tmp.data(), tmp.size());
  if (rc) return rc;
  HIPCHK(h, hipStreamSynchronize(h->stream));
  return 0;
}

// Host tables of the structured step of one grid, with local indices (grid node
// storage from 0, tiles from 0, cells from 0): tiles and their grid descriptors,
// special nodes, deferred nodes with their partial-force slots, sources, absorbing
// coefficients and inverse masses, and the split-fault nodes.
struct StructTables {
  std::vector<int4> tiles, grids;
  std::vector<int> spec_cnt, spec_idx;
  std::vector<DefNode> defs;
  std::vector<int> def_ref;      // their reference nodes (0-based)
  std::vector<int> part_off;
  std::vector<SrcEntry> dsrc;
  std::vector<double> dabso, dabson;
  std::vector<double> rmdef;     // [ndof][ndef]
  std::vector<unsigned char> fault_dmask;  // [npairs] Dirichlet after the fault: node 1 bits 0-1, node 2 bits 2-3
  std::vector<int> s_enode, ak_off, ak_idx;  // Stacey (see StructState)
  // recorded nodes inside tiles (TileArgs::mark_of, marks)
  std::vector<int> mark_of;
  std::vector<uint32_t> marks;
  // receivers at nodes (RecOut): (storage index, or deferred node, or 2 * pair + side; receiver)
  std::vector<std::pair<int, int>> rec_int, rec_def, rec_flt;
  std::vector<int> fault_def1, fault_def2;  // the pairs' nodes as k_deferred counts them (-1: one side)
  std::vector<int> fault_at;                // [side][pair]: their places in defs (one side: side 1 twice)
  std::vector<double> s_K;
};

// Partial forces of the deferred nodes: node g[i] (storage index, ascending) adds those at
// off[start[i] .. start[i] + cnt[i]), in this order.
struct Partials {
  std::vector<int> g, start, cnt, off;
};

// General path: every node adds the forces of its element points, in the order of the
// colours.  Their list is made on the device (on the host it took 20 ns per element point,
// as much as 400 steps of a 24,120-element mesh gain): slot[i] is the place of element point
// i among its node's, then each node's points are put in ascending order.
__global__ void k_gen_count(size_t n, const int* __restrict__ ibool, int* __restrict__ cnt, int* __restrict__ slot) {
  const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) slot[i] = atomicAdd(&cnt[ibool[i]], 1);
}
__global__ void k_gen_place(size_t n, const int* __restrict__ ibool, const int* __restrict__ start,
                            const int* __restrict__ slot, int* __restrict__ off) {
  const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) off[start[ibool[i]] + slot[i]] = (int)i;
}
__global__ void k_gen_defs(int n, const int* __restrict__ start, const int* __restrict__ cnt, int* __restrict__ off,
                           DefDev* __restrict__ def) {
  const int g = blockIdx.x * blockDim.x + threadIdx.x;
  if (g >= n) return;
  const int c = cnt[g];
  int* o = off + start[g];
  for (int i = 1; i < c; ++i) {
    const int x = o[i];
    int j = i;
    for (; j > 0 && o[j - 1] > x; --j) o[j] = o[j - 1];
    o[j] = x;
  }
  DefDev e{g, start[g], c, -1};
  if (c == 1 || c == 2) {  // offsets inline
    e.cnt |= 1 << 25;
    e.pstart = o[0];
    e.x = c == 2 ? o[1] : -1;
  }
  def[g] = e;
}
// the records of the nodes that have more than partial forces
__global__ void k_gen_put(int n, const DefDev* __restrict__ src, DefDev* __restrict__ def) {
  const int q = blockIdx.x * blockDim.x + threadIdx.x;
  if (q < n) def[src[q].g] = src[q];
}

template <typename T>
int prep_alloc(sem2d_solver* h, T** p, size_t n) {
  void* q = nullptr;
  HIPCHK(h, hipMalloc(&q, std::max<size_t>(n, 1) * sizeof(T)));
  h->st.prep_allocs.push_back(q);
  *p = (T*)q;
  return 0;
}

// node records and point lists on the device; start and cnt of every node on the host
int general_partials(sem2d_solver* h, std::vector<int>& start, std::vector<int>& cnt) {
  StructState& S = h->st;
  const size_t n = (size_t)h->nelem * h->np;
  const int nb = grid_for(n, 256), nn = h->npoin;
  if (n > (size_t)65536 * 256) return set_err(h, 5, "general path: too many element points");
  int *dcnt, *dstart, *slot;
  int rc;
  if ((rc = prep_alloc(h, &dcnt, nn)) || (rc = prep_alloc(h, &dstart, nn)) || (rc = prep_alloc(h, &slot, n))) return rc;
  if ((rc = prep_alloc(h, &S.part_off, n)) || (rc = prep_alloc(h, &S.gen_def, nn))) return rc;
  HIPCHK(h, hipMemsetAsync(dcnt, 0, (size_t)nn * sizeof(int), h->stream));
  k_gen_count<<<nb, 256, 0, h->stream>>>(n, h->ibool, dcnt, slot);
  start.resize(nn);
  cnt.resize(nn);
  HIPCHK(h, hipMemcpyAsync(cnt.data(), dcnt, (size_t)nn * sizeof(int), hipMemcpyDeviceToHost, h->stream));
  HIPCHK(h, hipStreamSynchronize(h->stream));
  int at = 0;
  for (int g = 0; g < nn; ++g) {
    start[g] = at;
    at += cnt[g];
    if (cnt[g] > 255) return set_err(h, 5, "prepare: more than 255 elements at a node");
  }
  HIPCHK(h, hipMemcpyAsync(dstart, start.data(), (size_t)nn * sizeof(int), hipMemcpyHostToDevice, h->stream));
  k_gen_place<<<nb, 256, 0, h->stream>>>(n, h->ibool, dstart, slot, S.part_off);
  k_gen_defs<<<grid_for(nn, 256), 256, 0, h->stream>>>(nn, dstart, dcnt, S.part_off, S.gen_def);
  HIPCHK(h, hipGetLastError());
  return 0;
}

// structured grids: the nodes of the tile perimeters and the source nodes inside tiles
int tile_partials(sem2d_solver* h, StructTables& X, Partials& P) {
  StructState& S = h->st;
  X.tiles = S.tiles;
  X.grids.assign(S.ntiles, make_int4(0, S.ROW, S.NZ1, 0));
  // special nodes: point-source nodes inside a tile patch
  std::vector<int> src_g;  // grid indices of source nodes
  for (const SrcEntry& e : h->src_host) src_g.push_back(S.gridx[e.node]);
  std::sort(src_g.begin(), src_g.end());
  src_g.erase(std::unique(src_g.begin(), src_g.end()), src_g.end());
  X.spec_cnt.assign(S.ntiles, 0);
  X.spec_idx.assign((size_t)S.ntiles * MAXSPECIAL, 0);
  // entries (g, tile, slot)
  struct Ent { int g, t, slot; };
  std::vector<Ent> ents;
  ents.reserve((size_t)S.ntiles * PERIM_MAX);
  for (int t = 0; t < S.ntiles; ++t) {
    const int4 tg = S.tiles[t];
    const int nxe = tg.z & 0xff, nze = (tg.z >> 8) & 0xff;
    const int PX = 4 * nxe + 1, PZ = 4 * nze + 1, X0 = 4 * tg.x, Z0 = tg.w;
    auto gi = [&](int Xn, int Zn) { return (int)storage_index(S, X0 + Xn, Z0 + Zn); };
    for (int Xn = 0; Xn < PX; ++Xn) ents.push_back({gi(Xn, 0), t, Xn});
    for (int Xn = 0; Xn < PX; ++Xn) ents.push_back({gi(Xn, PZ - 1), t, PX + Xn});
    for (int Zn = 1; Zn < PZ - 1; ++Zn) ents.push_back({gi(0, Zn), t, 2 * PX + Zn - 1});
    for (int Zn = 1; Zn < PZ - 1; ++Zn) ents.push_back({gi(PX - 1, Zn), t, 2 * PX + (PZ - 2) + Zn - 1});
    for (int g : src_g) {
      const int Xn = g % S.NX1 - X0, Zn = g / S.NX1 - Z0;
      if (Xn > 0 && Xn < PX - 1 && Zn > 0 && Zn < PZ - 1) {
        if (X.spec_cnt[t] >= MAXSPECIAL) return set_err(h, 5, "too many source nodes in one tile");
        X.spec_idx[(size_t)t * MAXSPECIAL + X.spec_cnt[t]] = Zn * PXM + Xn;
        ents.push_back({(int)storage_index(S, X0 + Xn, Z0 + Zn), t, PERIM_MAX + X.spec_cnt[t]});
        X.spec_cnt[t]++;
      }
    }
  }
  std::sort(ents.begin(), ents.end(), [](const Ent& a, const Ent& b) {
    return a.g != b.g ? a.g < b.g : a.t < b.t;
  });
  for (size_t i = 0; i < ents.size(); ++i) {
    if (i == 0 || ents[i].g != ents[i - 1].g) {
      P.g.push_back(ents[i].g);
      P.start.push_back((int)i);
      P.cnt.push_back(0);
    }
    ++P.cnt.back();
    P.off.push_back(ents[i].t * SLOTS + ents[i].slot);
  }
  return 0;
}

// Tables of the step kernels: of a structured grid, or of the general path, where every
// node is a deferred node and the partial forces are the element forces.
int struct_tables(sem2d_solver* h, StructTables& X) {
  StructState& S = h->st;
  const int nd = h->ndof;
  const int NG = h->ng;
  Partials P;
  if (S.on)
    if (int rc = tile_partials(h, X, P)) return rc;
  auto stored = [&](int ref) { return S.on ? S.gmap[ref] : ref; };
  // inverse map storage -> reference node, for sources / ABC / fault lookups
  std::vector<int> ginv(S.on ? S.NS : 0, -1);
  if (S.on)
    for (int k = 0; k < h->npoin; ++k) ginv[S.gmap[k]] = k;
  std::vector<char> extra((size_t)h->npoin, 0);  // nodes with sources (1) or absorbing terms (2)
  for (const SrcEntry& e : h->src_host) extra[e.node] |= 1;
  for (const AbsoHost& B : h->abso_host)
    for (int k : B.node) extra[k] |= 2;
  std::unordered_map<int, std::vector<int>> src_of;  // ref node -> src_host indices
  for (size_t q = 0; q < h->src_host.size(); ++q) src_of[h->src_host[q].node].push_back((int)q);
  std::unordered_map<int, std::vector<std::pair<int, int>>> abso_of;  // ref node -> (bc, k)
  for (size_t b = 0; b < h->abso_host.size(); ++b)
    for (size_t k = 0; k < h->abso_host[b].node.size(); ++k)
      abso_of[h->abso_host[b].node[k]].push_back({(int)b, (int)k});
  std::vector<char> is_fault((size_t)h->npoin, 0);
  for (int k : h->fault_n1) is_fault[k] = 1;
  for (int k : h->fault_n2) is_fault[k] = 1;
  // Dirichlet components per reference node: those applied by k_deferred (every
  // Dirichlet boundary at a node off the fault; at a fault node only those that act
  // before the fault) and those applied after the fault solve
  std::vector<unsigned char> dmask_def((size_t)h->npoin, 0), dmask_aft((size_t)h->npoin, 0);
  for (const auto& D : h->dirs)
    for (int k : D.node) {
      if (is_fault[k] && D.after_fault) dmask_aft[k] |= (unsigned char)D.comp;
      else dmask_def[k] |= (unsigned char)D.comp;
    }
  // Stacey: global list of boundary elements (in boundary order) and, per boundary and
  // boundary-local node, its element points e*NG+k in element order
  X.s_enode.clear();
  X.s_K.clear();
  std::vector<std::vector<std::vector<int>>> scon(h->abso_host.size());
  for (size_t b = 0; b < h->abso_host.size(); ++b) {
    const AbsoHost& B = h->abso_host[b];
    if (B.senode.empty()) continue;
    const int base = (int)(X.s_enode.size() / NG), nbe = (int)(B.senode.size() / NG);
    scon[b].assign(B.node.size(), {});
    for (int e = 0; e < nbe; ++e)
      for (int k = 0; k < NG; ++k) {
        const int bn = B.senode[(size_t)e * NG + k];
        X.s_enode.push_back(stored(B.node[bn]));
        scon[b][bn].push_back((base + e) * NG + k);
      }
    X.s_K.insert(X.s_K.end(), B.sK.begin(), B.sK.end());
  }
  X.ak_off.assign(1, 0);
  X.ak_idx.clear();
  std::vector<char> is_rec((size_t)h->npoin, 0);  // recorded reference nodes
  for (int k : h->rec_ref) is_rec[k] = 1;
  if (!S.on) {
    // the nodes that have more than partial forces; the records of the others are made on
    // the device
    std::vector<int> start, cnt;
    if (int rc = general_partials(h, start, cnt)) return rc;
    for (int g = 0; g < h->npoin; ++g)
      if (extra[g] || is_fault[g] || dmask_def[g] || dmask_aft[g] || is_rec[g]) {
        P.g.push_back(g);
        P.start.push_back(start[g]);
        P.cnt.push_back(cnt[g]);
      }
  }

  X.defs.clear();
  X.dsrc.clear();
  X.dabso.clear();
  X.dabson.clear();
  bool skew = false;
  for (const AbsoHost& B : h->abso_host) skew |= !B.nrm.empty();
  X.part_off = std::move(P.off);
  std::vector<int>& def_ref = X.def_ref;
  def_ref.resize(P.g.size());
  X.defs.reserve(P.g.size());
  for (size_t i = 0; i < P.g.size(); ++i) {
    DefNode n{};
    n.g = P.g[i];
    n.pstart = P.start[i];
    n.pcnt = P.cnt[i];
    const int ref = S.on ? ginv[n.g] : n.g;
    n.sstart = (int)X.dsrc.size();
    if (extra[ref] & 1)
      for (int q : src_of[ref]) X.dsrc.push_back(h->src_host[q]);
    n.scnt = (int)X.dsrc.size() - n.sstart;
    n.astart = (int)(X.dabso.size() / nd);
    if (extra[ref] & 2)
      for (auto& bk : abso_of[ref]) {
        const AbsoHost& B = h->abso_host[bk.first];
        const size_t nb = B.node.size();
        for (int c = 0; c < nd; ++c) X.dabso.push_back(B.C[(size_t)c * nb + bk.second]);
        if (skew)
          for (int c = 0; c < 2; ++c) X.dabson.push_back(B.nrm.empty() ? 0.0 : B.nrm[c * nb + bk.second]);
        if (!scon[bk.first].empty())
          for (int t : scon[bk.first][bk.second]) X.ak_idx.push_back(t);
        X.ak_off.push_back((int)X.ak_idx.size());
      }
    n.acnt = (int)(X.dabso.size() / nd) - n.astart;
    n.fault = is_fault[ref];
    n.dmask = dmask_def[ref];
    n.rec = is_rec[ref];
    n.rec_at = -1;
    X.defs.push_back(n);
    def_ref[i] = ref;
  }
  const size_t ndef = X.defs.size();
  {  // every Dirichlet node is a deferred node (tile perimeters hold the box's sides)
    size_t ndir_def = 0, ndir = 0;
    for (size_t q = 0; q < X.defs.size(); ++q) ndir_def += X.defs[q].dmask || dmask_aft[def_ref[q]] ? 1 : 0;
    for (size_t k = 0; k < dmask_def.size(); ++k) ndir += dmask_def[k] || dmask_aft[k] ? 1 : 0;
    if (ndir_def != ndir)
      return set_err(h, 5, "structured grid: %zu of the %zu Dirichlet nodes are not on tile edges", ndir_def, ndir);
  }
  X.fault_dmask.assign(h->fault_n1.size(), 0);
  for (size_t k = 0; k < h->fault_n1.size(); ++k) {
    X.fault_dmask[k] = dmask_aft[h->fault_n1[k]];
    if (!h->fault_n2.empty()) X.fault_dmask[k] |= (unsigned char)(dmask_aft[h->fault_n2[k]] << 2);
  }
  // places in defs of the fault's and the recorded nodes, by reference node
  std::unordered_map<int, int> at;
  for (size_t q = 0; q < ndef; ++q)
    if (is_rec[def_ref[q]] || is_fault[def_ref[q]]) at[def_ref[q]] = (int)q;
  auto def_of = [&](int ref) {  // as k_deferred counts them; -1: not deferred
    const auto f = at.find(ref);
    return f == at.end() ? -1 : (S.on ? f->second : ref);
  };
  X.fault_def1.clear();
  X.fault_def2.clear();
  std::unordered_map<int, int> flt_of;  // reference node -> 2 * pair + side
  for (size_t k = 0; k < h->fault_n1.size(); ++k) {
    const int r1 = h->fault_n1[k], r2 = h->fault_n2.empty() ? -1 : h->fault_n2[k];
    X.fault_def1.push_back(def_of(r1));
    X.fault_def2.push_back(r2 < 0 ? -1 : def_of(r2));
    flt_of[r1] = 2 * (int)k;
    if (r2 >= 0) flt_of[r2] = 2 * (int)k + 1;
  }
  X.rec_int.clear();
  X.rec_def.clear();
  X.rec_flt.clear();
  if (h->nrec && !h->rec_w)
    for (int r = 0; r < h->nrec; ++r) {
      const int ref = h->rec_ref[r];
      const auto f = flt_of.find(ref);
      if (f != flt_of.end()) X.rec_flt.push_back({f->second, r});
      else if (def_of(ref) >= 0) X.rec_def.push_back({def_of(ref), r});
      else X.rec_int.push_back({S.gmap[ref], r});
    }
  std::sort(X.rec_int.begin(), X.rec_int.end());
  std::sort(X.rec_def.begin(), X.rec_def.end());
  std::sort(X.rec_flt.begin(), X.rec_flt.end());
  for (int k = (int)X.rec_def.size() - 1; k >= 0; --k) X.defs[at[h->rec_ref[X.rec_def[k].second]]].rec_at = k;
  for (int k = (int)X.rec_flt.size() - 1; k >= 0; --k) X.defs[at[h->rec_ref[X.rec_flt[k].second]]].rec_at = k;
  X.fault_at.clear();
  for (int side = 0; side < 2; ++side)
    for (size_t k = 0; k < h->fault_n1.size(); ++k)
      X.fault_at.push_back(at[side && !h->fault_n2.empty() ? h->fault_n2[k] : h->fault_n1[k]]);
  // recorded nodes that are not deferred nodes: marks of the tile they lie in
  X.mark_of.assign(S.on ? S.ntiles : 0, -1);
  X.marks.clear();
  if (S.on) {
    for (int ref : h->rec_ref) {
      if (def_of(ref) >= 0) continue;
      const int Xg = S.gridx[ref] % S.NX1, Zg = S.gridx[ref] / S.NX1;
      int t = 0;
      tiles_at(S, Xg, Zg, [&](int u) { t = u; });  // one: the node is not on a tile edge
      const int4 tg = S.tiles[t];
      const int Xn = Xg - 4 * tg.x, Zn = Zg - tg.w;
      if (Xn <= 0 || Zn <= 0 || Xn >= 4 * (tg.z & 0xff) || Zn >= 4 * ((tg.z >> 8) & 0xff))
        return set_err(h, 5, "recorded node %d: not inside its tile", ref + 1);
      if (X.mark_of[t] < 0) {
        X.mark_of[t] = (int)(X.marks.size() / MARK_WORDS);
        X.marks.resize(X.marks.size() + MARK_WORDS, 0u);
      }
      const int p = Zn * PXM + Xn;
      X.marks[(size_t)X.mark_of[t] * MARK_WORDS + (p >> 5)] |= 1u << (p & 31);
    }
  }
  // every split-fault node must be a deferred node: k_deferred leaves those nodes
  // uncorrected and the lane of a fault pair finishes both its nodes; a fault node inside a
  // tile would be corrected by the tile kernel and again there
  {
    size_t nfault_def = 0;
    for (const DefNode& n : X.defs) nfault_def += n.fault ? 1 : 0;
    if (nfault_def != h->fault_n1.size() + h->fault_n2.size())
      return set_err(h, 5, "structured grid: %zu of the %zu split-fault nodes lie on tile edges; the fault "
                     "must follow a row of element edges (ezflt) for the structured path",
                     nfault_def, h->fault_n1.size() + h->fault_n2.size());
  }
  X.rmdef.assign(S.on ? (size_t)nd * ndef : 0, 0.0);  // the general path has it: rmass
  for (size_t q = 0; S.on && q < ndef; ++q)
    for (int c = 0; c < nd; ++c) X.rmdef[(size_t)c * ndef + q] = h->rmass_host[(size_t)c * h->npoin + def_ref[q]];
  return 0;
}

// Wavefronts of a fault's pairs (FaultOut): those of member m, whose pairs start at k0 and
// whose record places start at o0
void fault_waves(const FaultHost& F, int m, int k0, int o0, std::vector<int4>& wave, std::vector<int2>& member,
                 std::vector<int>& slot) {
  const int np = F.dev.np;
  member.push_back(make_int2((int)wave.size(), (np + 63) / 64));
  for (int k = 0; k < np; k += 64) wave.push_back(make_int4(k0 + k, std::min(64, np - k), m, 0));
  const size_t s0 = slot.size();
  slot.resize(s0 + np, -1);
  for (int o = 0; o < F.nout; ++o) slot[s0 + F.oix1 - 1 + (size_t)o * F.oixd] = o0 + o;
}

// Tiles a grid may have for a run of steps in one launch (k_run_steps): as many as there are
// compute units, one workgroup each.  A second one is not sure of a place on any of them: a
// workgroup of six wavefronts takes up to two places on each SIMD, and at the 134 to 254
// registers of the kernels a SIMD has two or three.  (The occupancy query says two workgroups
// for those of SH grids, but they were not resident together: 200 x 150 elements, 475 tiles,
// waited 443 ms to give up where two launches a step take 4.4 ms for 40 steps.)
constexpr int RUN_MAX_TILES = 256;

// Tables of k_run_steps for a grid without faults, element-point terms, Stacey terms,
// receivers inside elements and boundaries that are not flat (other grids: nbr stays null)
int run_tables(sem2d_solver* h, const StructTables& X) {
  StructState& S = h->st;
  S.run_ok = -1;
  if (!S.on || S.ntiles > RUN_MAX_TILES || h->flt.on || S.eta || S.b25 || S.s_nbe > 0 || S.dabson || h->rec_w ||
      h->coef_mode == COEF_PER_ELEM)
    return 0;
  // [ntiles][8] neighbours, [ntiles][SLOTS] deferred nodes, flags, count, fail
  const size_t at_slot = (size_t)S.ntiles * 8, at_flag = at_slot + (size_t)S.ntiles * SLOTS;
  const size_t at_count = at_flag + (size_t)S.ntiles * FLAG_STRIDE;
  std::vector<int> tab(at_count + 2, 0);
  std::fill(tab.begin(), tab.begin() + at_flag, -1);
  for (size_t q = 0; q < X.defs.size(); ++q) {
    const DefNode& n = X.defs[q];
    if (n.pcnt < 1 || n.pcnt > 4) return 0;
    for (int k = 0; k < n.pcnt; ++k) {
      const int o = X.part_off[n.pstart + k];
      tab[at_slot + o] = (int)q;
      int* nb = tab.data() + (size_t)(o / SLOTS) * 8;
      for (int l = 0; l < n.pcnt; ++l) {
        const int u = X.part_off[n.pstart + l] / SLOTS;
        int j = 0;
        while (j < 8 && nb[j] >= 0 && nb[j] != u) ++j;
        if (u == o / SLOTS) continue;
        if (j == 8) return 0;
        nb[j] = u;
      }
    }
  }
  int* p = nullptr;
  int rc = prep_upload(h, &p, tab.data(), tab.size());
  if (rc) return rc;
  HIPCHK(h, hipStreamSynchronize(h->stream));
  S.nbr = p, S.slot_def = p + at_slot;
  S.run_flag = (unsigned*)p + at_flag, S.run_count = (unsigned*)p + at_count;
  S.run_fail = p + at_count + 1;
  S.fpart2 = (char*)S.fpart + S.FPS * h->ndof * rsize(h);
  S.epoch = 0;
  S.run_ok = 0;
  return 0;
}

// Makes the tables of the step kernels and uploads them.
int prepare_structured(sem2d_solver* h) {
  StructState& S = h->st;
  HIPCHK(h, hipStreamSynchronize(h->stream));
  for (void* q : S.prep_allocs) hipFree(q);
  S.prep_allocs.clear();
  StructTables X;
  int rc = struct_tables(h, X);
  if (rc) return rc;
  S.ndef = S.on ? (int)X.defs.size() : h->npoin;
  if (S.on) {
    S.def_ref = X.def_ref;
    if ((rc = prep_upload(h, &S.tiles_dev, X.tiles.data(), X.tiles.size()))) return rc;
    if ((rc = prep_upload(h, &S.grids_dev, X.grids.data(), X.grids.size()))) return rc;
    if ((rc = prep_upload(h, &S.spec_cnt, X.spec_cnt.data(), X.spec_cnt.size()))) return rc;
    if ((rc = prep_upload(h, &S.spec_idx, X.spec_idx.data(), X.spec_idx.size()))) return rc;
    if ((rc = prep_upload(h, &S.mark_of, X.mark_of.data(), X.mark_of.size()))) return rc;
    if ((rc = prep_upload(h, &S.marks, X.marks.data(), X.marks.size()))) return rc;
  }
  {
    std::vector<DefDev> dn;
    std::vector<int4> dx;
    if (!pack_defs(X.defs, X.part_off, dn, dx))
      return set_err(h, 5, "prepare: more than 255 entries at a deferred node");
    DefDev* pn = nullptr;
    int4* px = nullptr;
    if ((rc = prep_upload(h, &pn, dn.data(), dn.size()))) return rc;
    if ((rc = prep_upload(h, &px, dx.data(), dx.size()))) return rc;
    std::vector<DefDev> fd;
    for (int i : X.fault_at) fd.push_back(dn[i]);
    DefDev* pf = nullptr;
    if ((rc = prep_upload(h, &pf, fd.data(), fd.size()))) return rc;
    S.fdef = pf;
    if (!S.on && !dn.empty())
      k_gen_put<<<grid_for(dn.size(), 256), 256, 0, h->stream>>>((int)dn.size(), pn, S.gen_def);
    HIPCHK(h, hipStreamSynchronize(h->stream));  // the packed copies are local
    S.defs.node = S.on ? pn : S.gen_def;
    S.defs.ext = px;
  }
  if (S.on && (rc = prep_upload(h, &S.part_off, X.part_off.data(), X.part_off.size()))) return rc;
  if ((rc = prep_upload(h, &S.dsrc, X.dsrc.data(), X.dsrc.size()))) return rc;
  if ((rc = prep_upload(h, &S.dabso, X.dabso.data(), X.dabso.size()))) return rc;
  S.dabson = nullptr;
  if (!X.dabson.empty() && (rc = prep_upload(h, &S.dabson, X.dabson.data(), X.dabson.size()))) return rc;
  if (S.on) {
    if ((rc = prep_upload_bulk(h, &S.rmdef, X.rmdef))) return rc;
  } else {
    S.rmdef = h->rmass;
  }
  S.FPS = S.on ? (size_t)S.ntiles * SLOTS : (size_t)h->nelem * h->np;
  S.w32 = true;
  if (S.on) {
    // per-cell arrays: the element coefficients and the element-point terms (if any)
    size_t ncell = h->coef_mode == COEF_SHARED ? (size_t)h->nelast * NP
                                               : (size_t)h->nelem * std::max(h->ndof, h->nelast) * NP;
    if (S.eta || S.b25) ncell = std::max(ncell, (size_t)h->nelem * NP);
    S.w32 = fits32(h->fstride, S.FPS, ncell, rsize(h));
  }
  void* fp = nullptr;
  // two arrays for the runs of steps of small grids (k_run_steps)
  HIPCHK(h, hipMalloc(&fp, std::max<size_t>(S.FPS * h->ndof, 1) * rsize(h) * (S.on && S.ntiles <= RUN_MAX_TILES ? 2 : 1)));
  S.prep_allocs.push_back(fp);
  S.fpart = fp;
  S.s_nbe = (int)(X.s_enode.size() / h->ng);
  if (S.s_nbe > 0) {
    if ((rc = prep_upload(h, &S.s_enode, X.s_enode.data(), X.s_enode.size()))) return rc;
    if ((rc = prep_upload(h, &S.s_K, X.s_K.data(), X.s_K.size()))) return rc;
    if ((rc = prep_upload(h, &S.ak_off, X.ak_off.data(), X.ak_off.size()))) return rc;
    if ((rc = prep_upload(h, &S.ak_idx, X.ak_idx.data(), X.ak_idx.size()))) return rc;
    void* q = nullptr;
    HIPCHK(h, hipMalloc(&q, X.s_enode.size() * 2 * sizeof(double)));
    S.prep_allocs.push_back(q);
    S.kxd = (double*)q;
  }
  auto up = [&](const int** p, const std::vector<int>& x) {
    int* q = nullptr;
    const int e = prep_upload(h, &q, x.data(), x.size());
    if (!e) hipStreamSynchronize(h->stream);  // x may be a local copy
    *p = q;
    return e;
  };
  auto up2 = [&](const int** p, const int** r, int* n, const std::vector<std::pair<int, int>>& x) {
    std::vector<int> a, b;
    for (auto& e : x) a.push_back(e.first), b.push_back(e.second);
    *n = (int)x.size();
    const int e = up(p, a);
    return e ? e : up(r, b);
  };
  S.rec = RecOut{};
  if (h->nrec && !h->rec_w) {
    S.rec.seis = h->seis;
    S.rec.nrec = h->nrec, S.rec.isamp = h->isamp, S.rec.nsamp = h->nsamp, S.rec.field = h->field;
    if ((rc = up2(&S.rec.int_g, &S.rec.int_r, &S.rec.nint, X.rec_int))) return rc;
    if ((rc = up2(&S.rec.def_q, &S.rec.def_r, &S.rec.ndefr, X.rec_def))) return rc;
    if ((rc = up2(&S.rec.flt_q, &S.rec.flt_r, &S.rec.nfltr, X.rec_flt))) return rc;
  }
  if (h->flt.on) {
    if ((rc = up(&h->flt.dev.def1, X.fault_def1))) return rc;
    if ((rc = up(&h->flt.dev.def2, X.fault_def2))) return rc;
    S.fo = FaultOut{};
    const FaultHost& FH = h->flt;
    std::vector<int4> wave;
    std::vector<int2> member;
    std::vector<int> slot;
    fault_waves(FH, 0, 0, 0, wave, member, slot);
    int4* wv = nullptr;
    int2* mb = nullptr;
    int* sl = nullptr;
    if ((rc = prep_upload(h, &wv, wave.data(), wave.size()))) return rc;
    if ((rc = prep_upload(h, &mb, member.data(), member.size()))) return rc;
    if ((rc = prep_upload(h, &sl, slot.data(), slot.size()))) return rc;
    S.fo.nwave = (int)wave.size(), S.fo.wave = wv, S.fo.member = mb, S.fo.slot = sl;
    void* q = nullptr;
    HIPCHK(h, hipMalloc(&q, (wave.size() * 6 + 1) * sizeof(double)));
    S.prep_allocs.push_back(q);
    S.fo.part = (double*)q;
    S.fo.cnt = (unsigned*)(S.fo.part + wave.size() * 6);
    HIPCHK(h, hipMemsetAsync(S.fo.cnt, 0, sizeof(double), h->stream));
    HIPCHK(h, hipStreamSynchronize(h->stream));  // the tables are local
    S.fo.nout = FH.nout, S.fo.nsamp = FH.nsamp, S.fo.rec = FH.rec;
    const size_t nside = (size_t)4 * h->ndof * h->fault_n1.size() * rsize(h);
    HIPCHK(h, hipMalloc(&h->flt.dev.side, nside));
    S.prep_allocs.push_back(h->flt.dev.side);
    HIPCHK(h, hipMemsetAsync(h->flt.dev.side, 0, nside, h->stream));
    h->flt.dev.dmask = nullptr;
    bool any = false;
    for (unsigned char m : X.fault_dmask) any |= m != 0;
    if (any) {
      unsigned char* pm = nullptr;
      if ((rc = prep_upload(h, &pm, X.fault_dmask.data(), X.fault_dmask.size()))) return rc;
      HIPCHK(h, hipStreamSynchronize(h->stream));
      h->flt.dev.dmask = pm;
    }
  }
  HIPCHK(h, hipStreamSynchronize(h->stream));
  if ((rc = run_tables(h, X))) return rc;
  S.ready = 1;
  return 0;
}

// The general path goes without tables until what they are made from changes.
void drop_tables(sem2d_solver* h) {
  StructState& S = h->st;
  hipStreamSynchronize(h->stream);
  for (void* q : S.prep_allocs) hipFree(q);
  S.prep_allocs.clear();
  (void)hipGetLastError();
  h->err.clear();
  S.ready = -1;
}

// Everything one structured step launches on: the device tables of one grid (a
// solver) or of many grids sharing the field arrays (a batch).
struct StepDev {
  int ndof = 0, nelast = 0, coef_mode = 0;
  size_t fstride = 0;
  void *d = nullptr, *v = nullptr, *a = nullptr;
  TileDev T{};
  bool w32 = false;  // field, partial-force and per-cell arrays below 4 GiB per component
  int s_nbe = 0;  // Stacey boundary elements (k_stacey_pre), their values passed to k_deferred
  const int* s_enode = nullptr;
  const double* s_K = nullptr;
  StaceyRefs SR{};
  int pipe_wgs = 0;  // persistent workgroups of the tile kernel (0: one per tile)
  const void *rmass0 = nullptr, *coefs = nullptr, *geom = nullptr;
  const void* nodemod = nullptr;  // per-node moduli (COEF_NODE), or null
  const void* elemmod = nullptr;  // per-element moduli (COEF_ELEM), or null
  const void *eta = nullptr, *b25 = nullptr;  // element-point terms (Kelvin-Voigt, 2.5D), or null
  void* fpart = nullptr;
  int ndef = 0;
  DefTable defs;
  const DefDev* fdef = nullptr;
  const int* part_off = nullptr;
  const SrcEntry* dsrc = nullptr;
  const double *dabso = nullptr, *dabson = nullptr;
  int ng = NG;
  const double* hg = nullptr;
  const void* rmdef = nullptr;
  const double* ampl = nullptr;
  int ampl_nt = 0;
  bool fault_on = false;
  FaultDev F{};
  FaultOut fo;
  RecOut recout;
  int* tick = nullptr;      // device step counter that the tile kernel moves on, or null
  const int* itp = nullptr;  // device step counter (graph replay) or null: step index by value
  hipStream_t stream = nullptr;
  bool pin = false;  // the state read is the predicted one (StepOut)
  StepOut out;
  void* rec = nullptr;  // where recorded nodes go (null: the a array)
  const int* mark_of = nullptr;
  const uint32_t* marks = nullptr;
  // out-of-place step (adjoint replay): read the state here, write it to d, v, a
  const void *din = nullptr, *vin = nullptr, *ain = nullptr;
};

StepDev step_dev(sem2d_solver* h) {
  StructState& S = h->st;
  StepDev X;
  X.ndof = h->ndof;
  X.nelast = h->nelast;
  X.coef_mode = h->coef_mode;
  X.fstride = h->fstride;
  X.d = h->d;
  X.v = h->v;
  X.a = h->a;
  X.T.ntiles = S.ntiles;
  X.T.tiles = S.tiles_dev;
  X.T.grids = S.grids_dev;
  X.w32 = S.w32;
  X.s_nbe = S.s_nbe;
  X.s_enode = S.s_enode;
  X.s_K = S.s_K;
  if (S.s_nbe > 0) X.SR = StaceyRefs{S.ak_off, S.ak_idx, S.kxd, S.on ? nullptr : S.s_K};
  X.T.spec_cnt = S.spec_cnt;
  X.T.spec_idx = S.spec_idx;
  X.mark_of = S.mark_of;
  X.marks = S.marks;
  X.T.NGp = h->fstride;
  X.T.FPS = S.FPS;
  X.pipe_wgs = S.pipe_wgs;
  X.rmass0 = S.rmass0;
  X.coefs = S.coefs;
  X.nodemod = S.nodemod;
  X.elemmod = S.elemmod;
  X.eta = S.eta;
  X.b25 = S.b25;
  X.geom = S.geom;
  X.fpart = S.fpart;
  X.ndef = S.ndef;
  X.defs = S.defs, X.fdef = S.fdef;
  X.part_off = S.part_off;
  X.dsrc = S.dsrc;
  X.dabso = S.dabso;
  X.dabson = S.dabson;
  X.ng = h->ng;
  X.hg = h->hg;
  X.rmdef = S.rmdef;
  X.ampl = h->ampl_dev;
  X.ampl_nt = h->ampl_nt;
  X.fault_on = h->flt.on;
  if (h->flt.on) X.F = h->flt.dev, X.fo = S.fo;
  X.recout = S.rec;
  X.stream = h->stream;
  return X;
}

// Tile kernel over all tiles: pipe_wgs persistent workgroups, or one per tile where there
// are fewer tiles (or pipe_wgs is 0).  Compact moduli are read once per node when the grid
// has them in that form.
template <typename R, int MODE>
TileArgs<R> tile_args(const StepDev& X, R dt, R c1, R c2, R c3, R c4) {
  TileArgs<R> A;
  A.d = (R*)X.d, A.v = (R*)X.v, A.a = (R*)X.a;
  A.din = (const R*)X.din, A.vin = (const R*)X.vin, A.ain = (const R*)X.ain;
  A.rmass0 = (const R*)X.rmass0;
  A.coefs = (const R*)(MODE == COEF_NODE ? X.nodemod : (MODE == COEF_ELEM ? X.elemmod : X.coefs));
  A.geom = (const R*)X.geom, A.eta = (const R*)X.eta, A.b25 = (const R*)X.b25;
  A.fpart = (R*)X.fpart;
  A.rec = (R*)(X.rec ? X.rec : X.a);
  A.S = X.T.NGp, A.FPS = X.T.FPS;
  A.tiles = X.T.tiles, A.grids = X.T.grids;
  A.spec_cnt = X.T.spec_cnt, A.spec_idx = X.T.spec_idx;
  A.mark_of = X.mark_of, A.marks = X.marks;
  A.tick = X.tick;
  A.out = X.out;
  A.ntiles = X.T.ntiles;
  A.dt = dt, A.c1 = c1, A.c2 = c2, A.c3 = c3, A.c4 = c4;
  return A;
}
template <typename R, int NDOF, int NELAST, int MODE, bool OOP, bool EP, bool PIN>
void launch_tile_p(const StepDev& X, R dt, R c1, R c2, R c3, R c4) {
  const int per_tile = (X.T.ntiles + 7) / 8 * 8;
  const int wgs = X.pipe_wgs > 0 ? std::min(X.pipe_wgs, per_tile) : per_tile;
  const TileArgs<R> A = tile_args<R, MODE>(X, dt, c1, c2, c3, c4);
  auto go = [&](auto w32) {
    k_tile_step<R, NDOF, NELAST, MODE, OOP, decltype(w32)::value, EP, PIN><<<wgs, TS_NT, 0, X.stream>>>(A);
  };
  if (X.w32) go(std::true_type{});
  else if constexpr (!PIN) go(std::false_type{});  // such grids keep to (d, v, a)
}

template <typename R, int NDOF, int NELAST, int MODE, bool OOP, bool EP>
void launch_tile_k(const StepDev& X, R dt, R c1, R c2, R c3, R c4) {
  if (X.pin) launch_tile_p<R, NDOF, NELAST, MODE, OOP, EP, true>(X, dt, c1, c2, c3, c4);
  else launch_tile_p<R, NDOF, NELAST, MODE, OOP, EP, false>(X, dt, c1, c2, c3, c4);
}

template <typename R, int NDOF, int NELAST, int MODE>
void launch_tile_t(const StepDev& X, R dt, R c1, R c2, R c3, R c4) {
  if constexpr (MODE == COEF_COMPACT) {
    // 400 x 400 P-SV elements, FP64: 50.3 us out of place with the moduli of every point,
    // 46.0 with those of every element (adjoint step 118.6 and 113.6)
    if (X.elemmod) {
      launch_tile_t<R, NDOF, NELAST, COEF_ELEM>(X, dt, c1, c2, c3, c4);
      return;
    }
    if (X.nodemod) {
      launch_tile_t<R, NDOF, NELAST, COEF_NODE>(X, dt, c1, c2, c3, c4);
      return;
    }
  }
  if constexpr ((MODE == COEF_COMPACT || MODE == COEF_NODE || MODE == COEF_ELEM) && NDOF == 2) {
    if (X.din) {  // out of place: the adjoint's forward and replay (P-SV, compact)
      launch_tile_k<R, NDOF, NELAST, MODE, true, false>(X, dt, c1, c2, c3, c4);
      return;
    }
  }
  if (X.eta || X.b25) launch_tile_k<R, NDOF, NELAST, MODE, false, true>(X, dt, c1, c2, c3, c4);
  else launch_tile_k<R, NDOF, NELAST, MODE, false, false>(X, dt, c1, c2, c3, c4);
}

template <typename R, int NDOF, int NELAST>
void launch_tile_m(const StepDev& X, R dt, R c1, R c2, R c3, R c4) {
  switch (X.coef_mode) {
    case COEF_SHARED: launch_tile_t<R, NDOF, NELAST, COEF_SHARED>(X, dt, c1, c2, c3, c4); break;
    case COEF_COMPACT: launch_tile_t<R, NDOF, NELAST, COEF_COMPACT>(X, dt, c1, c2, c3, c4); break;
    default: launch_tile_t<R, NDOF, NELAST, COEF_PER_ELEM>(X, dt, c1, c2, c3, c4);
  }
}
template <typename R>
DefArgs<R> def_args(const StepDev& X, int it, R dt, R c1, R c2, R c3, R c4) {
  DefArgs<R> A;
  A.ndef = X.ndef, A.defs = X.defs, A.part_off = X.part_off;
  A.fpart = (const R*)X.fpart, A.FPS = X.T.FPS;
  A.src = X.dsrc, A.ampl = X.ampl, A.nt = X.ampl_nt, A.it = it, A.itp = X.itp;
  A.abso = X.dabso, A.abson = X.dabson, A.rmdef = (const R*)X.rmdef;
  A.d = (R*)X.d, A.v = (R*)X.v, A.a = (R*)X.a, A.GS = X.fstride;
  A.dt = dt, A.c1 = c1, A.c2 = c2, A.c3 = c3, A.c4 = c4;
  A.so = X.out, A.recp = (R*)(X.rec ? X.rec : X.a);
  A.din = (const R*)X.din, A.vin = (const R*)X.vin, A.ain = (const R*)X.ain;
  A.SR = X.SR, A.rec = X.recout;
  A.rec.src = !X.out.final ? (const void*)A.recp : (A.rec.field == 0 ? X.d : (A.rec.field == 1 ? X.v : X.a));
  A.fdef = X.fdef;
  if (X.fault_on) A.F = X.F, A.fo = X.fo;
  return A;
}


// One step on the tables of a StepDev: the tiles, or (gen: the solver) the elements of the
// general path, then everything else in k_deferred.
template <typename R>
void launch_structured_step(const StepDev& X, int it, R dt, R c1, R c2, R c3, R c4, sem2d_solver* gen = nullptr) {
  if (gen) {
    ElemStep<R> E;
    E.fe = (R*)X.fpart;
    E.stride = X.T.FPS;
    E.a = (const R*)X.a;
    E.dt = dt, E.c1 = c1, E.c2 = c2;
    E.pin = X.pin;
    launch_force<R>(gen, (const R*)X.d, nullptr, (const R*)X.v, E);
  } else if (X.ndof == 2) launch_tile_m<R, 2, 6>(X, dt, c1, c2, c3, c4);
  else launch_tile_m<R, 1, 2>(X, dt, c1, c2, c3, c4);
  if (X.s_nbe > 0)  // Stacey terms from the previous step's state (boundary nodes are deferred)
    k_stacey_pre<R><<<(X.s_nbe * X.ng + 127) / 128, 128, 0, X.stream>>>(
        X.s_nbe, X.s_enode, X.SR.K ? nullptr : X.s_K, (const R*)(X.din ? X.din : X.d), (const R*)(X.din && X.vin ? X.vin : X.v),
        (const R*)(X.din && X.ain ? X.ain : X.a), X.fstride, dt, c1, (double*)X.SR.kxd, X.pin, X.ng,
        X.hg);
  const DefArgs<R> A = def_args<R>(X, it, dt, c1, c2, c3, c4);
  const int lanes = X.ndef + A.rec.nint + (X.fault_on ? A.fo.nwave * 64 : 0);
  auto deferred = [&](auto nd, auto oop, auto pin, auto flt) {
    k_deferred<R, decltype(nd)::value, decltype(oop)::value, decltype(pin)::value, decltype(flt)::value>
        <<<(lanes + 255) / 256, 256, 0, X.stream>>>(A);
  };
  using N1 = std::integral_constant<int, 1>;
  using N2 = std::integral_constant<int, 2>;
  const std::true_type yes{};
  const std::false_type no{};
  if (X.ndof == 2 && X.din) X.pin ? deferred(N2{}, yes, yes, no) : deferred(N2{}, yes, no, no);  // no faults
  else if (X.ndof == 2 && X.fault_on) X.pin ? deferred(N2{}, no, yes, yes) : deferred(N2{}, no, no, yes);
  else if (X.ndof == 2) X.pin ? deferred(N2{}, no, yes, no) : deferred(N2{}, no, no, no);
  else if (X.fault_on) X.pin ? deferred(N1{}, no, yes, yes) : deferred(N1{}, no, no, yes);
  else X.pin ? deferred(N1{}, no, yes, no) : deferred(N1{}, no, no, no);
}

// Predictor / corrector coefficients of one step: dp = d + dt v + c1 a, vp = v + c2 a,
// a' = f / M, v' = vp + c3 a', d' = dp + c4 a'.  Newmark (SRC/solver.f90:58-82):
// c1 = (1/2 - beta) dt^2, c2 = (1 - gamma) dt, c3 = gamma dt, c4 = beta dt^2.  Leapfrog
// (SRC/solver.f90:151-158: d = d + dt v_mid, v_mid = v_mid + dt a) is c1 = c2 = c4 = 0,
// c3 = dt.
template <typename R>
struct StepCoefs {
  R dt, c1, c2, c3, c4;
};
template <typename R>
StepCoefs<R> step_coefs(double dt, double beta, double gamma, int leapfrog) {
  if (leapfrog) return {(R)dt, (R)0, (R)0, (R)dt, (R)0};
  return {(R)dt, (R)((0.5 - beta) * dt * dt), (R)((1.0 - gamma) * dt), (R)(gamma * dt), (R)(beta * dt * dt)};
}

// Periodic boundaries (BC_PERIO_apply, SRC/bc_periodic.f90:78-90): the force of master
// node m[k] becomes f(m) + f(s), slave node s[k] takes it.  The pairs share no node.
template <typename R>
__global__ void k_periodic(int n, const int* __restrict__ m, const int* __restrict__ s, R* __restrict__ f,
                           int npoin, int ndof) {
  const int k = blockIdx.x * blockDim.x + threadIdx.x;
  if (k >= n) return;
  for (int c = 0; c < ndof; ++c) {
    const size_t o = (size_t)c * npoin;
    const R x = f[o + m[k]] + f[o + s[k]];
    f[o + m[k]] = x;
    f[o + s[k]] = x;
  }
}

// Polls of one wait of k_run_steps before it gives up (0.4 us or more each, 55 ms in all;
// a neighbour that is running is there within microseconds); SEM2D_RUN_SPINS sets it, 0 makes
// a launch give up where a neighbour is not there yet.
int run_spins() {
  const char* env = getenv("SEM2D_RUN_SPINS");
  return env ? std::max(0, atoi(env)) : 1 << 17;
}

// Steps from which a run of them is one launch of k_run_steps: the launch, its start and
// end and the check that it went through cost some 30 us more than two launches, and a step
// saves 8 (100 x 100 P-SV elements, FP64: 14.2 -> 6.0 us).
constexpr int RUN_MIN = 16;
// Steps h->it + 1 .. h->it + n from the predicted state to the final one in one launch;
// *done: whether they were taken (the state is unchanged otherwise)
template <typename R, int NDOF, int NELAST, int MODE>
int launch_run_k(sem2d_solver* h, const StepDev& X, int n, const StepCoefs<R>& K, bool* done) {
  StructState& S = h->st;
  *done = false;
  const void* kern = (const void*)k_run_steps<R, NDOF, NELAST, MODE>;
  if (S.run_ok == 0) {
    int dev = 0, ncu = 0, coop = 0, per = 0;
    HIPCHK(h, hipGetDevice(&dev));
    HIPCHK(h, hipDeviceGetAttribute(&ncu, hipDeviceAttributeMultiprocessorCount, dev));
    HIPCHK(h, hipDeviceGetAttribute(&coop, hipDeviceAttributeCooperativeLaunch, dev));
    HIPCHK(h, hipOccupancyMaxActiveBlocksPerMultiprocessor(&per, kern, TS_NT, 0));
    S.run_ok = coop && per > 0 && S.ntiles <= ncu ? 1 : -1;
    if (S.run_ok < 0) return 0;
  }
  HIPCHK(h, hipMemsetAsync(S.run_count, 0, sizeof(unsigned), h->stream));
  RunArgs<R> A;
  A.T = tile_args<R, MODE>(X, K.dt, K.c1, K.c2, K.c3, K.c4);
  A.D = def_args<R>(X, h->it + 1, K.dt, K.c1, K.c2, K.c3, K.c4);
  A.fpart2 = (R*)S.fpart2;
  A.nbr = S.nbr, A.slot_def = S.slot_def;
  A.flag = S.run_flag, A.arrived = S.run_count, A.fail = S.run_fail;
  A.epoch = S.epoch;
  A.nsteps = n;
  A.spins = run_spins();
  void* args[] = {&A};
  if (hipLaunchCooperativeKernel(kern, dim3(S.ntiles), dim3(TS_NT), args, 0, h->stream) != hipSuccess) {
    (void)hipGetLastError();  // one process at a time has the device's cooperative queue
    S.run_ok = -1;
    return 0;
  }
  S.epoch += n;
  int fail = 0;
  HIPCHK(h, hipMemcpyAsync(&fail, S.run_fail, sizeof(int), hipMemcpyDeviceToHost, h->stream));
  HIPCHK(h, hipStreamSynchronize(h->stream));
  if (fail) S.run_ok = -1;  // the device is shared with something that keeps tiles waiting
  ++(fail ? S.runs_given_up : S.runs_taken);
  *done = !fail;
  return 0;
}
template <typename R>
int launch_run(sem2d_solver* h, const StepDev& X, int n, const StepCoefs<R>& K, bool* done) {
  if (X.ndof == 2) {
    if (X.coef_mode == COEF_SHARED) return launch_run_k<R, 2, 6, COEF_SHARED>(h, X, n, K, done);
    if (X.elemmod) return launch_run_k<R, 2, 6, COEF_ELEM>(h, X, n, K, done);
    if (X.nodemod) return launch_run_k<R, 2, 6, COEF_NODE>(h, X, n, K, done);
    return launch_run_k<R, 2, 6, COEF_COMPACT>(h, X, n, K, done);
  }
  if (X.coef_mode == COEF_SHARED) return launch_run_k<R, 1, 2, COEF_SHARED>(h, X, n, K, done);
  if (X.elemmod) return launch_run_k<R, 1, 2, COEF_ELEM>(h, X, n, K, done);
  if (X.nodemod) return launch_run_k<R, 1, 2, COEF_NODE>(h, X, n, K, done);
  return launch_run_k<R, 1, 2, COEF_COMPACT>(h, X, n, K, done);
}

template <typename R>
int do_steps(sem2d_solver* h, int nsteps) {
  int rc = sync_sources(h);
  if (rc) return rc;
  const size_t n = (size_t)h->ndof * h->npoin;
  R* d = (R*)h->d;
  R* v = (R*)h->v;
  R* a = (R*)h->a;
  const StepCoefs<R> K = step_coefs<R>(h->dt, h->beta, h->gamma, h->leapfrog);
  const R dt = K.dt, c1 = K.c1, c2 = K.c2, c3 = K.c3, c4 = K.c4;
  const int gb = grid_for(n, 256);
  // The general path by elements and nodes (two launches a step) where its tables are there
  // or the call is long enough to pay for them: 24,120 elements NGLL 5 with ten
  // coefficients, 32 steps 2.2 ms against 1.7 by single launches, 64 steps 3.1 against 3.4,
  // 1000 steps 30 against 52; 800 elements NGLL 9, 64 steps 1.1 against 1.8 ms, 1000 steps 12
  // against 37.  Periodic boundaries, HHT-alpha, linear slip faults, incident waves and
  // Stacey terms joined at the ends keep the single launches, and so does what the tables cannot hold.
  bool tables = h->st.on || (!h->hht && !h->nper && !h->nlsf && (h->st.ready > 0 || (h->st.ready == 0 && nsteps >= 64)));
  for (auto& b : h->abso) tables = tables && !b.wxz && !b.ends;
  if (tables && !h->st.on && !h->st.ready) {  // room for the element forces and the node records
    const size_t pts = (size_t)h->nelem * h->np, need = pts * (h->ndof * rsize(h) + 8) + (size_t)h->npoin * 24;
    size_t fr = 0, tot = 0;
    tables = pts <= (size_t)65536 * 256 && hipMemGetInfo(&fr, &tot) == hipSuccess && need + need / 4 < fr;
  }
  if (tables && !h->st.ready && (rc = prepare_structured(h))) {
    if (h->st.on) return rc;
    // the general path: more entries at a node than a record counts, a fault whose pairs
    // share nodes, no memory left; the launches one by one need no tables
    drop_tables(h);
    tables = false;
  }
  if (h->flt.on && (rc = potency_reserve(h, h->flt.pot_rows + nsteps))) return rc;
  if (h->itinfo > 0 && (rc = info_reserve(h, h->info_rows + (h->it + nsteps) / h->itinfo - h->it / h->itinfo)))
    return rc;
  StepDev X;
  if (tables) X = step_dev(h);
  HIPCHK(h, hipEventRecord(h->ev0, h->stream));
  for (int s = 0; s < nsteps; ++s) {
    const int it = h->it + 1;
    if (tables && X.pin && h->st.run_ok >= 0) {
      // up to the call's last step or the next progress row
      int n = nsteps - s;
      if (h->itinfo > 0) n = std::min(n, h->itinfo - h->it % h->itinfo);
      bool done = false;
      if (n >= RUN_MIN && (rc = launch_run<R>(h, X, n, K, &done))) return rc;
      if (done) {
        for (int k = 1; k <= n; ++k)
          if (sampled(h, h->it + k)) h->taken = std::max(h->taken, (h->it + k) / h->isamp + 1);
        h->it += n;
        X.pin = false;
        record_info<R>(h, h->it);
        s += n - 1;
        continue;
      }
    }
    if (tables) {
      // the steps between hand the predicted state on (StepOut); the call's last step and
      // those with a progress row store d, v and a
      X.out.final = !X.w32 || s == nsteps - 1 || (h->itinfo > 0 && it % h->itinfo == 0);
      X.out.rec = !X.out.final && sampled(h, it) ? h->field : -1;
      if (h->flt.on) fault_out_step(h, it, X.fo);
      launch_structured_step<R>(X, it, dt, c1, c2, c3, c4, h->st.on ? nullptr : h);
      X.pin = !X.out.final;
      h->it = it;
      if (h->flt.on) fault_out_done(h, it);
      if (h->rec_w) record_receivers<R>(h, !X.out.final);
      else if (sampled(h, it)) h->taken = std::max(h->taken, it / h->isamp + 1);
      record_info<R>(h, it);
      continue;
    }
    // HHT-alpha: the forces, absorbing terms and sources see the fields at n + alpha
    R* df = d;
    R* vf = v;
    if (h->hht) {
      df = (R*)h->da;
      vf = (R*)h->va;
      k_predict_hht<R><<<gb, 256, 0, h->stream>>>(n, d, v, a, df, vf, dt, c1, c2, (R)h->alpha,
                                                  (R)(1.0 - h->alpha));
    } else {
      k_predict<R><<<gb, 256, 0, h->stream>>>(n, d, v, a, dt, c1, c2);
    }
    launch_force<R>(h, df, a, h->kv_eta ? vf : nullptr);
    if (!h->src_host.empty())
      k_sources<R><<<1, 64, 0, h->stream>>>((int)h->src_host.size(), h->src_dev, h->ampl_dev, h->ampl_nt, it, a,
                                           h->npoin);
    // periodic boundaries first among the boundary conditions (SRC/bc_gen.f90:273-275)
    if (h->nper)
      k_periodic<R><<<grid_for(h->nper, 128), 128, 0, h->stream>>>(h->nper, h->per_m, h->per_s, a, h->npoin,
                                                                  h->ndof);
    // the boundary conditions' time: it*dt, or t_alpha = it*dt + (alpha-1) dt for HHT-alpha
    // (SRC/main.f90:53, SRC/solver.f90:114-119)
    const double tbc = h->hht ? (double)it * h->dt + (h->alpha - 1.0) * h->dt : (double)it * h->dt;
    for (auto& b : h->abso) {
      if (b.wxz)
        k_abso_wave<R><<<grid_for(b.n, 128), 128, 0, h->stream>>>(b.n, h->ndof, b.node, b.C, b.wxz, b.wV, b.wT,
                                                                  b.wB, b.wp, tbc, vf, a, h->npoin);
      else if (b.nrm)
        k_abso_normal<R><<<grid_for(b.n, 128), 128, 0, h->stream>>>(b.n, b.node, b.C, b.nrm, vf, a, h->npoin);
      else
        k_abso<R><<<grid_for(b.n, 128), 128, 0, h->stream>>>(b.n, h->ndof, b.node, b.C, vf, a, h->npoin);
      if (b.nbe)
        k_stacey<R><<<grid_for(b.n, 128), 128, 0, h->stream>>>(b.n, b.node, b.soff, b.sidx, b.enode, b.K, df, a,
                                                                h->npoin, h->ng, h->hg);
    }
    // the other boundary conditions in their order (SRC/bc_gen.f90:273-281)
    for (auto& D : h->dirs)
      if (!D.after_fault)
        k_dirichlet<R><<<grid_for(D.node.size(), 128), 128, 0, h->stream>>>((int)D.node.size(), D.node_dev, D.comp,
                                                                           h->ndof, a, h->npoin);
    if (h->nlsf)
      k_lsf<R><<<grid_for(h->nlsf, 128), 128, 0, h->stream>>>(h->nlsf, h->ndof, h->lsf_n1, h->lsf_n2, h->lsf_nrm,
                                                             h->lsf_B, h->lsf_W1, h->lsf_W2, h->lsf_kt, h->lsf_kn,
                                                             df, a, h->npoin);
    if (h->flt.on)
        h->ndof == 2 ? (k_fault<R, 2><<<grid_for(h->flt.dev.np, 64), 64, 0, h->stream>>>(h->flt.dev, d, v, a, h->npoin, tbc))
                   : (k_fault<R, 1><<<grid_for(h->flt.dev.np, 64), 64, 0, h->stream>>>(h->flt.dev, d, v, a, h->npoin, tbc));
    for (auto& D : h->dirs)
      if (D.after_fault)
        k_dirichlet<R><<<grid_for(D.node.size(), 128), 128, 0, h->stream>>>((int)D.node.size(), D.node_dev, D.comp,
                                                                           h->ndof, a, h->npoin);
    k_correct<R><<<gb, 256, 0, h->stream>>>(n, d, v, a, (const R*)h->rmass, c3, c4);
    h->it = it;
    record_receivers<R>(h);
    record_fault(h);
    record_info<R>(h, it);
  }
  HIPCHK(h, hipEventRecord(h->ev1, h->stream));
  HIPCHK(h, hipGetLastError());
  HIPCHK(h, hipEventSynchronize(h->ev1));
  float ms = 0.f;
  HIPCHK(h, hipEventElapsedTime(&ms, h->ev0, h->ev1));
  h->last_ms = nsteps > 0 ? ms / nsteps : 0.0;
  if (h->flt.on) {
    int flag = 0;
    HIPCHK(h, hipMemcpy(&flag, h->flags, sizeof(int), hipMemcpyDeviceToHost));
    if (flag) return set_err(h, 20, "NR_Solver has exceeded the maximum iterations (200)");
  }
  if (h->itinfo > 0) {
    int cnt[2] = {0, 0};
    HIPCHK(h, hipMemcpy(cnt, h->info_cnt, sizeof cnt, hipMemcpyDeviceToHost));
    if (cnt[1]) return set_err(h, 21, "non-finite field values at step %d", cnt[1]);
  }
  return 0;
}

}  // namespace

extern "C" {

int sem2d_create(const sem2d_desc* s, sem2d_solver** out) {
  if (!s || !out) return 1;
  *out = nullptr;
  if (s->ngll < 3 || s->ngll > NGMAX) return 2;
  if (!(s->ndof == 1 || s->ndof == 2)) return 2;
  if (s->ndof == 2 && s->nelast != 6 && s->nelast != 10) return 2;
  if (s->ndof == 1 && s->nelast != 2 && s->nelast != 3) return 2;
  if (s->nelem <= 0 || s->npoin <= 0 || !s->ibool || !s->hprime || !s->rmass) return 2;
  if (s->coef_mode < 0 || s->coef_mode > 2) return 2;
  if (s->coef_mode == COEF_COMPACT &&
      (!s->lam_mu || !s->geom || !s->wgll || (s->nelast != 2 && s->nelast != 6) || s->ngll != NG))
    return 2;
  if (s->coef_mode != COEF_COMPACT && !s->coefs) return 2;
  sem2d_solver* h = new sem2d_solver();
  *out = h;
  h->ndof = s->ndof;
  h->nelem = s->nelem;
  h->npoin = s->npoin;
  h->nelast = s->nelast;
  h->coef_mode = s->coef_mode;
  h->fp32 = s->bulk_fp32 ? 1 : 0;
  h->dt = s->dt;
  h->beta = s->beta;
  h->gamma = s->gamma;
  h->ng = s->ngll;
  h->np = s->ngll * s->ngll;
  const int NG = h->ng, NP = h->np;  // this problem's NGLL from here on
  for (size_t k = 0; k < (size_t)s->nelem * NP; ++k)
    if (s->ibool[k] < 1 || s->ibool[k] > s->npoin) return set_err(h, 3, "ibool entry %zu out of range", k);
  h->elem_ibool.resize((size_t)s->nelem * NP);
  for (size_t k = 0; k < (size_t)s->nelem * NP; ++k) h->elem_ibool[k] = s->ibool[k] - 1;
  HIPCHK(h, hipStreamCreate(&h->stream));
  HIPCHK(h, hipEventCreate(&h->ev0));
  HIPCHK(h, hipEventCreate(&h->ev1));
  if (!scratch_on_device(h)) return 10;  // set-up of sem2d_compute_fint_noalloc's scratch
  std::vector<double> Hc((size_t)NP);
  for (int i = 0; i < NG; ++i)
    for (int j = 0; j < NG; ++j) Hc[i * NG + j] = s->hprime[j * NG + i];
  int rc = upload(h, &h->hg, Hc.data(), Hc.size());
  if (rc) return rc;
  // the NGLL = 5 kernels read H from constant memory (the same values for every problem)
  if (NG == sem2d::NG)
  {
    HIPCHK(h, hipMemcpyToSymbol(HIP_SYMBOL(c_H), Hc.data(), NP * sizeof(double), 0, hipMemcpyHostToDevice));
    const std::vector<float> Hf(Hc.begin(), Hc.end());
    HIPCHK(h, hipMemcpyToSymbol(HIP_SYMBOL(c_Hf), Hf.data(), NP * sizeof(float), 0, hipMemcpyHostToDevice));
  }
  if (s->coef_mode == COEF_COMPACT) {
    double W2[sem2d::NP];
    for (int j = 0; j < NG; ++j)
      for (int i = 0; i < NG; ++i) W2[j * NG + i] = s->wgll[i] * s->wgll[j];
    HIPCHK(h, hipMemcpyToSymbol(HIP_SYMBOL(c_W2), W2, sizeof W2, 0, hipMemcpyHostToDevice));
  }

  std::vector<int> colour;
  int ncol = 0;
  rc = build_colours(h, s, colour, ncol);
  if (rc) return rc;
  h->colour_start.assign(ncol + 1, 0);
  for (int e = 0; e < s->nelem; ++e) h->colour_start[colour[e] + 1]++;
  for (int c = 0; c < ncol; ++c) h->colour_start[c + 1] += h->colour_start[c];
  std::vector<int> pos(h->colour_start.begin(), h->colour_start.end() - 1);
  h->elem_order.assign(s->nelem, 0);
  for (int e = 0; e < s->nelem; ++e) h->elem_order[pos[colour[e]]++] = e;
  std::vector<int> ib((size_t)s->nelem * NP);
  for (int k = 0; k < s->nelem; ++k) {
    int e = h->elem_order[k];
    for (int p = 0; p < NP; ++p) ib[(size_t)k * NP + p] = s->ibool[(size_t)e * NP + p] - 1;
  }
  if ((rc = upload(h, &h->ibool, ib.data(), ib.size()))) return rc;
  const size_t per = h->coef_mode == COEF_COMPACT ? (size_t)h->ndof * NP : (size_t)h->nelast * NP;
  const double* rows = h->coef_mode == COEF_COMPACT ? s->lam_mu : s->coefs;
  std::vector<int> to(s->nelem);  // per-element arrays follow the colour-sorted element order
  for (int k = 0; k < s->nelem; ++k) to[h->elem_order[k]] = k;
  if (h->coef_mode == COEF_SHARED && (rc = upload_bulk(h, &h->coefs, s->coefs, (size_t)h->nelast * NP))) return rc;
  const size_t nf = (size_t)h->ndof * h->npoin;
  if ((rc = upload_bulk(h, &h->rmass, s->rmass, nf))) return rc;
  h->rmass_host.assign(s->rmass, s->rmass + nf);
  h->fstride = (size_t)h->npoin;
  // tile kernels: NGLL 5 and flat-element coefficients (nelast 6 or 2)
  if (NG == sem2d::NG && (h->nelast == 6 || h->nelast == 2) && structured_map(h, s)) {
    StructState& S = h->st;
    S.on = true;
    S.cell_elem.resize(s->nelem);
    for (int cell = 0; cell < s->nelem; ++cell) S.cell_elem[cell] = s->elem_of_cell[cell] - 1;
    h->fstride = S.NS;
    std::vector<double> rm0(S.NS, 0.0);
    for (int k = 0; k < h->npoin; ++k) rm0[S.gmap[k]] = s->rmass[k];
    if ((rc = upload_bulk(h, &S.rmass0, rm0.data(), rm0.size()))) return rc;
    if (h->coef_mode == COEF_SHARED) {
      S.coefs = h->coefs;
    } else {
      // per-element arrays in cell order (iz*nx + ix) as well
      std::vector<int> tc(s->nelem);
      for (int cell = 0; cell < s->nelem; ++cell) tc[S.cell_elem[cell]] = cell;
      if ((rc = upload_rows(h, rows, s->nelem, (int)per, {{&h->coefs, &to}, {&S.coefs, &tc}}))) return rc;
      if (h->coef_mode == COEF_COMPACT) {
        if ((rc = upload_rows(h, s->geom, s->nelem, 3, {{&h->geom, &to}, {&S.geom, &tc}}))) return rc;
        // the moduli once per element, if its points hold bitwise the same values (a medium
        // given by element)
        const int nde = h->ndof;
        const size_t nrow = (size_t)s->nelem * nde;
        bool flat = true;
        for (size_t r = 0; r < nrow && flat; ++r)
          for (int p = 1; p < NP && flat; ++p)
            flat = std::memcmp(s->lam_mu + r * NP, s->lam_mu + r * NP + p, sizeof(double)) == 0;
        std::vector<double> em(flat ? nrow : 0);
        for (size_t r = 0; r < em.size(); ++r) em[r] = s->lam_mu[r * NP];
        if (flat && (rc = upload_rows(h, em.data(), s->nelem, nde, {{&S.elemmod, &tc}}))) return rc;
        // the moduli once per node, if every element at a node holds bitwise the same
        // values there (a medium given as a function of position)
        const int nd = h->ndof;
        std::vector<double> nm(flat ? 0 : (size_t)nd * S.NS, 0.0);
        std::vector<unsigned char> seen(flat ? 0 : S.NS, 0);
        bool same = !flat;
        for (int e = 0; e < s->nelem && same; ++e)
          for (int p = 0; p < NP && same; ++p) {
            const size_t g = S.gmap[s->ibool[(size_t)e * NP + p] - 1];
            for (int c = 0; c < nd; ++c) {
              const double x = s->lam_mu[((size_t)e * nd + c) * NP + p];
              double& y = nm[(size_t)c * S.NS + g];
              if (!seen[g]) y = x;
              else if (std::memcmp(&x, &y, sizeof x) != 0) same = false;
            }
            seen[g] = 1;
          }
        if (same && (rc = upload_bulk(h, &S.nodemod, nm.data(), nm.size()))) return rc;
      }
    }
  }
  if (!h->st.on && h->coef_mode != COEF_SHARED) {
    if ((rc = upload_rows(h, rows, s->nelem, (int)per, {{&h->coefs, &to}}))) return rc;
    if (h->coef_mode == COEF_COMPACT && (rc = upload_rows(h, s->geom, s->nelem, 3, {{&h->geom, &to}}))) return rc;
  }
  const size_t nfs = (size_t)h->ndof * h->fstride;
  if ((rc = dev_alloc(h, (char**)&h->d, nfs * rsize(h)))) return rc;
  if ((rc = dev_alloc(h, (char**)&h->v, nfs * rsize(h)))) return rc;
  if ((rc = dev_alloc(h, (char**)&h->a, nfs * rsize(h)))) return rc;
  if ((rc = dev_alloc(h, &h->flags, 4))) return rc;
  if ((rc = dev_alloc(h, &h->info_acc, 2))) return rc;
  if ((rc = dev_alloc(h, &h->info_cnt, 2))) return rc;
  HIPCHK(h, hipMemsetAsync(h->info_acc, 0, 2 * sizeof(unsigned long long), h->stream));
  HIPCHK(h, hipMemsetAsync(h->info_cnt, 0, 2 * sizeof(int), h->stream));
  HIPCHK(h, hipMemsetAsync(h->d, 0, nfs * rsize(h), h->stream));
  HIPCHK(h, hipMemsetAsync(h->v, 0, nfs * rsize(h), h->stream));
  HIPCHK(h, hipMemsetAsync(h->a, 0, nfs * rsize(h), h->stream));
  HIPCHK(h, hipMemsetAsync(h->flags, 0, 4 * sizeof(int), h->stream));
  HIPCHK(h, hipStreamSynchronize(h->stream));
  return 0;
}

int sem2d_set_abso(sem2d_solver* h, int n, const int* node, const double* C) {
  if (!h) return 1;
  if (n <= 0 || !node || !C) return set_err(h, 3, "set_abso: empty boundary");
  std::vector<int> nd(n);
  for (int k = 0; k < n; ++k) {
    if (node[k] < 1 || node[k] > h->npoin) return set_err(h, 3, "set_abso: node out of range");
    nd[k] = node[k] - 1;
  }
  AbsoDev b;
  b.n = n;
  int rc = upload(h, &b.node, nd.data(), nd.size());
  if (rc) return rc;
  if ((rc = upload(h, &b.C, C, (size_t)h->ndof * n))) return rc;
  h->abso.push_back(b);
  AbsoHost ah;
  ah.node = nd;
  ah.C.assign(C, C + (size_t)h->ndof * n);
  h->abso_host.push_back(ah);
  h->st.ready = 0;
  return 0;
}

int sem2d_set_abso_normals(sem2d_solver* h, int n, const double* nrm) {
  if (!h) return 1;
  if (h->abso.empty()) return set_err(h, 3, "set_abso_normals: call sem2d_set_abso first");
  if (h->ndof != 2) return set_err(h, 3, "set_abso_normals: P-SV only");
  if (h->st.on)
    return set_err(h, 3, "set_abso_normals: a boundary that is not flat needs a solver on the general path");
  AbsoDev& ad = h->abso.back();
  if (!nrm || n != ad.n) return set_err(h, 3, "set_abso_normals: size differs from the boundary's");
  h->abso_host.back().nrm.assign(nrm, nrm + (size_t)2 * n);
  h->st.ready = 0;
  return upload(h, &ad.nrm, nrm, (size_t)2 * n);
}

int sem2d_set_abso_stacey(sem2d_solver* h, int nbe, const int* enode, const double* K) {
  if (!h) return 1;
  if (h->abso.empty()) return set_err(h, 3, "set_abso_stacey: call sem2d_set_abso first");
  if (h->ndof != 2) return set_err(h, 3, "set_abso_stacey: P-SV only");
  if (nbe < 1 || !enode || !K) return set_err(h, 3, "set_abso_stacey: empty");
  AbsoHost& ah = h->abso_host.back();
  AbsoDev& ad = h->abso.back();
  if (ad.nbe) return set_err(h, 3, "set_abso_stacey: this boundary already has its Stacey term");
  const int n = (int)ah.node.size();
  const int NG = h->ng;  // edge points per boundary element
  for (int k = 0; k < nbe * NG; ++k)
    if (enode[k] < 0 || enode[k] >= n) return set_err(h, 3, "set_abso_stacey: node out of range");
  ah.senode.assign(enode, enode + (size_t)nbe * NG);
  ah.sK.assign(K, K + (size_t)nbe * NG * 2);
  // general path: global nodes of the edge points, per boundary node its element points
  std::vector<int> eg((size_t)nbe * NG), off(n + 1, 0), idx((size_t)nbe * NG);
  for (int k = 0; k < nbe * NG; ++k) {
    eg[k] = ah.node[enode[k]];
    off[enode[k] + 1]++;
  }
  for (int q = 0; q < n; ++q) off[q + 1] += off[q];
  std::vector<int> fill(off.begin(), off.end() - 1);
  for (int k = 0; k < nbe * NG; ++k) idx[fill[enode[k]]++] = k;  // element order
  int rc;
  if ((rc = upload(h, &ad.enode, eg.data(), eg.size()))) return rc;
  if ((rc = upload(h, &ad.K, K, (size_t)nbe * NG * 2))) return rc;
  if ((rc = upload(h, &ad.soff, off.data(), off.size()))) return rc;
  if ((rc = upload(h, &ad.sidx, idx.data(), idx.size()))) return rc;
  ad.nbe = nbe;
  h->st.ready = 0;
  return 0;
}

static int use_general_path(sem2d_solver* h);

int sem2d_set_abso_periodic(sem2d_solver* h) {
  if (!h) return 1;
  if (h->abso.empty()) return set_err(h, 3, "set_abso_periodic: call sem2d_set_abso first");
  AbsoHost& ah = h->abso_host.back();
  AbsoDev& ad = h->abso.back();
  if (!ad.nbe) return set_err(h, 3, "set_abso_periodic: the boundary has no Stacey term");
  if (h->st.eta || h->st.b25)
    return set_err(h, 4, "set_abso_periodic: not with Kelvin-Voigt or 2.5D terms on a structured grid");
  int rc = use_general_path(h);
  if (rc) return rc;
  // both end nodes take the Stacey contributions of the first end node, then the last's
  // (SRC/bc_abso.f90:325-328)
  const int n = (int)ah.node.size(), NG = h->ng, nbe = ad.nbe;
  std::vector<std::vector<int>> lists(n);
  for (int k = 0; k < nbe * NG; ++k) lists[ah.senode[k]].push_back(k);  // element order
  std::vector<int> ends = lists[0];
  ends.insert(ends.end(), lists[n - 1].begin(), lists[n - 1].end());
  lists[0] = ends;
  lists[n - 1] = ends;
  std::vector<int> off(n + 1, 0), idx;
  for (int q = 0; q < n; ++q) {
    idx.insert(idx.end(), lists[q].begin(), lists[q].end());
    off[q + 1] = (int)idx.size();
  }
  if ((rc = upload(h, &ad.soff, off.data(), off.size()))) return rc;
  if ((rc = upload(h, &ad.sidx, idx.data(), idx.size()))) return rc;
  ad.ends = true;
  return 0;
}

int sem2d_set_force(sem2d_solver* h, int iglob, const double* dir, int* isrc) {
  if (!h) return 1;
  if (iglob < 1 || iglob > h->npoin) return set_err(h, 3, "set_force: node out of range");
  const int s = h->nsrc++;
  if (h->ndof == 1) {
    h->src_host.push_back({iglob - 1, 0, s, 1.0});
  } else {
    if (!dir) return set_err(h, 3, "set_force: dir required for P-SV");
    h->src_host.push_back({iglob - 1, 0, s, dir[0]});
    h->src_host.push_back({iglob - 1, 1, s, dir[1]});
  }
  h->stf.emplace_back();
  h->src_dirty = true;
  h->st.ready = 0;
  if (isrc) *isrc = s;
  return 0;
}

int sem2d_set_moment(sem2d_solver* h, int nel, const int* ixi, const int* ieta, const double* cxi,
                     const double* ceta, int* isrc) {
  if (!h) return 1;
  if (nel <= 0 || !ixi || !ieta || !cxi || !ceta) return set_err(h, 3, "set_moment: empty stencil");
  const int s = h->nsrc++;
  const int NG = h->ng;  // stencil points per element line
  for (int k = 0; k < nel; ++k) {
    // order of SRC/src_moment.f90:229-232: xi line (all components), then eta line
    for (int c = 0; c < h->ndof; ++c)
      for (int q = 0; q < NG; ++q) {
        int g = ixi[k * NG + q];
        if (g < 1 || g > h->npoin) return set_err(h, 3, "set_moment: node out of range");
        h->src_host.push_back({g - 1, c, s, cxi[((size_t)k * h->ndof + c) * NG + q]});
      }
    for (int c = 0; c < h->ndof; ++c)
      for (int q = 0; q < NG; ++q) {
        int g = ieta[k * NG + q];
        if (g < 1 || g > h->npoin) return set_err(h, 3, "set_moment: node out of range");
        h->src_host.push_back({g - 1, c, s, ceta[((size_t)k * h->ndof + c) * NG + q]});
      }
  }
  h->stf.emplace_back();
  h->src_dirty = true;
  h->st.ready = 0;
  if (isrc) *isrc = s;
  return 0;
}

int sem2d_set_stf(sem2d_solver* h, int isrc, int nt, const double* ampl) {
  if (!h) return 1;
  if (isrc < 0 || isrc >= h->nsrc) return set_err(h, 3, "set_stf: bad source index %d", isrc);
  if (nt < 0 || (nt > 0 && !ampl)) return set_err(h, 3, "set_stf: bad table");
  h->stf[isrc].assign(ampl, ampl + nt);
  h->src_dirty = true;
  return 0;
}

int sem2d_set_receivers(sem2d_solver* h, int nrec, const int* iglob, int isamp, int field, int nsamp) {
  if (!h) return 1;
  if (nrec <= 0 || !iglob || isamp < 1 || field < 0 || field > 2 || nsamp < 1)
    return set_err(h, 3, "set_receivers: bad arguments");
  std::vector<int> nd(nrec), ref(nrec);
  for (int r = 0; r < nrec; ++r) {
    if (iglob[r] < 1 || iglob[r] > h->npoin) return set_err(h, 3, "set_receivers: node out of range");
    nd[r] = ref[r] = iglob[r] - 1;
    if (h->st.on) nd[r] = h->st.gmap[nd[r]];
  }
  int rc = upload(h, &h->rec_node, nd.data(), nd.size());
  if (rc) return rc;
  h->rec_w = nullptr;
  h->rec_ref = std::move(ref);
  h->st.ready = 0;  // the tables mark the recorded nodes
  if ((rc = dev_alloc(h, &h->seis, (size_t)nsamp * h->ndof * nrec))) return rc;
  h->nrec = nrec;
  h->isamp = isamp;
  h->field = field;
  h->nsamp = nsamp;
  h->taken = 0;
  if (h->fp32) rc = record_receivers<float>(h);
  else rc = record_receivers<double>(h);
  HIPCHK(h, hipStreamSynchronize(h->stream));
  return rc;
}

// the fused tile kernels have neither the viscous nor the 2.5D term: a structured grid
// with either uses the general element path, with the fields in the reference numbering
static int use_general_path(sem2d_solver* h) {
  h->st.ready = 0;
  if (h->st.on) {
    h->st.on = false;
    h->fstride = (size_t)h->npoin;
    const size_t nfs = (size_t)h->ndof * h->fstride * rsize(h);
    HIPCHK(h, hipMemsetAsync(h->d, 0, nfs, h->stream));
    HIPCHK(h, hipMemsetAsync(h->v, 0, nfs, h->stream));
    HIPCHK(h, hipMemsetAsync(h->a, 0, nfs, h->stream));
  }
  return 0;
}

// per-element-point array in the colour-sorted element order of the general path
static int upload_elem_points(sem2d_solver* h, void** dst, const double* src) {
  const int NP = h->np;
  std::vector<double> e((size_t)h->nelem * NP);
  for (int k = 0; k < h->nelem; ++k)
    std::memcpy(&e[(size_t)k * NP], src + (size_t)h->elem_order[k] * NP, NP * sizeof(double));
  return upload_bulk(h, dst, e.data(), e.size());
}

// per-element-point array in cell order for the tile kernel of a structured grid
static int upload_cell_points(sem2d_solver* h, void** dst, const double* src) {
  StructState& S = h->st;
  const int NP = h->np;
  std::vector<double> c((size_t)h->nelem * NP);
  for (int cell = 0; cell < h->nelem; ++cell)
    std::memcpy(&c[(size_t)cell * NP], src + (size_t)S.cell_elem[cell] * NP, NP * sizeof(double));
  int rc = upload_bulk(h, dst, c.data(), c.size());
  if (rc) return rc;
  // one workgroup per CU: the variant's LDS allows no more
  int dev = 0, ncu = 256;
  if (hipGetDevice(&dev) == hipSuccess) hipDeviceGetAttribute(&ncu, hipDeviceAttributeMultiprocessorCount, dev);
  S.pipe_wgs = ((ncu + 7) / 8) * 8;
  S.ready = 0;
  return 0;
}

int sem2d_set_kelvin_voigt(sem2d_solver* h, const double* eta) {
  if (!h) return 1;
  if (!eta) return set_err(h, 3, "set_kelvin_voigt: null eta");
  if (h->it != 0 || h->nrec || h->flt.on || h->nsrc || !h->abso.empty())
    return set_err(h, 4, "set_kelvin_voigt: call it right after sem2d_create");
  if (h->st.on && (h->nelast == 6 || h->nelast == 2)) return upload_cell_points(h, &h->st.eta, eta);
  int rc = use_general_path(h);
  if (rc) return rc;
  return upload_elem_points(h, &h->kv_eta, eta);
}

int sem2d_set_25d(sem2d_solver* h, const double* beta) {
  if (!h) return 1;
  if (!beta) return set_err(h, 3, "set_25d: null beta");
  if (h->it != 0 || h->nrec || h->flt.on || h->nsrc || !h->abso.empty())
    return set_err(h, 4, "set_25d: call it right after sem2d_create");
  // the general element kernel's copy serves sem2d_compute_fint
  int rc = upload_elem_points(h, &h->beta25, beta);
  if (rc) return rc;
  if (h->st.on && (h->nelast == 6 || h->nelast == 2)) return upload_cell_points(h, &h->st.b25, beta);
  return use_general_path(h);
}

int sem2d_set_periodic(sem2d_solver* h, int n, const int* master, const int* slave) {
  if (!h) return 1;
  if (n <= 0 || !master || !slave) return set_err(h, 3, "set_periodic: bad arguments");
  if (h->it != 0 || h->nrec || h->flt.on || h->nsrc || !h->abso.empty())
    return set_err(h, 4, "set_periodic: call it right after sem2d_create");
  if (h->st.eta || h->st.b25 || h->kv_eta || h->beta25)
    return set_err(h, 4, "set_periodic: call it before sem2d_set_kelvin_voigt and sem2d_set_25d");
  if (h->nper) return set_err(h, 3, "set_periodic: one periodic boundary per solver");
  std::vector<char> mark(h->npoin, 0);
  std::vector<int> m(n), sl(n);
  for (int k = 0; k < n; ++k) {
    m[k] = master[k] - 1;
    sl[k] = slave[k] - 1;
    if (m[k] < 0 || m[k] >= h->npoin || sl[k] < 0 || sl[k] >= h->npoin || m[k] == sl[k] || mark[m[k]] ||
        mark[sl[k]])
      return set_err(h, 3, "set_periodic: nodes out of range or repeated");
    mark[m[k]] = mark[sl[k]] = 1;
  }
  // the pairs act on the reference numbering: the general element path
  int rc = use_general_path(h);
  if (rc) return rc;
  if ((rc = upload(h, &h->per_m, m.data(), n))) return rc;
  if ((rc = upload(h, &h->per_s, sl.data(), n))) return rc;
  h->nper = n;
  return 0;
}

int sem2d_set_receivers_interp(sem2d_solver* h, int nrec, const int* elem, const double* interp, int isamp,
                               int field, int nsamp) {
  if (!h) return 1;
  if (nrec <= 0 || !elem || !interp || isamp < 1 || field < 0 || field > 2 || nsamp < 1)
    return set_err(h, 3, "set_receivers_interp: bad arguments");
  if (h->elem_ibool.empty()) return set_err(h, 4, "set_receivers_interp: element table not kept");
  const int NP = h->np;
  std::vector<int> nd((size_t)nrec * NP), ref((size_t)nrec * NP);
  for (int r = 0; r < nrec; ++r) {
    if (elem[r] < 1 || elem[r] > h->nelem) return set_err(h, 3, "set_receivers_interp: element out of range");
    for (int k = 0; k < NP; ++k) {
      int g = h->elem_ibool[(size_t)(elem[r] - 1) * NP + k];
      nd[(size_t)r * NP + k] = h->st.on ? h->st.gmap[g] : g;
      ref[(size_t)r * NP + k] = g;
    }
  }
  h->rec_ref = std::move(ref);
  h->st.ready = 0;  // the tables mark the recorded nodes
  int rc = upload(h, &h->rec_node, nd.data(), nd.size());
  if (rc) return rc;
  if ((rc = upload(h, &h->rec_w, interp, (size_t)nrec * NP))) return rc;
  if ((rc = dev_alloc(h, &h->seis, (size_t)nsamp * h->ndof * nrec))) return rc;
  h->nrec = nrec;
  h->isamp = isamp;
  h->field = field;
  h->nsamp = nsamp;
  h->taken = 0;
  if (h->fp32) rc = record_receivers<float>(h);
  else rc = record_receivers<double>(h);
  HIPCHK(h, hipStreamSynchronize(h->stream));
  return rc;
}

int sem2d_set_fault(sem2d_solver* h, const sem2d_fault_desc* f, int nsamp) {
  if (!h) return 1;
  if (!f || f->npoin <= 0 || nsamp < 1) return set_err(h, 3, "set_fault: bad arguments");
  if (h->flt.on) return set_err(h, 3, "set_fault: only one fault per solver");
  if (h->nlsf) return set_err(h, 4, "set_fault: not combined with a linear slip fault");
  if (f->law < 1 || f->law > 3)
    return set_err(h, 3, "set_fault: law must be 1 (SWF), 2 (RSF) or 3 (time weakening, sem2d_set_fault_twf)");
  if ((f->law == 1 && (f->kind < 1 || f->kind > 3)) || (f->law == 2 && (f->kind < 1 || f->kind > 4)))
    return set_err(h, 3, "set_fault: invalid friction kind");
  if (f->oitd < 1 || f->oixd < 1 || f->oix1 < 1 || f->oixn > f->npoin || f->oixn < f->oix1)
    return set_err(h, 3, "set_fault: bad output decimation");
  const int np = f->npoin, nd = h->ndof;
  FaultHost& F = h->flt;
  FaultDev& D = F.dev;
  D.np = np;
  D.ndof = nd;
  // node2 == NULL: a fault with one side, on a domain boundary (symmetry; the
  // reference's bc2 and invM2 are then undefined, SRC/bc_dynflt.f90:256-259)
  const bool two = f->node2 != nullptr;
  if (two && !f->invM2) return set_err(h, 3, "set_fault: invM2 needed with node2");
  std::vector<int> n1(np), n2(np, -1);
  for (int k = 0; k < np; ++k) {
    if (f->node1[k] < 1 || f->node1[k] > h->npoin || (two && (f->node2[k] < 1 || f->node2[k] > h->npoin)))
      return set_err(h, 3, "set_fault: node out of range");
    n1[k] = f->node1[k] - 1;
    if (two) n2[k] = f->node2[k] - 1;
  }
  h->fault_n1 = n1;
  if (two) h->fault_n2 = n2;
  else h->fault_n2.clear();
  h->st.ready = 0;
  if (h->st.on)
    for (int k = 0; k < np; ++k) {
      n1[k] = h->st.gmap[n1[k]];
      if (two) n2[k] = h->st.gmap[n2[k]];
    }
  int rc;
  int* ip;
  double* dp;
  if ((rc = upload(h, &ip, n1.data(), np))) return rc;
  D.n1 = ip;
  if ((rc = upload(h, &ip, n2.data(), np))) return rc;
  D.n2 = ip;
#define UP(field, src, n)                           \
  if ((rc = upload(h, &dp, (src), (size_t)(n)))) return rc; \
  D.field = dp;
  UP(nrm, f->n1, 2 * np);
  UP(B, f->B, nd * np);
  UP(invM1, f->invM1, nd * np);
  std::vector<double> zero_m((size_t)nd * np, 0.0);
  UP(invM2, two ? f->invM2 : zero_m.data(), nd * np);
  UP(Z, f->Z, nd * np);
  UP(T0, f->T0, 2 * np);
  UP(coh, f->cohesion, np);
  std::vector<double> zero((size_t)2 * np, 0.0);
  const double* pp[6];
  for (int q = 0; q < 6; ++q) pp[q] = f->p[q] ? f->p[q] : zero.data();
  UP(p0, pp[0], np);
  UP(p1, pp[1], np);
  UP(p2, pp[2], np);
  UP(p3, pp[3], np);
  UP(p4, pp[4], np);
  UP(p5, pp[5], np);
  std::vector<double> Tc(np, 0.0), coeft(np, 0.0), mu(np), sig(np), th(np);
  for (int k = 0; k < np; ++k) th[k] = f->theta0 ? f->theta0[k] : 0.0;
  if (f->law == 2)
    for (int k = 0; k < np; ++k) {
      Tc[k] = pp[0][k] / pp[4][k];
      coeft[k] = std::exp(-h->dt / Tc[k]);
    }
  UP(Tc, Tc.data(), np);
  UP(coeft, coeft.data(), np);
  double* theta;
  if ((rc = upload(h, &theta, th.data(), np))) return rc;
  D.theta = theta;
  std::vector<double> V0((size_t)nd * np, 0.0);
  if (f->V0)
    for (int k = 0; k < np; ++k) V0[k] = f->V0[k];
  double *Dd, *Vd, *Td, *Tsd, *MUd, *Sd;
  if ((rc = upload(h, &Dd, zero.data(), (size_t)nd * np))) return rc;
  if ((rc = upload(h, &Vd, V0.data(), (size_t)nd * np))) return rc;
  if ((rc = upload(h, &Td, zero.data(), (size_t)2 * np))) return rc;
  if ((rc = upload(h, &Tsd, zero.data(), (size_t)2 * np))) return rc;
  // initial friction coefficient (SRC/bc_dynflt.f90:404-413), computed on the host
  for (int k = 0; k < np; ++k) {
    sig[k] = f->T0[np + k];
    const double dc = pp[0][k], mus = pp[1][k];
    if (f->law == 3) {  // time weakening alone: set by sem2d_set_fault_twf
      mu[k] = 1.7976931348623157e308;
    } else if (f->law == 1) {
      const double mud = pp[2][k], t = th[k];
      double m;
      if (f->kind == 1) m = mus - (mus - mud) * std::fmin(t / dc, 1.0);
      else if (f->kind == 2) m = mud - (mud - mus) * std::exp(-t / dc);
      else m = mud + (mus - mud) / std::pow(1.0 + t / dc, pp[4][k]);
      mu[k] = m + pp[3][k] * t;
    } else {
      const double a = pp[2][k], b = pp[3][k], vs = pp[4][k], v = V0[k], t = th[k];
      if (f->kind == 1) mu[k] = mus + a * std::fabs(v) / (std::fabs(v) + vs) - b * t / (t + dc);
      else if (f->kind <= 3)
        mu[k] = a * std::asinh(std::fabs(v) / (2.0 * vs) * std::exp((mus + b * std::log(vs * t / dc)) / a));
      else
        mu[k] = a * std::asinh(std::fabs(v) / (2.0 * vs) *
                               std::exp((mus + b * std::log(pp[5][k] * t / dc + 1)) / a));
    }
  }
  if ((rc = upload(h, &MUd, mu.data(), np))) return rc;
  if ((rc = upload(h, &Sd, sig.data(), np))) return rc;
#undef UP
  D.D = Dd;
  D.V = Vd;
  D.T = Td;
  D.Tstick = Tsd;
  D.MU = MUd;
  D.sigma = Sd;
  D.a2v = f->coefA2V;
  D.a2d = f->coefA2D;
  D.dt = h->dt;
  D.opening = f->allow_opening;
  D.law = f->law;
  D.kind = f->kind;
  D.healing = f->healing;
  D.nr_fail = h->flags;
  F.oit = f->oit;
  F.oitd = f->oitd;
  F.oix1 = f->oix1;
  F.oixn = f->oixn;
  F.oixd = f->oixd;
  F.nout = (f->oixn - f->oix1) / f->oixd + 1;
  F.nsamp = nsamp;
  F.taken = 0;
  if ((rc = dev_alloc(h, &F.rec, (size_t)nsamp * 6 * F.nout))) return rc;
  F.on = true;
  if ((rc = potency_reserve(h, 1024))) return rc;
  record_fault(h);
  HIPCHK(h, hipStreamSynchronize(h->stream));
  return 0;
}

int sem2d_step(sem2d_solver* h, int nsteps) {
  if (!h) return 1;
  if (nsteps < 0) return set_err(h, 3, "step: negative nsteps");
  return h->fp32 ? do_steps<float>(h, nsteps) : do_steps<double>(h, nsteps);
}

// device field (grid order when structured) -> host array in reference order
static int fetch_field(sem2d_solver* h, double* out, const void* dev) {
  const size_t n = (size_t)h->ndof * h->npoin;
  if (!h->st.on) return read_bulk(h, out, dev, n);
  const size_t S = h->fstride;
  std::vector<double> tmp((size_t)h->ndof * S);
  int rc = read_bulk(h, tmp.data(), dev, tmp.size());
  if (rc) return rc;
  for (int c = 0; c < h->ndof; ++c)
    for (int k = 0; k < h->npoin; ++k) out[(size_t)c * h->npoin + k] = tmp[(size_t)c * S + h->st.gmap[k]];
  return 0;
}

static int store_field(sem2d_solver* h, void* dev, const double* in) {
  const size_t n = (size_t)h->ndof * h->npoin;
  if (!h->st.on) return write_bulk(h, dev, in, n);
  const size_t S = h->fstride;
  std::vector<double> tmp((size_t)h->ndof * S, 0.0);
  for (int c = 0; c < h->ndof; ++c)
    for (int k = 0; k < h->npoin; ++k) tmp[(size_t)c * S + h->st.gmap[k]] = in[(size_t)c * h->npoin + k];
  return write_bulk(h, dev, tmp.data(), tmp.size());
}

int sem2d_fetch_fields(sem2d_solver* h, double* d, double* v, double* a) {
  if (!h) return 1;
  int rc = 0;
  if (d && (rc = fetch_field(h, d, h->d))) return rc;
  if (v && (rc = fetch_field(h, v, h->v))) return rc;
  if (a && (rc = fetch_field(h, a, h->a))) return rc;
  return 0;
}

int sem2d_set_fields(sem2d_solver* h, const double* d, const double* v, const double* a) {
  if (!h) return 1;
  int rc = 0;
  if (d && (rc = store_field(h, h->d, d))) return rc;
  if (v && (rc = store_field(h, h->v, v))) return rc;
  if (a && (rc = store_field(h, h->a, a))) return rc;
  return 0;
}

int sem2d_fetch_seismo(sem2d_solver* h, double* out, int* taken) {
  if (!h) return 1;
  if (h->nrec && out)
    HIPCHK(h, hipMemcpy(out, h->seis, (size_t)h->taken * h->ndof * h->nrec * sizeof(double), hipMemcpyDeviceToHost));
  if (taken) *taken = h->taken;
  return 0;
}

int sem2d_fetch_fault(sem2d_solver* h, double* out, int* taken) {
  if (!h) return 1;
  if (!h->flt.on) return set_err(h, 4, "fetch_fault: no fault");
  if (out)
    HIPCHK(h, hipMemcpy(out, h->flt.rec, (size_t)h->flt.taken * 6 * h->flt.nout * sizeof(double),
                        hipMemcpyDeviceToHost));
  if (taken) *taken = h->flt.taken;
  return 0;
}

int sem2d_set_fault_twf(sem2d_solver* h, int kind, const double* par, const double* coord) {
  if (!h) return 1;
  FaultHost& F = h->flt;
  if (!F.on) return set_err(h, 4, "set_fault_twf: call sem2d_set_fault first");
  if (h->it != 0) return set_err(h, 4, "set_fault_twf: the solver has already been stepped");
  if (kind < 1 || kind > 3 || !par || !coord) return set_err(h, 3, "set_fault_twf: bad arguments");
  FaultDev& D = F.dev;
  const int np = D.np;
  D.twf = kind;
  for (int q = 0; q < 9; ++q) D.tw[q] = par[q];
  double* xz = nullptr;
  int rc = upload(h, &xz, coord, (size_t)2 * np);
  if (rc) return rc;
  D.xz = xz;
  // initial friction (SRC/bc_dynflt.f90:404-413): the minimum with the time-weakening
  // coefficient at t = 0, or that coefficient alone (law 3); slip D = 0
  std::vector<double> mu(np);
  HIPCHK(h, hipMemcpy(mu.data(), D.MU, np * sizeof(double), hipMemcpyDeviceToHost));
  for (int k = 0; k < np; ++k) {
    const double mt = twf_mu(kind, par, coord[k], coord[np + k], 0.0, 0.0);
    mu[k] = D.law == 3 ? mt : std::fmin(mu[k], mt);
  }
  HIPCHK(h, hipMemcpy(D.MU, mu.data(), np * sizeof(double), hipMemcpyHostToDevice));
  if (F.taken)  // the friction row of the record of step 0, taken by sem2d_set_fault
    k_fault_record<<<grid_for(F.nout, 64), 64, 0, h->stream>>>(D, F.oix1, F.oixd, F.nout, F.rec);
  HIPCHK(h, hipStreamSynchronize(h->stream));
  return 0;
}

int sem2d_set_abso_wave(sem2d_solver* h, int n, const double* xz, const double* vdir, const double* tdir,
                        const double* B, const double* par) {
  if (!h) return 1;
  if (h->abso.empty()) return set_err(h, 3, "set_abso_wave: call sem2d_set_abso first");
  AbsoDev& ad = h->abso.back();
  if (n != ad.n || !xz || !vdir || !tdir || !B || !par) return set_err(h, 3, "set_abso_wave: bad arguments");
  if (h->it != 0) return set_err(h, 4, "set_abso_wave: the solver has already been stepped");
  if (h->st.eta || h->st.b25)
    return set_err(h, 4, "set_abso_wave: not with Kelvin-Voigt or 2.5D terms on a structured grid");
  int rc = use_general_path(h);  // the incident field acts on the reference numbering
  if (rc) return rc;
  if ((rc = upload(h, &ad.wxz, xz, (size_t)2 * n))) return rc;
  if ((rc = upload(h, &ad.wV, vdir, (size_t)h->ndof * n))) return rc;
  if ((rc = upload(h, &ad.wT, tdir, (size_t)h->ndof * n))) return rc;
  if ((rc = upload(h, &ad.wB, B, (size_t)n))) return rc;
  ad.wp = WavePar{par[0], par[1], par[2], par[3], par[4], par[5], par[6], par[7]};
  return 0;
}

int sem2d_set_lsf(sem2d_solver* h, int n, const int* node1, const int* node2, const double* nrm, const double* B,
                  const double* W1, const double* W2, double kt, double kn) {
  if (!h) return 1;
  if (n <= 0 || !node1 || !node2 || !nrm || !B || !W1 || !W2) return set_err(h, 3, "set_lsf: bad arguments");
  if (h->nlsf) return set_err(h, 3, "set_lsf: one linear slip fault per solver");
  if (h->it != 0) return set_err(h, 4, "set_lsf: the solver has already been stepped");
  if (h->flt.on || !h->dirs.empty())
    return set_err(h, 4, "set_lsf: not combined with a dynamic fault or Dirichlet boundaries");
  if (h->st.eta || h->st.b25)
    return set_err(h, 4, "set_lsf: not with Kelvin-Voigt or 2.5D terms on a structured grid");
  std::vector<int> a(n), b(n);
  for (int k = 0; k < n; ++k) {
    a[k] = node1[k] - 1;
    b[k] = node2[k] - 1;
    if (a[k] < 0 || a[k] >= h->npoin || b[k] < 0 || b[k] >= h->npoin)
      return set_err(h, 3, "set_lsf: node out of range");
  }
  int rc = use_general_path(h);
  if (rc) return rc;
  const size_t nd = (size_t)h->ndof * n;
  if ((rc = upload(h, &h->lsf_n1, a.data(), n)) || (rc = upload(h, &h->lsf_n2, b.data(), n)) ||
      (rc = upload(h, &h->lsf_nrm, nrm, (size_t)2 * n)) || (rc = upload(h, &h->lsf_B, B, nd)) ||
      (rc = upload(h, &h->lsf_W1, W1, nd)) || (rc = upload(h, &h->lsf_W2, W2, nd)))
    return rc;
  h->lsf_kt = kt;
  h->lsf_kn = kn;
  h->nlsf = n;
  return 0;
}

int sem2d_set_hht(sem2d_solver* h, double alpha) {
  if (!h) return 1;
  if (!(alpha >= 0.0 && alpha <= 1.0)) return set_err(h, 3, "set_hht: alpha must lie in [0, 1]");
  if (h->it != 0 || h->nrec || h->flt.on || h->nsrc || !h->abso.empty())
    return set_err(h, 4, "set_hht: call it right after sem2d_create");
  if (h->st.eta || h->st.b25 || h->kv_eta || h->beta25)
    return set_err(h, 4, "set_hht: call it before sem2d_set_kelvin_voigt and sem2d_set_25d");
  if (h->leapfrog) return set_err(h, 4, "set_hht: the solver is set to leapfrog");
  // the fields at n + alpha live in the reference numbering: the general element path
  int rc = use_general_path(h);
  if (rc) return rc;
  if (!h->da) {
    const size_t n = (size_t)h->ndof * h->npoin;
    if (h->fp32) {
      float *p1, *p2;
      if ((rc = dev_alloc(h, &p1, n)) || (rc = dev_alloc(h, &p2, n))) return rc;
      h->da = p1;
      h->va = p2;
    } else {
      double *p1, *p2;
      if ((rc = dev_alloc(h, &p1, n)) || (rc = dev_alloc(h, &p2, n))) return rc;
      h->da = p1;
      h->va = p2;
    }
  }
  h->hht = 1;
  h->alpha = alpha;
  return 0;
}

int sem2d_set_fault_normal(sem2d_solver* h, int kind, double coef, double v) {
  if (!h) return 1;
  FaultHost& F = h->flt;
  if (!F.on) return set_err(h, 4, "set_fault_normal: call sem2d_set_fault first");
  if (h->it != 0) return set_err(h, 4, "set_fault_normal: the solver has already been stepped");
  if (kind < 0 || kind > 3) return set_err(h, 3, "set_fault_normal: kind must be 0 to 3");
  F.dev.nor_kind = kind;
  F.dev.nor_coef = coef;
  F.dev.nor_v = v;
  return 0;
}

int sem2d_set_fault_sides(sem2d_solver* h, int on) {
  if (!h) return 1;
  FaultHost& F = h->flt;
  if (!F.on) return set_err(h, 4, "set_fault_sides: call sem2d_set_fault first");
  if (h->it != 0) return set_err(h, 4, "set_fault_sides: the solver has already been stepped");
  if (!on) {
    F.srec = nullptr;  // the block stays with the handle's allocations
    return 0;
  }
  int rc = dev_alloc(h, &F.srec, (size_t)F.nsamp * 4 * h->ndof * F.nout);
  if (rc) return rc;
  if (F.taken) record_sides(h, 0, 0);  // the record of step 0, taken by sem2d_set_fault
  HIPCHK(h, hipStreamSynchronize(h->stream));
  return 0;
}

int sem2d_fetch_fault_sides(sem2d_solver* h, double* out, int* nsamp_taken) {
  if (!h) return 1;
  FaultHost& F = h->flt;
  if (!F.on || !F.srec) return set_err(h, 4, "fetch_fault_sides: no per-side records (sem2d_set_fault_sides)");
  if (out)
    HIPCHK(h, hipMemcpy(out, F.srec, (size_t)F.taken * 4 * h->ndof * F.nout * sizeof(double),
                        hipMemcpyDeviceToHost));
  if (nsamp_taken) *nsamp_taken = F.taken;
  return 0;
}

int sem2d_fetch_potency(sem2d_solver* h, double* out, int* nrows) {
  if (!h) return 1;
  if (!h->flt.on) return set_err(h, 4, "fetch_potency: no fault");
  if (out && h->flt.pot_rows)
    HIPCHK(h, hipMemcpy(out, h->flt.pot, (size_t)h->flt.pot_rows * 2 * (h->ndof + 1) * sizeof(double),
                        hipMemcpyDeviceToHost));
  if (nrows) *nrows = h->flt.pot_rows;
  return 0;
}

int sem2d_fetch_fault_state(sem2d_solver* h, double* D, double* V, double* T, double* MU, double* Ts) {
  if (!h) return 1;
  if (!h->flt.on) return set_err(h, 4, "fetch_fault_state: no fault");
  const FaultDev& F = h->flt.dev;
  HIPCHK(h, hipStreamSynchronize(h->stream));
  const size_t nd = (size_t)F.ndof * F.np;
  if (D) HIPCHK(h, hipMemcpy(D, F.D, nd * sizeof(double), hipMemcpyDeviceToHost));
  if (V) HIPCHK(h, hipMemcpy(V, F.V, nd * sizeof(double), hipMemcpyDeviceToHost));
  if (T) HIPCHK(h, hipMemcpy(T, F.T, 2 * F.np * sizeof(double), hipMemcpyDeviceToHost));
  if (MU) HIPCHK(h, hipMemcpy(MU, F.MU, F.np * sizeof(double), hipMemcpyDeviceToHost));
  if (Ts) HIPCHK(h, hipMemcpy(Ts, F.Tstick, 2 * F.np * sizeof(double), hipMemcpyDeviceToHost));
  return 0;
}

int sem2d_compute_fint(sem2d_solver* h, const double* d, double* f) {
  if (!h) return 1;
  if (!d || !f) return set_err(h, 3, "compute_fint: null array");
  const size_t n = (size_t)h->ndof * h->npoin;
  void *dd = nullptr, *ff = nullptr;
  HIPCHK(h, hipMalloc(&dd, n * rsize(h)));
  HIPCHK(h, hipMalloc(&ff, n * rsize(h)));
  int rc = write_bulk(h, dd, d, n);
  if (!rc) {
    if (hipMemsetAsync(ff, 0, n * rsize(h), h->stream) != hipSuccess) rc = set_err(h, 10, "memset failed");
  }
  if (!rc) {
    if (h->fp32) launch_force<float>(h, (const float*)dd, (float*)ff);
    else launch_force<double>(h, (const double*)dd, (double*)ff);
    if (hipGetLastError() != hipSuccess) rc = set_err(h, 10, "force kernel launch failed");
  }
  if (!rc) rc = read_bulk(h, f, ff, n);
  hipFree(dd);
  hipFree(ff);
  return rc;
}

int sem2d_compute_fint_noalloc(sem2d_solver* h, const double* d, double* f) {
  if (!h) return 1;
  if (!d || !f) return set_err(h, 3, "compute_fint_noalloc: null array");
  const size_t n = (size_t)h->ndof * h->npoin;
  // 16 bytes of scratch per value.  FP64 fields: d at [0, 8n), f at [8n, 16n).  FP32
  // fields: the host d as doubles at [0, 8n), d as floats at [8n, 12n), f as floats at
  // [12n, 16n), then f as doubles back at [0, 8n) (the double d is consumed by then).
  if (n > NOALLOC_SCRATCH_BYTES / 16)
    return set_err(h, 3, "compute_fint_noalloc: ndof*npoin = %zu exceeds the scratch limit of %zu values",
                   n, NOALLOC_SCRATCH_BYTES / 16);
  unsigned char* base = (unsigned char*)scratch_on_device(h);
  if (!base) return 10;
  double* dd = (double*)base;
  const int nb = grid_for(n, 256);
  HIPCHK(h, hipMemcpyAsync(dd, d, n * sizeof(double), hipMemcpyHostToDevice, h->stream));
  double* out;
  if (h->fp32) {
    float* dr = (float*)(base + 8 * n);
    float* fr = (float*)(base + 12 * n);
    k_to_float<<<nb, 256, 0, h->stream>>>(dd, dr, n);
    k_fill<float><<<nb, 256, 0, h->stream>>>(fr, 0.0f, n);
    launch_force<float>(h, dr, fr);
    k_to_double<<<nb, 256, 0, h->stream>>>(fr, dd, n);
    out = dd;
  } else {
    double* fd = (double*)(base + 8 * n);
    k_fill<double><<<nb, 256, 0, h->stream>>>(fd, 0.0, n);
    launch_force<double>(h, dd, fd);
    out = fd;
  }
  if (hipGetLastError() != hipSuccess) return set_err(h, 10, "compute_fint_noalloc: kernel launch failed");
  HIPCHK(h, hipMemcpyAsync(f, out, n * sizeof(double), hipMemcpyDeviceToHost, h->stream));
  HIPCHK(h, hipStreamSynchronize(h->stream));
  return 0;
}

int sem2d_set_dirichlet(sem2d_solver* h, int n, const int* node, int comp) {
  if (!h) return 1;
  if (n <= 0 || !node) return set_err(h, 3, "set_dirichlet: empty boundary");
  if (comp < 1 || comp > 3 || (h->ndof == 1 && comp != 1))
    return set_err(h, 3, "set_dirichlet: comp must be 1 (component 1), 2 (component 2) or 3 (both; P-SV)");
  if (h->nlsf) return set_err(h, 4, "set_dirichlet: not combined with a linear slip fault");
  sem2d_solver::DirBC D;
  D.node.resize(n);
  for (int k = 0; k < n; ++k) {
    if (node[k] < 1 || node[k] > h->npoin) return set_err(h, 3, "set_dirichlet: node out of range");
    D.node[k] = node[k] - 1;
  }
  D.comp = comp;
  D.after_fault = h->flt.on;
  std::vector<int> dn(D.node);
  if (h->st.on)
    for (int& k : dn) k = h->st.gmap[k];
  int rc = upload(h, &D.node_dev, dn.data(), dn.size());
  if (rc) return rc;
  h->dirs.push_back(std::move(D));
  h->st.ready = 0;
  return 0;
}

int sem2d_set_time_scheme(sem2d_solver* h, int kind) {
  if (!h) return 1;
  if (kind != 0 && kind != 1) return set_err(h, 3, "set_time_scheme: kind must be 0 (newmark) or 1 (leapfrog)");
  if (kind == 1 && (h->beta != 0.0 || h->gamma != 0.5))
    return set_err(h, 3, "set_time_scheme: leapfrog needs beta = 0, gamma = 1/2 in the descriptor");
  if (h->it != 0) return set_err(h, 4, "set_time_scheme: the solver has already been stepped");
  if (kind == 1 && h->hht) return set_err(h, 4, "set_time_scheme: the solver is set to HHT-alpha");
  h->leapfrog = kind;
  return 0;
}

int sem2d_set_itinfo(sem2d_solver* h, int itinfo) {
  if (!h) return 1;
  if (itinfo < 0) return set_err(h, 3, "set_itinfo: negative interval");
  h->itinfo = itinfo;
  return 0;
}

int sem2d_field_info(sem2d_solver* h, double* vmax, double* dmax, int* nonfinite) {
  if (!h) return 1;
  const size_t n = (size_t)h->ndof * h->fstride;
  const int nb = (int)std::min<size_t>((n + 255) / 256, 4096);
  if (h->fp32)
    k_field_max<float><<<nb, 256, 0, h->stream>>>(n, (const float*)h->d, (const float*)h->v, (const float*)h->a,
                                                 h->info_acc, h->info_cnt);
  else
    k_field_max<double><<<nb, 256, 0, h->stream>>>(n, (const double*)h->d, (const double*)h->v,
                                                  (const double*)h->a, h->info_acc, h->info_cnt);
  unsigned long long acc[2];
  int cnt[2];
  HIPCHK(h, hipMemcpyAsync(acc, h->info_acc, sizeof acc, hipMemcpyDeviceToHost, h->stream));
  HIPCHK(h, hipMemcpyAsync(cnt, h->info_cnt, sizeof cnt, hipMemcpyDeviceToHost, h->stream));
  k_info_row<<<1, 64, 0, h->stream>>>(h->it, h->it * h->dt, h->info_acc, h->info_cnt, nullptr);
  HIPCHK(h, hipStreamSynchronize(h->stream));
  double x[2];
  std::memcpy(x, acc, sizeof x);
  if (vmax) *vmax = x[0];
  if (dmax) *dmax = x[1];
  if (nonfinite) *nonfinite = cnt[0];
  return 0;
}

int sem2d_fetch_info(sem2d_solver* h, double* rows, int* nrows) {
  if (!h) return 1;
  if (rows && h->info_rows)
    HIPCHK(h, hipMemcpy(rows, h->info, (size_t)h->info_rows * 4 * sizeof(double), hipMemcpyDeviceToHost));
  if (nrows) *nrows = h->info_rows;
  return 0;
}

int sem2d_set_tile_config(sem2d_solver* h, int threads, int wg_per_cu) {
  if (!h) return 1;
  if (!h->st.on) return set_err(h, 4, "set_tile_config: not a structured (MESH_CART) grid");
  if ((threads != 256 && threads != 512) || wg_per_cu > 4)
    return set_err(h, 3, "set_tile_config: threads must be 256 or 512 and wg_per_cu <= 4");
  StructState& S = h->st;
  int dev = 0, ncu = 256;
  if (hipGetDevice(&dev) == hipSuccess) hipDeviceGetAttribute(&ncu, hipDeviceAttributeMultiprocessorCount, dev);
  if (wg_per_cu < 0) wg_per_cu = tile_wgs_per_cu(h->fp32, h->ndof);  // automatic: the measured defaults
  S.pipe_wgs = ncu * wg_per_cu;
  S.pipe_wgs = ((S.pipe_wgs + 7) / 8) * 8;
  return 0;
}

int sem2d_run_counts(sem2d_solver* h, int* taken, int* given_up) {
  if (!h) return 1;
  if (taken) *taken = h->st.runs_taken;
  if (given_up) *given_up = h->st.runs_given_up;
  return 0;
}

int sem2d_get_step(sem2d_solver* h, int* it) {
  if (!h || !it) return 1;
  *it = h->it;
  return 0;
}

int sem2d_last_step_ms(sem2d_solver* h, double* ms) {
  if (!h || !ms) return 1;
  *ms = h->last_ms;
  return 0;
}

const char* sem2d_last_error(sem2d_solver* h) { return h ? h->err.c_str() : "null handle"; }

void sem2d_destroy(sem2d_solver* h) {
  if (!h) return;
  if (h->stream) hipStreamSynchronize(h->stream);
  if (h->adj) adj_free(h->adj);
  if (h->flt.pot) hipFree(h->flt.pot);
  if (h->info) hipFree(h->info);
  for (void* p : h->allocs) hipFree(p);
  for (void* p : h->st.prep_allocs) hipFree(p);
  for (auto& b : h->abso) { (void)b; }
  if (h->src_dev) hipFree(h->src_dev);
  if (h->ampl_dev) hipFree(h->ampl_dev);
  if (h->ev0) hipEventDestroy(h->ev0);
  if (h->ev1) hipEventDestroy(h->ev1);
  if (h->stream) hipStreamDestroy(h->stream);
  delete h;
}

}  // extern "C"

// ===========================================================================
// Batched ensemble: many independent structured scenarios advanced together.
//
// The member solvers' grids are laid side by side in one set of field arrays
// (member m's storage block starts at node_base[m]; component stride = the sum of
// the members' strides).  Tiles, deferred nodes, sources, absorbing coefficients
// and fault pairs of all members are concatenated with their indices offset, so
// one persistent tile launch and one deferred launch cover every scenario.  The
// step index lives in device memory (it_dev), which lets a captured hipGraph of a
// chunk of steps be replayed for the whole time loop.  Every member performs
// exactly the arithmetic of its own solver, so batch and one-by-one results are
// bitwise identical.
// ===========================================================================
namespace {

template <typename R>
__global__ void k_batch_record(const int* __restrict__ itp, int nrec, int ndof, const int* __restrict__ rec_node,
                               const R* __restrict__ field, size_t fstride, int isamp, int nsamp,
                               double* __restrict__ seis, FaultDev F, const int* __restrict__ fidx, int nout,
                               int oit0, int oitd, int fnsamp, double* __restrict__ frec) {
  const int q = blockIdx.x * blockDim.x + threadIdx.x;
  const int it = *itp;
  if (q < nrec && it % isamp == 0 && it / isamp < nsamp) {
    double* out = seis + (size_t)(it / isamp) * ndof * nrec;
    for (int c = 0; c < ndof; ++c) out[(size_t)c * nrec + q] = (double)field[(size_t)c * fstride + rec_node[q]];
  }
  if (q < nout && it >= oit0 && (it - oit0) % oitd == 0 && (it - oit0) / oitd < fnsamp) {
    double* out = frec + (size_t)((it - oit0) / oitd) * 6 * nout;
    const int k = fidx[q];
    out[0 * nout + q] = F.D[k];
    out[1 * nout + q] = F.V[k];
    out[2 * nout + q] = F.T[k];
    out[3 * nout + q] = F.T[F.np + k];
    out[4 * nout + q] = F.MU[k];
    out[5 * nout + q] = F.Tstick[k];
  }
}

}  // namespace

struct sem2d_batch {
  int n = 0;
  std::vector<sem2d_solver*> mem;
  int ndof = 0, nelast = 0, coef_mode = 0, fp32 = 0;
  double dt = 0, beta = 0, gamma = 0;
  int leapfrog = 0;
  hipStream_t stream = nullptr;
  hipEvent_t ev0 = nullptr, ev1 = nullptr;
  size_t fstride = 0;
  std::vector<size_t> node_base;
  std::vector<int> fault_base, rec_base, fout_base, src_base;
  StepDev X;
  int ncu = 256;
  // records
  int nrec = 0, isamp = 1, field = 1, nsamp = 0;
  int* rec_node = nullptr;
  double* seis = nullptr;
  int fnout = 0, oit0 = 0, oitd = 1, fnsamp = 0;
  int* fidx = nullptr;
  double* frec = nullptr;
  int* it_dev = nullptr;
  int* flags = nullptr;
  int it = 0;
  // potency rows: pot[member][pot_cap][2*(ndof+1)]; the row of the state after step s
  // is pot_shift + s (pot_shift + 1 rows precede the batch's first step)
  double* pot = nullptr;
  int pot_cap = 0, pot_shift = 0;
  // graph of a chunk of steps
  hipGraph_t graph = nullptr;
  hipGraphExec_t gexec = nullptr;
  int gsteps = 0;
  double last_ms = 0.0;
  std::string err;
  std::vector<void*> allocs;
};

namespace {

int berr(sem2d_batch* b, int code, const char* fmt, ...) {
  char buf[512];
  va_list ap;
  va_start(ap, fmt);
  vsnprintf(buf, sizeof buf, fmt, ap);
  va_end(ap);
  if (b) b->err = buf;
  return code;
}

#define BHIPCHK(b, call)                                                                  \
  do {                                                                                    \
    hipError_t e_ = (call);                                                               \
    if (e_ != hipSuccess)                                                                 \
      return berr(b, 10, "%s failed: %s (%s:%d)", #call, hipGetErrorString(e_), __FILE__, __LINE__); \
  } while (0)

template <typename T>
int balloc(sem2d_batch* b, T** p, size_t n) {
  void* q = nullptr;
  hipError_t e = hipMalloc(&q, std::max<size_t>(n, 1) * sizeof(T));
  if (e != hipSuccess) return berr(b, 11, "hipMalloc(%zu bytes): %s", n * sizeof(T), hipGetErrorString(e));
  b->allocs.push_back(q);
  *p = (T*)q;
  return 0;
}

template <typename T>
int bupload(sem2d_batch* b, T** p, const std::vector<T>& src) {
  int rc = balloc(b, p, src.size());
  if (rc) return rc;
  if (!src.empty())
    BHIPCHK(b, hipMemcpyAsync(*p, src.data(), src.size() * sizeof(T), hipMemcpyHostToDevice, b->stream));
  BHIPCHK(b, hipStreamSynchronize(b->stream));
  return 0;
}

int bupload_bulk(sem2d_batch* b, void** p, const std::vector<double>& src) {
  if (!b->fp32) return bupload(b, (double**)p, src);
  std::vector<float> tmp(src.begin(), src.end());
  return bupload(b, (float**)p, tmp);
}

// device -> host copy of n doubles
int bdown(sem2d_batch* b, std::vector<double>& dst, const double* src, size_t n) {
  dst.resize(n);
  if (n) BHIPCHK(b, hipMemcpy(dst.data(), src, n * sizeof(double), hipMemcpyDeviceToHost));
  return 0;
}

int check_members(sem2d_batch* b) {
  sem2d_solver* h0 = b->mem[0];
  for (int m = 0; m < b->n; ++m) {
    sem2d_solver* h = b->mem[m];
    if (!h) return berr(b, 3, "member %d is null", m);
    if (!h->st.on) return berr(b, 3, "member %d is not a structured (MESH_CART) grid", m);
    if (h->it != 0) return berr(b, 3, "member %d has already been stepped", m);
    if (h->ndof != h0->ndof || h->nelast != h0->nelast || h->coef_mode != h0->coef_mode || h->fp32 != h0->fp32)
      return berr(b, 3, "member %d: ndof, element kernel, coefficient mode and bulk precision must match", m);
    if (h->dt != h0->dt || h->beta != h0->beta || h->gamma != h0->gamma || h->leapfrog != h0->leapfrog)
      return berr(b, 3, "member %d: time step, time scheme and Newmark parameters must match", m);
    if (h->flt.on != h0->flt.on) return berr(b, 3, "member %d: either every member has a fault or none", m);
    if (h->flt.srec) return berr(b, 3, "member %d: per-side fault records (osides) are not batched", m);
    if (h->flt.on && h->flt.dev.twf) return berr(b, 3, "member %d: time-weakening friction is not batched", m);
    if (h->flt.on && h->flt.dev.nor_kind != 1)
      return berr(b, 3, "member %d: normal stress laws other than Coulomb are not batched", m);
    for (const AbsoHost& B : h->abso_host)
      if (!B.senode.empty()) return berr(b, 3, "member %d: Stacey boundaries are not batched", m);
    if (h->st.eta || h->st.b25) return berr(b, 3, "member %d: Kelvin-Voigt and 2.5D terms are not batched", m);
    if (h->flt.on && h->fault_n2.empty())
      return berr(b, 3, "member %d: faults with one side (on a domain boundary) are not batched", m);
    if (!h->dirs.empty()) return berr(b, 3, "member %d: Dirichlet boundaries are not batched", m);
    if (h->flt.on) {
      const FaultDev &F = h->flt.dev, &F0 = h0->flt.dev;
      if (F.law != F0.law || F.kind != F0.kind || F.opening != F0.opening || F.healing != F0.healing ||
          F.a2v != F0.a2v || F.a2d != F0.a2d)
        return berr(b, 3, "member %d: fault law, kind, opening, healing and time coefficients must match", m);
      const int oit0 = h->flt.oit - h->flt.taken * h->flt.oitd;
      const int oit00 = h0->flt.oit - h0->flt.taken * h0->flt.oitd;
      if (h->flt.oitd != h0->flt.oitd || oit0 != oit00)
        return berr(b, 3, "member %d: fault output times must match", m);
    }
  }
  return 0;
}

void batch_drop_graph(sem2d_batch* b);

// room for `rows` potency rows per member (outside any captured graph: a new buffer
// drops the graph, whose launches hold the old address).  The rows already recorded
// (pot_shift + 1 + it) move over; the first reservation takes them from the members.
int batch_pot_reserve(sem2d_batch* b, int rows) {
  if (rows <= b->pot_cap) return 0;
  const int cap = std::max(rows, 2 * b->pot_cap);
  const size_t nc = 2 * (size_t)(b->ndof + 1);
  const int have = b->pot ? b->pot_shift + 1 + b->it : b->pot_shift + 1;
  double* p = nullptr;
  BHIPCHK(b, hipMalloc(&p, (size_t)b->n * cap * nc * sizeof(double)));
  for (int m = 0; m < b->n; ++m) {
    const double* src = b->pot ? b->pot + (size_t)m * b->pot_cap * nc : b->mem[m]->flt.pot;
    if (have > 0)
      BHIPCHK(b, hipMemcpyAsync(p + (size_t)m * cap * nc, src, (size_t)have * nc * sizeof(double),
                                hipMemcpyDeviceToDevice, b->stream));
  }
  BHIPCHK(b, hipStreamSynchronize(b->stream));
  if (b->pot) hipFree(b->pot);
  b->pot = p;
  b->pot_cap = cap;
  b->X.fo.pot = p;
  b->X.fo.pot_cap = cap;
  batch_drop_graph(b);
  return 0;
}

// concatenate the device-resident per-member arrays that only exist on the device
int gather_fault(sem2d_batch* b) {
  const int nd = b->ndof;
  int np = 0;
  b->fault_base.assign(b->n, 0);
  for (int m = 0; m < b->n; ++m) {
    b->fault_base[m] = np;
    np += b->mem[m]->flt.dev.np;
  }
  FaultDev F = b->mem[0]->flt.dev;
  F.np = np;
  std::vector<int> n1, n2;
  std::vector<double> cat[22];
  // arrays and their row counts ([rows][np] layout)
  struct Arr { const double* FaultDev::*p; int rows; };
  const Arr arrs[] = {{&FaultDev::nrm, 2}, {&FaultDev::B, nd},    {&FaultDev::invM1, nd}, {&FaultDev::invM2, nd},
                      {&FaultDev::Z, nd},  {&FaultDev::T0, 2},    {&FaultDev::coh, 1},    {&FaultDev::p0, 1},
                      {&FaultDev::p1, 1},  {&FaultDev::p2, 1},    {&FaultDev::p3, 1},     {&FaultDev::p4, 1},
                      {&FaultDev::p5, 1},  {&FaultDev::Tc, 1},    {&FaultDev::coeft, 1}};
  struct State { double* FaultDev::*p; int rows; };
  const State states[] = {{&FaultDev::theta, 1}, {&FaultDev::D, nd},     {&FaultDev::V, nd}, {&FaultDev::T, 2},
                          {&FaultDev::Tstick, 2}, {&FaultDev::MU, 1},    {&FaultDev::sigma, 1}};
  const int na = sizeof(arrs) / sizeof(arrs[0]), ns = sizeof(states) / sizeof(states[0]);
  for (int q = 0; q < na; ++q) cat[q].assign((size_t)arrs[q].rows * np, 0.0);
  for (int q = 0; q < ns; ++q) cat[na + q].assign((size_t)states[q].rows * np, 0.0);
  for (int m = 0; m < b->n; ++m) {
    const FaultDev& Fm = b->mem[m]->flt.dev;
    const int nm = Fm.np, o = b->fault_base[m];
    std::vector<int> t1(nm), t2(nm);
    BHIPCHK(b, hipMemcpy(t1.data(), Fm.n1, nm * sizeof(int), hipMemcpyDeviceToHost));
    BHIPCHK(b, hipMemcpy(t2.data(), Fm.n2, nm * sizeof(int), hipMemcpyDeviceToHost));
    for (int k = 0; k < nm; ++k) {
      n1.push_back((int)(t1[k] + b->node_base[m]));
      n2.push_back((int)(t2[k] + b->node_base[m]));
    }
    std::vector<double> tmp;
    for (int q = 0; q < na + ns; ++q) {
      const int rows = q < na ? arrs[q].rows : states[q - na].rows;
      const double* src = q < na ? Fm.*(arrs[q].p) : Fm.*(states[q - na].p);
      int rc = bdown(b, tmp, src, (size_t)rows * nm);
      if (rc) return rc;
      for (int r = 0; r < rows; ++r)
        std::copy(tmp.begin() + (size_t)r * nm, tmp.begin() + (size_t)(r + 1) * nm, cat[q].begin() + (size_t)r * np + o);
    }
  }
  int rc;
  int* ip;
  if ((rc = bupload(b, &ip, n1))) return rc;
  F.n1 = ip;
  if ((rc = bupload(b, &ip, n2))) return rc;
  F.n2 = ip;
  for (int q = 0; q < na + ns; ++q) {
    double* dp;
    if ((rc = bupload(b, &dp, cat[q]))) return rc;
    if (q < na) F.*(arrs[q].p) = dp;
    else F.*(states[q - na].p) = dp;
  }
  F.nr_fail = b->flags;
  b->X.fault_on = true;
  b->X.F = F;
  // potency: the rows recorded before the batch (one per member at fault set-up; equal for
  // all members, none of which has been stepped)
  const int r0 = b->mem[0]->flt.pot_rows;
  for (int m = 0; m < b->n; ++m)
    if (b->mem[m]->flt.pot_rows != r0) return berr(b, 3, "member %d: potency rows differ from member 0's", m);
  if (r0 < 1) return berr(b, 3, "batch: members have no potency row of step 0");
  b->pot_shift = r0 - 1;
  if ((rc = batch_pot_reserve(b, r0))) return rc;
  // fault records: output nodes oix1:oixn:oixd of every member, member after member
  std::vector<int> fidx;
  b->fout_base.assign(b->n, 0);
  b->fnsamp = 0;
  for (int m = 0; m < b->n; ++m) {
    const FaultHost& H = b->mem[m]->flt;
    b->fout_base[m] = (int)fidx.size();
    for (int o = 0; o < H.nout; ++o) fidx.push_back(b->fault_base[m] + H.oix1 - 1 + o * H.oixd);
    b->fnsamp = std::max(b->fnsamp, H.nsamp);
  }
  b->fnout = (int)fidx.size();
  const FaultHost& H0 = b->mem[0]->flt;
  b->oitd = H0.oitd;
  b->oit0 = H0.oit - H0.taken * H0.oitd;
  if ((rc = bupload(b, &b->fidx, fidx))) return rc;
  if ((rc = balloc(b, &b->frec, (size_t)b->fnsamp * 6 * std::max(b->fnout, 1)))) return rc;
  return 0;
}

// the records of step 0, from the members' state
template <typename R>
void launch_batch_record(sem2d_batch* b) {
  const int nq = std::max(std::max(b->nrec, b->fnout), 1);
  const R* fld = (const R*)(b->field == 0 ? b->X.d : (b->field == 1 ? b->X.v : b->X.a));
  k_batch_record<R><<<grid_for(nq, 64), 64, 0, b->stream>>>(b->it_dev, b->nrec, b->ndof, b->rec_node, fld,
                                                            b->fstride, b->isamp, b->nsamp, b->seis, b->X.F,
                                                            b->fidx, b->fnout, b->oit0, b->oitd, b->fnsamp,
                                                            b->frec);
}

// nsteps steps that read the predicted state (pin) or (d, v, a); the last one stores the
// latter (final), the others the former (StepOut)
template <typename R>
void launch_batch_steps(sem2d_batch* b, int nsteps, bool pin, bool final) {
  const StepCoefs<R> K = step_coefs<R>(b->dt, b->beta, b->gamma, b->leapfrog);
  const R dt = K.dt, c1 = K.c1, c2 = K.c2, c3 = K.c3, c4 = K.c4;
  for (int s = 0; s < nsteps; ++s) {
    b->X.pin = b->X.w32 && (pin || s > 0);
    b->X.out.final = !b->X.w32 || (final && s == nsteps - 1);
    b->X.out.rec = !b->X.out.final && b->nrec ? b->field : -1;
    launch_structured_step<R>(b->X, 0, dt, c1, c2, c3, c4);
  }
}

void batch_drop_graph(sem2d_batch* b) {
  if (b->gexec) hipGraphExecDestroy(b->gexec);
  if (b->graph) hipGraphDestroy(b->graph);
  b->gexec = nullptr;
  b->graph = nullptr;
  b->gsteps = 0;
}

int batch_graph(sem2d_batch* b, int chunk) {
  if (b->gexec && b->gsteps == chunk) return 0;
  batch_drop_graph(b);
  BHIPCHK(b, hipStreamBeginCapture(b->stream, hipStreamCaptureModeThreadLocal));
  if (b->fp32) launch_batch_steps<float>(b, chunk, true, false);
  else launch_batch_steps<double>(b, chunk, true, false);
  BHIPCHK(b, hipStreamEndCapture(b->stream, &b->graph));
  BHIPCHK(b, hipGraphInstantiate(&b->gexec, b->graph, nullptr, nullptr, 0));
  b->gsteps = chunk;
  return 0;
}

// launch configuration of the tile kernel: workgroups per CU (0: one workgroup per tile)
void batch_set_config(sem2d_batch* b, int per_cu) {
  b->X.pipe_wgs = per_cu > 0 ? ((b->ncu * per_cu + 7) / 8) * 8 : 0;
  batch_drop_graph(b);
}

int batch_run(sem2d_batch* b, int nsteps, bool use_graph) {
  // the first and the last step apart (they read and store d, v, a), the graph's steps in
  // between hand the predicted state on
  const int mid = nsteps - 2, chunk = std::min(mid, 64);
  if (b->X.fault_on) {
    int rc = batch_pot_reserve(b, b->pot_shift + 1 + b->it + nsteps);
    if (rc) return rc;
  }
  if (use_graph && chunk > 0) {
    int rc = batch_graph(b, chunk);
    if (rc) return rc;
  }
  BHIPCHK(b, hipEventRecord(b->ev0, b->stream));
  auto direct = [&](int n, bool pin, bool final) {
    if (b->fp32) launch_batch_steps<float>(b, n, pin, final);
    else launch_batch_steps<double>(b, n, pin, final);
  };
  int done = 0;
  if (use_graph && chunk > 0) {
    direct(1, false, false);
    for (; done + chunk <= mid; done += chunk) BHIPCHK(b, hipGraphLaunch(b->gexec, b->stream));
    ++done;
  }
  if (done < nsteps) direct(nsteps - done, done > 0, true);
  BHIPCHK(b, hipEventRecord(b->ev1, b->stream));
  BHIPCHK(b, hipGetLastError());
  BHIPCHK(b, hipEventSynchronize(b->ev1));
  float ms = 0.f;
  BHIPCHK(b, hipEventElapsedTime(&ms, b->ev0, b->ev1));
  b->last_ms = nsteps > 0 ? ms / nsteps : 0.0;
  b->it += nsteps;
  if (b->X.fault_on) {
    int flag = 0;
    BHIPCHK(b, hipMemcpy(&flag, b->flags, sizeof(int), hipMemcpyDeviceToHost));
    if (flag) return berr(b, 20, "NR_Solver has exceeded the maximum iterations (200)");
  }
  return 0;
}

int rec_taken(const sem2d_batch* b) { return b->nrec ? std::min(b->nsamp, b->it / b->isamp + 1) : 0; }
int flt_taken(const sem2d_batch* b) {
  if (!b->X.fault_on || b->it < b->oit0) return 0;
  return std::min(b->fnsamp, (b->it - b->oit0) / b->oitd + 1);
}

}  // namespace

extern "C" {

int sem2d_batch_create(int n, sem2d_solver* const* members, sem2d_batch** out) {
  if (!out) return 1;
  *out = nullptr;
  if (n <= 0 || !members) return 2;
  sem2d_batch* b = new sem2d_batch();
  *out = b;
  b->n = n;
  b->mem.assign(members, members + n);
  int rc = check_members(b);
  if (rc) return rc;
  sem2d_solver* h0 = b->mem[0];
  b->ndof = h0->ndof;
  b->nelast = h0->nelast;
  b->coef_mode = h0->coef_mode;
  b->fp32 = h0->fp32;
  b->dt = h0->dt;
  b->beta = h0->beta;
  b->gamma = h0->gamma;
  b->leapfrog = h0->leapfrog;
  const int nd = b->ndof;
  const size_t rs = b->fp32 ? sizeof(float) : sizeof(double);
  BHIPCHK(b, hipStreamCreate(&b->stream));
  BHIPCHK(b, hipEventCreate(&b->ev0));
  BHIPCHK(b, hipEventCreate(&b->ev1));
  {
    int dev = 0;
    if (hipGetDevice(&dev) == hipSuccess) hipDeviceGetAttribute(&b->ncu, hipDeviceAttributeMultiprocessorCount, dev);
  }
  // member tables, concatenated
  StructTables A;
  std::vector<double> rmdef_c[2];
  std::vector<SrcEntry> dsrc;
  std::vector<double> ampl;
  int ampl_nt = 0, nsrc = 0;
  for (int m = 0; m < n; ++m) {
    sem2d_solver* h = b->mem[m];
    if ((rc = sync_sources(h))) return berr(b, rc, "member %d: %s", m, h->err.c_str());
    ampl_nt = std::max(ampl_nt, h->ampl_nt);
  }
  ampl_nt = std::max(ampl_nt, 1);  // every source owns a row of the table
  b->node_base.assign(n, 0);
  b->src_base.assign(n, 0);
  size_t nb = 0, cb = 0, shared_off = 0;
  int nrec = 0;
  for (int m = 0; m < n; ++m) {
    sem2d_solver* h = b->mem[m];
    StructTables X;
    if ((rc = struct_tables(h, X))) return berr(b, rc, "member %d: %s", m, h->err.c_str());
    b->node_base[m] = nb;
    const int tb = (int)A.tiles.size(), pb = (int)A.part_off.size(), sb = (int)A.dsrc.size();
    const int ab = (int)(A.dabso.size() / nd);
    const int cellw = b->coef_mode == COEF_SHARED ? (int)shared_off : (int)cb;
    if (nb + h->st.NS > 0x7fffffffULL || cb + h->nelem > 0x7fffffffULL) return berr(b, 5, "batch too large");
    for (size_t t = 0; t < X.tiles.size(); ++t) {
      A.tiles.push_back(X.tiles[t]);
      A.grids.push_back(make_int4((int)nb, X.grids[t].y, X.grids[t].z, cellw));
    }
    A.spec_cnt.insert(A.spec_cnt.end(), X.spec_cnt.begin(), X.spec_cnt.end());
    for (int r : X.mark_of) A.mark_of.push_back(r < 0 ? -1 : r + (int)(A.marks.size() / MARK_WORDS));
    A.marks.insert(A.marks.end(), X.marks.begin(), X.marks.end());
    {  // the lists of k_deferred, with the member's offsets
      const int db = (int)A.defs.size(), rb = nrec, fb = 2 * (int)A.fault_def1.size();
      const int rd = (int)A.rec_def.size(), rf = (int)A.rec_flt.size();
      for (DefNode& d : X.defs)
        if (d.rec_at >= 0) d.rec_at += d.fault ? rf : rd;
      for (int q : X.fault_def1) A.fault_def1.push_back(q + db);
      for (int q : X.fault_def2) A.fault_def2.push_back(q < 0 ? -1 : q + db);
      for (auto& e : X.rec_int) A.rec_int.push_back({e.first + (int)nb, e.second + rb});
      for (auto& e : X.rec_def) A.rec_def.push_back({e.first + db, e.second + rb});
      for (auto& e : X.rec_flt) A.rec_flt.push_back({e.first + fb, e.second + rb});
      nrec += h->nrec;
    }
    A.spec_idx.insert(A.spec_idx.end(), X.spec_idx.begin(), X.spec_idx.end());
    for (DefNode d : X.defs) {
      d.g += (int)nb;
      d.pstart += pb;
      d.sstart += sb;
      d.astart += ab;
      A.defs.push_back(d);
    }
    for (int po : X.part_off) A.part_off.push_back(po + tb * SLOTS);
    for (SrcEntry e : X.dsrc) {
      e.src += nsrc;
      A.dsrc.push_back(e);
    }
    A.dabso.insert(A.dabso.end(), X.dabso.begin(), X.dabso.end());
    const size_t ndef = X.defs.size();
    for (int c = 0; c < nd; ++c)
      rmdef_c[c].insert(rmdef_c[c].end(), X.rmdef.begin() + c * ndef, X.rmdef.begin() + (c + 1) * ndef);
    // source amplitude rows, padded to the common length
    b->src_base[m] = nsrc;
    for (int s = 0; s < h->nsrc; ++s) {
      std::vector<double> row(ampl_nt, 0.0);
      std::copy(h->stf[s].begin(), h->stf[s].end(), row.begin());
      ampl.insert(ampl.end(), row.begin(), row.end());
    }
    nsrc += h->nsrc;
    nb += h->st.NS;
    cb += h->nelem;
    shared_off += (size_t)h->nelast * NP;
  }
  b->fstride = nb;
  for (int c = 0; c < nd; ++c) {
    A.rmdef.insert(A.rmdef.end(), rmdef_c[c].begin(), rmdef_c[c].end());
  }
  StepDev& X = b->X;
  X.ndof = nd;
  X.nelast = b->nelast;
  X.coef_mode = b->coef_mode;
  X.fstride = nb;
  X.stream = b->stream;
  const int ntiles = (int)A.tiles.size();
  int4 *tiles, *grids;
  int *sc, *si, *po;
  DefDev* defs;
  int4* defx;
  SrcEntry* ds;
  double *dab, *amp;
  if ((rc = bupload(b, &tiles, A.tiles))) return rc;
  if ((rc = bupload(b, &grids, A.grids))) return rc;
  if ((rc = bupload(b, &sc, A.spec_cnt))) return rc;
  if ((rc = bupload(b, &si, A.spec_idx))) return rc;
  int* mo;
  uint32_t* mk;
  if ((rc = bupload(b, &mo, A.mark_of))) return rc;
  if ((rc = bupload(b, &mk, A.marks))) return rc;
  X.mark_of = mo;
  X.marks = mk;
  {
    std::vector<DefDev> dn;
    std::vector<int4> dx;
    if (!pack_defs(A.defs, A.part_off, dn, dx)) return berr(b, 5, "batch: more than 255 entries at a deferred node");
    if ((rc = bupload(b, &defs, dn))) return rc;
    if ((rc = bupload(b, &defx, dx))) return rc;
    std::vector<DefDev> fd;
    for (int q : A.fault_def1) fd.push_back(dn[q]);
    for (size_t k = 0; k < A.fault_def2.size(); ++k) fd.push_back(dn[A.fault_def2[k] < 0 ? A.fault_def1[k] : A.fault_def2[k]]);
    DefDev* pf = nullptr;
    if ((rc = bupload(b, &pf, fd))) return rc;
    X.fdef = pf;
  }
  if ((rc = bupload(b, &po, A.part_off))) return rc;
  if ((rc = bupload(b, &ds, A.dsrc))) return rc;
  if ((rc = bupload(b, &dab, A.dabso))) return rc;
  if (ampl.empty()) ampl.assign(1, 0.0);
  if ((rc = bupload(b, &amp, ampl))) return rc;
  void* rmdef;
  if ((rc = bupload_bulk(b, &rmdef, A.rmdef))) return rc;
  {
    X.w32 = fits32(nb, (size_t)ntiles * SLOTS,
                   b->coef_mode == COEF_SHARED ? shared_off : cb * std::max(nd, b->nelast) * NP, rs);
  }
  X.T.ntiles = ntiles;
  X.T.tiles = tiles;
  X.T.grids = grids;
  X.T.spec_cnt = sc;
  X.T.spec_idx = si;
  X.T.NGp = nb;
  X.T.FPS = (size_t)ntiles * SLOTS;
  X.ndef = (int)A.defs.size();
  X.defs.node = defs;
  X.defs.ext = defx;
  X.part_off = po;
  X.dsrc = ds;
  X.dabso = dab;
  X.rmdef = rmdef;
  X.ampl = amp;
  X.ampl_nt = ampl_nt;
  // bulk arrays: fields, inverse mass, coefficients, partial forces
  char *d, *v, *a, *rm0, *co, *ge = nullptr, *fp;
  if ((rc = balloc(b, &d, nd * nb * rs))) return rc;
  if ((rc = balloc(b, &v, nd * nb * rs))) return rc;
  if ((rc = balloc(b, &a, nd * nb * rs))) return rc;
  if ((rc = balloc(b, &rm0, nb * rs))) return rc;
  if ((rc = balloc(b, &fp, (size_t)nd * X.T.FPS * rs))) return rc;
  const size_t co_per = b->coef_mode == COEF_SHARED ? 0
                        : (b->coef_mode == COEF_COMPACT ? (size_t)nd * NP : (size_t)b->nelast * NP);
  const size_t co_n = b->coef_mode == COEF_SHARED ? shared_off : cb * co_per;
  if ((rc = balloc(b, &co, co_n * rs))) return rc;
  if (b->coef_mode == COEF_COMPACT && (rc = balloc(b, &ge, cb * 3 * rs))) return rc;
  size_t cofs = 0, gofs = 0;
  for (int m = 0; m < n; ++m) {
    sem2d_solver* h = b->mem[m];
    const size_t NS = h->st.NS, o = b->node_base[m];
    for (int c = 0; c < nd; ++c) {
      BHIPCHK(b, hipMemcpyAsync(d + (c * nb + o) * rs, (char*)h->d + c * NS * rs, NS * rs, hipMemcpyDeviceToDevice, b->stream));
      BHIPCHK(b, hipMemcpyAsync(v + (c * nb + o) * rs, (char*)h->v + c * NS * rs, NS * rs, hipMemcpyDeviceToDevice, b->stream));
      BHIPCHK(b, hipMemcpyAsync(a + (c * nb + o) * rs, (char*)h->a + c * NS * rs, NS * rs, hipMemcpyDeviceToDevice, b->stream));
    }
    BHIPCHK(b, hipMemcpyAsync(rm0 + o * rs, h->st.rmass0, NS * rs, hipMemcpyDeviceToDevice, b->stream));
    const size_t ncf = b->coef_mode == COEF_SHARED ? (size_t)h->nelast * NP : (size_t)h->nelem * co_per;
    BHIPCHK(b, hipMemcpyAsync(co + cofs * rs, h->st.coefs, ncf * rs, hipMemcpyDeviceToDevice, b->stream));
    cofs += ncf;
    if (ge) {
      BHIPCHK(b, hipMemcpyAsync(ge + gofs * rs, h->st.geom, (size_t)h->nelem * 3 * rs, hipMemcpyDeviceToDevice, b->stream));
      gofs += (size_t)h->nelem * 3;
    }
  }
  BHIPCHK(b, hipStreamSynchronize(b->stream));
  X.d = d;
  X.v = v;
  X.a = a;
  X.rmass0 = rm0;
  X.coefs = co;
  X.geom = ge;
  X.fpart = fp;
  if ((rc = balloc(b, &b->it_dev, 1))) return rc;
  if ((rc = balloc(b, &b->flags, 4))) return rc;
  const int zero4[4] = {0, 0, 0, 0};
  BHIPCHK(b, hipMemcpy(b->flags, zero4, sizeof zero4, hipMemcpyHostToDevice));
  BHIPCHK(b, hipMemcpy(b->it_dev, zero4, sizeof(int), hipMemcpyHostToDevice));
  X.itp = X.tick = b->it_dev;
  if (h0->flt.on) {
    if ((rc = gather_fault(b))) return rc;
    std::vector<int4> wave;
    std::vector<int2> member;
    std::vector<int> slot;
    for (int m = 0; m < n; ++m) fault_waves(b->mem[m]->flt, m, b->fault_base[m], b->fout_base[m], wave, member, slot);
    int *d1, *d2, *sl;
    int4* wv;
    int2* mb;
    if ((rc = bupload(b, &d1, A.fault_def1))) return rc;
    if ((rc = bupload(b, &d2, A.fault_def2))) return rc;
    if ((rc = bupload(b, &wv, wave))) return rc;
    if ((rc = bupload(b, &mb, member))) return rc;
    if ((rc = bupload(b, &sl, slot))) return rc;
    char* side;
    if ((rc = balloc(b, &side, (size_t)4 * nd * b->X.F.np * rs))) return rc;
    b->X.F.side = side;
    b->X.F.def1 = d1;
    b->X.F.def2 = d2;
    FaultOut& O = b->X.fo;
    O.nwave = (int)wave.size(), O.wave = wv, O.member = mb, O.slot = sl;
    if ((rc = balloc(b, &O.part, wave.size() * 6))) return rc;
    if ((rc = bupload(b, &O.cnt, std::vector<unsigned>(n, 0u)))) return rc;
    O.pot = b->pot, O.pot_cap = b->pot_cap, O.pot_row = b->pot_shift;
    O.rec = b->frec, O.nout = b->fnout, O.oit0 = b->oit0, O.oitd = b->oitd, O.nsamp = b->fnsamp;
  }
  // receivers: members with stations, member after member
  std::vector<int> rn;
  b->rec_base.assign(n, 0);
  for (int m = 0; m < n; ++m) {
    sem2d_solver* h = b->mem[m];
    b->rec_base[m] = (int)rn.size();
    if (!h->nrec) continue;
    if (h->rec_w) return berr(b, 3, "member %d: receivers inside elements (AtNode=F) are not batched", m);
    if (!rn.empty() && (h->isamp != b->isamp || h->field != b->field))
      return berr(b, 3, "member %d: receiver sampling and field must match", m);
    b->isamp = h->isamp;
    b->field = h->field;
    b->nsamp = std::max(b->nsamp, h->nsamp);
    std::vector<int> t(h->nrec);
    BHIPCHK(b, hipMemcpy(t.data(), h->rec_node, h->nrec * sizeof(int), hipMemcpyDeviceToHost));
    for (int g : t) rn.push_back(g + (int)b->node_base[m]);
  }
  b->nrec = (int)rn.size();
  if ((rc = bupload(b, &b->rec_node, rn))) return rc;
  if ((rc = balloc(b, &b->seis, (size_t)std::max(b->nsamp, 1) * nd * std::max(b->nrec, 1)))) return rc;
  if (b->nrec) {
    RecOut& P = X.recout;
    P.seis = b->seis, P.nrec = b->nrec, P.isamp = b->isamp, P.nsamp = b->nsamp, P.field = b->field;
    auto up2 = [&](const int** p, const int** r, int* cnt, const std::vector<std::pair<int, int>>& x) {
      std::vector<int> k, v;
      for (auto& e : x) k.push_back(e.first), v.push_back(e.second);
      *cnt = (int)x.size();
      int *pk = nullptr, *pv = nullptr;
      int e = bupload(b, &pk, k);
      if (!e) e = bupload(b, &pv, v);
      *p = pk, *r = pv;
      return e;
    };
    if ((rc = up2(&P.int_g, &P.int_r, &P.nint, A.rec_int))) return rc;
    if ((rc = up2(&P.def_q, &P.def_r, &P.ndefr, A.rec_def))) return rc;
    if ((rc = up2(&P.flt_q, &P.flt_r, &P.nfltr, A.rec_flt))) return rc;
  }
  // default launch configuration (sem2d_batch_tune measures the alternatives)
  batch_set_config(b, tile_wgs_per_cu(b->fp32, b->ndof));
  // records of step 0
  if (b->nrec || b->X.fault_on) {
    if (b->fp32) launch_batch_record<float>(b);
    else launch_batch_record<double>(b);
  }
  BHIPCHK(b, hipGetLastError());
  BHIPCHK(b, hipStreamSynchronize(b->stream));
  return 0;
}

int sem2d_batch_step(sem2d_batch* b, int nsteps) {
  if (!b) return 1;
  if (nsteps < 0) return berr(b, 3, "batch_step: negative nsteps");
  return batch_run(b, nsteps, true);
}

int sem2d_batch_tune(sem2d_batch* b, int trial_steps, int* choice) {
  if (!b) return 1;
  if (trial_steps < 1) return berr(b, 3, "batch_tune: trial_steps must be >= 1");
  // save the state the trials advance
  const size_t rs = b->fp32 ? sizeof(float) : sizeof(double);
  const size_t nf = (size_t)b->ndof * b->fstride * rs;
  std::vector<void*> saved;
  auto keep = [&](const void* src, size_t bytes) -> int {
    void* q = nullptr;
    BHIPCHK(b, hipMalloc(&q, std::max<size_t>(bytes, 1)));
    saved.push_back(q);
    BHIPCHK(b, hipMemcpyAsync(q, src, bytes, hipMemcpyDeviceToDevice, b->stream));
    return 0;
  };
  struct Blk { void* p; size_t bytes; };
  std::vector<Blk> blks = {{b->X.d, nf}, {b->X.v, nf}, {b->X.a, nf}, {b->it_dev, sizeof(int)}, {b->flags, 4 * sizeof(int)}};
  if (b->X.fault_on) {
    const FaultDev& F = b->X.F;
    const size_t np = F.np, ndp = (size_t)F.ndof * np;
    blks.push_back({F.theta, np * 8});
    blks.push_back({F.D, ndp * 8});
    blks.push_back({F.V, ndp * 8});
    blks.push_back({F.T, 2 * np * 8});
    blks.push_back({F.Tstick, 2 * np * 8});
    blks.push_back({F.MU, np * 8});
    blks.push_back({F.sigma, np * 8});
  }
  int rc = 0;
  for (auto& k : blks)
    if ((rc = keep(k.p, k.bytes))) break;
  const int it0 = b->it;
  const int cand[] = {2, 3, 4, 1, 0};  // workgroups per CU
  const int ncand = sizeof(cand) / sizeof(cand[0]);
  double best = 1e30;
  int ibest = 0;
  for (int q = 0; q < ncand && !rc; ++q) {
    batch_set_config(b, cand[q]);
    rc = batch_run(b, 1, false);  // warm-up
    if (!rc) rc = batch_run(b, trial_steps, false);
    if (!rc && b->last_ms < best) {
      best = b->last_ms;
      ibest = q;
    }
    // restore
    for (size_t k = 0; k < blks.size() && !rc; ++k)
      if (hipMemcpyAsync(blks[k].p, saved[k], blks[k].bytes, hipMemcpyDeviceToDevice, b->stream) != hipSuccess)
        rc = berr(b, 10, "batch_tune: restore failed");
    b->it = it0;
  }
  hipStreamSynchronize(b->stream);
  for (void* q : saved) hipFree(q);
  if (rc) return rc;
  batch_set_config(b, cand[ibest]);
  if (choice) *choice = ibest;
  return 0;
}

int sem2d_batch_set_config(sem2d_batch* b, int threads, int wg_per_cu) {
  if (!b) return 1;
  if ((threads != 256 && threads != 512) || wg_per_cu < 0 || wg_per_cu > 4)
    return berr(b, 3, "batch_set_config: threads must be 256 or 512 and 0 <= wg_per_cu <= 4");
  batch_set_config(b, wg_per_cu);
  return 0;
}

int sem2d_batch_config(sem2d_batch* b, int* threads, int* wgs, int* ntiles) {
  if (!b) return 1;
  if (threads) *threads = TS_NT;
  if (wgs) *wgs = b->X.pipe_wgs > 0 ? b->X.pipe_wgs : (b->X.T.ntiles + 7) / 8 * 8;
  if (ntiles) *ntiles = b->X.T.ntiles;
  return 0;
}

int sem2d_batch_fetch_fields(sem2d_batch* b, int m, double* d, double* v, double* a) {
  if (!b) return 1;
  if (m < 0 || m >= b->n) return berr(b, 3, "batch_fetch_fields: bad member %d", m);
  sem2d_solver* h = b->mem[m];
  const size_t NS = h->st.NS, o = b->node_base[m], rs = b->fp32 ? 4 : 8;
  BHIPCHK(b, hipStreamSynchronize(b->stream));
  double* outs[3] = {d, v, a};
  void* srcs[3] = {b->X.d, b->X.v, b->X.a};
  std::vector<char> raw(NS * rs);
  for (int q = 0; q < 3; ++q) {
    if (!outs[q]) continue;
    for (int c = 0; c < b->ndof; ++c) {
      BHIPCHK(b, hipMemcpy(raw.data(), (char*)srcs[q] + (c * b->fstride + o) * rs, NS * rs, hipMemcpyDeviceToHost));
      for (int k = 0; k < h->npoin; ++k) {
        const size_t g = h->st.gmap[k];
        outs[q][(size_t)c * h->npoin + k] = b->fp32 ? (double)((float*)raw.data())[g] : ((double*)raw.data())[g];
      }
    }
  }
  return 0;
}

int sem2d_batch_fetch_seismo(sem2d_batch* b, int m, double* out, int* taken) {
  if (!b) return 1;
  if (m < 0 || m >= b->n) return berr(b, 3, "batch_fetch_seismo: bad member %d", m);
  sem2d_solver* h = b->mem[m];
  const int tk = h->nrec ? std::min(rec_taken(b), h->nsamp) : 0;
  if (out && tk) {
    std::vector<double> all;
    int rc = bdown(b, all, b->seis, (size_t)tk * b->ndof * b->nrec);
    if (rc) return rc;
    for (int s = 0; s < tk; ++s)
      for (int c = 0; c < b->ndof; ++c)
        for (int r = 0; r < h->nrec; ++r)
          out[((size_t)s * b->ndof + c) * h->nrec + r] = all[((size_t)s * b->ndof + c) * b->nrec + b->rec_base[m] + r];
  }
  if (taken) *taken = tk;
  return 0;
}

int sem2d_batch_fetch_fault(sem2d_batch* b, int m, double* out, int* taken) {
  if (!b) return 1;
  if (m < 0 || m >= b->n) return berr(b, 3, "batch_fetch_fault: bad member %d", m);
  if (!b->X.fault_on) return berr(b, 4, "batch_fetch_fault: no fault");
  const FaultHost& H = b->mem[m]->flt;
  const int tk = std::min(flt_taken(b), H.nsamp);
  if (out && tk) {
    std::vector<double> all;
    int rc = bdown(b, all, b->frec, (size_t)tk * 6 * b->fnout);
    if (rc) return rc;
    for (int s = 0; s < tk; ++s)
      for (int q = 0; q < 6; ++q)
        for (int o = 0; o < H.nout; ++o)
          out[((size_t)s * 6 + q) * H.nout + o] = all[((size_t)s * 6 + q) * b->fnout + b->fout_base[m] + o];
  }
  if (taken) *taken = tk;
  return 0;
}

int sem2d_batch_fetch_fault_state(sem2d_batch* b, int m, double* D, double* V, double* T, double* MU, double* Ts) {
  if (!b) return 1;
  if (m < 0 || m >= b->n) return berr(b, 3, "batch_fetch_fault_state: bad member %d", m);
  if (!b->X.fault_on) return berr(b, 4, "batch_fetch_fault_state: no fault");
  BHIPCHK(b, hipStreamSynchronize(b->stream));
  const FaultDev& F = b->X.F;
  const int nm = b->mem[m]->flt.dev.np, o = b->fault_base[m], np = F.np;
  auto rows = [&](double* dst, const double* src, int nr) -> int {
    if (!dst) return 0;
    for (int r = 0; r < nr; ++r)
      BHIPCHK(b, hipMemcpy(dst + (size_t)r * nm, src + (size_t)r * np + o, nm * sizeof(double), hipMemcpyDeviceToHost));
    return 0;
  };
  int rc;
  if ((rc = rows(D, F.D, F.ndof))) return rc;
  if ((rc = rows(V, F.V, F.ndof))) return rc;
  if ((rc = rows(T, F.T, 2))) return rc;
  if ((rc = rows(MU, F.MU, 1))) return rc;
  if ((rc = rows(Ts, F.Tstick, 2))) return rc;
  return 0;
}

int sem2d_batch_fetch_potency(sem2d_batch* b, int m, double* out, int* nrows) {
  if (!b) return 1;
  if (m < 0 || m >= b->n) return berr(b, 3, "batch_fetch_potency: bad member %d", m);
  if (!b->X.fault_on) return berr(b, 4, "batch_fetch_potency: no fault");
  const int rows = b->pot_shift + 1 + b->it;
  const size_t nc = 2 * (size_t)(b->ndof + 1);
  if (out && rows)
    BHIPCHK(b, hipMemcpy(out, b->pot + (size_t)m * b->pot_cap * nc, (size_t)rows * nc * sizeof(double),
                         hipMemcpyDeviceToHost));
  if (nrows) *nrows = rows;
  return 0;
}

int sem2d_batch_get_step(sem2d_batch* b, int* it) {
  if (!b || !it) return 1;
  *it = b->it;
  return 0;
}

int sem2d_batch_last_step_ms(sem2d_batch* b, double* ms) {
  if (!b || !ms) return 1;
  *ms = b->last_ms;
  return 0;
}

const char* sem2d_batch_last_error(sem2d_batch* b) { return b ? b->err.c_str() : "null handle"; }

void sem2d_batch_destroy(sem2d_batch* b) {
  if (!b) return;
  if (b->stream) hipStreamSynchronize(b->stream);
  batch_drop_graph(b);
  for (void* p : b->allocs) hipFree(p);
  if (b->pot) hipFree(b->pot);
  if (b->ev0) hipEventDestroy(b->ev0);
  if (b->ev1) hipEventDestroy(b->ev1);
  if (b->stream) hipStreamDestroy(b->stream);
  delete b;
}

}  // extern "C"

// ===========================================================================
// Adjoint of the time loop with sqrt(N) checkpointing (structured P-SV grids,
// compact coefficients, beta = 0, no fault).
//
// forward:  from the zero state, nsteps steps; the state before every segment of
//           seg steps is kept (checkpoints); seismograms are recorded as usual.
// backward: for each segment, last first: the segment is replayed from its
//           checkpoint into seg+1 state slots, then the adjoint steps run from the
//           segment's last step down to its first, injecting dJ/d(seismogram) at the
//           sample steps and accumulating the sensitivities:
//             glam, gmu [cell]   dJ/d(lambda), dJ/d(mu) of each element (summed over
//                                its GLL points)
//             mbar [node]        dJ/dM (M the assembled mass, same for both components)
//             gabs [c][node]     dJ/dC_c at absorbing-boundary nodes (C the
//                                Clayton-Engquist coefficient, incl. its share c3*C
//                                of the modified mass)
// The host turns these into gradients with respect to per-element rho, lambda, mu
// (the chain rule through M = sum rho w J and C = sum rho c w |J1D|).
// ===========================================================================
struct AdjState {
  int nsteps = 0, seg = 0, nck = 0;
  // history mode: the displacement after every step (FP32 bulk: and the acceleration)
  // kept in device memory, so that the backward sweep needs no replay
  bool hist = false;
  char *H = nullptr, *AH = nullptr, *aN = nullptr;  // [nsteps+1] states; a after the last step
  void* hblock = nullptr;  // the history's device block (from or back to the history cache)
  size_t hbytes = 0;
  // injection plan of dJ/d(seismogram): distinct nodes, their contributions
  int nu = 0;
  int *unode = nullptr, *uoff = nullptr, *urec = nullptr;
  double* uw = nullptr;
  int* udef = nullptr;             // injection node of each deferred node, or -1
  unsigned char* utile = nullptr;  // tiles with an injection node in their patch
  size_t state_bytes = 0;  // d, v, a of one state
  std::vector<char*> ck, slot;
  char *ad = nullptr, *av = nullptr, *rmass = nullptr;  // av: the w of AdjNode
  double *glam = nullptr, *gmu = nullptr, *mbar = nullptr, *gabs = nullptr, *gseis = nullptr;
  std::vector<void*> allocs;
  double fwd_ms = 0, bwd_ms = 0;
};

// One reusable history block per process.  Releasing a block of this size (a hundred
// GB) and mapping a new one costs seconds, while a sequence of gradients (one adjoint
// state each) needs the same block again and again: a freed state's history block is
// kept here and handed to the next history plan that fits in it, until
// sem2d_adjoint_release.  A block in use by a live state is not shared.
struct HistCache {
  std::mutex m;
  void* p = nullptr;
  size_t bytes = 0;
  int dev = -1;
};
HistCache& hist_cache() {
  static HistCache c;
  return c;
}

// a block of at least `bytes` on the current device: the cached one if it fits, else a new
// one (the cached block released first); nullptr if the device has no room
void* hist_acquire(size_t bytes, size_t* got) {
  HistCache& c = hist_cache();
  std::lock_guard<std::mutex> lk(c.m);
  int dev = 0;
  (void)hipGetDevice(&dev);
  if (c.p && c.dev == dev && c.bytes >= bytes) {
    void* p = c.p;
    *got = c.bytes;
    c.p = nullptr;
    c.bytes = 0;
    return p;
  }
  if (c.p) {
    (void)hipFree(c.p);
    c.p = nullptr;
    c.bytes = 0;
  }
  void* p = nullptr;
  if (hipMalloc(&p, bytes) != hipSuccess) {
    (void)hipGetLastError();
    return nullptr;
  }
  *got = bytes;
  return p;
}

// size of the cached block usable on the current device (0: none)
size_t hist_cached_bytes() {
  HistCache& c = hist_cache();
  std::lock_guard<std::mutex> lk(c.m);
  int dev = 0;
  (void)hipGetDevice(&dev);
  return c.p && c.dev == dev ? c.bytes : 0;
}

void hist_return(void* p, size_t bytes) {
  HistCache& c = hist_cache();
  std::lock_guard<std::mutex> lk(c.m);
  int dev = 0;
  (void)hipGetDevice(&dev);
  if (c.p && c.bytes >= bytes) {  // keep the larger block
    (void)hipFree(p);
    return;
  }
  if (c.p) (void)hipFree(c.p);
  c.p = p;
  c.bytes = bytes;
  c.dev = dev;
}

void adj_free(AdjState* A) {
  for (void* p : A->allocs) hipFree(p);
  if (A->hblock) hist_return(A->hblock, A->hbytes);
  delete A;
}

namespace {

int adj_alloc(sem2d_solver* h, void** p, size_t bytes) {
  hipError_t e = hipMalloc(p, std::max<size_t>(bytes, 1));
  if (e != hipSuccess) return set_err(h, 11, "adjoint: hipMalloc(%zu bytes): %s", bytes, hipGetErrorString(e));
  h->adj->allocs.push_back(*p);
  return 0;
}

// Inverse mass per component in storage order for the adjoint: the single-component
// array of the tile kernels (k_adj_rmass), then the deferred nodes' own values
// (k_adj_rmass_def).
template <typename R>
__global__ void k_adj_rmass(size_t GS, int ndof, const R* __restrict__ rm0, R* __restrict__ out) {
  const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= GS) return;
  const R m = rm0[i];
  for (int c = 0; c < ndof; ++c) out[(size_t)c * GS + i] = m;
}
template <typename R>
__global__ void k_adj_rmass_def(int ndef, int ndof, DefTable defs, const R* __restrict__ rmdef, size_t GS,
                                R* __restrict__ out) {
  const int q = blockIdx.x * blockDim.x + threadIdx.x;
  if (q >= ndef) return;
  const size_t g = defs.node[q].g;
  for (int c = 0; c < ndof; ++c) out[(size_t)c * GS + g] = rmdef[(size_t)c * ndef + q];
}

// copy a whole state (d, v, a) between two state buffers or the solver's fields
int copy_state(sem2d_solver* h, char* dst_d, char* dst_v, char* dst_a, const char* d, const char* v, const char* a) {
  const size_t n = (size_t)h->ndof * h->fstride * rsize(h);
  HIPCHK(h, hipMemcpyAsync(dst_d, d, n, hipMemcpyDeviceToDevice, h->stream));
  HIPCHK(h, hipMemcpyAsync(dst_v, v, n, hipMemcpyDeviceToDevice, h->stream));
  HIPCHK(h, hipMemcpyAsync(dst_a, a, n, hipMemcpyDeviceToDevice, h->stream));
  return 0;
}

inline char* st_d(sem2d_solver* h, char* s) { (void)h; return s; }
inline char* st_v(sem2d_solver* h, char* s) { return s + (size_t)h->ndof * h->fstride * rsize(h); }
inline char* st_a(sem2d_solver* h, char* s) { return s + 2 * (size_t)h->ndof * h->fstride * rsize(h); }

// One adjoint tile step (dp, dn: d_{n-1}, d_{n+1} where the acceleration afw is not stored)
template <typename R>
void launch_adj_tile(sem2d_solver* h, const StepDev& X, const R* dfw, const R* afw, const R* dp, const R* dn,
                     R dt, R c1, R c2, R c3, double idt2, const InjectPlan& inj) {
  AdjState& A = *h->adj;
  StructState& S = h->st;
  AdjArgs<R> G;
  G.ad = (R*)A.ad, G.w = (R*)A.av;
  G.rmass = (const R*)A.rmass, G.dfw = dfw;
  G.x1 = afw ? afw : dp, G.x2 = afw ? nullptr : dn;
  G.coefs = (const R*)(S.elemmod ? S.elemmod : S.coefs), G.geom = (const R*)S.geom, G.fpart = (R*)S.fpart;
  G.glam = A.glam, G.gmu = A.gmu, G.mbar = A.mbar;
  G.S = h->fstride, G.FPS = S.FPS;
  G.tiles = X.T.tiles, G.grids = X.T.grids, G.spec_cnt = X.T.spec_cnt, G.spec_idx = X.T.spec_idx;
  G.ntiles = S.ntiles;
  G.dt = dt, G.c1 = c1, G.c2 = c2, G.c3 = c3, G.idt2 = idt2;
  G.inj = inj;
  // 32-bit offsets: the double mass-sensitivity array below 4 GiB too
  const bool w32 = S.w32 && h->fstride * sizeof(double) < (size_t(1) << 32);
  const int wgs = (S.ntiles + 7) / 8 * 8;
  auto go = [&](auto hist, auto el, auto w) {
    k_adj_step<R, decltype(hist)::value, decltype(el)::value, decltype(w)::value><<<wgs, TS_NT, 0, h->stream>>>(G);
  };
  const std::true_type yes{};
  const std::false_type no{};
  auto w = [&](auto hist, auto el) { w32 ? go(hist, el, yes) : go(hist, el, no); };
  if (afw) S.elemmod ? w(no, yes) : w(no, no);
  else S.elemmod ? w(yes, yes) : w(yes, no);
}

template <typename R>
int adj_backward(sem2d_solver* h, const double* gseis_host) {
  AdjState& A = *h->adj;
  StructState& S = h->st;
  const size_t GS = h->fstride, nf = (size_t)h->ndof * GS;
  const StepCoefs<R> K = step_coefs<R>(h->dt, h->beta, h->gamma, h->leapfrog);
  const R dt = K.dt, c1 = K.c1, c2 = K.c2, c3 = K.c3, c4 = K.c4;
  const size_t ns = (size_t)h->nsamp * h->ndof * h->nrec;
  if (h->nrec && gseis_host)
    HIPCHK(h, hipMemcpyAsync(A.gseis, gseis_host, ns * sizeof(double), hipMemcpyHostToDevice, h->stream));
  HIPCHK(h, hipMemsetAsync(A.ad, 0, nf * sizeof(R), h->stream));
  HIPCHK(h, hipMemsetAsync(A.av, 0, nf * sizeof(R), h->stream));
  HIPCHK(h, hipMemsetAsync(A.glam, 0, (size_t)h->nelem * sizeof(double), h->stream));
  HIPCHK(h, hipMemsetAsync(A.gmu, 0, (size_t)h->nelem * sizeof(double), h->stream));
  HIPCHK(h, hipMemsetAsync(A.mbar, 0, GS * sizeof(double), h->stream));
  HIPCHK(h, hipMemsetAsync(A.gabs, 0, (size_t)h->ndof * std::max(S.ndef, 1) * sizeof(double), h->stream));
  StepDev X = step_dev(h);
  X.recout = RecOut{};  // the replayed steps are not recorded again
  // the sample of step n, added to the state the step starts from
  auto plan_for = [&](int n) {
    InjectPlan P;
    if (!(h->nrec && n >= 1 && sampled(h, n))) return P;
    P.nu = A.nu;
    P.nrec = h->nrec;
    P.field = h->field;
    P.unode = A.unode;
    P.off = A.uoff;
    P.rec = A.urec;
    P.w = A.uw;
    P.g = A.gseis + (size_t)(n / h->isamp) * h->ndof * h->nrec;
    P.udef = A.udef;
    P.tile = A.utile;
    return P;
  };
  const int gd = (S.ndef + 255) / 256;
  HIPCHK(h, hipEventRecord(h->ev0, h->stream));
  if (A.hist) {
    // no replay: the forward displacements are all in memory
    const size_t nfb = nf * sizeof(R);
    const double idt = 1.0 / h->dt, idt2 = idt * idt;
    const int N = A.nsteps;
    for (int n = N; n >= 1; --n) {
      const R* dc = (const R*)(A.H + (size_t)n * nfb);
      const R* dp = (const R*)(A.H + (size_t)(n - 1) * nfb);
      const R* dn = n < N ? (const R*)(A.H + (size_t)(n + 1) * nfb) : nullptr;
      const R* af = A.AH ? (const R*)(A.AH + (size_t)n * nfb) : (n == N ? (const R*)A.aN : nullptr);
      const InjectPlan P = plan_for(n);
      launch_adj_tile<R>(h, X, dc, af, dp, dn, dt, c1, c2, c3, idt2, P);
      k_adj_deferred<R><<<gd, 256, 0, h->stream>>>(
          S.ndef, S.defs, S.part_off, (const R*)S.fpart, S.FPS, S.dabso, (const R*)S.rmdef, (R*)A.ad, (R*)A.av,
          GS, af, nullptr, nullptr, A.mbar, A.gabs, dt, c1, c2, c3, dc, dp, dn, idt, idt2, P);
    }
  }
  for (int k = A.hist ? -1 : A.nck - 1; k >= 0; --k) {
    const int s0 = k * A.seg, s1 = std::min(A.nsteps, s0 + A.seg), L = s1 - s0;
    // replay: slot[j] = state after step s0 + j
    char* s = A.slot[0];
    int rc = copy_state(h, st_d(h, s), st_v(h, s), st_a(h, s), st_d(h, A.ck[k]), st_v(h, A.ck[k]), st_a(h, A.ck[k]));
    if (rc) return rc;
    for (int j = 1; j <= L; ++j) {  // out of place: slot[j-1] -> slot[j]
      char* p = A.slot[j - 1];
      char* q = A.slot[j];
      X.din = st_d(h, p);
      X.vin = st_v(h, p);
      X.ain = st_a(h, p);
      X.d = st_d(h, q);
      X.v = st_v(h, q);
      X.a = st_a(h, q);
      launch_structured_step<R>(X, s0 + j, dt, c1, c2, c3, c4);
    }
    X.din = X.vin = X.ain = nullptr;
    // adjoint steps n = s1 .. s0+1
    for (int n = s1; n > s0; --n) {
      const int j = n - s0;
      const R* dfw = (const R*)st_d(h, A.slot[j]);
      const R* afw = (const R*)st_a(h, A.slot[j]);
      const InjectPlan P = plan_for(n);
      launch_adj_tile<R>(h, X, dfw, afw, nullptr, nullptr, dt, c1, c2, c3, 0.0, P);
      k_adj_deferred<R><<<gd, 256, 0, h->stream>>>(
          S.ndef, S.defs, S.part_off, (const R*)S.fpart, S.FPS, S.dabso, (const R*)S.rmdef, (R*)A.ad, (R*)A.av,
          GS, afw, (const R*)st_v(h, A.slot[j - 1]), (const R*)st_a(h, A.slot[j - 1]), A.mbar, A.gabs,
          dt, c1, c2, c3, nullptr, nullptr, nullptr, 0.0, 0.0, P);
    }
  }
  HIPCHK(h, hipEventRecord(h->ev1, h->stream));
  HIPCHK(h, hipGetLastError());
  HIPCHK(h, hipEventSynchronize(h->ev1));
  float ms = 0.f;
  HIPCHK(h, hipEventElapsedTime(&ms, h->ev0, h->ev1));
  A.bwd_ms = ms;
  return 0;
}

// Forward sweep of the history mode.  With beta = 0 the displacement after a step is the
// predicted one it started from, and the one the step hands on (StepOut) is that of the
// next: step n reads history slot n and writes slot n+1 (out of place, with the predicted
// velocity in place), so the history needs no copies; for FP32 fields the acceleration is
// stored into its own history.  The recorded nodes go through the solver's a array; the
// solver's own arrays receive the final state, and the acceleration after the last step
// is kept.
template <typename R>
int adj_forward_hist(sem2d_solver* h) {
  AdjState& A = *h->adj;
  const size_t nfb = (size_t)h->ndof * h->fstride * sizeof(R);
  const StepCoefs<R> K = step_coefs<R>(h->dt, h->beta, h->gamma, h->leapfrog);
  const R dt = K.dt, c1 = K.c1, c2 = K.c2, c3 = K.c3, c4 = K.c4;
  int rc = sync_sources(h);
  if (rc) return rc;
  StepDev X = step_dev(h);
  void *d0 = h->d, *a0 = h->a;
  auto Hn = [&](int n) { return (void*)(A.H + (size_t)n * nfb); };
  auto AHn = [&](int n) { return (void*)(A.AH + (size_t)n * nfb); };
  // d_0 and, from the zero initial state, the first predicted displacement
  HIPCHK(h, hipMemsetAsync(A.H, 0, 2 * nfb, h->stream));
  if (A.AH) HIPCHK(h, hipMemsetAsync(A.AH, 0, nfb, h->stream));
  HIPCHK(h, hipEventRecord(h->ev0, h->stream));
  X.pin = X.w32;
  X.out.accel = A.AH != nullptr;
  for (int n = 1; n <= A.nsteps; ++n) {
    const bool last = n == A.nsteps;
    X.din = Hn(X.pin ? n : n - 1);
    X.vin = nullptr;  // in place
    X.ain = A.AH ? AHn(n - 1) : nullptr;
    X.d = !X.pin ? Hn(n) : (last ? d0 : Hn(n + 1));
    X.a = A.AH ? AHn(n) : a0;
    X.out.final = last || !X.pin;
    X.rec = a0;
    X.out.rec = !X.out.final && sampled(h, n) ? h->field : -1;
    launch_structured_step<R>(X, n, dt, c1, c2, c3, c4);
    h->it = n;
    if (!h->rec_w) {
      if (sampled(h, n)) h->taken = std::max(h->taken, n / h->isamp + 1);
      continue;
    }
    if (X.out.final) {
      h->d = X.d;
      h->a = X.a;
    }
    rc = record_receivers<R>(h, !X.out.final);
    h->d = d0;
    h->a = a0;
    if (rc) return rc;
  }
  if (!X.pin) HIPCHK(h, hipMemcpyAsync(d0, Hn(A.nsteps), nfb, hipMemcpyDeviceToDevice, h->stream));
  if (A.AH) HIPCHK(h, hipMemcpyAsync(a0, AHn(A.nsteps), nfb, hipMemcpyDeviceToDevice, h->stream));
  if (A.aN) HIPCHK(h, hipMemcpyAsync(A.aN, a0, nfb, hipMemcpyDeviceToDevice, h->stream));
  HIPCHK(h, hipEventRecord(h->ev1, h->stream));
  HIPCHK(h, hipGetLastError());
  HIPCHK(h, hipEventSynchronize(h->ev1));
  float ms = 0.f;
  HIPCHK(h, hipEventElapsedTime(&ms, h->ev0, h->ev1));
  A.fwd_ms = ms;
  return 0;
}

}  // namespace

extern "C" {

int sem2d_adjoint_init(sem2d_solver* h, int nsteps, int seg) {
  if (!h) return 1;
  if (!h->st.on || h->ndof != 2 || h->coef_mode != COEF_COMPACT || h->nelast != 6)
    return set_err(h, 4, "adjoint: needs a structured P-SV grid with compact (lambda, mu) coefficients");
  if (h->beta != 0.0 || h->gamma != 0.5 || h->leapfrog)
    return set_err(h, 4, "adjoint: needs the explicit Newmark scheme (beta = 0, gamma = 1/2)");
  if (h->flt.on) return set_err(h, 4, "adjoint: faults are not differentiated");
  if (h->st.eta || h->st.b25) return set_err(h, 4, "adjoint: Kelvin-Voigt and 2.5D terms are not differentiated");
  for (const AbsoHost& B : h->abso_host)
    if (!B.senode.empty()) return set_err(h, 4, "adjoint: Stacey boundaries are not differentiated");
  if (nsteps < 1) return set_err(h, 3, "adjoint_init: nsteps must be >= 1");
  const bool autoplan = seg <= 0;
  if (seg <= 0) seg = (int)std::ceil(std::sqrt((double)nsteps));
  int rc;
  if (!h->st.ready && (rc = sync_sources(h))) return rc;
  if (!h->st.ready && (rc = prepare_structured(h))) return rc;
  if (h->adj) adj_free(h->adj);
  if (h->flt.pot) hipFree(h->flt.pot);
  h->adj = new AdjState();
  AdjState& A = *h->adj;
  A.nsteps = nsteps;
  A.seg = std::min(seg, nsteps);
  A.nck = (nsteps + A.seg - 1) / A.seg;
  const size_t nf = (size_t)h->ndof * h->fstride * rsize(h);
  A.state_bytes = 3 * nf;
  if (autoplan) {
    // history mode when every step's displacement (FP32 fields: and acceleration) fits in
    // free device memory, next to the adjoint's own arrays and a 4 GiB reserve
    const size_t hbytes = (size_t)(nsteps + 1) * nf * (h->fp32 ? 2 : 1);
    size_t fr = 0, tot = 0;
    const size_t cached = hist_cached_bytes();  // reusable, so counted as free
    if (hipMemGetInfo(&fr, &tot) == hipSuccess &&
        hbytes + 9 * nf + ((size_t)4 << 30) < fr + (cached >= hbytes ? hbytes : cached)) {
      size_t got = 0;
      void* p = hist_acquire(hbytes, &got);
      if (p) {
        A.hblock = p;
        A.hbytes = got;
        A.H = (char*)p;
        A.hist = true;
        if (h->fp32) {
          A.AH = A.H + (size_t)(nsteps + 1) * nf;
        } else {
          if ((rc = adj_alloc(h, &p, nf))) return rc;
          A.aN = (char*)p;
        }
        A.seg = nsteps;
        A.nck = 1;
      }  // else: checkpoints
    }
  }
  for (int k = 0; !A.hist && k < A.nck; ++k) {
    void* p;
    if ((rc = adj_alloc(h, &p, A.state_bytes))) return rc;
    A.ck.push_back((char*)p);
  }
  for (int k = 0; !A.hist && k <= A.seg; ++k) {
    void* p;
    if ((rc = adj_alloc(h, &p, A.state_bytes))) return rc;
    A.slot.push_back((char*)p);
  }
  void* p;
  if ((rc = adj_alloc(h, &p, nf))) return rc;
  A.ad = (char*)p;
  if ((rc = adj_alloc(h, &p, nf))) return rc;
  A.av = (char*)p;
  if ((rc = adj_alloc(h, &p, (size_t)h->nelem * sizeof(double)))) return rc;
  A.glam = (double*)p;
  if ((rc = adj_alloc(h, &p, (size_t)h->nelem * sizeof(double)))) return rc;
  A.gmu = (double*)p;
  if ((rc = adj_alloc(h, &p, h->fstride * sizeof(double)))) return rc;
  A.mbar = (double*)p;
  if ((rc = adj_alloc(h, &p, (size_t)h->ndof * std::max(h->st.ndef, 1) * sizeof(double)))) return rc;
  A.gabs = (double*)p;
  if ((rc = adj_alloc(h, &p, (size_t)std::max(h->nsamp, 1) * h->ndof * std::max(h->nrec, 1) * sizeof(double))))
    return rc;
  A.gseis = (double*)p;
  // injection plan: the receivers' nodes (or element nodes with weights), grouped by
  // node, contributions in receiver order
  if (h->nrec) {
    const int per = h->rec_w ? h->np : 1;
    std::vector<int> rn((size_t)h->nrec * per);
    std::vector<double> rw((size_t)h->nrec * per, 1.0);
    HIPCHK(h, hipMemcpy(rn.data(), h->rec_node, rn.size() * sizeof(int), hipMemcpyDeviceToHost));
    if (h->rec_w) HIPCHK(h, hipMemcpy(rw.data(), h->rec_w, rw.size() * sizeof(double), hipMemcpyDeviceToHost));
    std::map<int, std::vector<std::pair<int, double>>> by;  // node -> (receiver, weight)
    for (int r = 0; r < h->nrec; ++r)
      for (int k = 0; k < per; ++k) by[rn[(size_t)r * per + k]].push_back({r, rw[(size_t)r * per + k]});
    std::vector<int> un, off(1, 0), rec;
    std::vector<double> w;
    for (auto& kv : by) {
      un.push_back(kv.first);
      for (auto& e : kv.second) {
        rec.push_back(e.first);
        w.push_back(e.second);
      }
      off.push_back((int)rec.size());
    }
    A.nu = (int)un.size();
    void* q;
    if ((rc = adj_alloc(h, &q, un.size() * sizeof(int)))) return rc;
    A.unode = (int*)q;
    if ((rc = adj_alloc(h, &q, off.size() * sizeof(int)))) return rc;
    A.uoff = (int*)q;
    if ((rc = adj_alloc(h, &q, rec.size() * sizeof(int)))) return rc;
    A.urec = (int*)q;
    if ((rc = adj_alloc(h, &q, w.size() * sizeof(double)))) return rc;
    A.uw = (double*)q;
    HIPCHK(h, hipMemcpy(A.unode, un.data(), un.size() * sizeof(int), hipMemcpyHostToDevice));
    HIPCHK(h, hipMemcpy(A.uoff, off.data(), off.size() * sizeof(int), hipMemcpyHostToDevice));
    HIPCHK(h, hipMemcpy(A.urec, rec.data(), rec.size() * sizeof(int), hipMemcpyHostToDevice));
    HIPCHK(h, hipMemcpy(A.uw, w.data(), w.size() * sizeof(double), hipMemcpyHostToDevice));
    // injection nodes that are deferred nodes (storage index of deferred node q:
    // gmap[def_ref[q]]), and the tiles with an injection node in their patch
    const StructState& S = h->st;
    std::unordered_map<int, int> u_at;  // injection node -> u (a few entries)
    for (int u = 0; u < (int)un.size(); ++u) u_at[un[u]] = u;
    std::vector<int> udef(std::max(S.ndef, 1), -1);
    for (int q = 0; q < S.ndef; ++q) {
      auto it = u_at.find(S.gmap[S.def_ref[q]]);
      if (it != u_at.end()) udef[q] = it->second;
    }
    std::vector<unsigned char> utile(S.ntiles, 0);
    for (int ref : h->rec_ref)
      tiles_at(S, S.gridx[ref] % S.NX1, S.gridx[ref] / S.NX1, [&](int t) { utile[t] = 1; });
    if ((rc = adj_alloc(h, &q, udef.size() * sizeof(int)))) return rc;
    A.udef = (int*)q;
    if ((rc = adj_alloc(h, &q, utile.size()))) return rc;
    A.utile = (unsigned char*)q;
    HIPCHK(h, hipMemcpy(A.udef, udef.data(), udef.size() * sizeof(int), hipMemcpyHostToDevice));
    HIPCHK(h, hipMemcpy(A.utile, utile.data(), utile.size(), hipMemcpyHostToDevice));
  }
  // inverse mass of both components in storage order.  The tile kernels' single-
  // component array holds it at every node whose components are equal; the deferred
  // nodes' per-component array covers the others (absorbing-boundary nodes), so the
  // device assembles it from those two when every node with unequal components is a
  // deferred node (else from the host copy).
  if ((rc = adj_alloc(h, &p, nf))) return rc;
  A.rmass = (char*)p;
  const StructState& S = h->st;
  bool dev_ok = true;
  {
    std::vector<char> isdef(h->npoin, 0);
    for (int q = 0; q < S.ndef; ++q) isdef[S.def_ref[q]] = 1;
    const double* rh = h->rmass_host.data();
    for (int c = 1; c < h->ndof && dev_ok; ++c)
      for (int k = 0; k < h->npoin; ++k)
        if (rh[(size_t)c * h->npoin + k] != rh[k] && !isdef[k]) {
          dev_ok = false;
          break;
        }
  }
  if (dev_ok) {
    const size_t GS = h->fstride;
    if (h->fp32) {
      k_adj_rmass<float><<<grid_for(GS, 256), 256, 0, h->stream>>>(GS, h->ndof, (const float*)S.rmass0,
                                                                  (float*)A.rmass);
      if (S.ndef > 0)
        k_adj_rmass_def<float><<<grid_for(S.ndef, 256), 256, 0, h->stream>>>(
            S.ndef, h->ndof, S.defs, (const float*)S.rmdef, GS, (float*)A.rmass);
    } else {
      k_adj_rmass<double><<<grid_for(GS, 256), 256, 0, h->stream>>>(GS, h->ndof, (const double*)S.rmass0,
                                                                    (double*)A.rmass);
      if (S.ndef > 0)
        k_adj_rmass_def<double><<<grid_for(S.ndef, 256), 256, 0, h->stream>>>(
            S.ndef, h->ndof, S.defs, (const double*)S.rmdef, GS, (double*)A.rmass);
    }
    HIPCHK(h, hipGetLastError());
    HIPCHK(h, hipStreamSynchronize(h->stream));
  } else {
    std::vector<double> rm((size_t)h->ndof * h->fstride, 0.0);
    for (int c = 0; c < h->ndof; ++c)
      for (int k = 0; k < h->npoin; ++k)
        rm[(size_t)c * h->fstride + h->st.gmap[k]] = h->rmass_host[(size_t)c * h->npoin + k];
    if ((rc = write_bulk(h, A.rmass, rm.data(), rm.size()))) return rc;
  }
  return 0;
}

int sem2d_adjoint_forward(sem2d_solver* h) {
  if (!h) return 1;
  if (!h->adj) return set_err(h, 4, "adjoint_forward: call sem2d_adjoint_init first");
  AdjState& A = *h->adj;
  const size_t nf = (size_t)h->ndof * h->fstride * rsize(h);
  HIPCHK(h, hipMemsetAsync(h->d, 0, nf, h->stream));
  HIPCHK(h, hipMemsetAsync(h->v, 0, nf, h->stream));
  HIPCHK(h, hipMemsetAsync(h->a, 0, nf, h->stream));
  h->it = 0;
  h->taken = 0;
  int rc = h->fp32 ? record_receivers<float>(h) : record_receivers<double>(h);
  if (rc) return rc;
  if (A.hist) return h->fp32 ? adj_forward_hist<float>(h) : adj_forward_hist<double>(h);
  double ms = 0;
  for (int k = 0; k < A.nck; ++k) {
    char* c = A.ck[k];
    if ((rc = copy_state(h, st_d(h, c), st_v(h, c), st_a(h, c), (char*)h->d, (char*)h->v, (char*)h->a))) return rc;
    const int L = std::min(A.seg, A.nsteps - k * A.seg);
    rc = h->fp32 ? do_steps<float>(h, L) : do_steps<double>(h, L);
    if (rc) return rc;
    ms += h->last_ms * L;
  }
  A.fwd_ms = ms;
  return 0;
}

int sem2d_adjoint_backward(sem2d_solver* h, const double* gseis) {
  if (!h) return 1;
  if (!h->adj) return set_err(h, 4, "adjoint_backward: call sem2d_adjoint_init first");
  if (h->it != h->adj->nsteps) return set_err(h, 4, "adjoint_backward: run sem2d_adjoint_forward first");
  return h->fp32 ? adj_backward<float>(h, gseis) : adj_backward<double>(h, gseis);
}

int sem2d_adjoint_fetch(sem2d_solver* h, double* glam, double* gmu, double* gmass, double* gabso) {
  if (!h) return 1;
  if (!h->adj) return set_err(h, 4, "adjoint_fetch: call sem2d_adjoint_init first");
  AdjState& A = *h->adj;
  StructState& S = h->st;
  HIPCHK(h, hipStreamSynchronize(h->stream));
  std::vector<double> tmp;
  if (glam || gmu) {
    tmp.resize(h->nelem);
    for (int q = 0; q < 2; ++q) {
      double* out = q == 0 ? glam : gmu;
      if (!out) continue;
      HIPCHK(h, hipMemcpy(tmp.data(), q == 0 ? A.glam : A.gmu, h->nelem * sizeof(double), hipMemcpyDeviceToHost));
      for (int cell = 0; cell < h->nelem; ++cell) out[S.cell_elem[cell]] = tmp[cell];
    }
  }
  if (gmass) {
    tmp.resize(h->fstride);
    HIPCHK(h, hipMemcpy(tmp.data(), A.mbar, h->fstride * sizeof(double), hipMemcpyDeviceToHost));
    for (int k = 0; k < h->npoin; ++k) gmass[k] = tmp[S.gmap[k]];
  }
  if (gabso) {
    std::fill(gabso, gabso + (size_t)h->ndof * h->npoin, 0.0);
    tmp.resize((size_t)h->ndof * std::max(S.ndef, 1));
    HIPCHK(h, hipMemcpy(tmp.data(), A.gabs, tmp.size() * sizeof(double), hipMemcpyDeviceToHost));
    for (int c = 0; c < h->ndof; ++c)
      for (int q = 0; q < S.ndef; ++q) gabso[(size_t)c * h->npoin + S.def_ref[q]] = tmp[(size_t)c * S.ndef + q];
  }
  return 0;
}

int sem2d_adjoint_release(void) {
  HistCache& c = hist_cache();
  std::lock_guard<std::mutex> lk(c.m);
  if (c.p) {
    hipError_t e = hipFree(c.p);
    c.p = nullptr;
    c.bytes = 0;
    if (e != hipSuccess) return 10;
  }
  return 0;
}

int sem2d_adjoint_plan(sem2d_solver* h, int* history, int* seg) {
  if (!h) return 1;
  if (!h->adj) return set_err(h, 4, "adjoint_plan: call sem2d_adjoint_init first");
  if (history) *history = h->adj->hist ? 1 : 0;
  if (seg) *seg = h->adj->seg;
  return 0;
}

int sem2d_adjoint_timing(sem2d_solver* h, double* fwd_ms, double* bwd_ms) {
  if (!h) return 1;
  if (!h->adj) return set_err(h, 4, "adjoint_timing: call sem2d_adjoint_init first");
  if (fwd_ms) *fwd_ms = h->adj->fwd_ms;
  if (bwd_ms) *bwd_ms = h->adj->bwd_ms;
  return 0;
}

}  // extern "C"
