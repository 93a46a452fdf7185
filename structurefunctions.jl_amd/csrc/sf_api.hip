// sf_api.hip -- host side of libsfmi355x.so: validation, bin tables, work items, launches.
//
// Validation mirrors what the reference checks before its O(N^2) loop:
//   _validate_array_shape          src/Calculations/shapes.jl:67-105  (D in {2,3}, W, N match)
//   _assert_counts_representable   src/Calculations/serial.jl:111-120 (N(N-1)/2 fits the count type)
//   pair_geometry_for              src/HelperFunctions.jl:390-417     (known metric only)
//   operator validity              src/StructureFunctionTypes.jl:43-151
// plus the preconditions the reference assumes silently: edges sorted (searchsortedfirst on an
// unsorted vector is meaningless) and, for the flat squared plan (BinEdges.jl:440), non-negative.
#include <hip/hip_runtime.h>

#include <math.h>
#include <stdarg.h>
#include <stdio.h>
#include <string.h>

#include <algorithm>
#include <map>
#include <string>
#include <tuple>
#include <vector>

#include "../../include/sfmi355x.h"
#include "sf_internal.h"

namespace sfk {
// kernel launchers (sf_kernels.hip)
hipError_t launch_prep(int G, int D, bool mixed, int geom_code, const void *prep_slices,
                       int n_slices, int64_t max_n, double *rec64, float *rec32, int nz, void *const *zp,
                       const int64_t *zb, hipStream_t st);
hipError_t launch_hist(int G, int D, bool J, bool mixed, bool sload, bool near, const Params &P, int grid,
                       int block, size_t smem, hipStream_t st);
hipError_t launch_recheck(int G, int D, bool J, const Params &P, int grid, hipStream_t st);
hipError_t launch_merge_checked(const double *src_s, const unsigned long long *src_c, double *dst_s,
                                unsigned long long *dst_c, int64_t n,
                                const unsigned long long *pcount, int64_t cap, int *flag,
                                hipStream_t st);
hipError_t launch_zero(void *p, int64_t bytes, hipStream_t st);
hipError_t launch_absmax(int count, const double *const *x, const int64_t *n, double *out, hipStream_t st);
hipError_t launch_derive_sp(double *s, unsigned long long *c, int64_t nbins, hipStream_t st);
hipError_t launch_eval_math(int fn, int64_t n, const double *a, const double *b, double *out,
                            hipStream_t st);
size_t cull_workspace_bytes(int64_t N);
hipError_t launch_cull(const double *x, int64_t N, int W, int D, int geom, double reach, int bits, void *ws,
                       int32_t *perm, double *info, float *gbox, hipStream_t st);
hipError_t launch_cull_count(const float *gbox, int64_t N, double *info, double reach, int K, hipStream_t st);
hipError_t launch_cull_units(const float *gbox, int64_t N, double *info, double reach, int K, int slice, Item *units,
                             int64_t n, hipStream_t st);
int hist_occupancy(int G, int D, bool J, bool mixed, int opk, bool sload, bool fx, int block,
                   size_t smem);
int hist_opk(const Params &P, int G, bool mixed);
int strip_occupancy(int G, int D, int opk, int block, size_t smem);
struct PrepSliceHost {
  const double *x, *u;
  int64_t N, pt_off;
  const int32_t *perm;
  int64_t mul;
};
}  // namespace sfk

using namespace sfk;

// Device scratch of the allocation-free entry (sf_hist_batch_device_noalloc): records, bin tables,
// work items, accumulators and the re-bin queue of one call, carved in that order.  One copy per
// device, held until the process ends; every call on a device shares it.
static __device__ __align__(256) char scratch[SF_NOALLOC_SCRATCH_BYTES];

namespace {

// A bump allocator over a caller-provided device region (the allocation-free entry's scratch).
struct Arena {
  char *base = nullptr;
  size_t cap = 0, used = 0;
  bool split = false;  // a call that did not fit, but would in parts (see plan_build)
};

template <typename T>
struct DevBuf {
  T *p = nullptr;
  size_t cap = 0;  // elements
  bool borrowed = false;  // p points into an Arena: never freed
  // the next n elements of the arena (256-byte aligned); hipErrorOutOfMemory when they do not fit
  hipError_t take(size_t n, Arena &a) {
    if (p && !borrowed) return hipErrorInvalidValue;  // would leak an owned allocation
    const size_t want = std::max<size_t>(n, 1);
    const size_t off = (a.used + 255) & ~(size_t)255;
    if (off > a.cap || want > (a.cap - off) / sizeof(T)) return hipErrorOutOfMemory;
    p = (T *)(a.base + off);
    cap = want;
    borrowed = true;
    a.used = off + want * sizeof(T);
    return hipSuccess;
  }
  hipError_t ensure(size_t n) {
    if (borrowed) return hipErrorInvalidValue;
    if (n <= cap && p) return hipSuccess;
    if (p) {
      hipError_t e = hipFree(p);
      p = nullptr;
      cap = 0;
      if (e != hipSuccess) return e;
    }
    size_t want = std::max<size_t>(n, 1);
    hipError_t e = hipMalloc((void **)&p, want * sizeof(T));
    if (e == hipSuccess) cap = want;
    return e;
  }
  void release() {
    if (p && !borrowed) (void)hipFree(p);
    p = nullptr;
    cap = 0;
    borrowed = false;
  }
};

// Page-locked host memory for one kind of transfer, kept by a context.  `done` follows the last
// copy out of it: the buffer is not written before that copy has ended.
struct Stage {
  char *p = nullptr;
  size_t cap = 0;
  hipEvent_t done = nullptr;
  bool busy = false;
  hipError_t acquire(size_t n) {
    if (busy) {
      const hipError_t e = hipEventSynchronize(done);
      if (e != hipSuccess) return e;
      busy = false;
    }
    if (n <= cap && p) return hipSuccess;
    if (p) (void)hipHostFree(p);
    p = nullptr;
    cap = 0;
    const size_t want = std::max<size_t>(n, 1 << 16);
    const hipError_t e = hipHostMalloc((void **)&p, want, hipHostMallocDefault);
    if (e == hipSuccess) cap = want;
    return e;
  }
  // copies the first n bytes to the device and marks the buffer busy until that has happened
  hipError_t send(void *dst, size_t n, hipStream_t st) {
    hipError_t e = hipSuccess;
    if (!done) e = hipEventCreateWithFlags(&done, hipEventDisableTiming);
    if (e == hipSuccess) e = hipMemcpyAsync(dst, p, n, hipMemcpyHostToDevice, st);
    if (e == hipSuccess) {
      busy = true;
      e = hipEventRecord(done, st);
      if (e != hipSuccess) {  // no event to wait for: wait here
        busy = false;
        (void)hipStreamSynchronize(st);
      }
    }
    return e;
  }
  void release() {
    if (busy) (void)hipEventSynchronize(done);
    if (p) (void)hipHostFree(p);
    if (done) (void)hipEventDestroy(done);
    p = nullptr;
    cap = 0;
    done = nullptr;
    busy = false;
  }
};
// Larger transfers go from and to pageable memory: the copy through a staging buffer would cost
// more than the driver's handling of a pageable one, and the kept memory stays bounded.
inline constexpr size_t kStageMax = 1 << 20;

// largest |v| (NaN ignored): several running maxima, because one is a chain of dependent compares
double abs_max(const double *v, int64_t n) {
  double m[8] = {};
  int64_t k = 0;
  for (; k + 8 <= n; k += 8)
    for (int l = 0; l < 8; ++l) m[l] = std::max(m[l], fabs(v[k + l]));
  for (; k < n; ++k) m[0] = std::max(m[0], fabs(v[k]));
  for (int l = 1; l < 8; ++l) m[0] = std::max(m[0], m[l]);
  return m[0];
}

bool jl_isless(double a, double b) {
  if (a != a) return false;
  if (b != b) return true;
  if (a < b) return true;
  if (a == b) return signbit(a) && !signbit(b);
  return false;
}

int op_order(const sf_problem &p) {
  switch (p.op) {
    case SF_OP_PROJECTED: return p.nl + p.nt;
    case SF_OP_S2: return 2;
    case SF_OP_S3: return 3;
    case SF_OP_T2COMP: return 2;
    case SF_OP_L1T2COMP: return 3;
    case SF_OP_SINGLE_PASS: return 3;
    default: return p.nl;
  }
}

float round_down_f(long double x) {
  float f = (float)x;
  if ((long double)f > x) f = nextafterf(f, -INFINITY);
  return f;
}
float round_up_f(long double x) {
  float f = (float)x;
  if ((long double)f < x) f = nextafterf(f, INFINITY);
  return f;
}

// Cell partition of the positive key axis: binades [2^elo, 2^ehi) cut into 2^M cells each.
struct Partition {
  int M;
  int elo, ehi;
  int ncell() const { return (ehi - elo) << M; }
  // lower bound of cell c (c = 0 also stands for everything below): (1 + m / 2^M) 2^e, exact
  double low(int c) const {
    const int e = elo + (c >> M);
    const uint64_t m = (uint64_t)(c & ((1 << M) - 1));
    const uint64_t bits = ((uint64_t)(e + 1023) << 52) | (m << (52 - M));
    double v;
    memcpy(&v, &bits, sizeof v);
    return v;
  }
};

Partition make_partition(const std::vector<long double> &keys, int cap_cells, int Mmax) {
  long double mn = INFINITY, mx = 0;
  for (long double k : keys)
    if (k > 0 && k < INFINITY) {
      mn = std::min(mn, k);
      mx = std::max(mx, k);
    }
  Partition P;
  if (!(mn < INFINITY)) {  // no positive finite key
    P.elo = 0;
    P.ehi = 1;
    P.M = 0;
    return P;
  }
  int e0, e1;
  frexpl(mn, &e0);  // mn in [2^(e0-1), 2^e0)
  frexpl(mx, &e1);
  P.elo = e0 - 2;   // one spare binade below the smallest key
  P.ehi = e1 + 1;   // and above the largest
  P.elo = std::max(P.elo, -1020);
  P.ehi = std::min(P.ehi, 1020);
  P.M = 0;
  for (int M = Mmax; M >= 0; --M) {
    if (((P.ehi - P.elo) << M) <= cap_cells) {
      P.M = M;
      break;
    }
  }
  return P;
}

}  // namespace

namespace {
// A plan holds everything one batch shape needs on the device: per-point records, bin tables,
// work items, accumulators and the re-bin queue.  Building it does the host work and the
// uploads; launching it enqueues kernels only, so a launch can be captured into a hipGraph and
// replayed while the caller rewrites x/u in place (time slices).
struct Plan {
  sf_ctx *ctx = nullptr;
  int n = 0, G = 0, D = 0, geom_code = 0, ncell = 0, S64 = 0, F32 = 0;
  int nout = 0;  // output slices (n is the internal slice count: six per slice for 2D single pass)
  bool J = false, mixed = false, sload = false, sp = false, fx = false;
  bool rec_f = false;      // its binary64 kernel reads prep64s's records, which lie in rec32
  int block = 256, tj = 256, copies = 1, grid = 1, ncell_max = 1, n_items = 0;
  int strip = 0;            // B-strip launch (fields per strip), 0: off
  int qcap64 = 0;           // binary64 kernel: LDS queue entries per workgroup
  int n_items64 = 0;        // B-strip: the per-slice items the binary64 kernel runs instead
  int64_t total_pts = 0, max_n = 0, total_pairs = 0, cap = 0;
  Params P{};
  DevBuf<double> rec64;
  DevBuf<float> rec32;
  DevBuf<char> tables;  // slices, items, tables, edges and record sources: one upload
  const PrepSliceHost *prep = nullptr;
  const Item *items64 = nullptr;
  // accumulators: sums, counts, the re-bin queue's count, the work counter and the overflow flag,
  // in one piece (one clear; a host call reads sums, counts and queue count in one copy)
  DevBuf<char> acc;
  double *acc_s = nullptr;
  unsigned long long *acc_c = nullptr;
  unsigned long long *pcount = nullptr;
  int *counter = nullptr;
  int *flag = nullptr;
  size_t acc_bytes = 0;
  DevBuf<Pending> pending;
  DevBuf<float> gboxes;   // boxes of the record groups of culled slices
  DevBuf<Item> units;     // culled slices' work units, slice after slice
  int n_units = 0, near_grid = 1, jchunk = 1;
  DevBuf<int32_t> perm;   // spatial order of the binary32 records (culling)
  bool culled = false;    // some slice is evaluated by its work units, not by items
  Arena *arena = nullptr;  // set: every buffer is taken from this region (no device allocation)
  // fused outputs: 1D operators evaluated with the main (joint) one, their accumulators and the
  // caller's outputs they merge into
  int n1d = 0, mcopies = 0;
  DevBuf<double> msums;
  DevBuf<unsigned long long> mcounts;
  double *mdst_s[kMaxFused] = {};
  unsigned long long *mdst_c[kMaxFused] = {};
  hipGraphExec_t graph = nullptr;
  double *g_sums = nullptr;
  unsigned long long *g_counts = nullptr;
  hipStream_t g_stream = nullptr;
  void release() {
    if (graph) (void)hipGraphExecDestroy(graph);
    graph = nullptr;
    rec64.release(); rec32.release(); tables.release(); acc.release(); pending.release();
    perm.release();
    gboxes.release();
    units.release();
    msums.release();
    mcounts.release();
  }
};

}  // namespace

namespace {
// Launch shape of the histogram kernel; 0 keeps the built-in choice.  block: threads per
// workgroup (rows of an i-tile); j_chunk: columns per work item; bpc: workgroups per CU; variant:
// column records through LDS (1), scalar loads (2) or B-strips (3); copies: privatised copies of
// the LDS histogram (1D: lane groups, a power of two up to 64; joint: 1 or 2, by lane halves);
// layout: joint histogram slots value-bin fastest (1) or distance-bin fastest (2), odd row stride.
struct Tuning {
  int block = 0, j_chunk = 0, bpc = 0, variant = 0, copies = 0, layout = 0;
  bool any() const { return block || j_chunk || bpc || variant || copies || layout; }
};

// Autotuner key: (geometry, D, joint, precision code, operator class, 2D single-pass planes,
// log2 of the pair count of the caller's slices, n_dist, n_val).  Shared by the tuner and the
// plan builder so that an entry the tuner stores is the one a later call looks up.
using TuneKey = std::tuple<int, int, int, int, int, int, int, int, int>;
int hist_opk_of(const sf_problem &p0) {
  Params Pk{};
  Pk.op = p0.op;
  Pk.nl = p0.nl;
  Pk.nt = p0.nt;
  Pk.n_val = p0.n_val;
  Pk.nmom = (p0.op == SF_OP_SINGLE_PASS && p0.n_val == 0) ? 4 : 1;
  return hist_opk(Pk, -1, true);
}
TuneKey tune_key(const sf_problem &p0, int64_t input_pairs) {
  int lg = 0;
  for (int64_t v = input_pairs; v > 1; v >>= 1) ++lg;
  const int G = p0.geometry == SF_GEOM_FLAT ? kFlat : kSphere;
  return TuneKey(G, p0.D, p0.n_val > 0 ? 1 : 0, p0.precision, hist_opk_of(p0),
                 sp2d(p0.op, p0.n_val) ? 1 : 0, lg, p0.n_dist, p0.n_val);
}
}  // namespace

struct sf_ctx {
  int device = 0;
  hipStream_t stream = nullptr;
  int n_cu = 0;
  size_t max_smem = 0;
  int clock_khz = 0;   // peak shader clock
  std::string err;
  int64_t stats[8] = {0, 0, 0, 0, 0, 0, 0, 0};
  hipEvent_t ev[4] = {nullptr, nullptr, nullptr, nullptr};
  bool ev_pending = false;
  Tuning tune;  // sf_set_tuning override (all zero: none)
  // largest re-bin queue a call of this context has needed (entries): later plans start there
  int64_t queue_hint = 0;
  // autotuner cache: the call's shape (tune_key) -> the fastest launch shape measured for it
  std::map<TuneKey, Tuning> tuned;
  // device buffers: host-input staging and the plan reused by one-shot calls
  DevBuf<double> d_x, d_u;
  DevBuf<char> d_out;   // host calls of several outputs: their device sums and counts
  DevBuf<double> d_max;  // coordinate magnitudes (partial maxima)
  Stage up_xu, up_tab, down;  // host calls' inputs, every call's tables, read-backs
  Plan oneshot;
  // the allocation-free entry: its plan (buffers borrowed from the scratch array) and this
  // device's address of the array
  Plan noalloc;
  char *scratch_ptr = nullptr;
  Plan fused;  // the fused-output entry's plan
  // spatial sort and culling: device workspace, and each slice's information (launch_cull)
  DevBuf<char> cull_ws;
  DevBuf<double> cull_info;

  int fail(int code, const char *fmt, ...) {
    char buf[512];
    va_list ap;
    va_start(ap, fmt);
    vsnprintf(buf, sizeof buf, fmt, ap);
    va_end(ap);
    err = buf;
    return code;
  }
};

#define HIPCHK(expr)                                                                    \
  do {                                                                                  \
    hipError_t e_ = (expr);                                                             \
    if (e_ != hipSuccess)                                                               \
      return ctx->fail(SF_E_DEVICE, "%s failed: %s", #expr, hipGetErrorString(e_));     \
  } while (0)

namespace {

// A LinearBinEdges rule must describe the materialised edge vector it comes with: n edges (plus
// -Inf / +Inf when padded), first and last edges equal to its fields, a finite non-negative step.
int validate_rule(sf_ctx *ctx, const sf_bin_rule *r, int nbins, const double *edges, const char *what) {
  if (r->kind != SF_RULE_LINEAR) return ctx->fail(SF_E_ARG, "%s: unknown bin rule kind %d", what, r->kind);
  if (r->padded != 0 && r->padded != 1) return ctx->fail(SF_E_ARG, "%s: padded must be 0 or 1", what);
  const int64_t want = r->padded ? r->n + 1 : r->n - 1;
  if (r->n < 2 || want != nbins)
    return ctx->fail(SF_E_DIM, "%s: LinearBinEdges of length %lld does not give %d bins", what, (long long)r->n, nbins);
  if (!(r->first_edge > -INFINITY && r->last_edge < INFINITY && r->first_edge <= r->last_edge))
    return ctx->fail(SF_E_ARG, "%s: LinearBinEdges needs finite first <= last", what);
  if (!(r->step_val >= 0.0 && r->step_val < INFINITY) || r->inv_step != r->inv_step)
    return ctx->fail(SF_E_ARG, "%s: LinearBinEdges needs a finite non-negative step", what);
  const int o = r->padded ? 1 : 0;
  if (edges[o] != r->first_edge || edges[o + r->n - 1] != r->last_edge)
    return ctx->fail(SF_E_ARG, "%s: the edge vector does not hold the LinearBinEdges range", what);
  if (r->padded && !(edges[0] == -INFINITY && edges[nbins] == INFINITY))
    return ctx->fail(SF_E_ARG, "%s: a padded rule needs -Inf and +Inf around the range", what);
  return SF_OK;
}

int validate_one(sf_ctx *ctx, const sf_problem *p, bool host_ptrs, int idx) {
  if (!p) return ctx->fail(SF_E_ARG, "slice %d: null problem", idx);
  if (p->D != 2 && p->D != 3)
    return ctx->fail(SF_E_DIM, "expected spatial/velocity dimension D=2 or D=3 on axis 1; got D=%d", p->D);
  if (p->geometry == SF_GEOM_FLAT) {
    if (p->W != p->D)
      return ctx->fail(SF_E_DIM,
                       "this geometry locates a point with %d coordinate(s) on axis 1 of x, but got "
                       "size(x,1)=%d (velocity dimension D=%d from size(u,1))", p->D, p->W, p->D);
  } else if (p->geometry == SF_GEOM_SPHERE_DEG || p->geometry == SF_GEOM_SPHERE_RAD) {
    if (p->W != 2)
      return ctx->fail(SF_E_DIM,
                       "this geometry locates a point with 2 coordinate(s) on axis 1 of x, but got "
                       "size(x,1)=%d (velocity dimension D=%d from size(u,1))", p->W, p->D);
    if (p->geometry == SF_GEOM_SPHERE_DEG && !(p->radius > 0.0 && p->radius < INFINITY))
      return ctx->fail(SF_E_ARG, "Haversine radius must be positive and finite; got %g", p->radius);
  } else {
    return ctx->fail(SF_E_ARG, "no pair geometry is defined for geometry code %d", p->geometry);
  }
  if (p->N < 0) return ctx->fail(SF_E_DIM, "N must be non-negative; got %lld", (long long)p->N);
  if (p->N >= (1LL << 31) - 4096)
    return ctx->fail(SF_E_UNSUPPORTED, "N=%lld exceeds this backend's 2^31 point limit", (long long)p->N);
  if (p->N > 0 && (!p->x || !p->u)) return ctx->fail(SF_E_ARG, "slice %d: null x or u", idx);
  switch (p->op) {
    case SF_OP_PROJECTED:
      if (p->nl < 0 || p->nt < 0 || p->nl + p->nt > 3)
        return ctx->fail(SF_E_UNSUPPORTED,
                         "ProjectedStructureFunctionType{%d,%d}: this backend supports NL,NT >= 0, NL+NT <= 3",
                         p->nl, p->nt);
      break;
    case SF_OP_S2: case SF_OP_S3: case SF_OP_T2COMP: case SF_OP_L1T2COMP:
      break;
    case SF_OP_FULLVEC:
      if (p->nl < 1 || p->nl > 3)
        return ctx->fail(SF_E_UNSUPPORTED, "FullVectorStructureFunctionType{%d}: NF must be 1..3", p->nl);
      break;
    case SF_OP_SINGLE_PASS:  // n_val > 0: the 2D form, six edge vectors (checked below)
      break;
    default:
      return ctx->fail(SF_E_ARG, "unknown operator code %d (derived operators are not pairwise)", p->op);
  }
  if (p->n_dist < 1 || !p->dist_edges)
    return ctx->fail(SF_E_ARG, "distance_bins must have at least 2 edges");
  for (int k = 0; k <= p->n_dist; ++k) {
    const double e = p->dist_edges[k];
    if (e != e) return ctx->fail(SF_E_ARG, "distance_bins contains NaN");
    if (k > 0 && jl_isless(e, p->dist_edges[k - 1]))
      return ctx->fail(SF_E_ARG, "distance_bins must be sorted ascending");
  }
  if (p->geometry == SF_GEOM_FLAT)
    for (int k = 0; k <= p->n_dist; ++k)
      if (p->dist_edges[k] < 0.0 && !(k == 0 && p->dist_edges[0] == -INFINITY))
        return ctx->fail(SF_E_ARG,
                         "Euclidean distance_bins must be non-negative (squared-distance plan); only a "
                         "leading -Inf (InfPaddedBinEdges catch-all) is allowed");
  if (p->n_val < 0) return ctx->fail(SF_E_ARG, "n_val must be >= 0");
  if (p->n_val > 0) {
    if (!p->val_edges) return ctx->fail(SF_E_ARG, "value_bins missing");
    // the single pass's 2D form carries one edge vector per invariant, back to back
    const int nvec = sp2d(p->op, p->n_val) ? kSpRows : 1;
    for (int t = 0; t < nvec; ++t) {
      const double *ve = p->val_edges + (size_t)t * (p->n_val + 1);
      for (int k = 0; k <= p->n_val; ++k) {
        const double e = ve[k];
        if (e != e) return ctx->fail(SF_E_ARG, "value_bins contains NaN");
        if (k > 0 && jl_isless(e, ve[k - 1]))
          return ctx->fail(SF_E_ARG, "value_bins must be sorted ascending");
      }
    }
  }
  if (p->precision != SF_PREC_FP64 && p->precision != SF_PREC_MIXED && p->precision != SF_PREC_MIXED_FIXED)
    return ctx->fail(SF_E_ARG, "precision must be SF_PREC_FP64, SF_PREC_MIXED or SF_PREC_MIXED_FIXED");
  if (p->count_bits != 32 && p->count_bits != 64)
    return ctx->fail(SF_E_ARG, "count_bits must be 32 or 64");
  if (p->semantics != SF_SEM_POINT && p->semantics != SF_SEM_BATCH)
    return ctx->fail(SF_E_ARG, "semantics must be SF_SEM_POINT or SF_SEM_BATCH");
  if (p->dist_rule) {
    const int rc = validate_rule(ctx, p->dist_rule, p->n_dist, p->dist_edges, "distance_bins");
    if (rc) return rc;
  }
  if (p->val_rule) {
    if (p->n_val == 0) return ctx->fail(SF_E_ARG, "val_rule given without value_bins");
    if (p->op == SF_OP_SINGLE_PASS)
      return ctx->fail(SF_E_UNSUPPORTED, "the single pass's 2D form takes explicit value edge vectors only");
    const int rc = validate_rule(ctx, p->val_rule, p->n_val, p->val_edges, "value_bins");
    if (rc) return rc;
  }
  const unsigned __int128 pairs = (unsigned __int128)p->N * (unsigned __int128)(p->N > 0 ? p->N - 1 : 0) / 2;
  const unsigned __int128 cmax = p->count_bits == 32 ? 0xffffffffull : 0xffffffffffffffffull;
  if (pairs > cmax)
    return ctx->fail(SF_E_COUNT,
                     "count_eltype=UInt%d cannot represent the worst-case pair count for N=%lld; "
                     "pass count_eltype=UInt64 or Int64.", p->count_bits, (long long)p->N);
  if (host_ptrs && p->geometry == SF_GEOM_SPHERE_RAD) {
    for (int64_t k = 0; k < 2 * p->N; ++k)
      if (fabs(p->x[k]) > 1.6e6)
        return ctx->fail(SF_E_UNSUPPORTED, "SphericalAngle coordinates beyond |1.6e6| rad are not supported");
  }
  return SF_OK;
}

int validate_batch(sf_ctx *ctx, int n, const sf_problem *s, bool host_ptrs) {
  if (n < 0) return ctx->fail(SF_E_ARG, "n_slices must be >= 0");
  if (n > 0 && !s) return ctx->fail(SF_E_ARG, "null slices");
  for (int k = 0; k < n; ++k) {
    int rc = validate_one(ctx, &s[k], host_ptrs, k);
    if (rc) return rc;
    if (k > 0) {
      const sf_problem &a = s[0], &b = s[k];
      if (a.D != b.D || a.W != b.W || a.geometry != b.geometry || a.op != b.op || a.nl != b.nl ||
          a.nt != b.nt || a.n_dist != b.n_dist || a.n_val != b.n_val || a.precision != b.precision ||
          a.semantics != b.semantics ||
          (a.geometry == SF_GEOM_SPHERE_DEG && a.radius != b.radius))
        return ctx->fail(SF_E_ARG, "slice %d: all slices must share D, geometry, operator, bin counts and precision", k);
    }
  }
  return SF_OK;
}

// Host-side tables for one slice.
struct SliceTables {
  std::vector<Cell> tab64, tab32;
  std::vector<double> dedges;  // exact keys
  Slice desc{};
  double crowd = 0;  // share of the keys that the table leaves uncertain (the edges' own intervals aside)
};

// binary64 decision points of a LinearBinEdges rule lie within this distance of the edge values
long double rule_slack(const sf_bin_rule *r) {
  if (!r) return 0.0L;
  return ldexpl(1.0L, -48) * (fabsl((long double)r->first_edge) + fabsl((long double)r->last_edge));
}

LinRule lin_rule_of(const sf_bin_rule *r) {
  LinRule L{};
  if (!r) return L;
  L.on = 1;
  L.padded = r->padded;
  L.n = r->n;
  L.f = r->first_edge;
  L.l = r->last_edge;
  L.inv = r->inv_step;
  L.step = r->step_val;
  return L;
}

// the kernels' lin_rule_bin
int lin_rule_bin_host(const LinRule &r, double x, int nb) {
  const double c = -r.f * r.inv;
  const double t = std::fma(x, r.inv, c), n = (double)r.n;
  const double fi = std::fmin(std::fmax(std::floor(t) + 1.0, 1.0), n);
  int k = (int)fi + (std::fma(fi - 1.0, r.step, r.f) < x ? 1 : 0);
  if (x <= r.f) k = 1;
  if (x > r.l) k = (int)r.n + 1;
  if (!r.padded) --k;
  if (r.padded && x <= -INFINITY) k = 0;
  return x != x ? nb + 1 : k;
}

void build_tables(const sf_problem &p, double xmax, SliceTables &T) {
  const int nE = p.n_dist + 1;
  const bool flat = p.geometry == SF_GEOM_FLAT;
  const long double R = flat ? 1.0L : (p.geometry == SF_GEOM_SPHERE_DEG ? (long double)p.radius : 1.0L);
  // ---- binary64 exact keys and table
  T.dedges.resize(nE);
  std::vector<long double> k64(nE);
  for (int k = 0; k < nE; ++k) {
    const double e = p.dist_edges[k];
    // flat, point-field kernels: squared edges (a leading -Inf, InfPaddedBinEdges' underflow
    // edge, stays -Inf); flat, batch-leading kernels: the edges themselves (r = sqrt(r^2) is
    // binned); sphere: the edges themselves, -0.0 -> +0.0 (keys are > 0)
    if (flat) T.dedges[k] = p.semantics == SF_SEM_BATCH ? e : (e == -INFINITY ? e : e * e);
    else T.dedges[k] = e == 0.0 ? 0.0 : e;
    k64[k] = T.dedges[k];
  }
  Partition P64 = make_partition(k64, 1024, 6);
  const int n64 = P64.ncell();
  T.tab64.resize(n64);
  int b64 = 0;  // edges below the cell: they ascend, and so do the cells
  for (int c = 0; c < n64; ++c) {
    const double low = P64.low(c);  // cell bounds are exact binary64 values
    // (keys below the window, c = 0: only non-positive edges are below them)
    while (b64 < nE && (c == 0 ? T.dedges[b64] <= 0.0 : T.dedges[b64] < low)) ++b64;
    T.tab64[c].bx = b64;
    T.tab64[c].lo = INFINITY;
    T.tab64[c].hi = INFINITY;
    T.tab64[c].blo = 0;
  }
  // ---- binary32 keys: flat r^2 = e^2; sphere chord^2 = (2 sin(e / 2R))^2
  std::vector<long double> C(nE);
  for (int k = 0; k < nE; ++k) {
    const long double e = p.dist_edges[k];
    if (flat) {
      C[k] = (e == -INFINITY) ? e : e * e;
    } else if (e <= 0) {
      C[k] = e;
    } else {
      const long double th = std::min(e / R, (long double)M_PIl);
      const long double c = 2.0L * sinl(0.5L * th);
      C[k] = c * c;
    }
  }
  // margins: relative 2^-18 (64 ulp) plus an absolute term for the hi/lo split of the inputs
  const long double drel = ldexpl(1.0L, -20);
  const long double e1 = flat ? ldexpl(1.0L, -44) * std::max((long double)xmax, 1e-300L) : ldexpl(1.0L, -44);
  // a LinearBinEdges rule decides within a few binary64 ulps of max(|first|, |last|) of each
  // materialised edge (its rounding of the step, 1 / step and the two multiply-adds); the margin
  // covers 2^-48 (|first| + |last|), in key-space units
  const long double dr = rule_slack(p.dist_rule) / R;
  std::vector<float> lo(nE), hi(nE);
  for (int k = 0; k < nE; ++k) {
    if (C[k] == INFINITY) { lo[k] = INFINITY; hi[k] = INFINITY; continue; }
    const long double a = 2.0L * sqrtl(fabsl(C[k])) * (e1 + dr) + (e1 + dr) * (e1 + dr) + 1e-30L;
    lo[k] = round_down_f(C[k] - fabsl(C[k]) * drel - a);
    hi[k] = round_up_f(C[k] + fabsl(C[k]) * drel + a);
  }
  std::vector<long double> ckeys(C.begin(), C.end());
  Partition P32 = make_partition(ckeys, kCell32Max, 6);
  // keep every cell's lower bound representable in binary32
  P32.elo = std::max(P32.elo, -125);
  P32.ehi = std::min(P32.ehi, 127);
  if (P32.ehi <= P32.elo) P32.ehi = P32.elo + 1;
  // Nearly coincident points: the binary32 records carry positions as hi + lo (2^-48 relative), a
  // direction error of 2^-48 / separation that below a separation of 2^-22 (sphere: radians; flat:
  // times max|x|) would outgrow the value bound's margin and the reference's own binary64 accuracy
  // (2^-53 / separation); below 1e-30 products of tiny differences underflow.  Nearly antipodal
  // points, within 2^-10 rad: sin(separation) and the error bound's 1 / sin lose their accuracy.
  const float close = flat ? round_up_f(std::max(1e-30L, ldexpl((long double)xmax * (long double)xmax, -44)))
                           : 0x1p-44f;
  const float anti = 4.0f - 0x1p-20f;
  double top = flat ? 0.0 : 4.0;  // largest key that matters (flat: that of the last finite edge)
  for (int k = 0; flat && k < nE; ++k)
    if (C[k] < INFINITY) top = std::max(top, (double)C[k]);
  // The table of n32 cells from their bounds: cell c holds keys in [Flo[c], Fhi[c]] at most (both
  // ascend).  Per cell: the edges whose intervals end below it, and the number (and the index, where
  // it is one) of those that meet it, from each edge's first and last cell.  Returns the length of
  // key in [0, top] that its cells leave uncertain, the edges' own intervals aside: those that hold
  // several edges, or one edge beside the nearly coincident keys.
  // On the sphere a quarter of it is the share of evenly spread pairs that will be re-binned.
  auto fill = [&](const std::vector<float> &Flo, const std::vector<float> &Fhi) {
    const int n32 = (int)Flo.size();
    double lost = 0.0;
    auto length = [&](double a, double b) { return std::max(0.0, std::min(top, b) - std::max(0.0, a)); };
    T.tab32.resize(n32);
    std::vector<int> dbelow(n32 + 1, 0), dmeet(n32 + 1, 0), dwhich(n32 + 1, 0);
    for (int k = 0; k < nE; ++k) {
      if (C[k] == -INFINITY) { ++dbelow[0]; continue; }  // -Inf: below every key
      const int c0 = (int)(std::partition_point(Fhi.begin(), Fhi.end(), [&](float Fn) { return lo[k] >= Fn; }) -
                           Fhi.begin());
      const int c1 = (int)(std::partition_point(Flo.begin(), Flo.end(), [&](float Fc) { return !(hi[k] < Fc); }) -
                           Flo.begin());
      ++dbelow[c1];
      if (c0 < c1) {
        ++dmeet[c0];
        --dmeet[c1];
        dwhich[c0] += k;
        dwhich[c1] -= k;
      }
    }
    for (int c = 0, below = 0, nint = 0, which = 0; c < n32; ++c) {
      const float Fc = Flo[c], Fn = Fhi[c];
      below += dbelow[c];
      nint += dmeet[c];
      which += dwhich[c];
      Cell &cl = T.tab32[c];
      cl.bx = 0;
      cl.blo = below;
      if (nint == 0) {
        cl.lo = INFINITY;
        cl.hi = INFINITY;
      } else if (nint == 1) {
        cl.lo = lo[which];
        cl.hi = hi[which];
      } else {
        cl.lo = -INFINITY;
        cl.hi = INFINITY;
        lost += length(Fc, Fn);
      }
      // keys that the kernels leave to the exact sequence wherever a bin holds them: those of nearly
      // coincident points (below `close`) and on the sphere of nearly antipodal ones
      if (Fc < close) {
        if (nint == 0) {
          if (below > 0 && below < nE) {
            cl.lo = -INFINITY;
            cl.hi = close;
            cl.blo = below - 1;
          }
        } else if (nint == 1 && hi[which] <= close) {  // an edge at or near zero
          cl.lo = -INFINITY;
          cl.hi = close;
        } else if (!(nint == 1 && below == 0 && lo[which] > close)) {  // (else nothing counted below the edge)
          cl.lo = -INFINITY;
          cl.hi = INFINITY;
          if (nint == 1 && Fn > close) lost += length(Fc, Fn);
        }
      }
      // (keys past the last edge are in no bin: an axis that ends below `anti` has none of the latter)
      const int under = below + (nint == 1 && hi[which] < anti);
      if (!flat && below + nint > 0 && under < nE && Fn > anti && Fc < 8.0f) {
        cl.lo = nint == 0 ? anti : std::min(cl.lo, anti);
        cl.hi = INFINITY;
      }
    }
    return lost;
  };
  // the length of key that fill would return for the plain table of P32's binades, M bits each
  auto lost_of = [&](int M) {
    const Partition Q{M, P32.elo, P32.ehi};
    auto cell = [&](float v) {
      int32_t bits;
      memcpy(&bits, &v, sizeof bits);
      return std::min(std::max((bits >> (23 - M)) - ((Q.elo + 127) << M), 0), Q.ncell() - 1);
    };
    auto low = [&](int c) { return c > 0 ? Q.low(c) : 0.0; };
    auto high = [&](int c) { return c + 1 < Q.ncell() ? std::min(top, Q.low(c + 1)) : top; };
    const int cc = cell(close);
    double len = 0.0;
    int seen = -1, counted = -1;  // last cell that an edge so far meets, last one counted
    int below_c = 0, n_c = 0, k_c = 0;  // edges below cell cc; in it, and the last of those
    for (int k = 0; k < nE; ++k) {
      if (!(std::fabs(C[k]) < INFINITY)) {
        below_c += C[k] < 0;
        continue;
      }
      const int c0 = cell(lo[k]), c1 = cell(hi[k]);
      for (int c = std::max(c0, counted + 1); c <= std::min(seen, c1); ++c) {
        len += std::max(0.0, high(c) - low(c));
        counted = c;
      }
      seen = std::max(seen, c1);
      below_c += c1 < cc;
      if (c0 <= cc && cc <= c1) {
        ++n_c;
        k_c = k;
      }
    }
    if (n_c == 1 && low(cc) < close && hi[k_c] > close && (below_c > 0 || lo[k_c] <= close))
      len += std::max(0.0, high(cc) - low(cc));
    return len;
  };
  // the coarsest cells that keep the edges as far apart as the finest that fit, and away from the nearly
  // coincident keys (a leading -Inf edge and a second one at a power of two): a wave's lanes then share
  // more of them (reads of one cell are broadcasts, of two cells in one bank a conflict), and
  // the LDS that they leave holds more copies of a 1D histogram, or another workgroup: du_L^2 over 64
  // log bins, flat 2D, N = 65536, 112 cells for 896 and 32 copies for 16: kernel 1934 -> 1729 us
  const double crowd = lost_of(P32.M);
  for (int M = 0; M < P32.M; ++M)
    if (lost_of(M) <= crowd) P32.M = M;
  const int np = P32.ncell();  // <= kCell32Max: at most 252 binades, M chosen to fit
  std::vector<float> Flo(np, -INFINITY), Fhi(np, INFINITY);
  for (int c = 1; c < np; ++c) Fhi[c - 1] = Flo[c] = (float)P32.low(c);
  (void)fill(Flo, Fhi);
  T.crowd = crowd / std::max(top, 1e-300);
  int mir = 0;
  // (its five instructions a pair cost 4 %, a share of 0.8 % re-binned 40 % and more; it can be larger
  // than the plain table by up to 16 KB of LDS, which a histogram of thousands of bins may not leave)
  if (!flat && p.precision == SF_PREC_FP64 && crowd > 0.004 && nE <= kCell32Max) {
    // mirrored table (cell32m): `mir` cells for keys below 2, the rest by m = 4 - key below 2 downwards.
    // The smallest cells are those of the edge next to zero or next to 4 (keys within 2^-20 of 4 are
    // uncertain anyway: nearly antipodal).
    long double near = 2.0L;
    for (int k = 0; k < nE; ++k) {
      if (C[k] > 0 && C[k] < near) near = C[k];
      if (C[k] < 4.0L - 0x1p-20L && 4.0L - C[k] < near) near = 4.0L - C[k];
    }
    int elo = 0;
    while (elo > -120 && ldexpl(1.0L, elo + 1) > near) --elo;
    Partition H;
    H.elo = elo;
    H.ehi = 1;
    H.M = 6;
    while (H.M > 0 && 2 * H.ncell() > kCell32Max) --H.M;
    if (2 * H.ncell() <= kCell32Max) {
      const std::vector<Cell> plain = T.tab32;
      mir = H.ncell();
      Flo.assign(2 * mir, -INFINITY);
      Fhi.assign(2 * mir, INFINITY);
      for (int c = 0; c < mir; ++c) {
        if (c > 0) Flo[c] = (float)H.low(c);
        Fhi[c] = c + 1 < mir ? (float)H.low(c + 1) : 2.0f;
        // m in [low(c), low(c + 1)), the first from below everything: one unit outwards
        const int q = 2 * mir - 1 - c;
        Flo[q] = nextafterf((float)(4.0 - (c + 1 < mir ? H.low(c + 1) : 2.0)), -INFINITY);
        if (c > 0) Fhi[q] = nextafterf((float)(4.0 - H.low(c)), INFINITY);
      }
      if (fill(Flo, Fhi) < 0.5 * crowd) {
        P32 = H;
      } else {  // (a smallest edge so small that the cells of two halves are too wide)
        mir = 0;
        T.tab32 = plain;
      }
    }
  }
  const int n32 = (int)T.tab32.size();
  Slice &s = T.desc;
  s.drule = lin_rule_of(p.dist_rule);
  s.vrule = p.n_val > 0 ? lin_rule_of(p.val_rule) : LinRule{};
  s.M64 = P64.M;
  s.ncell64 = n64;
  s.base64 = ((int64_t)(P64.elo + 1023) << P64.M);  // cell 0 starts at 2^elo
  s.M32 = P32.M;
  s.ncell32 = n32;
  s.mir = mir;
  s.base32 = ((P32.elo + 127) << P32.M);
  // value axis
  s.v_uniform = 0;
  s.v_negzero = 0;
  s.vzero = kNoZeroBin;
  s.v0 = 0; s.vinv = 0; s.v0f = 0; s.vinvf = 0; s.vtc = 0; s.vslack = 0; s.vabs = 0; s.vslackt = 0; s.vtcu = 0; s.veps2 = 0;
  s.v_fx = 0; s.vwf = 0; s.vsf = 0; s.fxc1 = 0; s.fxc0 = 0; s.plane = 0; s.vsmall = 0; s.gz = 0;
  s.v_log = 0; s.vk0 = 0; s.vl0f = 0; s.vlinvf = 0;
  if (p.n_val > 0) {
    const int nv = p.n_val;
    const double *E = p.val_edges;
    for (int k = 0; k <= nv; ++k) if (E[k] == 0.0 && signbit(E[k])) s.v_negzero++;
    if (!s.v_negzero && !(p.op == SF_OP_PROJECTED && p.nl == 0 && p.nt == 0)) {
      s.vzero = -1;
      if (s.vrule.on) s.vzero += lin_rule_bin_host(s.vrule, 0.0, nv);
      else
        for (int k = 0; k <= nv; ++k) s.vzero += E[k] < 0.0;
    }
    const double v0 = E[0], v1 = E[nv];
    if (v0 > -INFINITY && v1 < INFINITY && v1 > v0) {
      const long double w = ((long double)v1 - v0) / nv;
      long double dev = 0;
      for (int k = 0; k <= nv; ++k) dev = std::max(dev, fabsl(((long double)E[k] - v0) / w - k));
      if (dev < 0.25L) {
        s.v_uniform = 1;
        s.v0 = v0;
        s.vinv = (double)(1.0L / w);
        s.v0f = (float)v0;
        s.vinvf = (float)(1.0L / w);
        // exact product of two binary32 numbers, rounded once; with the roundings of v0 and of
        // 1 / w to binary32 it is within 3 * 2^-24 |v0 / w| (and terms of second order) of
        // -v0 / w, which the slack's 4u (1 + |v0 / w|) covers
        s.vtc = (float)(-(double)s.v0f * (double)s.vinvf);
        // slack in t units: edge non-uniformity + rounding of v0 and 1/w in binary32
        const long double u = ldexpl(1.0L, -24);
        s.vslack = round_up_f(dev + 4.0L * u * (1.0L + fabsl((long double)v0 / w)) + 4.0L * u * nv + 1e-6L +
                              rule_slack(p.val_rule) / w);
        // a value in range has |t| < nv + 1: the rounding of t and of t + eps, t - eps (u |t| each, of which
        // two meet an edge).  Twice this (8u |t| at its largest) left a quarter more pairs to the re-bin
        // where the values crowd at an edge in the middle of the axis
        s.vslackt = round_up_f((long double)s.vslack + 4.0L * u * (nv + 2));
        // one margin for every value in range (|t| < nv + 1): 16u |t| covers the rounding of the
        // multiply-add, of the value and of the sums vtc + margin and t - floor(t)
        const long double eps = (long double)s.vslack + 24.0L * u * (nv + 2) + 4.0L * u * fabsl((long double)s.vtc);
        s.vtcu = (float)((long double)s.vtc + eps);
        s.veps2 = round_up_f(2.0L * eps);
        // fixed-point joint cells need every value of bin g within [-1/64, 1 + 1/64] widths of
        // the binary32 grid point fmaf(g, vwf, v0f)
        if (dev < 1.0L / 64) {
          s.v_fx = 1;
          s.vwf = (float)w;
          s.vsf = kFxScale / s.vwf;
          s.fxc1 = (float)((double)s.vwf * (double)s.vsf);
          s.fxc0 = (float)(8388608.0 + (double)kFxBias - (double)s.v0f * (double)s.vsf);
          // a certified bin g of a value with |v| < w/4 is within half a bin of [-w/4, w/4] (the
          // binary32 value's error is below half a bin, or the pair is re-binned), so g - gz is
          // 1 .. 3 with gz = floor((-w/4 - v0)/w) - 2; the kZeroBins = 5 cells gz .. gz + 4 leave
          // a bin of margin on either side
          s.vsmall = (float)(0.25L * w);
          const long double gzl = floorl((-0.25L * w - (long double)v0) / w) - 2.0L;
          s.gz = (int32_t)std::max(-1.0e9L, std::min(1.0e9L, gzl));
        }
      }
    }
    if (!s.v_uniform) s.vslack = (float)ldexpl(1.0L, -21);  // relative slack for binary32 edges
    s.vabs = round_up_f(2.0L * rule_slack(p.val_rule));
    if (!s.v_uniform) {
      // log-spaced from the first positive edge on (a leading 0 or negative edges allowed): the
      // binary32 kernel guesses the bin from log2(v) and walks to it; the walk alone decides, so
      // the guess only needs to be close
      int k0 = 0;
      while (k0 <= nv && !(E[k0] > 0.0)) ++k0;
      if (k0 + 3 <= nv && E[nv] < INFINITY) {
        const long double l0 = log2l((long double)E[k0]), l1 = log2l((long double)E[nv]);
        const long double st = (l1 - l0) / (nv - k0);
        long double dev = 0;
        for (int k = k0; k <= nv; ++k) dev = std::max(dev, fabsl((log2l((long double)E[k]) - l0) / st - (k - k0)));
        if (st > 0 && dev < 0.25L) {
          s.v_log = 1;
          s.vk0 = k0;
          s.vl0f = (float)l0;
          s.vlinvf = (float)(1.0L / st);
        }
      }
    }
  }
}

// whether build_tables gives both slices of a batch (validate_batch: one geometry, operator and bin
// counts) the same tables
bool same_tables(const sf_problem &a, double xa, const sf_problem &b, double xb) {
  auto rule = [](const sf_bin_rule *r, const sf_bin_rule *q) {
    return r == q || (r && q && r->kind == q->kind && r->padded == q->padded && r->n == q->n &&
                      r->first_edge == q->first_edge && r->last_edge == q->last_edge &&
                      r->inv_step == q->inv_step && r->step_val == q->step_val);
  };
  auto edges = [](const double *e, const double *f, int n) {
    return e == f || memcmp(e, f, sizeof(double) * n) == 0;
  };
  return xa == xb && rule(a.dist_rule, b.dist_rule) && edges(a.dist_edges, b.dist_edges, a.n_dist + 1) &&
         (a.n_val == 0 || (rule(a.val_rule, b.val_rule) && edges(a.val_edges, b.val_edges, a.n_val + 1)));
}

int64_t pairs_of(int64_t n) { return n > 1 ? n * (n - 1) / 2 : 0; }

// output cells per slice: (n_dist), (n_dist, n_val), or (6, n_dist) for the single pass
int out_cells(const sf_problem &p) {
  if (p.op == SF_OP_SINGLE_PASS) return kSpRows * p.n_dist * (p.n_val > 0 ? p.n_val : 1);
  return p.n_dist * (p.n_val > 0 ? p.n_val : 1);
}

// _sp1d_derive_rows! (serial_single_pass.jl:208-219) on host memory
void derive_sp_host(double *s, uint64_t *c, int64_t nbins) {
  for (int64_t b = 0; b < nbins; ++b) {
    double *col = s + kSpRows * b;
    uint64_t *cc = c + kSpRows * b;
    col[2] = col[0] - col[1];
    col[5] = col[3] - col[4];
    for (int t = 1; t < kSpRows; ++t) cc[t] = cc[0];
  }
}

}  // namespace

// ----------------------------------------------------------------------------------------------
// C ABI
// ----------------------------------------------------------------------------------------------
extern "C" int sf_create(int device, sf_ctx **out) {
  if (!out) return SF_E_ARG;
  *out = nullptr;
  int ndev = 0;
  if (hipGetDeviceCount(&ndev) != hipSuccess || ndev <= 0) return SF_E_DEVICE;
  if (device < 0 || device >= ndev) return SF_E_ARG;
  sf_ctx *ctx = new sf_ctx();
  ctx->device = device;
  if (hipSetDevice(device) != hipSuccess) { delete ctx; return SF_E_DEVICE; }
  hipDeviceProp_t prop;
  if (hipGetDeviceProperties(&prop, device) != hipSuccess) { delete ctx; return SF_E_DEVICE; }
  ctx->n_cu = prop.multiProcessorCount;
  ctx->max_smem = prop.sharedMemPerBlock;
  ctx->clock_khz = prop.clockRate;
  int v = 0;
  if (hipDeviceGetAttribute(&v, hipDeviceAttributeMaxSharedMemoryPerBlock, device) == hipSuccess && v > 0)
    ctx->max_smem = (size_t)v;
  if (hipStreamCreate(&ctx->stream) != hipSuccess) { delete ctx; return SF_E_DEVICE; }
  // this device's copy of the allocation-free entry's scratch array (the array's name is a host
  // stand-in; only this address is used on the host)
  if (hipGetSymbolAddress((void **)&ctx->scratch_ptr, HIP_SYMBOL(scratch)) != hipSuccess) {
    ctx->scratch_ptr = nullptr;
    (void)hipGetLastError();
  }
  *out = ctx;
  return SF_OK;
}

extern "C" void sf_destroy(sf_ctx *ctx) {
  if (!ctx) return;
  (void)hipSetDevice(ctx->device);
  (void)hipStreamSynchronize(ctx->stream);
  ctx->d_x.release();
  ctx->d_u.release();
  ctx->d_out.release();
  ctx->d_max.release();
  ctx->up_xu.release();
  ctx->up_tab.release();
  ctx->down.release();
  ctx->oneshot.release();
  ctx->noalloc.release();
  ctx->fused.release();
  ctx->cull_ws.release();
  ctx->cull_info.release();
  for (int k = 0; k < 4; ++k)
    if (ctx->ev[k]) (void)hipEventDestroy(ctx->ev[k]);
  (void)hipStreamDestroy(ctx->stream);
  delete ctx;
}

extern "C" const char *sf_last_error(const sf_ctx *ctx) { return ctx ? ctx->err.c_str() : "null context"; }

extern "C" int sf_device_info(sf_ctx *ctx, int64_t out[4]) {
  if (!ctx || !out) return SF_E_ARG;
  out[0] = ctx->n_cu;
  out[1] = ctx->clock_khz;
  out[2] = (int64_t)ctx->max_smem;
  out[3] = 64;
  return SF_OK;
}

extern "C" int sf_last_stats(sf_ctx *ctx, int64_t out[8]) {
  if (!ctx || !out) return SF_E_ARG;
  if (ctx->ev_pending) {
    ctx->ev_pending = false;
    float t01 = 0, t12 = 0, t03 = 0;
    if (hipEventSynchronize(ctx->ev[3]) == hipSuccess) {
      (void)hipEventElapsedTime(&t01, ctx->ev[0], ctx->ev[1]);
      (void)hipEventElapsedTime(&t12, ctx->ev[1], ctx->ev[2]);
      (void)hipEventElapsedTime(&t03, ctx->ev[0], ctx->ev[3]);
    }
    ctx->stats[4] = (int64_t)(t01 * 1e6);
    ctx->stats[5] = (int64_t)(t12 * 1e6);
    ctx->stats[6] = (int64_t)(t03 * 1e6);
  }
  for (int k = 0; k < 8; ++k) out[k] = ctx->stats[k];
  return SF_OK;
}

extern "C" int sf_check(int32_t n_slices, const sf_problem *slices, char *msg, int32_t msg_len) {
  sf_ctx tmp;  // carries the message only; no device state is touched
  const int rc = validate_batch(&tmp, n_slices, slices, true);
  if (msg && msg_len > 0) {
    strncpy(msg, tmp.err.c_str(), (size_t)msg_len - 1);
    msg[msg_len - 1] = 0;
  }
  return rc;
}

extern "C" int sf_eval_math(sf_ctx *ctx, int32_t fn, int64_t n, const double *a, const double *b,
                            double *out) {
  if (!ctx) return SF_E_ARG;
  if (fn < 0 || fn > 4 || n < 0 || (n > 0 && (!a || !out))) return ctx->fail(SF_E_ARG, "bad arguments");
  if ((fn == 2 || fn == 4) && n > 0 && !b) return ctx->fail(SF_E_ARG, "fn needs b");
  if (n == 0) return SF_OK;
  HIPCHK(hipSetDevice(ctx->device));
  const int nout = (fn <= 1) ? 2 : 1;
  DevBuf<double> da, db, dout;
  HIPCHK(da.ensure((size_t)n));
  HIPCHK(db.ensure((size_t)n));
  HIPCHK(dout.ensure((size_t)n * nout));
  hipStream_t st = ctx->stream;
  HIPCHK(hipMemcpyAsync(da.p, a, sizeof(double) * n, hipMemcpyHostToDevice, st));
  if (b) HIPCHK(hipMemcpyAsync(db.p, b, sizeof(double) * n, hipMemcpyHostToDevice, st));
  HIPCHK(launch_eval_math(fn, n, da.p, db.p, dout.p, st));
  HIPCHK(hipMemcpyAsync(out, dout.p, sizeof(double) * n * nout, hipMemcpyDeviceToHost, st));
  HIPCHK(hipStreamSynchronize(st));
  da.release(); db.release(); dout.release();
  return SF_OK;
}

extern "C" int sf_set_tuning(sf_ctx *ctx, int32_t block, int32_t j_chunk, int32_t blocks_per_cu,
                             int32_t variant, int32_t copies, int32_t layout) {
  if (!ctx) return SF_E_ARG;
  if (block != 0 && (block < 64 || block > 1024 || block % 64 != 0))
    return ctx->fail(SF_E_ARG, "block must be 0 or a multiple of 64 in [64, 1024]");
  if (j_chunk < 0 || blocks_per_cu < 0) return ctx->fail(SF_E_ARG, "tuning values must be >= 0");
  if (variant < 0 || variant > 3) return ctx->fail(SF_E_ARG, "variant must be 0, 1, 2 or 3");
  if (copies < 0 || copies > 64 || (copies & (copies - 1)) != 0)
    return ctx->fail(SF_E_ARG, "copies must be 0 or a power of two up to 64");
  if (layout < 0 || layout > 2) return ctx->fail(SF_E_ARG, "layout must be 0, 1 or 2");
  ctx->tune = Tuning{block, j_chunk, blocks_per_cu, variant, copies, layout};
  return SF_OK;
}

namespace {

// ---- spatial sort and culling ----------------------------------------------------------------
// When every distance edge of a slice is finite, a pair farther apart than the last edge is not
// counted.  Points are put in Morton (Z-curve) order of their key-space coordinates (flat: x;
// sphere: the unit vector), so that consecutive points are spatially compact, and only those blocks
// of 64 rows and one or two groups of kGroup columns are evaluated whose bounding boxes are not
// farther apart than the last edge: the slice's work units, which the device lists (launch_cull).
// Only the binary32 records are reordered (each keeps its caller index); the binary64 records, and
// with them every re-binned pair, stay in the caller's order.
struct CullInfo {
  bool tried = false, active = false;
  double reach = 0;       // largest counted distance in key-space units
  int64_t units = 0;
  int rstep = 1;          // row blocks of 64 rstep records
};

// Starts the spatial order, group boxes and number of work units of one slice on the device
// (launch_cull), where culling may be worth it: the record order goes to perm (device, N entries).
int cull_start(sf_ctx *ctx, const sf_problem &p, const double *dx, double xmax, int rows, hipStream_t st, CullInfo &ci,
               int32_t *perm, double *info_d, float *gbox) {
  const int64_t N = p.N;
  const double emax = p.dist_edges[p.n_dist];
  if (N < 4 * (int64_t)rows || N > (1LL << 30) || !(emax < INFINITY)) return SF_OK;
  const bool flat = p.geometry == SF_GEOM_FLAT;
  // largest distance in key-space units: flat |dx|; sphere chord 2 sin(theta / 2)
  double reach;
  if (flat) {
    reach = std::max(emax, 0.0);
  } else {
    const double R = p.geometry == SF_GEOM_SPHERE_DEG ? p.radius : 1.0;
    const double th = std::min(std::max(emax, 0.0) / R, M_PI);
    reach = 2.0 * sin(0.5 * th);
  }
  // cheap refusals before touching the data: the sphere's extent is at most 2, a flat slice's
  // at most 2 max|x| (when the caller measured it)
  if (!flat && reach >= 1.0) return SF_OK;
  if (flat && xmax > 0 && reach >= xmax) return SF_OK;
  // 8 bits of the Morton key per axis where its cells (the extent's 1/256 at most) are a quarter of the
  // reach or less: finer ones leave the boxes what they are (N = 262144 points of the sphere, reach
  // 0.05 rad: 206e6 pairs evaluated, 204e6 with 10), and the sort takes two passes, not three
  const double ext = flat ? 2.0 * xmax : 2.0;
  const int bits = ext > 0 && ext <= 64.0 * reach ? 8 : 10;
  const int geom = flat ? 0 : (p.geometry == SF_GEOM_SPHERE_DEG ? 1 : 2);
  HIPCHK(ctx->cull_ws.ensure(cull_workspace_bytes(N)));
  HIPCHK(launch_cull(dx, N, p.W, p.D, geom, reach, bits, ctx->cull_ws.p, perm, info_d, gbox, st));
  ci.tried = true;
  ci.reach = reach;
  return SF_OK;
}

// Whether culling may be worth it, from launch_cull's info, and whether the units of wide row blocks are
// to be counted (ci.rstep).  Joint histograms of points on a surface: rows that lie side by side in the
// spatial order send many lanes to one cell where the reach holds thousands of points, and LDS atomics to one
// address serialize.  The waves of a block of 1024 rows take rows 16 apart; but the block's box is larger,
// and more columns are in its reach.  (1D histograms have copies for that.  In space, points as close have
// boxes that much wider: blocks of 1024 rows took 1.4 to 2.0 times as long at N = 65536.)
void cull_rows(const sf_problem &p, bool J, const double *info, int rows, CullInfo &ci) {
  if (!ci.tried || p.N < 4 * (int64_t)rows) return;
  if (info[6] != 0.0) return;  // non-finite coordinates: no culling
  // worth it only if the reach is small against the extent
  double ext = 0;
  for (int k = 0; k < 3; ++k) ext = std::max(ext, info[3 + k] - info[k]);
  if (!(info[9] < 0.5 * ext)) return;
  uint64_t units;
  memcpy(&units, &info[8], sizeof units);
  ci.active = true;
  ci.units = (int64_t)std::min<uint64_t>(units, 1ull << 31);
  // (from 4096 columns in reach of a row block on: below, wide blocks do not pay, and counting them would)
  if (J && p.W == 2 && ci.units > p.N) ci.rstep = kWideRows;
}

// The row blocks (launch_cull_count's number against launch_cull's), and whether the units leave out
// enough: most of their pairs are counted, which makes them slower than the pairs of whole tiles.  Measured
// (flat 2D, 3D, sphere; N = 16384 to 262144; reaches of 0.5 to 35 % of the domain):
//   wide blocks pay up to 1.5 (fixed-point cells) or 2.0 (binary64 cells) times the units of narrow ones
//   share of all pairs at which units and whole tiles take as long: 1D 0.75; joint, narrow blocks, 0.4 .. 0.55
//   (fixed point) and 0.25 .. 0.4 (binary64 cells), in space 0.8; wide blocks 0.63 .. 0.8 (fixed point), and
//   for binary64 cells from 0.37 at 1.17 times the narrow units over 0.45 (1.35) to 0.7 (2.0)
// Joint du_L, flat 2D, N = 200000, 40 x 64 bins, binary64 cells, ms, narrow / wide / whole tiles: reach 10 %
// 6.7 / 5.2 / 19.4, 20 % 22.5 / 14.8 / 19.6, 35 % 54.7 / 34.2 / 20.5; fixed point, 25 %: 15.5 / 11.5 / 18.4.
void cull_decide(const sf_problem &p, bool J, bool fx, const double *info, CullInfo &ci) {
  double most = !J ? 0.75 : (p.W == 3 ? 0.75 : (fx ? 0.5 : 0.33));
  if (ci.rstep > 1) {
    uint64_t units;
    memcpy(&units, &info[11], sizeof units);
    const double times = (double)units / (double)std::max<int64_t>(ci.units, 1);
    if (times <= (fx ? 1.5 : 2.0)) {
      ci.units = (int64_t)std::min<uint64_t>(units, 1ull << 31);
      most = fx ? 0.65 : 0.35 + 0.42 * (times - 1.15);
    } else {
      ci.rstep = 1;
    }
  }
  if ((double)ci.units * 4096.0 > most * (double)pairs_of(p.N) || ci.units > (1 << 30)) ci.active = false;
}

// Stride of the binary32 record order: record k holds point (k * mul) mod N.  Points that the
// caller stores next to each other (a drifter track, a grid row) tend to fall in the same
// (distance, value) cell against a common column point, so a wave whose 64 rows are neighbours
// sends most of its LDS atomics to one or two cells and they serialize.  A stride near N times
// the golden ratio conjugate (a Kronecker sequence) hands each wave rows spread over the whole
// slice.  The pair set and the cells are unchanged; only the order of the additions differs.
int64_t interleave_mul(int64_t N) {
  if (N < 128) return 0;
  int64_t m = (int64_t)((double)N * 0.6180339887498949);
  auto gcd = [](int64_t a, int64_t b) {
    while (b) {
      const int64_t t = a % b;
      a = b;
      b = t;
    }
    return a;
  };
  while (gcd(m, N) != 1) ++m;
  return m;
}

// Fused outputs: the 1D operators a fused plan evaluates besides its main operator.
struct MultiSpec {
  int n1d = 0;
  int op[kMaxFused] = {}, nl[kMaxFused] = {}, nt[kMaxFused] = {};
};

// a plan buffer: allocated, or (allocation-free entry) taken from the plan's arena
#define PLBUF(buf, n)                                                                             \
  do {                                                                                            \
    const hipError_t e_ = pl.arena ? (buf).take((size_t)(n), *pl.arena) : (buf).ensure((size_t)(n)); \
    if (e_ == hipErrorOutOfMemory && pl.arena)                                                    \
      return ctx->fail(SF_E_UNSUPPORTED,                                                          \
                       "this call needs more device scratch than the allocation-free entry's %llu MiB " \
                       "(at %s); use sf_hist_batch_device", (unsigned long long)(SF_NOALLOC_SCRATCH_BYTES >> 20), #buf); \
    if (e_ != hipSuccess) return ctx->fail(SF_E_DEVICE, "%s: %s", #buf, hipGetErrorString(e_));   \
  } while (0)

// Host work and uploads for one batch.  x/u of each slice are device pointers.
int plan_build(sf_ctx *ctx, Plan &pl, int n_in, const sf_problem *sl_in, const double *const *dx_in,
               const double *const *du_in, const double *xmax_in, hipStream_t st, bool cull,
               const MultiSpec *multi = nullptr, bool wide = false) {
  // the single pass's 2D form runs every input slice as six plane slices (one joint histogram per
  // invariant, its own value edges); plane t of input slice s writes output cells t, t + 6, ...
  const bool planes = sp2d(sl_in[0].op, sl_in[0].n_val);
  std::vector<sf_problem> ex_sl;
  std::vector<const double *> ex_x, ex_u;
  std::vector<double> ex_m;
  int n = n_in;
  const sf_problem *sl = sl_in;
  const double *const *dx = dx_in;
  const double *const *du = du_in;
  const double *xmax = xmax_in;
  if (planes) {
    for (int s = 0; s < n_in; ++s) {
      for (int t = 0; t < kSpRows; ++t) {
        sf_problem q = sl_in[s];
        q.val_edges = sl_in[s].val_edges + (size_t)t * (sl_in[s].n_val + 1);
        ex_sl.push_back(q);
        ex_x.push_back(dx_in[s]);
        ex_u.push_back(du_in[s]);
        ex_m.push_back(xmax_in[s]);
      }
    }
    n = kSpRows * n_in;
    sl = ex_sl.data();
    dx = ex_x.data();
    du = ex_u.data();
    xmax = ex_m.data();
  }
  const sf_problem &p0 = sl[0];
  pl.ctx = ctx;
  pl.n = n;
  pl.nout = n_in;
  const bool flat = p0.geometry == SF_GEOM_FLAT;
  pl.G = flat ? kFlat : kSphere;
  pl.D = p0.D;
  pl.geom_code = p0.geometry;
  pl.J = p0.n_val > 0;
  pl.mixed = p0.precision != SF_PREC_FP64;
  pl.ncell = out_cells(p0);  // per input slice
  pl.sp = p0.op == SF_OP_SINGLE_PASS && !planes;
  pl.n1d = multi ? multi->n1d : 0;
  // B-strip: slices that share positions (the auxiliary axes of one field: same x, N, edges) and
  // bin 1D histograms in binary32 evaluate each pair's geometry once for up to kStripMax fields.
  // Opt-in (tuning variant 3): the per-slice 1D kernel with 16 histogram copies outruns it (eight
  // sphere fields, N = 65536: 828 against 609 Gpairs/s), its column velocities being LDS reads.
  pl.strip = 0;
  if (ctx->tune.variant == 3 && p0.precision != SF_PREC_FP64 && p0.n_val == 0 &&
      p0.op != SF_OP_SINGLE_PASS && n_in >= 2) {
    bool same = true;
    for (int s = 1; s < n && same; ++s)
      same = sl[s].x == p0.x && sl[s].N == p0.N && xmax[s] == xmax[0] &&
             memcmp(sl[s].dist_edges, p0.dist_edges, sizeof(double) * (p0.n_dist + 1)) == 0 &&
             (sl[s].dist_rule == nullptr) == (p0.dist_rule == nullptr) &&
             (!p0.dist_rule || memcmp(sl[s].dist_rule, p0.dist_rule, sizeof(sf_bin_rule)) == 0);
    if (same) pl.strip = kStripMax;
  }
  const int strip = pl.strip;
  pl.S64 = rec_d64(pl.G, pl.D);
  pl.F32 = rec_f32(pl.G, pl.D);
  const int G = pl.G, D = pl.D, ncell = pl.ncell, S64 = pl.S64, F32 = pl.F32;
  const bool J = pl.J, mixed = pl.mixed;

  // ---- records
  pl.total_pts = 0;
  pl.max_n = 0;
  pl.total_pairs = 0;
  std::vector<PrepSliceHost> prep(n);
  for (int s = 0; s < n; ++s) {
    prep[s].x = dx[s];
    prep[s].u = du[s];
    prep[s].N = sl[s].N;
    prep[s].pt_off = pl.total_pts;
    prep[s].perm = nullptr;
    // (the binary64 kernel's spherical records: joint histograms only, whose atomics the order
    // spreads; 1D ones keep their lane-group copies and adjacent rows, see tile_row)
    prep[s].mul = (mixed || (G == kSphere && J)) ? interleave_mul(sl[s].N) : 0;
    pl.total_pts += sl[s].N;
    pl.max_n = std::max<int64_t>(pl.max_n, sl[s].N);
    pl.total_pairs += pairs_of(sl[s].N);
  }
  PLBUF(pl.rec64, ((size_t)pl.total_pts * S64 + 16));
  // + one record (F32 <= 16): the binary32 pair loop requests the record after its last column
  // (sphere: the binary64 difference form's records, kF64Rec doubles per point, share the buffer)
  static_assert(kF64Rec * 2 == rec_f32(kSphere, 2) && kF64Rec * 2 == rec_f32(kSphere, 3), "record sizes");
  const bool rec_f = pl.rec_f = G == kSphere && fast64(J, hist_opk_of(p0));
  if (mixed || (rec_f && !pl.arena)) PLBUF(pl.rec32, ((size_t)pl.total_pts * F32 + 16));

  // ---- spatial sort and culling (binary32 kernel, one-shot calls): started here, so that the device
  // works on it while the tables are built
  std::vector<CullInfo> cinfo(n);
  std::vector<int64_t> grp(n);  // first group box of each slice
  bool cull_tried = false;
  if (cull && mixed && !strip) {
    int64_t groups = 0;
    for (int s = 0; s < n; ++s) {
      grp[s] = groups;
      groups += (sl[s].N + kGroup - 1) / kGroup;
    }
    // the record order of slice s lands at pl.perm + pt_off (used only where culling is active)
    PLBUF(pl.perm, ((size_t)pl.total_pts));
    PLBUF(pl.gboxes, ((size_t)groups * 6));
    HIPCHK(ctx->cull_info.ensure((size_t)n * kCullInfo));
    for (int s = 0; s < n; ++s) {
      const int rc = cull_start(ctx, sl[s], dx[s], xmax[s], J ? 768 : 256, st, cinfo[s], pl.perm.p + prep[s].pt_off,
                                ctx->cull_info.p + (size_t)s * kCullInfo, pl.gboxes.p + (size_t)grp[s] * 6);
      if (rc) return rc;
      cull_tried = cull_tried || cinfo[s].tried;
    }
  }

  // ---- tables
  std::vector<Slice> sdesc(n);
  std::vector<Cell> cells;
  std::vector<double> dedges, vedges;
  std::vector<float> vedges32;
  int ncell_max = 1;
  double crowd = 0.0;
  SliceTables T;
  for (int s = 0; s < n; ++s) {
    // (slices of one call mostly bin by the same edges: a table is built where they differ)
    if (s == 0 || !same_tables(sl[s - 1], xmax[s - 1], sl[s], xmax[s])) {
      T = SliceTables();
      build_tables(sl[s], xmax[s], T);
    }
    crowd = std::max(crowd, T.crowd);
    Slice d = T.desc;
    d.N = sl[s].N;
    d.pt_off = prep[s].pt_off;
    for (int k = 0; k < pl.n1d; ++k)  // (a fused output of another value than zero at rest)
      if (multi->op[k] == SF_OP_PROJECTED && multi->nl[k] == 0 && multi->nt[k] == 0) d.vzero = kNoZeroBin;
    d.out_off = planes ? (int64_t)(s / kSpRows) * ncell + s % kSpRows : (int64_t)s * ncell;
    d.plane = planes ? s % kSpRows : 0;
    d.xerr = flat ? round_up_f(ldexpl((long double)xmax[s], -28)) : 0.0f;
    d.strip_n = (strip && s % strip == 0) ? std::min(strip, n - s) : 0;
    d.tab_off = (int32_t)cells.size();
    cells.insert(cells.end(), T.tab64.begin(), T.tab64.end());
    d.tab32_off = (int32_t)cells.size();
    cells.insert(cells.end(), T.tab32.begin(), T.tab32.end());
    d.dedge_off = (int32_t)dedges.size();
    dedges.insert(dedges.end(), T.dedges.begin(), T.dedges.end());
    d.vedge_off = (int32_t)vedges.size();
    if (J) {
      for (int k = 0; k <= p0.n_val; ++k) {
        vedges.push_back(sl[s].val_edges[k]);
        vedges32.push_back((float)sl[s].val_edges[k]);
      }
    }
    // (the binary64 table is read by the batch-leading flat operators without a difference form only)
    ncell_max = std::max(ncell_max, flat && p0.semantics == SF_SEM_BATCH ? std::max(d.ncell64, d.ncell32) : d.ncell32);
    sdesc[s] = d;
  }
  if (vedges.empty()) { vedges.push_back(0.0); vedges32.push_back(0.0f); }
  pl.ncell_max = ncell_max;
  // fixed-point joint cells (binary32 kernel, one operator, value edges uniform in every slice)
  pl.fx = p0.precision == SF_PREC_MIXED_FIXED && J && !pl.sp;
  for (int s = 0; s < n && pl.fx; ++s) pl.fx = sdesc[s].v_uniform && sdesc[s].v_fx;

  // ---- launch geometry: one histogram per workgroup; small 1D histograms get 256-thread workgroups with
  // per-lane interleaved copies (several workgroups per CU)
  // launch shape: explicit tuning (sf_set_tuning) > autotuned entry for this key > defaults
  Params Pk{};
  Pk.op = p0.op;
  Pk.nl = p0.nl;
  Pk.nt = p0.nt;
  Pk.n_val = p0.n_val;
  Pk.nmom = pl.sp ? 4 : 1;
  Pk.n1d = pl.n1d;
  const int nmom = Pk.nmom;
  Tuning tn = ctx->tune;
  // the autotuner times one-operator launches; a fused launch (more LDS, more work per pair) keeps
  // the built-in shapes rather than a shape tuned for its main operator alone
  if (!tn.any() && pl.n1d == 0) {
    int64_t in_pairs = 0;
    for (int s = 0; s < n_in; ++s) in_pairs += pairs_of(sl_in[s].N);
    const auto it = ctx->tuned.find(tune_key(sl_in[0], in_pairs));
    if (it != ctx->tuned.end()) tn = it->second;
  }
  const int t_block = tn.block, t_jchunk = tn.j_chunk, t_bpc = tn.bpc, t_variant = tn.variant;
  // joint histograms: chosen below, when the LDS they need is known
  // 1D single pass: 512 threads (its 36-byte slots fill the LDS at two or three workgroups per CU;
  // more waves per workgroup then pay: flat 2D 595 against 492 Gpairs/s, sphere 644 against 529).
  // One-operator 1D kernels keep 256: 512 gained 5 % on flat 2D at N = 262144, nothing at 65536,
  // and lost on small slices (N = 4096: 51 against 88; the 256 ragged slices: 1019 against 1031)
  // Fused 1D outputs without a joint one: 512 threads (their histograms, 16 copies each, fill the
  // LDS at two or three workgroups per CU, like the single pass's)
  int block = t_block ? t_block : (J || pl.sp || pl.n1d) ? 512 : 256;
  // column records staged per LDS chunk; the fixed-point joint launch keeps two workgroups per CU
  const int tj = std::min(block, (pl.fx || strip) ? 128 : 256);
  // column records: variant 1 stages them through LDS, variant 2 reads them with scalar loads
  // (binary32 kernel only); 0 picks the default, scalar loads: joint histograms measured 212 vs
  // 204 Gpairs/s at N = 65536 (they also keep the record out of VGPRs, which the two-workgroup
  // fixed-point launch needs); 1D histograms with 16 copies, N = 262144, sphere 974 vs 908 and
  // flat 2D 1158 vs 958 (no LDS stage: more workgroups per CU)
  const bool sload = mixed && !strip && t_variant != 1;
  // a B-strip stages every field's column records; the binary64 kernel stages none (scalar loads)
  const int stage_bytes = (sload || !mixed) ? 0 : tj * F32 * 4 * (strip ? strip : 1);
  int copies = 1;
  if (!J) {
    // per-lane-group copies of a 1D histogram (lanes l and l + copies share one): 16 measured
    // best on both binary32 1D kernels (flat 2D du_L^2 at N = 65536: 636 / 643 / 840 / 708 / 597
    // Gpairs/s for 64 / 32 / 16 / 8 / 4 copies; sphere at N = 262144: 601 / 605 / 890 / 732 / 610).
    // A fused launch without a joint output does not use this histogram (its outputs have their
    // own): one copy.
    copies = pl.n1d ? 1 : (tn.copies ? tn.copies : 16);
    while (copies > 1 &&
           (size_t)smem_layout(p0.n_dist, 0, ncell_max, stage_bytes, copies, nmom, 0, 0, strip).total * 2 > ctx->max_smem)
      copies >>= 1;
  } else if (mixed && tn.copies == 2) {
    copies = 2;  // joint histogram privatised by lane halves (binary32 kernel only)
  }
  const int jlayout = (J && tn.layout) ? tn.layout : 1;
  // fused 1D outputs: 16 lane-group copies of their histograms (lanes l, l + 16, l + 32, l + 48
  // share one), fewer only if the LDS cannot hold them.  Their binary64 LDS atomics bound the
  // fused kernel (one per output and pair): beside the sphere's 64 x 96 joint histogram, 4, 8, 16
  // and 32 copies measured 199, 176, 169 and 169 ms for four 1D outputs at N = 262144
  int mcop = 0;
  if (pl.n1d) {
    mcop = 16;
    while (mcop > 1 && (size_t)smem_layout(p0.n_dist, p0.n_val, ncell_max, stage_bytes, copies, nmom, pl.fx, 0,
                                           strip, jlayout, pl.n1d, mcop).total > ctx->max_smem)
      mcop >>= 1;
  }
  pl.mcopies = mcop;
  const SmemLayout L0 = smem_layout(p0.n_dist, p0.n_val, ncell_max, stage_bytes, copies, nmom, pl.fx, 0, strip,
                                    jlayout, pl.n1d, mcop);
  // the binary64 kernel keeps one copy of a joint histogram, and queues the pairs it evaluates by
  // the reference's sequence: kRareQueue entries per wave, fewer (or none: such pairs are then
  // evaluated as they come) where the LDS does not hold them
  // (it reads its column records with scalar loads: no LDS stage)
  auto rare_queue = [&](int blk) {
    int q = kRareQueue * (blk / 64);
    while (q > 0 && (size_t)smem_layout(p0.n_dist, p0.n_val, ncell_max, 0, J ? 1 : copies, nmom, 0, q, 0,
                                        jlayout).total > ctx->max_smem)
      q = q > blk / 64 ? q / 2 : 0;
    return q;
  };
  const SmemLayout L64 = smem_layout(p0.n_dist, p0.n_val, ncell_max, 0, J ? 1 : copies, nmom, 0, 0, 0,
                                     jlayout);
  if ((size_t)std::max(L0.total, L64.total) > ctx->max_smem)
    return ctx->fail(SF_E_UNSUPPORTED,
                     "histogram of %d cells needs %d bytes of LDS; the device allows %zu per workgroup",
                     ncell, std::max(L0.total, L64.total), ctx->max_smem);
  auto occupancy = [&](int blk, size_t bytes) {
    const int nb = strip ? strip_occupancy(G, D, hist_opk(Pk, G, mixed), blk, bytes)
                         : hist_occupancy(G, D, J, mixed, hist_opk(Pk, G, mixed), sload, pl.fx, blk, bytes);
    // LDS is handed out in units of 1280 bytes, which the runtime's figure leaves out (max_smem is a
    // CU's: 128 of them): a re-bin queue sized to the last byte had cost a workgroup per CU (flat 3D
    // du_L^2, 100 bins, N = 98304, 512 threads: 4.94 ms, now 4.24)
    const size_t unit = ctx->max_smem / 128;
    return std::min(nb, (int)(128 / std::max<size_t>(1, (bytes + unit - 1) / unit)));
  };
  // binary32 kernel: LDS bytes with a re-bin queue of q entries; and the entries that the queue needs
  // where table cells hold several edges: room for four groups of 32 columns' worth of their pairs, of
  // few such pairs for twelve.  A group that does not fit goes to the global queue by itself, and the
  // waves of the device wait for one counter.  Linear axes up to pi on the sphere, N = 98304: 100 bins
  // (3.9 % of the pairs) 34.4 -> 13.6 ms, 50 bins (0.8 %) 10.0 -> 7.3; twelve groups of 3.9 % cost 16.9.
  auto bytes32 = [&](int q) {
    return (size_t)smem_layout(p0.n_dist, p0.n_val, ncell_max, stage_bytes, copies, nmom, pl.fx, q, strip, jlayout,
                               pl.n1d, mcop).total;
  };
  // Third-order operators: their values crowd at zero (a cube's density grows as v^(-2/3)), and where the
  // axis has an edge there, up to 5 % of the pairs are uncertain on the sphere (cubes; du_L^2 du_T 2.5 %)
  // and 2.4 % on flat fields.  Every reservation in the global queue takes its counter 12 ns, so that a wave
  // needs room for three groups of 32 columns: 160 entries where they cost no threads per CU, for cubes
  // on the sphere 300 at any price.  Kernel ms with room for 32 / now, sphere, N = 40000: du_T^3, 64 x 64 bins,
  // binary32 4.81 (two workgroups of 512) / 2.19 (one of 1024); fixed point, 48 x 64 bins, du_T^3 4.87 / 1.87,
  // du_L^2 du_T 4.83 / 1.73.  Flat 2D du_L^3, binary32, 64 x 64: 2.22 / 1.80; with one workgroup of 1024
  // in place of two of 768 it would be 2.26 for 1.70 (fixed point).
  bool third = false;
  if (J && ((p0.op == SF_OP_PROJECTED && p0.nl + p0.nt == 3) || p0.op == SF_OP_S3 || p0.op == SF_OP_L1T2COMP))
    for (int s = 0; s < n && !third; ++s)
      for (int k = 0; k <= p0.n_val && !third; ++k)
        third = std::fabs(sl[s].val_edges[k]) * p0.n_val < 0.0625 * (sl[s].val_edges[p0.n_val] - sl[s].val_edges[0]);
  const bool cubes = third && G == kSphere && p0.op == SF_OP_PROJECTED && (p0.nl == 3 || p0.nt == 3);
  double room = cubes ? 300.0 : (third ? 160.0 : 32.0);
  auto queue_need = [&](int blk) {
    if (!mixed) return 0;
    // (32 entries a wave at least: a size that leaves no room for a queue beside one workgroup more per CU
    // had every queued pair wait for the global counter, fixed point, 48 x 80 bins 2.25 -> 4.27 ms)
    const double each = crowd > 0.001 ? 2048.0 * crowd : 0.0;
    const double wave = std::max(room, std::max(4.0 * each, std::min(12.0 * each, 160.0)));
    int q = 64;
    while (q < wave * (blk / 64) && q < kQueueCap) q = third ? q + 64 : 2 * q;
    while (q > 0 && bytes32(q) > ctx->max_smem) q = q > 64 ? q / 128 * 64 : 0;
    if (third || each == 0.0 || q == 0) return q;
    // Fewer where these cost more threads than their reservations: a pair takes about 0.6 + 10 / w ps
    // with w waves on each CU (joint twice that), and a reservation for G groups 12 ns / 2048 G.  A
    // group as large as all that is left for the queue gains nothing by it.  Four groups' room at any
    // price (one workgroup per CU) / now: flat 3D, linear, 150 bins, N = 60000, 2.3 % of the pairs, 8.1 / 4.8 ms;
    // sphere, 200 bins, 51 %, done again in binary64 with the same shape, 51.2 / 34.4 ms.
    int best = 0;
    double least = 1e300;
    int most = 0;
    for (int r = 32 * (blk / 64); r <= q; r *= 2) {
      const int w = occupancy(blk, bytes32(r)) * (blk / 64);
      most = std::max(most, w);
      if (2 * w < most || w == 0) break;
      // (flat: the crowded keys are the largest ones, which few pairs have; 5 % at most)
      const double groups = std::max(1.0, floor(r / (blk / 64) / (G == kFlat ? std::min(each, 102.4) : each)));
      const double t = std::max((J ? 2.0 : 1.0) * (0.6 + 10.0 / w), 6.0 / groups);
      if (t < least) {
        least = t;
        best = r;
      }
    }
    return best > 0 ? best : q;
  };
  auto resident = [&](int blk) {  // workgroups of blk threads per CU
    return std::max(1, occupancy(blk, mixed ? bytes32(queue_need(blk))
                                            : (size_t)smem_layout(p0.n_dist, p0.n_val, ncell_max, 0, copies, nmom, 0,
                                                                  rare_queue(blk), 0, jlayout).total));
  };
  if (!t_block && J) {
    // joint histograms: the workgroup that leaves most waves on a CU, the smallest of those (more of
    // them end and begin at different times, and share fewer slots).  Three of 512 threads against two of
    // 768, fixed point, N = 98304, flat 2D: 4.71 / 4.93 ms at 40 x 64 bins, 4.91 / 5.06 at 20 x 32; two of
    // 512 against one of 1024, sphere, N = 65536, 40 x 64 bins: binary64 3.64 / 4.04, binary32 3.10 /
    // 3.34; fused, 40 x 48: 10.1 / 10.6.  64 x 96 bins keep two of 768 (fixed point) and one of 1024.
    auto most_threads = [&] {
      int most = 0;
      for (const int blk : {512, 768, 1024}) {
        const int threads = resident(blk) * blk;
        if (threads > most) {
          most = threads;
          block = blk;
        }
      }
      return most;
    };
    const int threads = most_threads();
    if (third && !cubes) {
      room = 32.0;
      if (most_threads() <= threads) {
        room = 160.0;
        (void)most_threads();
      }
    }
  }
  const int qcap64 = rare_queue(block);
  pl.qcap64 = qcap64;
  int bpc = resident(block);
  if (!J && !strip && pl.n1d == 0 && !tn.copies && copies == 16 && pl.total_pairs >= 100000000) {
    // 32 copies where they cost no workgroup per CU: two lanes of a wave share one, not four, and a
    // half wave's atomics never meet (N = 98304, 20 bins: flat 2D du_L^2 3.53 -> 3.29 ms, 3D 4.02 -> 3.94,
    // sphere 4.57 -> 4.47; 64 bins, where five fit instead of six: 3.32 -> 3.44); in calls of a few
    // hundred microseconds clearing and summing them costs as much (N = 4096: 144 us, 148 with 32)
    const size_t need64 = (size_t)smem_layout(p0.n_dist, 0, ncell_max, 0, 32, nmom, 0, qcap64).total;
    const size_t need = mixed ? (size_t)smem_layout(p0.n_dist, 0, ncell_max, stage_bytes, 32, nmom, 0,
                                                        queue_need(block)).total : need64;
    if (std::max(need, need64) <= ctx->max_smem && occupancy(block, need) >= bpc) copies = 32;
  }
  // binary32 kernel: the LDS re-bin queue, as large as fits without costing a workgroup per CU more
  // (0: every queued pair takes the global queue's atomic)
  int qcap = 0;
  if (mixed) {
    for (int q = kQueueCap; q >= 64 && qcap == 0; q >>= 1)
      if (bytes32(q) <= ctx->max_smem && occupancy(block, bytes32(q)) >= bpc) qcap = q;
    qcap = std::max(qcap, queue_need(block));
  }
  if (t_bpc) bpc = std::min(bpc, t_bpc);
  const int max_blocks = bpc * ctx->n_cu;

  // ---- work items: (slice, i-tile, j-chunk); slices in descending N
  int jchunk = t_jchunk;
  if (jchunk <= 0) {
    // Large calls: 16 items per resident workgroup, in whole tiles.  Smaller ones: an item's fixed
    // cost against the workgroups that it leaves idle at the end, which is least at a width that goes
    // with the root of the call's (row tile, column) count.  Measured, against one tile at least: host
    // du_L^2 at N = 777 107 / 153 us (binary64; 10 items then; sphere 122 / 195), N = 4096 157 / 200;
    // joint du_L at N = 16384 binary64 385 / 550.
    // The planes of a 2D single pass: their pairs that share a cell serialize, so an item's time varies
    // most, and narrow items pay at every size (sphere, N = 12000: 2.03 ms at 128 columns, 2.4 at 256,
    // 6.9 at 1024; N = 3000: 0.50 ms, 0.56 at 32 columns).
    const double cols = (double)pl.total_pairs / block;  // columns of all row tiles
    const double large = std::min(std::max(cols / (16.0 * max_blocks), (double)block), 64.0 * block);
    const double small = sp2d(p0.op, p0.n_val) ? std::max(128.0, cols / (64.0 * max_blocks))
                                               : std::max(16.0, sqrt(cols) / 3.0);
    // (wide: as few items as there can be, where the allocation-free entry's scratch is short)
    const int jc = wide ? 64 * block : (int)std::min(large, small);
    const int unit = jc >= block ? block : 16;
    jchunk = (jc + unit - 1) / unit * unit;
  }
  // fixed-point cells: one item must stay below the flush limit (the LDS histogram is flushed
  // between items only)
  if (pl.fx) jchunk = std::max(1, std::min<int>(jchunk, (int)(kFxFlushLimit / block)));
  // culling, second part (scalar-loaded columns only): which slices, and their work units
  pl.culled = false;
  pl.n_units = 0;
  if (cull_tried && sload) {
    const size_t bytes = sizeof(double) * kCullInfo * (size_t)n;
    const bool pinned = bytes <= kStageMax;
    std::vector<double> own(pinned ? 0 : (size_t)n * kCullInfo);
    if (pinned) HIPCHK(ctx->down.acquire(bytes));
    double *info = pinned ? (double *)ctx->down.p : own.data();
    auto read = [&]() -> int {
      HIPCHK(hipMemcpyAsync(info, ctx->cull_info.p, bytes, hipMemcpyDeviceToHost, st));
      HIPCHK(hipStreamSynchronize(st));
      return SF_OK;
    };
    int rc = read();
    if (rc) return rc;
    bool again = false;
    for (int s = 0; s < n; ++s) {
      cull_rows(sl[s], J, info + (size_t)s * kCullInfo, block, cinfo[s]);
      if (!cinfo[s].active || cinfo[s].rstep == 1) continue;
      HIPCHK(launch_cull_count(pl.gboxes.p + (size_t)grp[s] * 6, sl[s].N, ctx->cull_info.p + (size_t)s * kCullInfo,
                               cinfo[s].reach, cinfo[s].rstep, st));
      again = true;
    }
    if (again && (rc = read())) return rc;
    int64_t units = 0;
    for (int s = 0; s < n; ++s) {
      if (cinfo[s].active) cull_decide(sl[s], J, pl.fx, info + (size_t)s * kCullInfo, cinfo[s]);
      if (units + cinfo[s].units > (1LL << 30)) cinfo[s].active = false;
      if (!cinfo[s].active) continue;
      units += cinfo[s].units;
      prep[s].perm = pl.perm.p + prep[s].pt_off;
      pl.culled = true;
    }
    pl.n_units = (int)units;
    if (units > 0) {
      PLBUF(pl.units, (size_t)units);
      units = 0;
      for (int s = 0; s < n; ++s) {
        if (!cinfo[s].active || cinfo[s].units == 0) continue;
        HIPCHK(launch_cull_units(pl.gboxes.p + (size_t)grp[s] * 6, sl[s].N, ctx->cull_info.p + (size_t)s * kCullInfo,
                                 cinfo[s].reach, cinfo[s].rstep, s, pl.units.p + units, cinfo[s].units, st));
        units += cinfo[s].units;
      }
    }
    const int waves = block / 64;
    pl.near_grid = std::max(1, std::min(max_blocks, (pl.n_units + waves - 1) / waves));
  }
  std::vector<int> order(n);
  for (int s = 0; s < n; ++s) order[s] = s;
  std::stable_sort(order.begin(), order.end(), [&](int a, int b) { return sl[a].N > sl[b].N; });
  std::vector<Item> items, items64;
  for (int s : order) {
    if (cinfo[s].active) continue;  // its work units are listed on the device
    const int64_t N = sl[s].N;
    const int64_t jc = jchunk;
    const size_t first = items.size();
    for (int64_t i0 = 0; i0 < N - 1; i0 += block) {
      for (int64_t j0 = i0; j0 < N; j0 += jc) {
        Item it;
        it.slice = s;
        it.i0 = (int32_t)i0;
        it.j0 = (int32_t)j0;
        it.j1 = (int32_t)std::min<int64_t>(N, j0 + jc);
        // a B-strip's items belong to its leading slice
        if (!strip || s % strip == 0) items.push_back(it);
        if (strip) items64.push_back(it);
      }
    }
    // full items of the slice first (a diagonal item costs its full rectangle): the short last
    // column range of every row tile and the short last row tile end the queue, so workgroups
    // finish together (a linear-time partition; a one-shot call builds its items every time)
    const int64_t rows = block;
    std::stable_partition(items.begin() + first, items.end(), [N, rows, jc](const Item &a) {
      return N - a.i0 >= rows && a.j1 - a.j0 == jc;
    });
  }
  if (pl.fx) {
    // every item must fit the fixed-point cells' exact range (checked, not assumed)
    for (const Item &it : items)
      if ((int64_t)block * (int64_t)(it.j1 - it.j0) > kFxFlushLimit)
        return ctx->fail(SF_E_DEVICE, "internal: work item of %d x %d pair updates exceeds the fixed-point flush limit",
                         block, it.j1 - it.j0);
  }
  pl.n_items = (int)items.size();  // (none: every slice is culled)
  if (items.empty()) items.push_back(Item{0, 0, 0, 0});
  if (strip && items64.empty()) items64.push_back(Item{0, 0, 0, 0});
  pl.n_items64 = (int)items64.size();
  pl.grid = std::max(1, std::min(pl.n_items, max_blocks));
  pl.block = block;
  pl.jchunk = jchunk;
  pl.tj = tj;
  pl.copies = copies;
  pl.sload = sload;

  // ---- upload: every table in one copy
  struct Part {
    const void *src;
    size_t bytes, off;
  };
  Part parts[] = {{sdesc.data(), sizeof(Slice) * n, 0},
                  {items.data(), sizeof(Item) * items.size(), 0},
                  {cells.data(), sizeof(Cell) * cells.size(), 0},
                  {dedges.data(), sizeof(double) * dedges.size(), 0},
                  {vedges.data(), sizeof(double) * vedges.size(), 0},
                  {vedges32.data(), sizeof(float) * vedges32.size(), 0},
                  {prep.data(), sizeof(PrepSliceHost) * n, 0},
                  {items64.data(), sizeof(Item) * items64.size(), 0}};
  size_t total = 0;
  for (Part &q : parts) {
    q.off = total;
    total = (total + q.bytes + 255) & ~(size_t)255;
  }
  const size_t acells = (size_t)pl.nout * ncell;
  pl.acc_bytes = 16 * acells + 4 * sizeof(unsigned long long) + 8 * sizeof(int);
  if (pl.arena) {
    // Calls that the allocation-free entry took when slices' descriptions were smaller and row tiles
    // larger (at most a sixteenth of the scratch together) run in parts where they do not fit; and so
    // do spherical binary64 ones whose second records (64 bytes a point) do not fit beside the rest.
    const size_t need = ((pl.arena->used + 255) & ~(size_t)255) + total + ((pl.acc_bytes + 255) & ~(size_t)255) +
                        (mixed ? 1024 * sizeof(Pending) : 0);
    const size_t more = !mixed && rec_f ? ((size_t)pl.total_pts * F32 + 16) * sizeof(float) : 0;
    pl.arena->split = need + more > pl.arena->cap && need <= pl.arena->cap + pl.arena->cap / 16;
  }
  PLBUF(pl.tables, total);
  PLBUF(pl.acc, pl.acc_bytes);
  if (!mixed && rec_f && pl.arena) PLBUF(pl.rec32, ((size_t)pl.total_pts * F32 + 16));
  {
    // from page-locked memory, without waiting for it (the allocation-free entry keeps none)
    const bool pinned = !pl.arena && total <= kStageMax;
    std::vector<char> own(pinned ? 0 : total);
    if (pinned) HIPCHK(ctx->up_tab.acquire(total));
    char *h = pinned ? ctx->up_tab.p : own.data();
    for (const Part &q : parts)
      if (q.bytes) memcpy(h + q.off, q.src, q.bytes);
    if (pinned) {
      HIPCHK(ctx->up_tab.send(pl.tables.p, total, st));
    } else {
      HIPCHK(hipMemcpyAsync(pl.tables.p, h, total, hipMemcpyHostToDevice, st));
      HIPCHK(hipStreamSynchronize(st));
    }
  }
  char *tb = pl.tables.p;
  pl.prep = (const PrepSliceHost *)(tb + parts[6].off);
  pl.items64 = (const Item *)(tb + parts[7].off);
  pl.acc_s = (double *)pl.acc.p;
  pl.acc_c = (unsigned long long *)(pl.acc_s + acells);
  pl.pcount = pl.acc_c + acells;
  pl.counter = (int *)(pl.pcount + 4);
  pl.flag = pl.counter + 4;
  if (pl.n1d) {
    PLBUF(pl.msums, ((size_t)pl.n1d * pl.nout * p0.n_dist));
    PLBUF(pl.mcounts, ((size_t)pl.n1d * pl.nout * p0.n_dist));
  }

  pl.cap = 0;
  if (mixed) {
    pl.cap = std::max<int64_t>(1LL << 22, pl.total_pairs / 2000);
    pl.cap = std::min<int64_t>(pl.cap, 1LL << 27);
    pl.cap = std::max<int64_t>(pl.cap, std::min<int64_t>(ctx->queue_hint, kQueueMax));
    if (pl.arena) {
      // the re-bin queue gets the rest of the scratch (an overflow is redone in binary64)
      const size_t off = (pl.arena->used + 255) & ~(size_t)255;
      const int64_t room = off < pl.arena->cap ? (int64_t)((pl.arena->cap - off) / sizeof(Pending)) : 0;
      pl.cap = std::min<int64_t>(pl.cap, room);
      if (pl.cap < 1024)
        return ctx->fail(SF_E_UNSUPPORTED,
                         "this call leaves no room for the re-bin queue in the allocation-free entry's "
                         "%llu MiB scratch; use sf_hist_batch_device", (unsigned long long)(SF_NOALLOC_SCRATCH_BYTES >> 20));
    }
    PLBUF(pl.pending, ((size_t)pl.cap));
  }

  Params &P = pl.P;
  P = Params{};
  P.slices = (const Slice *)(tb + parts[0].off);
  P.items = (const Item *)(tb + parts[1].off);
  P.n_items = pl.n_items;
  P.block_rows = block;
  P.counter = pl.counter;
  P.rec64 = pl.rec64.p;
  P.rec32 = pl.rec32.p;
  P.cells = (const Cell *)(tb + parts[2].off);
  P.dedges = (const double *)(tb + parts[3].off);
  P.vedges = (const double *)(tb + parts[4].off);
  P.vedges32 = (const float *)(tb + parts[5].off);
  P.sums = pl.acc_s;
  P.counts = pl.acc_c;
  P.pending = pl.pending.p;
  P.pending_count = pl.pcount;
  P.pending_cap = pl.cap;
  P.stats = nullptr;
  P.ncell_max = ncell_max;
  P.tj = tj;
  P.copies = copies;
  P.jlayout = jlayout;
  P.stage_bytes = stage_bytes;
  P.n_dist = p0.n_dist;
  P.n_val = p0.n_val;
  P.op = p0.op;
  P.nl = p0.nl;
  P.nt = p0.nt;
  P.order = op_order(p0);
  P.radius = (p0.geometry == SF_GEOM_SPHERE_DEG) ? p0.radius : 1.0;
  // |dv| <= vcoef * (|u_i| + |u_j|)^order * amp  (flat amp = 1; sphere amp = 1 + c^2 / sin(sigma))
  P.vcoef = (float)ldexp(16.0 * std::max(1, P.order), -24);
  P.nmom = nmom;
  P.fx = pl.fx ? 1 : 0;
  P.qcap = qcap;
  P.qw = qcap / (block / 64);
  P.bl = (flat && p0.semantics == SF_SEM_BATCH) ? 1 : 0;
  P.strip = strip;
  P.n1d = pl.n1d;
  P.mcopies = mcop;
  P.n_slices = pl.nout;
  P.mab_a = P.mab_b = 0;
  for (int k = 0; k < pl.n1d; ++k) {
    P.mop[k] = multi->op[k];
    P.mnl[k] = multi->nl[k];
    P.mnt[k] = multi->nt[k];
    int a = 0, b = 0;
    if (!fused_basis_index(multi->op[k], multi->nl[k], multi->nt[k], &a, &b))
      return ctx->fail(SF_E_DEVICE, "internal: fused output %d is not a basis product", k);
    P.mab_a |= (uint32_t)a << (4 * k);
    P.mab_b |= (uint32_t)b << (4 * k);
  }  // unused outputs: fields 0, 1 * 1
  P.ja = P.jb = 0;
  if (pl.n1d && J && !fused_basis_index(p0.op, p0.nl, p0.nt, &P.ja, &P.jb))
    return ctx->fail(SF_E_DEVICE, "internal: the fused joint operator is not a basis product");
  P.msums = pl.n1d ? pl.msums.p : nullptr;
  P.mcounts = pl.n1d ? pl.mcounts.p : nullptr;
  P.flush_limit = pl.fx ? kFxFlushLimit : 0x7fffffffLL;
  return SF_OK;
}

// Kernel-only launch sequence: records from the current x/u, zeroed accumulators, histogram,
// re-bin (mixed), merge into out (skipped, with *flag set, if the re-bin queue overflowed).
// ev (optional) brackets the histogram and re-bin kernels for timing.
int plan_launch(Plan &pl, bool use_mixed, double *out_s, unsigned long long *out_c, hipStream_t st,
                hipEvent_t *ev) {
  sf_ctx *ctx = pl.ctx;
  if (pl.total_pairs == 0) return SF_OK;
  const int64_t ncells = (int64_t)pl.nout * pl.ncell;
  const int64_t mcells = (int64_t)pl.n1d * pl.nout * pl.P.n_dist;
  if (pl.n1d && !use_mixed)  // fused outputs exist in the binary32 kernel only
    return ctx->fail(SF_E_UNSUPPORTED, "internal: fused outputs launched on the binary64 kernel");
  {
    // records; accumulators, queue count, work counter and overflow flag, and the fused ones cleared
    void *zp[kZeroSetMax] = {pl.acc.p};
    int64_t zb[kZeroSetMax] = {(int64_t)pl.acc_bytes};
    int nz = 1;
    if (pl.n1d) {
      zp[nz] = pl.msums.p;
      zb[nz++] = (int64_t)sizeof(double) * mcells;
      zp[nz] = pl.mcounts.p;
      zb[nz++] = (int64_t)sizeof(unsigned long long) * mcells;
    }
    HIPCHK(launch_prep(pl.G, pl.D, use_mixed, pl.geom_code, pl.prep, pl.n, pl.max_n, pl.rec64.p,
                       use_mixed || pl.rec_f ? pl.rec32.p : nullptr, nz, zp, zb, st));
  }
  const bool use_sload = use_mixed && pl.sload;
  const int stage = (use_sload || !use_mixed) ? 0 : pl.tj * pl.F32 * 4;
  Params P = pl.P;
  P.stage_bytes = stage;
  if (!use_mixed) {  // the binary64 kernel keeps binary64 sums and 32-bit counts, no queue
    P.fx = 0;
    if (P.n_val > 0) P.copies = 1;
    P.qcap = pl.qcap64;
    P.qw = pl.qcap64 / (pl.block / 64);
    P.flush_limit = 0x7fffffffLL;
    if (pl.strip) {  // one slice at a time
      P.strip = 0;
      P.items = pl.items64;
      P.n_items = pl.n_items64;
    }
  }
  const int stage_mixed = stage * ((use_mixed && pl.strip) ? pl.strip : 1);
  P.stage_bytes = stage_mixed;
  const SmemLayout L = smem_layout(P.n_dist, P.n_val, P.ncell_max, stage_mixed, P.copies, P.nmom, P.fx, P.qcap,
                                   P.strip, P.jlayout, P.n1d, P.mcopies);
  if (ev) HIPCHK(hipEventRecord(ev[0], st));
  if (P.n_items > 0)
    HIPCHK(launch_hist(pl.G, pl.D, pl.J, use_mixed, use_sload, false, P, pl.grid, pl.block, (size_t)L.total, st));
  if (use_mixed && pl.n_units > 0) {  // culled slices: their work units instead of items
    Params Pu = P;
    Pu.items = pl.units.p;
    Pu.n_items = pl.n_units;
    HIPCHK(launch_hist(pl.G, pl.D, pl.J, true, true, true, Pu, pl.near_grid, pl.block, (size_t)L.total, st));
  }
  if (ev) HIPCHK(hipEventRecord(ev[1], st));
  // four 256-thread workgroups per CU: the re-bin is a latency-bound gather (2D single pass,
  // 2.7e8 queued pairs: 22.6 / 16.7 / 19.6 ms with one / four / eight per CU)
  if (use_mixed) HIPCHK(launch_recheck(pl.G, pl.D, pl.J, P, 4 * ctx->n_cu, st));
  if (ev) HIPCHK(hipEventRecord(ev[2], st));
  // (a fused call without a joint output passes no out_s / out_c, a host call reads acc)
  if (out_s)
    HIPCHK(launch_merge_checked(pl.acc_s, pl.acc_c, out_s, out_c, ncells,
                                use_mixed ? pl.pcount : nullptr, pl.cap, pl.flag, st));
  const int64_t per = (int64_t)pl.nout * pl.P.n_dist;
  for (int k = 0; k < pl.n1d; ++k)
    HIPCHK(launch_merge_checked(pl.msums.p + k * per, pl.mcounts.p + k * per, pl.mdst_s[k], pl.mdst_c[k], per,
                                pl.pcount, pl.cap, pl.flag, st));
  if (pl.sp && out_s) HIPCHK(launch_derive_sp(out_s, out_c, (int64_t)pl.nout * pl.P.n_dist, st));
  if (ev) HIPCHK(hipEventRecord(ev[3], st));
  return SF_OK;
}

// work items of a plan's launch; culled slices: the number of items that their units' pairs would fill
int64_t work_items(const Plan &pl) {
  const int64_t item = (int64_t)pl.block * pl.jchunk;
  return pl.n_items + ((int64_t)pl.n_units * 4096 + item - 1) / item;
}

// One-shot: build (into the context's cached plan, reusing its buffers), launch, and on a
// re-bin queue overflow redo the call with the binary64 kernel.  h_acc (host calls; out_s and out_c
// are null then): receives the accumulators (sums, then counts) instead of a merge, read with the
// queue's count in one copy.
int run_batch(sf_ctx *ctx, int n, const sf_problem *sl, const double *const *dx,
              const double *const *du, const double *xmax, double *out_s,
              unsigned long long *out_c, hipStream_t st, std::vector<char> *h_acc = nullptr) {
  Plan &pl = ctx->oneshot;
  int rc = plan_build(ctx, pl, n, sl, dx, du, xmax, st, true);
  if (rc) return rc;
  for (int k = 0; k < 8; ++k) ctx->stats[k] = 0;
  ctx->stats[0] = pl.total_pairs;
  ctx->stats[2] = work_items(pl);
  ctx->stats[3] = std::max(pl.n_items > 0 ? pl.grid : 0, pl.n_units > 0 ? pl.near_grid : 0);
  ctx->stats[7] = pl.block;
  ctx->ev_pending = false;
  if (pl.total_pairs == 0) return SF_OK;
  for (int k = 0; k < 4; ++k)
    if (!ctx->ev[k]) HIPCHK(hipEventCreate(&ctx->ev[k]));
  rc = plan_launch(pl, pl.mixed, out_s, out_c, st, ctx->ev);
  if (rc) return rc;
  unsigned long long pc = 0;
  const size_t acells = 16 * (size_t)pl.nout * pl.ncell;  // bytes of sums and counts
  auto fetch = [&]() -> int {
    const size_t from = h_acc ? 0 : acells, bytes = acells + sizeof(pc) - from;
    const bool pinned = bytes <= kStageMax;
    if (pinned) HIPCHK(ctx->down.acquire(bytes));
    if (h_acc) h_acc->resize(bytes);
    char *h = pinned ? ctx->down.p : h_acc->data();
    HIPCHK(hipMemcpyAsync(h, pl.acc.p + from, bytes, hipMemcpyDeviceToHost, st));
    HIPCHK(hipStreamSynchronize(st));
    if (h_acc && pinned) memcpy(h_acc->data(), h, bytes);
    memcpy(&pc, h + (acells - from), sizeof(pc));
    return SF_OK;
  };
  if (pl.mixed || h_acc) {
    rc = fetch();
    if (rc) return rc;
  }
  if (pl.mixed) {
    ctx->stats[1] = (int64_t)pc;
    if ((int64_t)pc > pl.cap && (int64_t)pc <= kQueueMax) {
      // the merge was skipped: the queue now knows its size, so grow it and run the binary32
      // kernel once more (and remember the size for later calls of this context)
      ctx->queue_hint = std::max<int64_t>(ctx->queue_hint, std::min<int64_t>((int64_t)pc + pc / 4, kQueueMax));
      pl.cap = ctx->queue_hint;
      HIPCHK(pl.pending.ensure((size_t)pl.cap));
      pl.P.pending = pl.pending.p;
      pl.P.pending_cap = pl.cap;
      rc = plan_launch(pl, true, out_s, out_c, st, ctx->ev);
      if (rc) return rc;
      rc = fetch();
      if (rc) return rc;
      ctx->stats[1] = (int64_t)pc;
    }
    if ((int64_t)pc > pl.cap) {
      // the merge was skipped; redo everything with the binary64 kernel (which evaluates every
      // pair in the caller's order: rebuild the work items without culling first)
      if (pl.culled) {
        rc = plan_build(ctx, pl, n, sl, dx, du, xmax, st, false);
        if (rc) return rc;
      }
      rc = plan_launch(pl, false, out_s, out_c, st, ctx->ev);
      if (rc) return rc;
      if (h_acc && (rc = fetch())) return rc;
    }
  }
  ctx->ev_pending = true;
  return SF_OK;
}

// Coordinate magnitudes max|x| (times scale) of a batch of device slices, for the binary32 kernels'
// margins; zero where no binary32 kernel on flat points needs them.  Partial maxima are reduced on the
// device (a read-back of x cost 0.25 ms of a 2.3 ms call at N = 65536, 2D) into d_part: at least
// kMaxParts doubles a slice, or null for a buffer of the context's.
int coord_max(sf_ctx *ctx, int n, const sf_problem *sl, hipStream_t st, double scale, std::vector<double> &xmax,
              double *d_part = nullptr) {
  xmax.assign((size_t)n, 0.0);
  if (sl[0].precision == SF_PREC_FP64 || sl[0].geometry != SF_GEOM_FLAT) return SF_OK;
  std::vector<const double *> x;
  std::vector<int64_t> len;
  for (int s = 0; s < n; ++s)
    if (sl[s].N > 0) {
      x.push_back(sl[s].x);
      len.push_back((int64_t)sl[s].W * sl[s].N);
    }
  if (x.empty()) return SF_OK;
  const size_t np = x.size() * kMaxParts;
  const bool pinned = !d_part && sizeof(double) * np <= kStageMax;
  if (!d_part) {
    HIPCHK(ctx->d_max.ensure(np));
    d_part = ctx->d_max.p;
  }
  std::vector<double> own(pinned ? 0 : np);
  if (pinned) HIPCHK(ctx->down.acquire(sizeof(double) * np));
  double *h = pinned ? (double *)ctx->down.p : own.data();
  HIPCHK(launch_absmax((int)x.size(), x.data(), len.data(), d_part, st));
  HIPCHK(hipMemcpyAsync(h, d_part, sizeof(double) * np, hipMemcpyDeviceToHost, st));
  HIPCHK(hipStreamSynchronize(st));
  size_t k = 0;
  for (int s = 0; s < n; ++s)
    if (sl[s].N > 0) {
      xmax[s] = scale * abs_max(h + k, kMaxParts);
      k += kMaxParts;
    }
  return SF_OK;
}

// whether host slice s has the positions of the slice before it (auxiliary axes share them)
bool shares_x(const sf_problem *sl, int s) {
  return s > 0 && sl[s].x == sl[s - 1].x && sl[s].N == sl[s - 1].N && sl[s].W == sl[s - 1].W;
}

// Host slices' x and u to the device (ctx->d_x, ctx->d_u): small ones together through page-locked
// memory, shared positions once.
int send_inputs(sf_ctx *ctx, int n, const sf_problem *sl, hipStream_t st, std::vector<const double *> &px,
                std::vector<const double *> &pu) {
  int64_t tx = 0, tu = 0;
  for (int s = 0; s < n; ++s) {
    tx += shares_x(sl, s) ? 0 : (int64_t)sl[s].W * sl[s].N;
    tu += (int64_t)sl[s].D * sl[s].N;
  }
  const bool pinned = sizeof(double) * (size_t)(tx + tu) <= kStageMax;
  if (pinned) {
    HIPCHK(ctx->d_x.ensure((size_t)(tx + tu) + 2));
    HIPCHK(ctx->up_xu.acquire(sizeof(double) * (size_t)(tx + tu)));
  } else {
    HIPCHK(ctx->d_x.ensure((size_t)tx + 2));
    HIPCHK(ctx->d_u.ensure((size_t)tu + 2));
  }
  double *h = (double *)ctx->up_xu.p;
  int64_t ox = 0, ou = 0;
  for (int s = 0; s < n; ++s) {
    const bool same = shares_x(sl, s);
    const int64_t nx = same ? 0 : (int64_t)sl[s].W * sl[s].N, nu = (int64_t)sl[s].D * sl[s].N;
    px[s] = same ? px[s - 1] : ctx->d_x.p + ox;
    pu[s] = pinned ? ctx->d_x.p + tx + ou : ctx->d_u.p + ou;
    if (pinned) {
      if (nx) memcpy(h + ox, sl[s].x, sizeof(double) * nx);
      if (nu) memcpy(h + tx + ou, sl[s].u, sizeof(double) * nu);
    } else {
      if (nx) HIPCHK(hipMemcpyAsync(ctx->d_x.p + ox, sl[s].x, sizeof(double) * nx, hipMemcpyHostToDevice, st));
      if (nu) HIPCHK(hipMemcpyAsync(ctx->d_u.p + ou, sl[s].u, sizeof(double) * nu, hipMemcpyHostToDevice, st));
    }
    ox += nx;
    ou += nu;
  }
  if (pinned && tx + tu > 0) HIPCHK(ctx->up_xu.send(ctx->d_x.p, sizeof(double) * (size_t)(tx + tu), st));
  return SF_OK;
}

int host_entry(sf_ctx *ctx, int n, const sf_problem *sl, double *sums, uint64_t *counts) {
  ctx->err.clear();
  int rc = validate_batch(ctx, n, sl, true);
  if (rc) return rc;
  if (n == 0) return SF_OK;
  if (!sums || !counts) return ctx->fail(SF_E_ARG, "null sums or counts");
  HIPCHK(hipSetDevice(ctx->device));
  hipStream_t st = ctx->stream;
  const sf_problem &p0 = sl[0];
  const int ncell = out_cells(p0);
  std::vector<const double *> px(n), pu(n);
  std::vector<double> xmax(n, 0.0);
  rc = send_inputs(ctx, n, sl, st, px, pu);
  if (rc) return rc;
  for (int s = 0; s < n; ++s) xmax[s] = shares_x(sl, s) ? xmax[s - 1] : abs_max(sl[s].x, (int64_t)sl[s].W * sl[s].N);
  std::vector<char> acc;
  rc = run_batch(ctx, n, sl, px.data(), pu.data(), xmax.data(), nullptr, nullptr, st, &acc);
  if (rc) return rc;
  const size_t cells = (size_t)n * ncell;
  if (acc.empty()) acc.assign(16 * cells, 0);  // no pairs: nothing was launched
  const double *hs = (const double *)acc.data();
  const uint64_t *hc = (const uint64_t *)(hs + cells);
  for (size_t k = 0; k < cells; ++k) {
    sums[k] += hs[k];
    counts[k] += hc[k];
  }
  if (p0.op == SF_OP_SINGLE_PASS && p0.n_val == 0) derive_sp_host(sums, counts, (int64_t)n * p0.n_dist);
  return SF_OK;
}

}  // namespace

extern "C" int sf_hist(sf_ctx *ctx, const sf_problem *p, double *sums, uint64_t *counts) {
  if (!ctx) return SF_E_ARG;
  return host_entry(ctx, 1, p, sums, counts);
}

extern "C" int sf_hist_batch(sf_ctx *ctx, int32_t n_slices, const sf_problem *slices, double *sums,
                             uint64_t *counts) {
  if (!ctx) return SF_E_ARG;
  return host_entry(ctx, n_slices, slices, sums, counts);
}

extern "C" int sf_hist_batch_device(sf_ctx *ctx, int32_t n, const sf_problem *sl, double *d_sums,
                                    uint64_t *d_counts, void *stream) {
  if (!ctx) return SF_E_ARG;
  ctx->err.clear();
  int rc = validate_batch(ctx, n, sl, false);
  if (rc) return rc;
  if (n == 0) return SF_OK;
  if (!d_sums || !d_counts) return ctx->fail(SF_E_ARG, "null sums or counts");
  HIPCHK(hipSetDevice(ctx->device));
  hipStream_t st = stream ? (hipStream_t)stream : ctx->stream;
  std::vector<const double *> px(n), pu(n);
  std::vector<double> xmax;
  for (int s = 0; s < n; ++s) {
    px[s] = sl[s].x;
    pu[s] = sl[s].u;
  }
  rc = coord_max(ctx, n, sl, st, 1.0, xmax);
  if (rc) return rc;
  return run_batch(ctx, n, sl, px.data(), pu.data(), xmax.data(), d_sums,
                   (unsigned long long *)d_counts, st);
}

extern "C" int sf_hist_device(sf_ctx *ctx, const sf_problem *p, double *d_sums, uint64_t *d_counts,
                              void *stream) {
  return sf_hist_batch_device(ctx, 1, p, d_sums, d_counts, stream);
}

// ----------------------------------------------------------------------------------------------
// fused outputs: one pair evaluation, several operators
// ----------------------------------------------------------------------------------------------
// What a fused call does with its outputs: each output's own problems (validated as its own call
// would be), the joint output fused into the launch (-1: none), the fused 1D outputs in launch
// order, and the outputs that run as their own calls (binary64 precision: all of them; else those
// whose binary32 value is not a product of two basis values, FullVector{1} and {3}).
struct FusedSetup {
  std::vector<std::vector<sf_problem>> per;
  int joint = -1;
  std::vector<int> ids;
  std::vector<int> separate;
  MultiSpec ms;
  const std::vector<sf_problem> &main() const { return per[joint >= 0 ? joint : ids[0]]; }
  bool launch() const { return joint >= 0 || !ids.empty(); }
};

int fused_setup(sf_ctx *ctx, int32_t n, const sf_problem *sl, int32_t n_out, const sf_output *outs,
                FusedSetup &fs) {
  if (n_out < 1 || !outs) return ctx->fail(SF_E_ARG, "a fused call needs at least one output");
  int joint = -1, n1 = 0;
  for (int k = 0; k < n_out; ++k) {
    if (outs[k].op == SF_OP_SINGLE_PASS)
      return ctx->fail(SF_E_ARG, "output %d: the single pass is not a fused output (it is its own fused form)", k);
    if (outs[k].n_val > 0) {
      if (joint >= 0) return ctx->fail(SF_E_UNSUPPORTED, "a fused call takes at most one joint output");
      joint = k;
    } else {
      ++n1;
    }
  }
  if (n1 > SF_MAX_FUSED) return ctx->fail(SF_E_UNSUPPORTED, "a fused call takes at most %d 1D outputs", SF_MAX_FUSED);
  fs.per.assign((size_t)n_out, {});
  for (int k = 0; k < n_out; ++k) {
    fs.per[k].assign(sl, sl + std::max(n, 0));
    for (sf_problem &q : fs.per[k]) {
      q.op = outs[k].op;
      q.nl = outs[k].nl;
      q.nt = outs[k].nt;
      q.n_val = outs[k].n_val;
      if (outs[k].n_val == 0 || outs[k].val_edges) {  // else each slice's own value edges
        q.val_edges = outs[k].val_edges;
        q.val_rule = outs[k].val_rule;
      }
    }
    const int rc = validate_batch(ctx, n, fs.per[k].data(), false);
    if (rc) return rc;
  }
  fs.joint = -1;
  fs.ids.clear();
  fs.separate.clear();
  fs.ms = MultiSpec();
  if (n > 0 && sl[0].precision == SF_PREC_FP64) {
    for (int k = 0; k < n_out; ++k) fs.separate.push_back(k);
    return SF_OK;
  }
  int a = 0, b = 0;
  if (joint >= 0) {
    if (fused_basis_index(outs[joint].op, outs[joint].nl, outs[joint].nt, &a, &b)) fs.joint = joint;
    else fs.separate.push_back(joint);
  }
  for (int k = 0; k < n_out; ++k) {
    if (k == joint) continue;
    if (!fused_basis_index(outs[k].op, outs[k].nl, outs[k].nt, &a, &b)) {
      fs.separate.push_back(k);
      continue;
    }
    fs.ms.op[fs.ms.n1d] = outs[k].op;
    fs.ms.nl[fs.ms.n1d] = outs[k].nl;
    fs.ms.nt[fs.ms.n1d] = outs[k].nt;
    ++fs.ms.n1d;
    fs.ids.push_back(k);
  }
  return SF_OK;
}

extern "C" int sf_hist_multi_device(sf_ctx *ctx, int32_t n, const sf_problem *sl, int32_t n_out,
                                    const sf_output *outs, double *const *d_sums, uint64_t *const *d_counts,
                                    void *stream) {
  if (!ctx) return SF_E_ARG;
  ctx->err.clear();
  if (n_out < 1 || !outs || !d_sums || !d_counts) return ctx->fail(SF_E_ARG, "a fused call needs at least one output");
  for (int k = 0; k < n_out; ++k)
    if (!d_sums[k] || !d_counts[k]) return ctx->fail(SF_E_ARG, "output %d: null sums or counts", k);
  FusedSetup fs;
  int rc = fused_setup(ctx, n, sl, n_out, outs, fs);
  if (rc) return rc;
  if (n == 0) return SF_OK;
  HIPCHK(hipSetDevice(ctx->device));
  hipStream_t st = stream ? (hipStream_t)stream : ctx->stream;
  for (int k : fs.separate) {
    rc = sf_hist_batch_device(ctx, n, fs.per[k].data(), d_sums[k], d_counts[k], st);
    if (rc) return rc;
  }
  if (!fs.launch()) return SF_OK;
  const std::vector<int> &separate = fs.separate;
  const std::vector<std::vector<sf_problem>> &per = fs.per;
  const int joint = fs.joint;
  Plan &pl = ctx->fused;
  for (size_t j = 0; j < fs.ids.size(); ++j) {
    pl.mdst_s[j] = d_sums[fs.ids[j]];
    pl.mdst_c[j] = (unsigned long long *)d_counts[fs.ids[j]];
  }
  // the plan's main problem: the joint output's (its value bins), or the first 1D output's,
  // whose own histogram then stays unused
  const std::vector<sf_problem> &main = fs.main();
  std::vector<const double *> px(n), pu(n);
  std::vector<double> xmax;
  for (int s = 0; s < n; ++s) {
    px[s] = sl[s].x;
    pu[s] = sl[s].u;
  }
  rc = coord_max(ctx, n, sl, st, 1.0, xmax);
  if (rc) return rc;
  rc = plan_build(ctx, pl, n, main.data(), px.data(), pu.data(), xmax.data(), st, true, &fs.ms);
  if (rc) return rc;
  for (int k = 0; k < 8; ++k) ctx->stats[k] = 0;
  ctx->stats[0] = pl.total_pairs;
  ctx->stats[2] = work_items(pl);
  ctx->stats[3] = std::max(pl.n_items > 0 ? pl.grid : 0, pl.n_units > 0 ? pl.near_grid : 0);
  ctx->stats[7] = pl.block;
  ctx->ev_pending = false;
  if (pl.total_pairs == 0) return SF_OK;
  for (int k = 0; k < 4; ++k)
    if (!ctx->ev[k]) HIPCHK(hipEventCreate(&ctx->ev[k]));
  double *js = joint >= 0 ? d_sums[joint] : nullptr;
  unsigned long long *jc = joint >= 0 ? (unsigned long long *)d_counts[joint] : nullptr;
  unsigned long long pc = 0;
  for (int attempt = 0; attempt < 2; ++attempt) {
    rc = plan_launch(pl, true, js, jc, st, ctx->ev);
    if (rc) return rc;
    HIPCHK(hipMemcpyAsync(&pc, pl.pcount, sizeof(pc), hipMemcpyDeviceToHost, st));
    HIPCHK(hipStreamSynchronize(st));
    ctx->stats[1] = (int64_t)pc;
    if ((int64_t)pc <= pl.cap || (int64_t)pc > kQueueMax) break;
    // the merges were skipped: grow the re-bin queue to the size reached and run again
    ctx->queue_hint = std::max<int64_t>(ctx->queue_hint, std::min<int64_t>((int64_t)pc + pc / 4, kQueueMax));
    pl.cap = ctx->queue_hint;
    HIPCHK(pl.pending.ensure((size_t)pl.cap));
    pl.P.pending = pl.pending.p;
    pl.P.pending_cap = pl.cap;
  }
  ctx->ev_pending = true;
  if ((int64_t)pc > pl.cap) {
    // still too many pairs to re-bin: every fused output with the binary64 kernel, one after
    // the other (the separate outputs are done)
    for (int k = 0; k < n_out; ++k) {
      if (std::find(separate.begin(), separate.end(), k) != separate.end()) continue;
      std::vector<sf_problem> q = per[k];
      for (sf_problem &e : q) e.precision = SF_PREC_FP64;
      rc = sf_hist_batch_device(ctx, n, q.data(), d_sums[k], d_counts[k], st);
      if (rc) return rc;
    }
  }
  return SF_OK;
}

// Host-pointer form: x, u and the outputs are host memory (staged like sf_hist_batch).
extern "C" int sf_hist_multi(sf_ctx *ctx, int32_t n, const sf_problem *sl, int32_t n_out, const sf_output *outs,
                             double *const *sums, uint64_t *const *counts) {
  if (!ctx) return SF_E_ARG;
  ctx->err.clear();
  if (n < 0 || (n > 0 && !sl)) return ctx->fail(SF_E_ARG, "bad slices");
  if (n_out < 1 || n_out > SF_MAX_FUSED + 1 || !outs || !sums || !counts)
    return ctx->fail(SF_E_ARG, "a fused call needs 1 to %d outputs", SF_MAX_FUSED + 1);
  {
    // the host arrays are checked here; each output's operator and bins by sf_hist_multi_device
    std::vector<sf_problem> chk(sl, sl + n);
    for (sf_problem &q : chk) {
      q.op = outs[0].op;
      q.nl = outs[0].nl;
      q.nt = outs[0].nt;
      q.n_val = outs[0].n_val;
      if (outs[0].n_val == 0 || outs[0].val_edges) {
        q.val_edges = outs[0].val_edges;
        q.val_rule = outs[0].val_rule;
      }
    }
    const int rc = validate_batch(ctx, n, chk.data(), true);
    if (rc) return rc;
  }
  if (n == 0) return SF_OK;
  HIPCHK(hipSetDevice(ctx->device));
  hipStream_t st = ctx->stream;
  std::vector<const double *> px(n), pu(n);
  int rc = send_inputs(ctx, n, sl, st, px, pu);
  if (rc) return rc;
  std::vector<sf_problem> dev(sl, sl + n);
  for (int s = 0; s < n; ++s) {
    dev[s].x = px[s];
    dev[s].u = pu[s];
  }
  // outputs: every output's sums, then every output's counts, in one kept buffer
  std::vector<int64_t> cells((size_t)n_out);
  size_t total = 0;
  for (int k = 0; k < n_out; ++k) {
    cells[k] = (int64_t)n * sl[0].n_dist * (outs[k].n_val > 0 ? outs[k].n_val : 1);
    total += (size_t)cells[k];
  }
  const size_t bytes = 16 * total;
  HIPCHK(ctx->d_out.ensure(bytes));
  std::vector<double *> ds((size_t)n_out);
  std::vector<uint64_t *> dc((size_t)n_out);
  size_t off = 0;
  for (int k = 0; k < n_out; ++k) {
    ds[k] = (double *)ctx->d_out.p + off;
    dc[k] = (uint64_t *)ctx->d_out.p + total + off;
    off += (size_t)cells[k];
  }
  HIPCHK(launch_zero(ctx->d_out.p, (int64_t)bytes, st));
  rc = sf_hist_multi_device(ctx, n, dev.data(), n_out, outs, ds.data(), dc.data(), st);
  if (rc) return rc;
  const bool pinned = bytes <= kStageMax;
  std::vector<char> own(pinned ? 0 : bytes);
  if (pinned) HIPCHK(ctx->down.acquire(bytes));
  char *h = pinned ? ctx->down.p : own.data();
  HIPCHK(hipMemcpyAsync(h, ctx->d_out.p, bytes, hipMemcpyDeviceToHost, st));
  HIPCHK(hipStreamSynchronize(st));
  const double *hs = (const double *)h;
  const uint64_t *hc = (const uint64_t *)h + total;
  off = 0;
  for (int k = 0; k < n_out; ++k) {
    for (int64_t c = 0; c < cells[k]; ++c) {
      sums[k][c] += hs[off + c];
      counts[k][c] += hc[off + c];
    }
    off += (size_t)cells[k];
  }
  return SF_OK;
}

// ----------------------------------------------------------------------------------------------
// allocation-free entry: every device buffer of the call comes from one static array per device
// ----------------------------------------------------------------------------------------------
extern "C" int sf_hist_batch_device_noalloc(sf_ctx *ctx, int32_t n, const sf_problem *sl, double *d_sums,
                                            uint64_t *d_counts, void *stream) {
  if (!ctx) return SF_E_ARG;
  ctx->err.clear();
  int rc = validate_batch(ctx, n, sl, false);
  if (rc) return rc;
  if (n == 0) return SF_OK;
  if (!d_sums || !d_counts) return ctx->fail(SF_E_ARG, "null sums or counts");
  if (!ctx->scratch_ptr) return ctx->fail(SF_E_DEVICE, "the scratch array has no address on this device");
  // the records alone must fit in half of it (checked before any device work; the tables, items,
  // accumulators, the queue and the binary64 difference form's own records as the plan takes them)
  int64_t pts = 0;
  for (int s = 0; s < n; ++s) pts += sl[s].N;
  const int G = sl[0].geometry == SF_GEOM_FLAT ? kFlat : kSphere;
  const int64_t rec_bytes = pts * (8 * rec_d64(G, sl[0].D) + (sl[0].precision != SF_PREC_FP64 ? 4 * rec_f32(G, sl[0].D) : 0));
  if (rec_bytes > (int64_t)(SF_NOALLOC_SCRATCH_BYTES / 2))
    return ctx->fail(SF_E_UNSUPPORTED,
                     "%lld points need %lld bytes of records, more than half of the allocation-free entry's "
                     "%llu MiB scratch; use sf_hist_batch_device", (long long)pts, (long long)rec_bytes,
                     (unsigned long long)(SF_NOALLOC_SCRATCH_BYTES >> 20));
  HIPCHK(hipSetDevice(ctx->device));
  hipStream_t st = stream ? (hipStream_t)stream : ctx->stream;
  std::vector<const double *> px(n), pu(n);
  std::vector<double> xmax;
  for (int s = 0; s < n; ++s) {
    px[s] = sl[s].x;
    pu[s] = sl[s].u;
  }
  // the partial maxima take the head of the scratch before the plan does (they are read back here;
  // their bytes are fewer than those of the slices' descriptions)
  static_assert(sizeof(double) * kMaxParts <= sizeof(Slice), "partial maxima of a slice");
  if (sizeof(Slice) * (size_t)n > SF_NOALLOC_SCRATCH_BYTES)
    return ctx->fail(SF_E_UNSUPPORTED,
                     "%d slices need more device scratch than the allocation-free entry's %llu MiB; use "
                     "sf_hist_batch_device", n, (unsigned long long)(SF_NOALLOC_SCRATCH_BYTES >> 20));
  rc = coord_max(ctx, n, sl, st, 1.0, xmax, (double *)ctx->scratch_ptr);
  if (rc) return rc;
  for (int k = 0; k < 8; ++k) ctx->stats[k] = 0;
  ctx->ev_pending = false;
  // slices a .. b - 1 in one launch; where they do not fit, in halves, one after the other on the stream
  const int ncell = out_cells(sl[0]);
  auto run = [&](auto &&self, int a, int b, bool wide) -> int {
    Plan &pl = ctx->noalloc;
    Arena arena{ctx->scratch_ptr, (size_t)SF_NOALLOC_SCRATCH_BYTES, 0};
    pl.arena = &arena;
    // no culling: its sort workspace would be another buffer
    int rc = plan_build(ctx, pl, b - a, sl + a, px.data() + a, pu.data() + a, xmax.data() + a, st, false, nullptr, wide);
    pl.arena = nullptr;
    if (rc == SF_E_UNSUPPORTED && arena.split) {
      if (b - a == 1) return wide ? rc : self(self, a, b, true);
      const int m = a + (b - a) / 2;
      rc = self(self, a, m, false);
      return rc ? rc : self(self, m, b, false);
    }
    if (rc) return rc;
    ctx->stats[0] += pl.total_pairs;
    ctx->stats[2] += work_items(pl);
    ctx->stats[3] = std::max<int64_t>(ctx->stats[3], pl.n_items > 0 ? pl.grid : 0);
    ctx->stats[7] = pl.block;
    if (pl.total_pairs == 0) return SF_OK;
    double *ds = d_sums + (size_t)a * ncell;
    unsigned long long *dc = (unsigned long long *)d_counts + (size_t)a * ncell;
    rc = plan_launch(pl, pl.mixed, ds, dc, st, nullptr);
    if (rc) return rc;
    if (pl.mixed) {
      unsigned long long pc = 0;
      HIPCHK(hipMemcpyAsync(&pc, pl.pcount, sizeof(pc), hipMemcpyDeviceToHost, st));
      HIPCHK(hipStreamSynchronize(st));
      ctx->stats[1] += (int64_t)pc;
      // the queue overflowed its share of the scratch: the merge was skipped, redo in binary64
      if ((int64_t)pc > pl.cap) rc = plan_launch(pl, false, ds, dc, st, nullptr);
    }
    return rc;
  };
  rc = run(run, 0, n, false);
  if (!rc) ctx->err.clear();
  return rc;
}

// ----------------------------------------------------------------------------------------------
// plans: build once, execute many times (optionally as a captured hipGraph)
// ----------------------------------------------------------------------------------------------
struct sf_plan {
  sf_ctx *ctx = nullptr;
  Plan pl;
  hipStream_t last_stream = nullptr;
  double *last_s = nullptr;
  unsigned long long *last_c = nullptr;
  // fused plan (sf_plan_create_multi): its outputs' problems and launch positions, and the last
  // execution's destinations (for the binary64 redo after a re-bin queue overflow)
  int n_out = 0;
  FusedSetup fs;
  std::vector<double *> last_ms;
  std::vector<unsigned long long *> last_mc;
};

// Waits for the upload that plan_build leaves running on st: a plan is executed on whatever stream the
// caller names (and is captured into a graph there), which nothing else orders after st.
static int plan_ready(sf_ctx *ctx, hipStream_t st) {
  HIPCHK(hipStreamSynchronize(st));
  return SF_OK;
}

extern "C" int sf_plan_create(sf_ctx *ctx, int32_t n, const sf_problem *sl, sf_plan **out) {
  if (!ctx || !out) return SF_E_ARG;
  *out = nullptr;
  ctx->err.clear();
  int rc = validate_batch(ctx, n, sl, false);
  if (rc) return rc;
  if (n == 0) return ctx->fail(SF_E_ARG, "a plan needs at least one slice");
  HIPCHK(hipSetDevice(ctx->device));
  hipStream_t st = ctx->stream;
  std::vector<const double *> px(n), pu(n);
  std::vector<double> xmax;
  for (int s = 0; s < n; ++s) {
    px[s] = sl[s].x;
    pu[s] = sl[s].u;
  }
  // coordinate magnitude for the binary32 margin; later contents must stay within 2x of it
  rc = coord_max(ctx, n, sl, st, 2.0, xmax);
  if (rc) return rc;
  sf_plan *plan = new sf_plan();
  plan->ctx = ctx;
  // no culling in plans: the positions behind x may change between executions
  rc = plan_build(ctx, plan->pl, n, sl, px.data(), pu.data(), xmax.data(), st, false);
  if (!rc) rc = plan_ready(ctx, st);
  if (rc) {
    plan->pl.release();
    delete plan;
    return rc;
  }
  *out = plan;
  return SF_OK;
}

extern "C" int sf_plan_execute(sf_plan *plan, double *d_sums, uint64_t *d_counts, void *stream,
                               int32_t use_graph) {
  if (!plan) return SF_E_ARG;
  sf_ctx *ctx = plan->ctx;
  if (plan->n_out) return ctx->fail(SF_E_ARG, "a fused plan: use sf_plan_execute_multi");
  if (!d_sums || !d_counts) return ctx->fail(SF_E_ARG, "null sums or counts");
  HIPCHK(hipSetDevice(ctx->device));
  hipStream_t st = stream ? (hipStream_t)stream : ctx->stream;
  Plan &pl = plan->pl;
  unsigned long long *dc = (unsigned long long *)d_counts;
  plan->last_stream = st;
  plan->last_s = d_sums;
  plan->last_c = dc;
  if (!use_graph) return plan_launch(pl, pl.mixed, d_sums, dc, st, nullptr);
  if (!pl.graph || pl.g_sums != d_sums || pl.g_counts != dc || pl.g_stream != st) {
    if (pl.graph) {
      HIPCHK(hipGraphExecDestroy(pl.graph));
      pl.graph = nullptr;
    }
    hipGraph_t g = nullptr;
    HIPCHK(hipStreamBeginCapture(st, hipStreamCaptureModeThreadLocal));
    const int rc = plan_launch(pl, pl.mixed, d_sums, dc, st, nullptr);
    const hipError_t e = hipStreamEndCapture(st, &g);
    if (rc) {
      if (g) (void)hipGraphDestroy(g);
      return rc;
    }
    if (e != hipSuccess) return ctx->fail(SF_E_DEVICE, "graph capture failed: %s", hipGetErrorString(e));
    const hipError_t e2 = hipGraphInstantiate(&pl.graph, g, nullptr, nullptr, 0);
    (void)hipGraphDestroy(g);
    if (e2 != hipSuccess) {
      pl.graph = nullptr;
      return ctx->fail(SF_E_DEVICE, "graph instantiation failed: %s", hipGetErrorString(e2));
    }
    pl.g_sums = d_sums;
    pl.g_counts = dc;
    pl.g_stream = st;
  }
  HIPCHK(hipGraphLaunch(pl.graph, st));
  return SF_OK;
}

extern "C" int sf_plan_create_multi(sf_ctx *ctx, int32_t n, const sf_problem *sl, int32_t n_out,
                                    const sf_output *outs, sf_plan **out) {
  if (!ctx || !out) return SF_E_ARG;
  *out = nullptr;
  ctx->err.clear();
  if (n <= 0) return ctx->fail(SF_E_ARG, "a plan needs at least one slice");
  sf_plan *plan = new sf_plan();
  plan->ctx = ctx;
  plan->n_out = n_out;
  int rc = fused_setup(ctx, n, sl, n_out, outs, plan->fs);
  if (!rc && !plan->fs.separate.empty())
    rc = ctx->fail(SF_E_UNSUPPORTED,
                   "a fused plan needs a binary32 precision and outputs that fuse (output %d does not: "
                   "binary64, or FullVector{1}/{3}); make one plan per output instead",
                   plan->fs.separate[0]);
  if (rc) {
    delete plan;
    return rc;
  }
  HIPCHK(hipSetDevice(ctx->device));
  hipStream_t st = ctx->stream;
  std::vector<const double *> px(n), pu(n);
  std::vector<double> xmax;
  for (int s = 0; s < n; ++s) {
    px[s] = sl[s].x;
    pu[s] = sl[s].u;
  }
  // later contents must stay within 2x of the coordinate magnitude read now
  rc = coord_max(ctx, n, sl, st, 2.0, xmax);
  // no culling in plans: the positions behind x may change between executions
  if (!rc) rc = plan_build(ctx, plan->pl, n, plan->fs.main().data(), px.data(), pu.data(), xmax.data(), st, false,
                           &plan->fs.ms);
  if (!rc) rc = plan_ready(ctx, st);
  if (rc) {
    plan->pl.release();
    delete plan;
    return rc;
  }
  *out = plan;
  return SF_OK;
}

extern "C" int sf_plan_execute_multi(sf_plan *plan, double *const *d_sums, uint64_t *const *d_counts, void *stream,
                                     int32_t use_graph) {
  if (!plan) return SF_E_ARG;
  sf_ctx *ctx = plan->ctx;
  if (plan->n_out == 0) return ctx->fail(SF_E_ARG, "not a fused plan (use sf_plan_execute)");
  if (!d_sums || !d_counts) return ctx->fail(SF_E_ARG, "null output arrays");
  for (int k = 0; k < plan->n_out; ++k)
    if (!d_sums[k] || !d_counts[k]) return ctx->fail(SF_E_ARG, "output %d: null sums or counts", k);
  HIPCHK(hipSetDevice(ctx->device));
  hipStream_t st = stream ? (hipStream_t)stream : ctx->stream;
  Plan &pl = plan->pl;
  const FusedSetup &fs = plan->fs;
  bool moved = false;
  for (size_t j = 0; j < fs.ids.size(); ++j) {
    moved |= pl.mdst_s[j] != d_sums[fs.ids[j]] || pl.mdst_c[j] != (unsigned long long *)d_counts[fs.ids[j]];
    pl.mdst_s[j] = d_sums[fs.ids[j]];
    pl.mdst_c[j] = (unsigned long long *)d_counts[fs.ids[j]];
  }
  double *js = fs.joint >= 0 ? d_sums[fs.joint] : nullptr;
  unsigned long long *jc = fs.joint >= 0 ? (unsigned long long *)d_counts[fs.joint] : nullptr;
  plan->last_stream = st;
  plan->last_ms.assign(d_sums, d_sums + plan->n_out);
  plan->last_mc.assign((unsigned long long *const *)d_counts, (unsigned long long *const *)d_counts + plan->n_out);
  if (!use_graph) return plan_launch(pl, true, js, jc, st, nullptr);
  if (!pl.graph || moved || pl.g_sums != js || pl.g_counts != jc || pl.g_stream != st) {
    if (pl.graph) {
      HIPCHK(hipGraphExecDestroy(pl.graph));
      pl.graph = nullptr;
    }
    hipGraph_t g = nullptr;
    HIPCHK(hipStreamBeginCapture(st, hipStreamCaptureModeThreadLocal));
    const int rc = plan_launch(pl, true, js, jc, st, nullptr);
    const hipError_t e = hipStreamEndCapture(st, &g);
    if (rc) {
      if (g) (void)hipGraphDestroy(g);
      return rc;
    }
    if (e != hipSuccess) return ctx->fail(SF_E_DEVICE, "graph capture failed: %s", hipGetErrorString(e));
    const hipError_t e2 = hipGraphInstantiate(&pl.graph, g, nullptr, nullptr, 0);
    (void)hipGraphDestroy(g);
    if (e2 != hipSuccess) {
      pl.graph = nullptr;
      return ctx->fail(SF_E_DEVICE, "graph instantiation failed: %s", hipGetErrorString(e2));
    }
    pl.g_sums = js;
    pl.g_counts = jc;
    pl.g_stream = st;
  }
  HIPCHK(hipGraphLaunch(pl.graph, st));
  return SF_OK;
}

extern "C" int sf_plan_sync(sf_plan *plan, int32_t *redone) {
  if (!plan) return SF_E_ARG;
  sf_ctx *ctx = plan->ctx;
  if (redone) *redone = 0;
  if (!plan->last_stream) return SF_OK;
  HIPCHK(hipSetDevice(ctx->device));
  Plan &pl = plan->pl;
  HIPCHK(hipStreamSynchronize(plan->last_stream));
  if (!pl.mixed || pl.total_pairs == 0) return SF_OK;
  int flag = 0;
  HIPCHK(hipMemcpy(&flag, pl.flag, sizeof(int), hipMemcpyDeviceToHost));
  if (flag && plan->n_out) {
    // a fused plan's last execute overflowed the re-bin queue and left every output untouched:
    // each output with the binary64 kernel
    for (int k = 0; k < plan->n_out; ++k) {
      std::vector<sf_problem> q = plan->fs.per[k];
      for (sf_problem &e : q) e.precision = SF_PREC_FP64;
      const int rc = sf_hist_batch_device(ctx, (int)q.size(), q.data(), plan->last_ms[k],
                                          (uint64_t *)plan->last_mc[k], plan->last_stream);
      if (rc) return rc;
    }
    HIPCHK(hipStreamSynchronize(plan->last_stream));
    if (redone) *redone = 1;
  } else if (flag) {
    // the last execute overflowed the re-bin queue and left the outputs untouched
    const int rc = plan_launch(pl, false, plan->last_s, plan->last_c, plan->last_stream, nullptr);
    if (rc) return rc;
    HIPCHK(hipStreamSynchronize(plan->last_stream));
    if (redone) *redone = 1;
  }
  return SF_OK;
}

extern "C" void sf_plan_destroy(sf_plan *plan) {
  if (!plan) return;
  (void)hipSetDevice(plan->ctx->device);
  if (plan->last_stream) (void)hipStreamSynchronize(plan->last_stream);
  plan->pl.release();
  delete plan;
}

// ----------------------------------------------------------------------------------------------
// autotuner
// ----------------------------------------------------------------------------------------------
extern "C" int sf_autotune(sf_ctx *ctx, int32_t n, const sf_problem *sl, int32_t out[6]) {
  if (!ctx) return SF_E_ARG;
  ctx->err.clear();
  int rc = validate_batch(ctx, n, sl, false);
  if (rc) return rc;
  if (n == 0) return ctx->fail(SF_E_ARG, "nothing to tune");
  HIPCHK(hipSetDevice(ctx->device));
  const sf_problem &p0 = sl[0];
  const bool J = p0.n_val > 0, mixed = p0.precision != SF_PREC_FP64;
  const bool fx = p0.precision == SF_PREC_MIXED_FIXED && J;
  const int ncell = out_cells(p0);
  DevBuf<double> ts;
  DevBuf<unsigned long long> tc;
  HIPCHK(ts.ensure((size_t)n * ncell));
  HIPCHK(tc.ensure((size_t)n * ncell));
  const Tuning saved = ctx->tune;
  std::vector<const double *> px(n), pu(n);
  std::vector<double> xmax(n, 0.0);
  for (int s = 0; s < n; ++s) {
    px[s] = sl[s].x;
    pu[s] = sl[s].u;
    xmax[s] = 1.0;  // timing only: margins do not change the work, results are discarded
  }
  // device time of one call with launch shape c (a warm-up call first)
  auto time_of = [&](const Tuning &c, double *t) {
    ctx->tune = c;
    for (int rep = 0; rep < 2; ++rep) {
      const int r = run_batch(ctx, n, sl, px.data(), pu.data(), xmax.data(), ts.p, tc.p, ctx->stream);
      if (r) return r;
      int64_t st[8];
      sf_last_stats(ctx, st);
      *t = (double)st[6];
    }
    return SF_OK;
  };
  // coordinate search: threads per workgroup x column variant, then the histogram's privatised
  // copies and (joint) slot layout, then the column-range length
  std::vector<Tuning> stage1;
  const int blocks[4] = {256, 512, 768, 1024};
  for (int b : blocks) {
    if (J && b < 512) continue;
    if (!J && b > 512) continue;
    if (J && b == 768 && !fx) continue;  // 768: the fixed-point cells' two-workgroup launch
    for (int v = (mixed ? 1 : 0); v <= (mixed ? 2 : 0); ++v) stage1.push_back(Tuning{b, 0, 0, v, 0, 0});
  }
  double best = 1e300;
  Tuning best_c = stage1.front();
  auto consider = [&](const Tuning &c) {
    double t = 0;
    const int r = time_of(c, &t);
    if (r == SF_E_UNSUPPORTED) return SF_OK;  // shape does not fit this device: skip it
    if (r) return r;
    if (t < best) {
      best = t;
      best_c = c;
    }
    return SF_OK;
  };
  for (const Tuning &c : stage1)
    if ((rc = consider(c))) break;
  if (!rc) {
    std::vector<Tuning> stage2;
    if (!J) {
      for (int cp : {4, 8, 32}) {
        Tuning c = best_c;
        c.copies = cp;
        stage2.push_back(c);
      }
    } else if (mixed) {
      for (int cp : {1, 2})
        for (int lay : {1, 2}) {
          if (cp == 1 && lay == 1) continue;  // the built-in choice, already timed
          Tuning c = best_c;
          c.copies = cp;
          c.layout = lay;
          stage2.push_back(c);
        }
    }
    for (const Tuning &c : stage2)
      if ((rc = consider(c))) break;
  }
  if (!rc) {
    const int b = best_c.block ? best_c.block : 256;
    for (int sc : {2, 8}) {
      Tuning c = best_c;
      c.j_chunk = sc * b;
      if ((rc = consider(c))) break;
    }
  }
  ctx->tune = saved;
  ts.release();
  tc.release();
  if (rc) return rc;
  int64_t total = 0;
  for (int s = 0; s < n; ++s) total += pairs_of(sl[s].N);
  ctx->tuned[tune_key(p0, total)] = best_c;
  if (out) {
    out[0] = best_c.block;
    out[1] = best_c.j_chunk;
    out[2] = best_c.bpc;
    out[3] = best_c.variant;
    out[4] = best_c.copies;
    out[5] = best_c.layout;
  }
  return SF_OK;
}
