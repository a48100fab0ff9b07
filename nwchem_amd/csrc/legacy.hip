// legacy.hip -- the reference's per-call GPU surface, MI355X-native.
//
// Drop-in for the functions of the same names in src/tce/ccsd_t/sd_t_total.cu
// (27 contraction entry points, compute_en_, dev_mem_s_/dev_mem_d_,
// dev_release_), memory.cu (initmemmodule_/finalizememmodule_ and the
// size-keyed device pool behind them) and hybrid.c (check_device_,
// device_init_).  The drivers ccsd_t_gpu.F / ccsd_t_singles_gpu.F /
// ccsd_t_doubles_gpu.F call these unchanged: operand blocks arrive as host
// arrays per call, results accumulate into library-owned device tiles, and
// compute_en_ reduces a task's tiles to {E[T], E(T)}.
//
// Differences in mechanism (not in results): one library stream instead of a
// stream created and destroyed per call; operands staged through a reusable
// pinned buffer; one contraction kernel, and one for small calls, parameterised
// by the strides of the family (d1, d2, s1) and variant instead of 25
// hand-expanded kernels; a two-pass deterministic energy reduction instead of
// one-thread blocks and a host-side sum.  Errors are recorded (tce_t_last_error)
// and reported on stderr rather than calling exit(1).
#include <hip/hip_runtime.h>
#include <rocblas/rocblas.h>

#include <algorithm>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <map>
#include <mutex>
#include <set>

#include "internal.h"

namespace tce_t {

static thread_local std::string g_err;
void set_error(const std::string &msg) { g_err = msg; }

namespace {

// ------------------------------------------------------------ device pool --
// memory.cu keeps freed blocks in per-size free lists until
// finalizememmodule; the same policy here (exact-size reuse).
struct Pool {
  std::map<size_t, std::set<void *>> free_list;
  std::map<void *, size_t> live;
  bool init = false;
  void *get(size_t bytes) {
    auto it = free_list.find(bytes);
    if (it != free_list.end() && !it->second.empty()) {
      void *p = *it->second.begin();
      it->second.erase(it->second.begin());
      if (it->second.empty()) free_list.erase(it);
      live[p] = bytes;
      return p;
    }
    void *p = nullptr;
    if (hipMalloc(&p, bytes) != hipSuccess) {
      // morecore (memory.cu:40-52): flush the free lists and retry once
      (void)hipGetLastError();
      clear();
      if (hipMalloc(&p, bytes) != hipSuccess) return nullptr;
    }
    live[p] = bytes;
    return p;
  }
  void put(void *p) {
    auto it = live.find(p);
    if (it == live.end()) return;
    free_list[it->second].insert(p);
    live.erase(it);
  }
  void clear() {
    for (auto &kv : free_list)
      for (void *p : kv.second) (void)hipFree(p);
    free_list.clear();
  }
};

struct Legacy {
  std::mutex mu;
  Pool pool;
  hipStream_t stream = nullptr;
  int backend = -1;                  // TCE_T_LEGACY_DIRECT / _TTGT (-1: from the environment)
  rocblas_handle blas = nullptr;     // TTGT: DGEMM on the library stream
  double *t3_d = nullptr, *t3_s = nullptr;  // task tiles (doubles, singles)
  long dims_d[6] = {0}, dims_s[6] = {0};    // h1,h2,h3,p4,p5,p6 of each tile
  double *pinned = nullptr;
  size_t pinned_bytes = 0;
  bool failed = false;
};
Legacy &L() {
  static Legacy s;
  return s;
}

bool ok(hipError_t e, const char *what) {
  if (e == hipSuccess) return true;
  char buf[256];
  snprintf(buf, sizeof buf, "%s: %s", what, hipGetErrorString(e));
  set_error(buf);
  fprintf(stderr, "tce_t legacy: %s\n", buf);
  L().failed = true;
  return false;
}

bool ensure_stream() {
  if (L().stream) return true;
  return ok(hipStreamCreateWithFlags(&L().stream, hipStreamNonBlocking), "hipStreamCreate");
}

int backend_of(Legacy &S) {
  if (S.backend < 0) {
    const char *e = getenv("TCE_T_LEGACY");
    S.backend = (e && !strcmp(e, "ttgt")) ? TCE_T_LEGACY_TTGT : TCE_T_LEGACY_DIRECT;
  }
  return S.backend;
}

bool ensure_blas(Legacy &S) {
  if (S.blas) return true;
  if (rocblas_create_handle(&S.blas) != rocblas_status_success ||
      rocblas_set_stream(S.blas, S.stream) != rocblas_status_success) {
    set_error("rocBLAS handle for the TTGT back end");
    fprintf(stderr, "tce_t legacy: %s\n", g_err.c_str());
    S.failed = true;
    return false;
  }
  return true;
}

// Row-index codes of the reference kernels' loop variables.
enum { P4 = 0, P5 = 1, P6 = 2, H1 = 3, H2 = 4, H3 = 5 };

// Output layouts (Fortran order, fastest first) and signs of the 27
// variants: the triplesx declarations and update signs of
// ccsd_t_kernels_omp.F:5-1198 (the GPU kernels of sd_t_total.cu write the
// same layouts).
const int kS1L[9][6] = {{H3, H2, H1, P6, P5, P4}, {H3, H1, H2, P6, P5, P4}, {H1, H3, H2, P6, P5, P4},
                        {H3, H2, H1, P6, P4, P5}, {H3, H1, H2, P6, P4, P5}, {H1, H3, H2, P6, P4, P5},
                        {H3, H2, H1, P4, P6, P5}, {H3, H1, H2, P4, P6, P5}, {H1, H3, H2, P4, P6, P5}};
const int kS1S[9] = {+1, -1, +1, -1, +1, -1, +1, -1, +1};
const int kD1L[9][6] = {{H3, H2, H1, P6, P5, P4}, {H3, H1, H2, P6, P5, P4}, {H1, H3, H2, P6, P5, P4},
                        {H3, H2, H1, P5, P4, P6}, {H3, H1, H2, P5, P4, P6}, {H1, H3, H2, P5, P4, P6},
                        {H3, H2, H1, P5, P6, P4}, {H3, H1, H2, P5, P6, P4}, {H1, H3, H2, P5, P6, P4}};
const int kD1S[9] = {-1, +1, -1, -1, +1, -1, +1, -1, +1};
const int kD2L[9][6] = {{H3, H2, H1, P6, P5, P4}, {H2, H1, H3, P6, P5, P4}, {H2, H3, H1, P6, P5, P4},
                        {H3, H2, H1, P6, P4, P5}, {H2, H1, H3, P6, P4, P5}, {H2, H3, H1, P6, P4, P5},
                        {H3, H2, H1, P4, P6, P5}, {H2, H1, H3, P4, P6, P5}, {H2, H3, H1, P4, P6, P5}};
const int kD2S[9] = {-1, -1, +1, +1, +1, -1, -1, -1, +1};

// One call: the output tile's extents and row codes in its own (layout)
// order, operand strides by row code and the contraction.
struct CallArgs {
  long dimL[6];   // extents in output order
  int codeL[6];   // row code at each output position
  long total;     // elements of the output tile
  long K;         // contraction length (1 for s1)
  // operand strides by row code (elements), contraction stride = 1 or 0
  long sa[6], sb[6];
  long ka, kb;    // stride of the contraction index in a / b
  double sign;
};

// The direct contraction.  Every variant's layout has the three hole indices
// first (the block of F = h1 h2 h3 contiguous elements) and the three particle
// indices after them, one to two of them on each operand.  A thread owns one
// element of the hole block at TA x TB places of the particle indices, TA of
// one that sits on the a operand and TB of one that sits on b: TA + TB operand
// loads feed TA TB multiply-adds, and lanes read and write consecutive
// elements of t3.  The d1/d2 operands are packed first (pack_operands): the
// hole indices fastest, in the output's order, then the contraction index, so
// that lanes read consecutive operand elements too (t2sub and the d2 v2sub
// have the contraction index fastest: every lane on a line of its own).
// Bound: HBM, 16 bytes per element of t3 (read and written on each call; the
// operands stay in L2), at tiles of 12^3 x 24^3 elements 82 us at the 4.7 TB/s
// of a plain copy.  Time per call there: one element per thread, with two
// loads per multiply-add and six 64-bit divisions per element, 584 us on
// average; 4 x 4 tiles on the operands as they come s1 74, d1 117 to 208, d2
// 215 to 528 us; packed (4 to 10 us
// more) s1 74, d1 114, d2 164 us.
constexpr int TA = 4, TB = 4;
struct DirectArgs {
  unsigned F, d0, d1;          // hole block, its two fastest extents
  long fa[3], fb[3];           // operand strides of the hole indices
  int na, nb;                  // extents of the two tiled particle indices
  unsigned tiles_a, tiles_b;   // tiles of them
  long a_sa, b_sb;             // their operand strides
  long a_t, b_t, c_t;          // strides of the particle indices in t3
  long c_sa, c_sb;             // operand strides of the third one
  unsigned threads, nc;        // per place of the third index; its extent
  int K;
  long ka, kb;
  double sign;
};

// Whether operand a (t1sub / t2sub) of a family has the index.
bool on_a(int family, int code) {
  return code == P4 || code == H1 || (family == 1 && code == P5) || (family == 2 && code == H2);
}

// A packed copy of one operand: dims in the packed order (holes in the
// output's order, contraction index, particles), source strides.
struct PackArgs {
  unsigned n;
  unsigned ext[5];
  long src[5];
};
struct PackPair {
  PackArgs p[2];  // a, b
  long at[2];     // source offsets (elements)
  long to[2];     // packed offsets
};

__global__ void __launch_bounds__(256) pack_operands(PackPair P, const double *__restrict__ in,
                                                     double *__restrict__ out) {
  const PackArgs &p = P.p[blockIdx.y];
  const unsigned x = blockIdx.x * 256u + threadIdx.x;
  if (x >= p.n) return;
  unsigned r = x;
  long o = 0;
#pragma unroll
  for (int q = 0; q < 5; ++q) {
    const unsigned v = r % p.ext[q];
    r /= p.ext[q];
    o += v * p.src[q];
  }
  out[P.to[blockIdx.y] + x] = in[P.at[blockIdx.y] + o];
}

// The packed form of a call's operand (a or b): fills p and replaces the
// operand's strides in c.
PackArgs pack_args(CallArgs &c, int family, bool a) {
  PackArgs p;
  long *st = a ? c.sa : c.sb;
  long &ks = a ? c.ka : c.kb;
  int q = 0;
  long at = 1;
  auto dim = [&](long ext, long &stride) {
    p.ext[q] = (unsigned)ext;
    p.src[q++] = stride;
    stride = at;
    at *= ext;
  };
  for (int k = 0; k < 3; ++k)
    if (on_a(family, c.codeL[k]) == a) dim(c.dimL[k], st[c.codeL[k]]);
  dim(c.K, ks);
  for (int k = 3; k < 6; ++k)
    if (on_a(family, c.codeL[k]) == a) dim(c.dimL[k], st[c.codeL[k]]);
  p.n = (unsigned)at;
  for (; q < 5; ++q) p.ext[q] = 1, p.src[q] = 0;
  return p;
}

DirectArgs direct_args(const CallArgs &c, int family) {
  DirectArgs d;
  long stride[6], s = 1;
  for (int q = 0; q < 6; ++q) stride[q] = s, s *= c.dimL[q];
  d.F = (unsigned)(c.dimL[0] * c.dimL[1] * c.dimL[2]);
  d.d0 = (unsigned)c.dimL[0], d.d1 = (unsigned)c.dimL[1];
  for (int q = 0; q < 3; ++q) d.fa[q] = c.sa[c.codeL[q]], d.fb[q] = c.sb[c.codeL[q]];
  int qa = -1, qb = -1, qc = -1;
  for (int q = 3; q < 6; ++q) {
    const bool a = on_a(family, c.codeL[q]);
    if (a && qa < 0) qa = q;
    else if (!a && qb < 0) qb = q;
    else qc = q;
  }
  d.na = (int)c.dimL[qa], d.nb = (int)c.dimL[qb];
  d.tiles_a = (unsigned)((d.na + TA - 1) / TA), d.tiles_b = (unsigned)((d.nb + TB - 1) / TB);
  d.a_sa = c.sa[c.codeL[qa]], d.b_sb = c.sb[c.codeL[qb]];
  d.a_t = stride[qa], d.b_t = stride[qb], d.c_t = stride[qc];
  d.c_sa = c.sa[c.codeL[qc]], d.c_sb = c.sb[c.codeL[qc]];
  d.threads = (unsigned)((long)d.F * d.tiles_a * d.tiles_b);
  d.nc = (unsigned)c.dimL[qc];
  d.K = (int)c.K;
  d.ka = c.ka, d.kb = c.kb;
  d.sign = c.sign;
  return d;
}

__global__ void __launch_bounds__(256) contract_kernel(DirectArgs c, double *__restrict__ t3,
                                                       const double *__restrict__ a,
                                                       const double *__restrict__ b) {
  const unsigned x = blockIdx.x * 256u + threadIdx.x;
  if (x >= c.threads) return;
  unsigned r = x / c.F;
  const unsigned o = x - r * c.F;
  const unsigned i0 = o % c.d0, i12 = o / c.d0, i1 = i12 % c.d1, i2 = i12 / c.d1;
  const int pb = (int)(r % c.tiles_b) * TB;
  r /= c.tiles_b;
  const int pa = (int)r * TA;
  const long pc = blockIdx.y;
  const double *ap[TA], *bp[TB];
  const long oa = i0 * c.fa[0] + i1 * c.fa[1] + i2 * c.fa[2] + pc * c.c_sa;
  const long ob = i0 * c.fb[0] + i1 * c.fb[1] + i2 * c.fb[2] + pc * c.c_sb;
#pragma unroll
  for (int u = 0; u < TA; ++u) ap[u] = a + oa + min(pa + u, c.na - 1) * c.a_sa;
#pragma unroll
  for (int v = 0; v < TB; ++v) bp[v] = b + ob + min(pb + v, c.nb - 1) * c.b_sb;
  double *t = t3 + o + pa * c.a_t + pb * c.b_t + pc * c.c_t;
  double old[TA][TB], acc[TA][TB];
#pragma unroll
  for (int u = 0; u < TA; ++u)
#pragma unroll
    for (int v = 0; v < TB; ++v) {
      acc[u][v] = 0.0;
      old[u][v] = pa + u < c.na && pb + v < c.nb ? t[u * c.a_t + v * c.b_t] : 0.0;
    }
#pragma unroll 4
  for (int k = 0; k < c.K; ++k) {
    double av[TA], bv[TB];
#pragma unroll
    for (int u = 0; u < TA; ++u) av[u] = ap[u][k * c.ka];
#pragma unroll
    for (int v = 0; v < TB; ++v) bv[v] = bp[v][k * c.kb];
#pragma unroll
    for (int u = 0; u < TA; ++u)
#pragma unroll
      for (int v = 0; v < TB; ++v) acc[u][v] = fma(av[u], bv[v], acc[u][v]);
  }
#pragma unroll
  for (int u = 0; u < TA; ++u)
#pragma unroll
    for (int v = 0; v < TB; ++v)
      if (pa + u < c.na && pb + v < c.nb)
        t[u * c.a_t + v * c.b_t] = old[u][v] + c.sign * acc[u][v];
}

// The same with one element a thread, in t3's own order, on the operands as they
// come: calls too small to fill the chip with tiles.
__global__ void __launch_bounds__(256) contract_elements(CallArgs c, double *__restrict__ t3,
                                                         const double *__restrict__ a,
                                                         const double *__restrict__ b) {
  const unsigned o = blockIdx.x * 256u + threadIdx.x;
  if (o >= c.total) return;
  unsigned r = o;
  long oa = 0, ob = 0;
#pragma unroll
  for (int q = 0; q < 6; ++q) {
    const unsigned n = (unsigned)c.dimL[q], v = r % n;
    r /= n;
    oa += v * c.sa[c.codeL[q]];
    ob += v * c.sb[c.codeL[q]];
  }
  double acc = 0.0;
  for (long k = 0; k < c.K; ++k) acc = fma(a[oa + k * c.ka], b[ob + k * c.kb], acc);
  t3[o] += c.sign * acc;
}

// How a call runs.  Tiles pay from 2^20 elements (s1) or 2^22 multiply-adds
// (d1, d2) on; below, their fewer threads and the packing launch cost more than
// they save.  Time of a call, elements / tiles (h holes and p particles each,
// contraction over one of them): s1 h=6,p=12 25.6 / 26.6 us, 10,10 29.8 / 28.6,
// 8,16 39 / 31; d1 1,8 18.3 / 23.1, 6,12 28.4 / 31.6, 3,40 37.9 / 34.5, 10,10 41.2
// / 37.8; d2 1,8 19 / 24, 3,16 30 / 35, 6,12 35.1 / 34.6, 5,16 48 / 38, 8,16 107 / 49.
// Packing gains through the hole indices; a block of one hole triple has none
// (d2 1,100 414 us packed, 405 not).  The tiled kernels count in 32 bits and put
// one particle index in grid.y, which ends at 65535.
struct Route {
  bool tiled, pack;
};
Route route_of(const CallArgs &c, int family, long na, long nb) {
  long x = 1, third = 1;
  bool a = false, b = false;
  for (int q = 0; q < 6; ++q) {
    const bool on = q >= 3 && on_a(family, c.codeL[q]);
    const bool tile = q >= 3 && (on ? !a : !b);
    if (q >= 3 && !tile) third = c.dimL[q];
    else x *= tile ? (c.dimL[q] + 3) / 4 : c.dimL[q];
    if (q >= 3) (on ? a : b) = true;
  }
  const long most = 0xffffff00l;
  Route r;
  r.tiled = c.total * std::max(c.K, 1l) >= (family == 0 ? 1l << 20 : 1l << 22) && third <= 65535 &&
            x <= most;
  r.pack = r.tiled && family != 0 && c.K > 0 && c.dimL[0] * c.dimL[1] * c.dimL[2] > 1 &&
           na <= most && nb <= most;
  return r;
}

// TTGT back end (the alternative of sd_t_total_ttlg.cu: GEMM plus
// transposes): the d1/d2 contraction as one DGEMM into C[m + M n] (rocBLAS,
// FP64 matrix cores), m and n the output indices that sit on the t2 and the
// v2 operand; this kernel adds C into the task tile in the variant's layout
// (the transpose).  Strides of C by row code in c.sa; c.sb, c.ka, c.kb and
// c.K unused.
__global__ void __launch_bounds__(256) permute_add_kernel(CallArgs c, double *__restrict__ t3,
                                                          const double *__restrict__ C) {
  long o = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (o >= c.total) return;
  long r = o, oc = 0;
#pragma unroll
  for (int q = 0; q < 6; ++q) {
    long v = r % c.dimL[q];
    r /= c.dimL[q];
    oc += v * c.sa[c.codeL[q]];
  }
  t3[o] += c.sign * C[oc];
}

// family: 0 = s1, 1 = d1, 2 = d2.  dims by row code; K contraction length.
// host_t3 == nullptr: accumulate into the library's device tile of the task
// (the GPU surface); otherwise into the caller's host triplesx (the CPU
// surface), staged through the device for the call.
void launch_call(int family, int n, const long dims[6], long K, const double *ha, long na,
                 const double *hb, long nb, bool singles, double *host_t3 = nullptr) {
  Legacy &S = L();
  std::lock_guard<std::mutex> lk(S.mu);
  if (!ensure_stream()) return;
  double *t3 = host_t3 ? nullptr : (singles ? S.t3_s : S.t3_d);
  if (!host_t3 && !t3) {
    set_error("sd_t kernel called before dev_mem_s_/dev_mem_d_");
    fprintf(stderr, "tce_t legacy: %s\n", g_err.c_str());
    S.failed = true;
    return;
  }
  const int *Lo = family == 0 ? kS1L[n - 1] : family == 1 ? kD1L[n - 1] : kD2L[n - 1];
  int sign = family == 0 ? kS1S[n - 1] : family == 1 ? kD1S[n - 1] : kD2S[n - 1];
  CallArgs c;
  c.total = 1;
  for (int q = 0; q < 6; ++q) {
    c.codeL[q] = Lo[q];
    c.dimL[q] = dims[Lo[q]];
    c.total *= c.dimL[q];
  }
  // The task tile holds exactly these elements (same extents, permuted).
  const long *td = singles ? S.dims_s : S.dims_d;
  long tsize = td[0] * td[1] * td[2] * td[3] * td[4] * td[5];
  if (!host_t3 && tsize != c.total) {
    set_error("operand dimensions do not match the task tile");
    fprintf(stderr, "tce_t legacy: %s\n", g_err.c_str());
    S.failed = true;
    return;
  }
  c.K = K;
  c.sign = (double)sign;
  for (int q = 0; q < 6; ++q) c.sa[q] = c.sb[q] = 0;
  long p4d = dims[P4], p5d = dims[P5], p6d = dims[P6], h1d = dims[H1], h2d = dims[H2], h3d = dims[H3];
  if (family == 0) {  // t1sub(p4,h1), v2sub(h3,h2,p6,p5)
    c.sa[P4] = 1;
    c.sa[H1] = p4d;
    c.sb[H3] = 1;
    c.sb[H2] = h3d;
    c.sb[P6] = h3d * h2d;
    c.sb[P5] = h3d * h2d * p6d;
    c.ka = c.kb = 0;
  } else if (family == 1) {  // t2sub(h7,p4,p5,h1), v2sub(h3,h2,p6,h7)
    c.ka = 1;
    c.sa[P4] = K;
    c.sa[P5] = K * p4d;
    c.sa[H1] = K * p4d * p5d;
    c.sb[H3] = 1;
    c.sb[H2] = h3d;
    c.sb[P6] = h3d * h2d;
    c.kb = h3d * h2d * p6d;
  } else {  // t2sub(p7,p4,h1,h2), v2sub(p7,h3,p6,p5)
    c.ka = 1;
    c.sa[P4] = K;
    c.sa[H1] = K * p4d;
    c.sa[H2] = K * p4d * h1d;
    c.kb = 1;
    c.sb[H3] = K;
    c.sb[P6] = K * h3d;
    c.sb[P5] = K * h3d * p6d;
  }
  (void)p5d;
  // Stage both operands through one pinned buffer, copy, launch.  The
  // synchronisation before returning keeps the caller's MA stack semantics
  // (operands may be popped right after the call).
  size_t bytes = (size_t)(na + nb) * sizeof(double);
  if (bytes > S.pinned_bytes) {
    if (S.pinned) (void)hipHostFree(S.pinned);
    S.pinned = nullptr;
    S.pinned_bytes = 0;
    if (!ok(hipHostMalloc((void **)&S.pinned, bytes), "hipHostMalloc")) return;
    S.pinned_bytes = bytes;
  }
  memcpy(S.pinned, ha, na * sizeof(double));
  memcpy(S.pinned + na, hb, nb * sizeof(double));
  Route route = route_of(c, family, na, nb);
  if (family != 0 && backend_of(S) != TCE_T_LEGACY_DIRECT) route.pack = false;
  // packed copies go behind the operands
  double *dops = (double *)S.pool.get(route.pack ? 2 * bytes : bytes);
  if (!dops && route.pack) {
    (void)hipGetLastError();
    route.pack = false;
    dops = (double *)S.pool.get(bytes);
  }
  if (!dops) {
    set_error("device pool allocation failed");
    S.failed = true;
    return;
  }
  if (!ok(hipMemcpyAsync(dops, S.pinned, bytes, hipMemcpyHostToDevice, S.stream), "H2D")) return;
  const size_t tbytes = (size_t)c.total * sizeof(double);
  if (host_t3) {
    t3 = (double *)S.pool.get(tbytes);
    if (!t3) {
      set_error("device pool allocation failed");
      S.failed = true;
      S.pool.put(dops);
      return;
    }
    // pageable copies: the caller's array is read and written in place
    if (!ok(hipMemcpyAsync(t3, host_t3, tbytes, hipMemcpyHostToDevice, S.stream), "H2D t3")) return;
  }
  int threads = 256;
  long blocks = (c.total + threads - 1) / threads;
  double *dC = nullptr;
  if (family != 0 && backend_of(S) == TCE_T_LEGACY_TTGT && ensure_blas(S)) {
    // m: the indices on t2sub, n: those on v2sub (C[m + M n])
    long M, N;
    CallArgs p = c;
    for (int q = 0; q < 6; ++q) p.sa[q] = 0;
    if (family == 2) {  // t2sub(p7,p4,h1,h2), v2sub(p7,h3,p6,p5)
      M = p4d * h1d * h2d, N = h3d * p6d * p5d;
      p.sa[P4] = 1, p.sa[H1] = p4d, p.sa[H2] = p4d * h1d;
      p.sa[H3] = M, p.sa[P6] = M * h3d, p.sa[P5] = M * h3d * p6d;
    } else {  // t2sub(h7,p4,p5,h1), v2sub(h3,h2,p6,h7)
      M = p4d * p5d * h1d, N = h3d * h2d * p6d;
      p.sa[P4] = 1, p.sa[P5] = p4d, p.sa[H1] = p4d * p5d;
      p.sa[H3] = M, p.sa[H2] = M * h3d, p.sa[P6] = M * h3d * h2d;
    }
    dC = (double *)S.pool.get((size_t)M * N * sizeof(double));
    if (!dC) {
      set_error("device pool allocation failed");
      S.failed = true;
      S.pool.put(dops);
      if (host_t3) S.pool.put(t3);
      return;
    }
    const double one = 1.0, zero = 0.0;
    const rocblas_status st =
        family == 2
            ? rocblas_dgemm(S.blas, rocblas_operation_transpose, rocblas_operation_none, (int)M,
                            (int)N, (int)K, &one, dops, (int)K, dops + na, (int)K, &zero, dC, (int)M)
            : rocblas_dgemm(S.blas, rocblas_operation_transpose, rocblas_operation_transpose,
                            (int)M, (int)N, (int)K, &one, dops, (int)K, dops + na, (int)N, &zero,
                            dC, (int)M);
    if (st != rocblas_status_success) {
      set_error("rocblas_dgemm failed");
      fprintf(stderr, "tce_t legacy: %s\n", g_err.c_str());
      S.failed = true;
      return;
    }
    hipLaunchKernelGGL(permute_add_kernel, dim3((unsigned)blocks), dim3(threads), 0, S.stream, p,
                       t3, dC);
    if (!ok(hipGetLastError(), "permute_add_kernel launch")) return;
  } else {
    const double *ops = dops;
    if (route.pack) {
      PackPair P;
      P.p[0] = pack_args(c, family, true);
      P.p[1] = pack_args(c, family, false);
      P.at[0] = P.to[0] = 0;
      P.at[1] = P.to[1] = na;
      double *packed = dops + na + nb;
      hipLaunchKernelGGL(pack_operands, dim3((std::max(P.p[0].n, P.p[1].n) + 255) / 256, 2),
                         dim3(256), 0, S.stream, P, dops, packed);
      if (!ok(hipGetLastError(), "pack_operands launch")) return;
      ops = packed;
    }
    if (route.tiled) {
      const DirectArgs da = direct_args(c, family);
      hipLaunchKernelGGL(contract_kernel, dim3((da.threads + 255) / 256, da.nc), dim3(256), 0,
                         S.stream, da, t3, ops, ops + na);
    } else {
      hipLaunchKernelGGL(contract_elements, dim3((unsigned)blocks), dim3(threads), 0, S.stream, c,
                         t3, ops, ops + na);
    }
    if (!ok(hipGetLastError(), "contract_kernel launch")) return;
  }
  if (host_t3 && !ok(hipMemcpyAsync(host_t3, t3, tbytes, hipMemcpyDeviceToHost, S.stream), "D2H t3"))
    return;
  ok(hipStreamSynchronize(S.stream), "contract_kernel");
  S.pool.put(dops);
  if (dC) S.pool.put(dC);
  if (host_t3) S.pool.put(t3);
}

// Energy of one task tile, layout (h3 fastest, h2, h1, p6, p5, p4 slowest)
// as in ccsd_t_dot.F:89-110; first pass: one partial pair per block.  The
// orbital energies of the six tiles are e1..e6 (h1, h2, h3, p4, p5, p6).
// A unit of work is one particle triple by up to kEnChunk elements of its
// hole block, whose e_h1 + e_h2 + e_h3 sit in LDS; where the hole block leaves
// half of the threads idle or more, as many triples as the threads hold (a
// single hole orbital, 64 particles each: one triple at a time 259 us for the
// call, 256 at a time 32; one element a thread in turn 115).
// Bound: HBM, 16 bytes per element.  With five 64-bit divisions per element to
// find its indices, 24e6 elements took 147 us; their bytes take 82 us.
constexpr int kEnChunk = 2048;
__device__ __forceinline__ void energy_block(long h1d, long h2d, long h3d, long p4d, long p5d,
                                             long p6d, const double *__restrict__ e1,
                                             const double *__restrict__ e2,
                                             const double *__restrict__ e3,
                                             const double *__restrict__ e4,
                                             const double *__restrict__ e5,
                                             const double *__restrict__ e6, double factor,
                                             const double *__restrict__ t3d,
                                             const double *__restrict__ t3s,
                                             double *__restrict__ part) {
  __shared__ double eh[kEnChunk];
  const long F = h1d * h2d * h3d, P = p4d * p5d * p6d;
  const int per = F > 0 && F <= 128 ? 256 / (int)F : 1;  // triples of a unit
  const int mine = per > 1 ? (int)threadIdx.x / (int)F : 0;
  const int first = (int)threadIdx.x - mine * (int)F, step = per > 1 ? (int)F : 256;
  const long groups = (P + per - 1) / per, units = (F + kEnChunk - 1) / kEnChunk * groups;
  double s1 = 0.0, s2 = 0.0;
  long cur = -1;
  for (long u = blockIdx.x; u < units; u += gridDim.x) {
    const long chunk = u / groups, pt = (u - chunk * groups) * per + mine, f0 = chunk * kEnChunk;
    const int n = (int)(F - f0 < kEnChunk ? F - f0 : kEnChunk);
    if (chunk != cur) {  // uniform
      __syncthreads();
      for (int f = threadIdx.x; f < n; f += blockDim.x) {
        const long x = f0 + f, r = x / h3d;
        eh[f] = e1[r / h2d] + e2[r % h2d] + e3[x - r * h3d];
      }
      __syncthreads();
      cur = chunk;
    }
    if (mine >= per || pt >= P) continue;  // groups share the one chunk: no barrier ahead
    const long p45 = pt / p6d;
    const double denom_0 = -(e4[p45 / p5d] + e5[p45 % p5d] + e6[pt - p45 * p6d]);
    const double *d = t3d + pt * F + f0, *s = t3s + pt * F + f0;
#pragma unroll 4
    for (int f = first; f < n; f += step) {
      const double doub = d[f], sing = s[f];
      const double denom = doub * factor / (eh[f] + denom_0);
      s1 += denom * doub;
      s2 += denom * (doub + sing);
    }
  }
  __shared__ double r1[256], r2[256];
  r1[threadIdx.x] = s1;
  r2[threadIdx.x] = s2;
  __syncthreads();
  for (int w = 128; w > 0; w >>= 1) {
    if ((int)threadIdx.x < w) {
      r1[threadIdx.x] += r1[threadIdx.x + w];
      r2[threadIdx.x] += r2[threadIdx.x + w];
    }
    __syncthreads();
  }
  if (threadIdx.x == 0) {
    part[2 * blockIdx.x] = r1[0];
    part[2 * blockIdx.x + 1] = r2[0];
  }
}

// compute_en_: the six energy vectors packed in one device buffer.
__global__ void __launch_bounds__(256) energy_partial(
    long h1d, long h2d, long h3d, long p4d, long p5d, long p6d, const double *__restrict__ ev,
    double factor, const double *__restrict__ t3d, const double *__restrict__ t3s,
    double *__restrict__ part) {
  const double *e1 = ev, *e2 = e1 + h1d, *e3 = e2 + h2d, *e4 = e3 + h3d, *e5 = e4 + p4d, *e6 = e5 + p5d;
  energy_block(h1d, h2d, h3d, p4d, p5d, p6d, e1, e2, e3, e4, e5, e6, factor, t3d, t3s, part);
}

// tce_t_compute_en_noalloc: six separate device vectors.
__global__ void __launch_bounds__(256) energy_partial_split(
    long h1d, long h2d, long h3d, long p4d, long p5d, long p6d, const double *__restrict__ e1,
    const double *__restrict__ e2, const double *__restrict__ e3, const double *__restrict__ e4,
    const double *__restrict__ e5, const double *__restrict__ e6, double factor,
    const double *__restrict__ t3d, const double *__restrict__ t3s, double *__restrict__ part) {
  energy_block(h1d, h2d, h3d, p4d, p5d, p6d, e1, e2, e3, e4, e5, e6, factor, t3d, t3s, part);
}

// Grid of the energy reduction: compute_en_ and tce_t_compute_en_noalloc
// both run energy_partial on this many blocks, so their sums are the same.
constexpr int kEnBlocks = 1024;
constexpr int kEnThreads = 256;

// The block partials of tce_t_compute_en_noalloc: 2 doubles per block,
// 16 KiB, one copy per device for the life of the process.  Every call
// writes all of them before reading them, so nothing needs clearing between
// calls.  Host code never passes this name to a kernel (in host code it is
// a stand-in, not a device address); it uses the address
// hipGetSymbolAddress gives on each device.
constexpr size_t kScratchDoubles = 2 * kEnBlocks;
static __device__ __align__(256) double scratch[kScratchDoubles];

// Second pass: fixed-order sum of the block partials, one workgroup (one
// thread over the 1024 pairs took 86 us, a chain of dependent loads and adds).
__global__ void __launch_bounds__(256) energy_final(const double *__restrict__ part, int nblk,
                                                    double *__restrict__ out) {
  __shared__ double r1[256], r2[256];
  double a = 0.0, b = 0.0;
  for (int i = threadIdx.x; i < nblk; i += 256) {
    a += part[2 * i];
    b += part[2 * i + 1];
  }
  r1[threadIdx.x] = a;
  r2[threadIdx.x] = b;
  __syncthreads();
  for (int w = 128; w > 0; w >>= 1) {
    if ((int)threadIdx.x < w) {
      r1[threadIdx.x] += r1[threadIdx.x + w];
      r2[threadIdx.x] += r2[threadIdx.x + w];
    }
    __syncthreads();
  }
  if (threadIdx.x == 0) {
    out[0] = r1[0];
    out[1] = r2[0];
  }
}

void alloc_tile(bool singles, const long d[6]) {
  Legacy &S = L();
  std::lock_guard<std::mutex> lk(S.mu);
  if (!ensure_stream()) return;
  size_t n = (size_t)d[0] * d[1] * d[2] * d[3] * d[4] * d[5];
  double *&t = singles ? S.t3_s : S.t3_d;
  long *dims = singles ? S.dims_s : S.dims_d;
  if (t) S.pool.put(t);
  t = (double *)S.pool.get(n * sizeof(double));
  if (!t) {
    set_error("device tile allocation failed");
    fprintf(stderr, "tce_t legacy: %s\n", g_err.c_str());
    S.failed = true;
    return;
  }
  for (int q = 0; q < 6; ++q) dims[q] = d[q];
  ok(hipMemsetAsync(t, 0, n * sizeof(double), S.stream), "hipMemset t3");
}

int local_rank() {
  const char *vars[] = {"OMPI_COMM_WORLD_LOCAL_RANK", "MPI_LOCALRANKID", "SLURM_LOCALID",
                        "LOCAL_RANK"};
  for (const char *v : vars) {
    const char *s = getenv(v);
    if (s && *s) return atoi(s);
  }
  return 0;
}

}  // namespace
}  // namespace tce_t

using namespace tce_t;

extern "C" const char *tce_t_last_error(void) { return g_err.c_str(); }

// ------------------------------------------------------ entry points -------
#define S1_ENTRY(N)                                                                       \
  extern "C" void sd_t_s1_##N##_cuda_(long *h1d, long *h2d, long *h3d, long *p4d,        \
                                      long *p5d, long *p6d, double *t3, double *t1,      \
                                      double *v2) {                                      \
    (void)t3;                                                                             \
    long dims[6] = {*p4d, *p5d, *p6d, *h1d, *h2d, *h3d};                                  \
    launch_call(0, N, dims, 1, t1, (*p4d) * (*h1d), v2, (*h3d) * (*h2d) * (*p6d) * (*p5d), \
                true);                                                                    \
  }
#define D1_ENTRY(N)                                                                       \
  extern "C" void sd_t_d1_##N##_cuda_(long *h1d, long *h2d, long *h3d, long *h7d,        \
                                      long *p4d, long *p5d, long *p6d, double *t3,       \
                                      double *t2, double *v2) {                          \
    (void)t3;                                                                             \
    long dims[6] = {*p4d, *p5d, *p6d, *h1d, *h2d, *h3d};                                  \
    launch_call(1, N, dims, *h7d, t2, (*h7d) * (*p4d) * (*p5d) * (*h1d), v2,              \
                (*h3d) * (*h2d) * (*p6d) * (*h7d), false);                                \
  }
#define D2_ENTRY(N)                                                                       \
  extern "C" void sd_t_d2_##N##_cuda_(long *h1d, long *h2d, long *h3d, long *p4d,        \
                                      long *p5d, long *p6d, long *p7d, double *t3,       \
                                      double *t2, double *v2) {                          \
    (void)t3;                                                                             \
    long dims[6] = {*p4d, *p5d, *p6d, *h1d, *h2d, *h3d};                                  \
    launch_call(2, N, dims, *p7d, t2, (*p7d) * (*p4d) * (*h1d) * (*h2d), v2,              \
                (*p7d) * (*h3d) * (*p6d) * (*p5d), false);                                \
  }
#define ALL9(M) M(1) M(2) M(3) M(4) M(5) M(6) M(7) M(8) M(9)
ALL9(S1_ENTRY)
ALL9(D1_ENTRY)
ALL9(D2_ENTRY)

// The CPU surface (ccsd_t_kernels_omp.F argument order: h3d, h2d, h1d, p6d,
// p5d, p4d[, h7d / p7d]): the same contractions accumulated into the
// caller's host triplesx (not zeroed), for the CPU drivers
// (ccsd_t_singles_l.F, offl_ccsd_t_doubles_l.F) and their other callers.
#define S1_CPU(N)                                                                          \
  extern "C" void sd_t_s1_##N##_(long *h3d, long *h2d, long *h1d, long *p6d, long *p5d,    \
                                 long *p4d, double *triplesx, double *t1sub, double *v2sub) { \
    long dims[6] = {*p4d, *p5d, *p6d, *h1d, *h2d, *h3d};                                   \
    launch_call(0, N, dims, 1, t1sub, (*p4d) * (*h1d), v2sub,                              \
                (*h3d) * (*h2d) * (*p6d) * (*p5d), true, triplesx);                        \
  }
#define D1_CPU(N)                                                                          \
  extern "C" void sd_t_d1_##N##_(long *h3d, long *h2d, long *h1d, long *p6d, long *p5d,    \
                                 long *p4d, long *h7d, double *triplesx, double *t2sub,   \
                                 double *v2sub) {                                          \
    long dims[6] = {*p4d, *p5d, *p6d, *h1d, *h2d, *h3d};                                   \
    launch_call(1, N, dims, *h7d, t2sub, (*h7d) * (*p4d) * (*p5d) * (*h1d), v2sub,         \
                (*h3d) * (*h2d) * (*p6d) * (*h7d), false, triplesx);                       \
  }
#define D2_CPU(N)                                                                          \
  extern "C" void sd_t_d2_##N##_(long *h3d, long *h2d, long *h1d, long *p6d, long *p5d,    \
                                 long *p4d, long *p7d, double *triplesx, double *t2sub,   \
                                 double *v2sub) {                                          \
    long dims[6] = {*p4d, *p5d, *p6d, *h1d, *h2d, *h3d};                                   \
    launch_call(2, N, dims, *p7d, t2sub, (*p7d) * (*p4d) * (*h1d) * (*h2d), v2sub,         \
                (*p7d) * (*h3d) * (*p6d) * (*p5d), false, triplesx);                       \
  }
ALL9(S1_CPU)
ALL9(D1_CPU)
ALL9(D2_CPU)

extern "C" void dev_mem_d_(long *h1d, long *h2d, long *h3d, long *p4d, long *p5d, long *p6d) {
  long d[6] = {*h1d, *h2d, *h3d, *p4d, *p5d, *p6d};
  alloc_tile(false, d);
}
extern "C" void dev_mem_s_(long *h1d, long *h2d, long *h3d, long *p4d, long *p5d, long *p6d) {
  long d[6] = {*h1d, *h2d, *h3d, *p4d, *p5d, *p6d};
  alloc_tile(true, d);
}
extern "C" void dev_release_(void) {
  Legacy &S = L();
  std::lock_guard<std::mutex> lk(S.mu);
  if (S.stream) (void)hipStreamSynchronize(S.stream);
  if (S.t3_d) S.pool.put(S.t3_d);
  if (S.t3_s) S.pool.put(S.t3_s);
  S.t3_d = S.t3_s = nullptr;
}
extern "C" void initmemmodule_(void) {
  Legacy &S = L();
  std::lock_guard<std::mutex> lk(S.mu);
  S.pool.init = true;
}
extern "C" void finalizememmodule_(void) {
  Legacy &S = L();
  std::lock_guard<std::mutex> lk(S.mu);
  if (S.stream) (void)hipStreamSynchronize(S.stream);
  S.pool.clear();
  S.pool.init = false;
}

extern "C" void compute_en_(double *factor, double *energy, double *eval1, double *eval2,
                            double *eval3, double *eval4, double *eval5, double *eval6, long *h1d,
                            long *h2d, long *h3d, long *p4d, long *p5d, long *p6d, double *host1,
                            double *host2) {
  (void)host1;
  (void)host2;
  Legacy &S = L();
  std::lock_guard<std::mutex> lk(S.mu);
  energy[0] = energy[1] = 0.0;
  if (!ensure_stream()) return;
  if (!S.t3_d || !S.t3_s) {
    set_error("compute_en_ called without device tiles");
    fprintf(stderr, "tce_t legacy: %s\n", g_err.c_str());
    S.failed = true;
    return;
  }
  long d[6] = {*h1d, *h2d, *h3d, *p4d, *p5d, *p6d};
  long ne = d[0] + d[1] + d[2] + d[3] + d[4] + d[5];
  const int nblk = kEnBlocks, threads = kEnThreads;
  size_t bytes = (ne + 2 * nblk + 2) * sizeof(double);
  double *dbuf = (double *)S.pool.get(bytes);
  if (!dbuf) {
    set_error("device pool allocation failed");
    S.failed = true;
    return;
  }
  // Orbital energies of the six tiles, packed h1,h2,h3,p4,p5,p6.
  if (S.pinned_bytes < (size_t)(ne + 2) * sizeof(double)) {
    if (S.pinned) (void)hipHostFree(S.pinned);
    S.pinned = nullptr;
    S.pinned_bytes = 0;
    if (!ok(hipHostMalloc((void **)&S.pinned, (ne + 2) * sizeof(double)), "hipHostMalloc")) return;
    S.pinned_bytes = (ne + 2) * sizeof(double);
  }
  double *src[6] = {eval1, eval2, eval3, eval4, eval5, eval6};
  long at = 0;
  for (int q = 0; q < 6; ++q) {
    memcpy(S.pinned + at, src[q], d[q] * sizeof(double));
    at += d[q];
  }
  if (!ok(hipMemcpyAsync(dbuf, S.pinned, ne * sizeof(double), hipMemcpyHostToDevice, S.stream), "H2D"))
    return;
  double *part = dbuf + ne, *out = part + 2 * nblk;
  hipLaunchKernelGGL(energy_partial, dim3(nblk), dim3(threads), 0, S.stream, d[0], d[1], d[2], d[3],
                     d[4], d[5], dbuf, *factor, S.t3_d, S.t3_s, part);
  hipLaunchKernelGGL(energy_final, dim3(1), dim3(kEnThreads), 0, S.stream, part, nblk, out);
  if (!ok(hipGetLastError(), "energy launch")) return;
  if (!ok(hipMemcpyAsync(S.pinned, out, 2 * sizeof(double), hipMemcpyDeviceToHost, S.stream), "D2H"))
    return;
  if (!ok(hipStreamSynchronize(S.stream), "energy")) return;
  energy[0] = S.pinned[0];
  energy[1] = S.pinned[1];
  S.pool.put(dbuf);
}

// ------------------------------------------------ no-allocation energy -----
namespace tce_t {
namespace {
constexpr int kMaxDevices = 64;
std::mutex g_scratch_mu;
double *g_scratch[kMaxDevices] = {nullptr};  // device address of `scratch` per device

// Address of this device's `scratch` (looked up once per device, with the
// device current); nullptr on failure.
double *scratch_on(int dev) {
  if (dev < 0 || dev >= kMaxDevices) return nullptr;
  std::lock_guard<std::mutex> lk(g_scratch_mu);
  if (!g_scratch[dev]) {
    void *p = nullptr;
    if (hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)) != hipSuccess || !p) {
      (void)hipGetLastError();
      return nullptr;
    }
    g_scratch[dev] = (double *)p;
  }
  return g_scratch[dev];
}
}  // namespace
}  // namespace tce_t

extern "C" int tce_t_compute_en_noalloc(double factor, const double *t3d, const double *t3s,
                                        const double *eval1, const double *eval2,
                                        const double *eval3, const double *eval4,
                                        const double *eval5, const double *eval6, long h1d,
                                        long h2d, long h3d, long p4d, long p5d, long p6d,
                                        double *energy, void *stream) {
  if (!t3d || !t3s || !eval1 || !eval2 || !eval3 || !eval4 || !eval5 || !eval6 || !energy) {
    set_error("tce_t_compute_en_noalloc: NULL pointer");
    return TCE_T_ERR_ARG;
  }
  const long d[6] = {h1d, h2d, h3d, p4d, p5d, p6d};
  long total = 1;
  for (long x : d) {
    if (x <= 0 || total > (1L << 62) / x) {
      set_error("tce_t_compute_en_noalloc: tile extents must be positive and their product "
                "below 2^62");
      return TCE_T_ERR_ARG;
    }
    total *= x;
  }
  // the partials of kEnBlocks blocks fill the fixed scratch array exactly
  static_assert(2 * kEnBlocks <= (int)kScratchDoubles, "scratch holds every block partial");
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess) {
    (void)hipGetLastError();
    set_error("tce_t_compute_en_noalloc: hipGetDevice failed");
    return TCE_T_ERR_HIP;
  }
  double *part = scratch_on(dev);
  if (!part) {
    set_error("tce_t_compute_en_noalloc: hipGetSymbolAddress(scratch) failed");
    return TCE_T_ERR_HIP;
  }
  hipStream_t st = (hipStream_t)stream;
  hipLaunchKernelGGL(energy_partial_split, dim3(kEnBlocks), dim3(kEnThreads), 0, st, h1d, h2d, h3d,
                     p4d, p5d, p6d, eval1, eval2, eval3, eval4, eval5, eval6, factor, t3d, t3s,
                     part);
  hipLaunchKernelGGL(energy_final, dim3(1), dim3(kEnThreads), 0, st, part, kEnBlocks, energy);
  const hipError_t e = hipGetLastError();
  if (e != hipSuccess) {
    set_error(std::string("tce_t_compute_en_noalloc launch: ") + hipGetErrorString(e));
    return TCE_T_ERR_HIP;
  }
  return TCE_T_OK;
}

extern "C" int check_device_(long *icuda) { return local_rank() < *icuda ? 1 : 0; }

extern "C" int device_init_(long *icuda, long *cuda_device_number) {
  int n = 0;
  if (hipGetDeviceCount(&n) != hipSuccess) n = 0;
  if (n < *icuda) {
    printf("Warning: Please check whether you have %ld cuda devices per node\n", *icuda);
    fflush(stdout);
    *cuda_device_number = 30;
  } else {
    (void)hipSetDevice(local_rank());
  }
  return 1;
}

extern "C" int tce_t_legacy_backend(int backend) {
  Legacy &S = L();
  std::lock_guard<std::mutex> lk(S.mu);
  if (backend == TCE_T_LEGACY_QUERY) return backend_of(S);
  if (backend != TCE_T_LEGACY_DIRECT && backend != TCE_T_LEGACY_TTGT) return TCE_T_ERR_ARG;
  S.backend = backend;
  return backend;
}

// Sticky failure flag of the per-call surface (the reference exits instead).
extern "C" int tce_t_legacy_status(void) {
  Legacy &S = L();
  int f = S.failed ? TCE_T_ERR_HIP : TCE_T_OK;
  S.failed = false;
  return f;
}
