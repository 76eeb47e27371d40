// gd_runtime.hip -- host runtime of the C ABI: device selection, packing a
// complex into the device layout of gd_device.h, tiling, kernel launches,
// the plain one-job docking path, energy evaluation and accept records.
// Batching and serving build on the same job objects (gd_batch.hip).
//
// Reference call sequence replaced (src/backend_gpu/backend_gpu.cu:64-133,
// prepair.C:12-135): CopyH2D of a 6.3 MiB Complex per job, one launch for
// the initial energies, one launch + blocking D2H of records per dump.  Here
// a job's tables are packed once into device memory sized to the job, the
// replica state never leaves the device, and the MC steps between two exchange
// points or dump ends are one launch of the stepping kernel, or each a pair-,
// reduce- and finish-kernel launch (dock_run says which).
#include <hip/hip_runtime.h>

#include <algorithm>
#include <atomic>
#include <chrono>
#include <cmath>
#include <limits>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <map>
#include <mutex>
#include <string>
#include <vector>

#include "../../include/geauxdock_amd.h"
#include "gd_device.h"
#include "gd_internal.h"
#include "gd_tiling_table.h"

// kernels (gd_kernels.hip)
template <int LC>
__global__ void gd_pair_kernel(const GdJob *, const GdItem *, int, int, int);
__global__ void gd_pair_kernel_split(const GdJob *, const GdItem *, int, int, int);
__global__ void gd_eval_setup_kernel(const GdJob, GdJob *, const int *, const float *, int);
__global__ void gd_reduce_kernel(const GdJob *, const GdBlock *);
__global__ void gd_finish_kernel(const GdJob *, const GdBlock *, int, int, const int *, int *);
template <int LC>
__global__ void gd_chain_kernel(const GdChain);
template <bool BACK>
__global__ void gd_keep_kernel(const GdJob *, const GdBlock *, unsigned *, const unsigned *, unsigned);
__global__ void gd_start_job_kernel(const GdJob, GdJob *);
__global__ void gd_pack_kernel(const GdPackList);
__global__ void gd_exchange_kernel(const GdJob *, const GdExch *, int);
__global__ void gd_move_draws_kernel(uint64_t, uint32_t, int, GdScale6, int, uint32_t, int, float *);
__global__ void gd_clock_kernel(long long, float, long long *, float *);
__global__ void gd_copy_kernel(const float4 *, float4 *, size_t);
__global__ void gd_swap_propose_kernel(const GdJob *, const GdBlock *, int, const int *, int);
__global__ void gd_swap_accept_kernel(const GdJob *, const GdBlock *, int, const int *, int, int,
                                      const int *);

namespace gdr {

static thread_local std::string g_err;
static int g_device = -1;
static int g_cu = 0;
static int g_wall_khz = 100000;  // rate of the constant-rate counter
static std::mutex g_mu;

void set_error(const std::string &s) { g_err = s; }
const char *last_error() { return g_err.c_str(); }

gd_status hip_fail(hipError_t e, const char *what) {
  char buf[256];
  std::snprintf(buf, sizeof buf, "%s: %s", what, hipGetErrorString(e));
  set_error(buf);
  (void)hipGetLastError();  // reported here: the runtime keeps it for the next check of a launch
  return GD_ERR_HIP;
}

KTimer::~KTimer() {
  for (auto e : ev) hipEventDestroy(e);
}
gd_status KTimer::begin(hipStream_t s) {
  if (used + 2 > (int)ev.size()) {
    hipEvent_t a, b;
    hipError_t e;
    // timing-only events: without the system-scope fence a record costs no
    // L2 writeback and invalidate (about 5 us per record on MI355X, paid by
    // the work around it); the elapsed times are read after a stream
    // synchronisation, so no event needs to order memory
    if ((e = hipEventCreateWithFlags(&a, hipEventDisableSystemFence)) != hipSuccess ||
        (e = hipEventCreateWithFlags(&b, hipEventDisableSystemFence)) != hipSuccess)
      return hip_fail(e, "hipEventCreateWithFlags");
    ev.push_back(a);
    ev.push_back(b);
  }
  hipError_t e = hipEventRecord(ev[used], s);
  return e == hipSuccess ? GD_OK : hip_fail(e, "hipEventRecord");
}
gd_status KTimer::end(hipStream_t s) {
  hipError_t e = hipEventRecord(ev[used + 1], s);
  used += 2;
  return e == hipSuccess ? GD_OK : hip_fail(e, "hipEventRecord");
}
gd_status KTimer::collect() {
  for (int i = 0; i + 1 < used; i += 2) {
    float t = 0.0f;
    hipError_t e = hipEventElapsedTime(&t, ev[i], ev[i + 1]);
    if (e != hipSuccess) return hip_fail(e, "hipEventElapsedTime");
    ms += t;
    ++n;
  }
  if (used >= 4) {
    float t = 0.0f;
    hipError_t e = hipEventElapsedTime(&t, ev[0], ev[used - 2]);
    if (e != hipSuccess) return hip_fail(e, "hipEventElapsedTime");
    first_to_last_ms += t;
  }
  used = 0;
  return GD_OK;
}

// Pair-phase timer of the multi-stream plain path: per sampled MC step, the
// span from the first start to the last end of its parts' launches (events on
// every part's stream), every event timed from one reference recorded earlier
// on the first stream (so no elapsed time is negative).
struct SpanTimer {
  std::vector<hipEvent_t> ev;
  int used = 0;
  hipEvent_t ref = nullptr;
  double ms = 0.0;
  int n = 0;
  ~SpanTimer() {
    for (auto e : ev) hipEventDestroy(e);
    if (ref) hipEventDestroy(ref);
  }
  hipEvent_t next() {
    if (used == (int)ev.size()) {
      hipEvent_t e;
      if (hipEventCreateWithFlags(&e, hipEventDisableSystemFence) != hipSuccess) return nullptr;
      ev.push_back(e);
    }
    return ev[used++];
  }
  gd_status mark_ref(hipStream_t s) {
    if (!ref && hipEventCreateWithFlags(&ref, hipEventDisableSystemFence) != hipSuccess)
      return hip_fail(hipErrorOutOfMemory, "hipEventCreate");
    const hipError_t e = hipEventRecord(ref, s);
    return e == hipSuccess ? GD_OK : hip_fail(e, "hipEventRecord");
  }
  gd_status record(hipStream_t s) {  // per sample: start and end of every part's launch
    hipEvent_t e = next();
    if (!e) return hip_fail(hipErrorOutOfMemory, "hipEventCreate");
    const hipError_t r = hipEventRecord(e, s);
    return r == hipSuccess ? GD_OK : hip_fail(r, "hipEventRecord");
  }
  double parts_ms = 0.0, first_a = -1.0, last_a = -1.0;
  int n_part_launches = 0;
  gd_status collect(int np) {  // after every part's stream is synchronised
    for (int i = 0; i + 2 * np - 1 < used; i += 2 * np) {
      float t0 = 0.0f, t_lo = 0.0f, t_hi = 0.0f;
      for (int k = 0; k < np; ++k) {
        float a, b;
        hipError_t e = hipEventElapsedTime(&a, ref, ev[i + 2 * k]);
        if (e == hipSuccess) e = hipEventElapsedTime(&b, ref, ev[i + 2 * k + 1]);
        if (e != hipSuccess) return hip_fail(e, "hipEventElapsedTime");
        if (k == 0) t0 = t_lo = a, t_hi = b;
        t_lo = std::min(t_lo, a);
        t_hi = std::max(t_hi, b);
        parts_ms += b - a;
        ++n_part_launches;
      }
      ms += t_hi - t_lo;
      ++n;
      if (first_a < 0.0) first_a = t0;
      last_a = t0;
    }
    used = 0;
    return GD_OK;
  }
};

int device() { return g_device; }
int n_cu() { return g_cu; }

gd_status ensure_device() {
  if (g_device >= 0) {
    hipError_t e = hipSetDevice(g_device);
    return e == hipSuccess ? GD_OK : hip_fail(e, "hipSetDevice");
  }
  return gd_init(0);
}

// ---- device arena: one hipMalloc per job, carved into 256-byte aligned pieces
struct Arena {
  size_t off = 0;
  std::vector<std::pair<void **, size_t>> reqs;
  template <class T>
  void add(T **p, size_t n) {
    reqs.push_back({(void **)p, (n * sizeof(T) + 255) / 256 * 256});
    off += reqs.back().second;
  }
  gd_status commit(void **base) {
    *base = nullptr;
    if (off == 0) return GD_OK;
    hipError_t e = hipMalloc(base, off);
    if (e != hipSuccess) return hip_fail(e, "hipMalloc");
    size_t o = 0;
    for (auto &r : reqs) {
      *r.first = (char *)*base + o;
      o += r.second;
    }
    return GD_OK;
  }
};

// Exact float threshold T on r^2 such that sqrtf(r2) <= pmf0  <=>  r2 <= T
// (the reference tests dst - pmf0 <= 0 with dst = sqrtf(r2),
// energy_prt_v1.C:88,100).  sqrtf is correctly rounded and monotone.
static float sqrt_threshold(float pmf0) {
  if (!(pmf0 >= 0.0f)) return -1.0f;  // never true for r2 >= 0
  float x = (float)((double)pmf0 * (double)pmf0);
  while (std::sqrt(x) > pmf0) x = std::nextafter(x, 0.0f);
  for (;;) {
    const float n = std::nextafter(x, INFINITY);
    if (std::sqrt(n) <= pmf0 && std::isfinite(n))
      x = n;
    else
      break;
  }
  return x;
}

// Far-field threshold on r^2 for one (ligand type, point type) pair: from it on
// the PMF exponent (6 - r/2)(r - pmf0) log2(e) stays below -26 (so 1 + exp2 of it
// rounds to 1 in FP32 even with the kernel's rounding of the exponent) and
// el1 r >= 1 (the electrostatic factor is 1/(el1 r)); both hold for every larger r
// because the exponent decreases beyond r = 6 + pmf0/2.  Rounded up.
float far_r2_threshold(double pmf0, double el1) {
  if (!(el1 > 0.0)) return std::numeric_limits<float>::infinity();
  const double log2e = 1.44269504088896340736;
  // -log2(e)/2 r^2 + log2(e)(6 + pmf0/2) r - 6 log2(e) pmf0 + 26 = 0, larger root
  const double qa = -0.5 * log2e, qb = log2e * (6.0 + 0.5 * pmf0), qc = -6.0 * log2e * pmf0 + 26.0;
  const double disc = qb * qb - 4.0 * qa * qc;
  double r = disc > 0.0 ? (-qb - std::sqrt(disc)) / (2.0 * qa) : 6.0 + 0.5 * pmf0;
  r = std::max(r, 6.0 + 0.5 * pmf0) * (1.0 + 1e-6);
  while (log2e * (6.0 - 0.5 * r) * (r - pmf0) > -26.0) r *= 1.0 + 1e-6;
  r = std::max(r, (1.0 / el1) * (1.0 + 1e-6));
  const float f = (float)(r * r);
  return (double)f >= r * r ? f : std::nextafter(f, std::numeric_limits<float>::infinity());
}

// The row threshold of the pair loop's near branch: the far-field threshold
// raised to cover the terms that branch also holds, so that a wave whose lanes
// are all beyond it skips exact zeros only:
//   hydrophobic, r^2 <= 81; psp, r^2 <= psp_thr (negative: no psp term);
//   H-bond (hb), hdb1 2^-q with q = ((r - hdb0) c)^2, c = hdb1 sqrt(log2(e)/2):
//   2^-q is exactly 0 in FP32 for q >= 151, and q >= 160 from r = hdb0 + sqrt(160) / c on.
static float near_r2_threshold(double pmf0, double el1, float psp_thr, bool hb, double hdb0,
                               double c) {
  double r2n = far_r2_threshold(pmf0, el1);
  r2n = std::max(r2n, 81.0 * (1.0 + 1e-6));
  if (psp_thr >= 0.0f) r2n = std::max(r2n, (double)psp_thr * (1.0 + 1e-6));
  if (hb && c > 0.0) {
    const double rh = hdb0 + std::sqrt(160.0) / c;
    r2n = std::max(r2n, rh * rh * (1.0 + 1e-5));
  }
  float f = (float)r2n;
  if ((double)f < r2n) f = std::nextafter(f, std::numeric_limits<float>::infinity());
  return f;
}

// ---------------------------------------------------------------------------
// Tiling: ligand chunk size lc (kernel template), protein tile ptile.  Looked
// up by size bucket in the tuned table (gd_tiling_table.h), else the rule
// below; either way a function of the job (and the device's CU count) only, so
// a job's reduction order, and hence its bits, is the same in every process,
// alone or in a batch.
int lg2_floor(int x) {
  int b = 0;
  while (b < 30 && (2 << b) <= x) ++b;
  return b;
}

// One-job tilings are keyed on the ligand's 4-atom chunk count, ceil(L / 4):
// on two streams the best tile count keeps each half-launch's items (chunks x
// tile groups x replica blocks) near the machine's group slots, so it follows
// the chunk count exactly rather than a size class of L.
int chunk_key(int L) { return (std::max(1, L) + 3) / 4; }

static const GdTuned *tuned_entry(int mode, int L, int P, int R) {
  const int lgL = mode == GD_TUNE_PLAIN ? chunk_key(L) : lg2_floor(std::max(1, L)),
            lgP = lg2_floor(std::max(1, P)), lgR = lg2_floor(std::max(1, R));
  for (const GdTuned &t : kTunedTable) {
    if (t.mode != mode) continue;
    if (mode == GD_TUNE_WAVES ||
        (t.lgL == lgL && t.lgP == lgP && (mode == GD_TUNE_SHARED || t.lgR == lgR)))
      return &t;
  }
  return nullptr;
}

// ptile giving at least nP tiles of P points (the kernel rounds nP up to a
// multiple of GD_GROUP)
static int ptile_for_tiles(int P, int nP) {
  nP = std::max(1, std::min(nP, P));
  return (P + nP - 1) / nP;
}

void default_tiling(int L, int P, int R, int &lc, int &ptile) {
  if (const GdTuned *t = tuned_entry(GD_TUNE_PLAIN, L, P, R)) {
    lc = t->lc;
    ptile = ptile_for_tiles(P, t->value);
    return;
  }
  // 4 atoms per wave keeps the pair kernel at ~62 VGPRs (8 waves per SIMD);
  // ~22 waves per SIMD over the launch (about three waves per slot) balanced
  // per-tile overhead (KDE and MCS shares, partial sums) against the launch's
  // tail in a sweep of tile counts on a 3000-point, 1760-replica job
  lc = 4;
  const int nL = (L + lc - 1) / lc;
  const int nblk = (R + 63) / 64;
  const int simds = 4 * (g_cu > 0 ? g_cu : 256);
  const int target_waves = 22 * simds;
  int nP = std::max(1, target_waves / std::max(1, nblk * nL));
  nP = std::min(nP, std::max(1, P / 16));
  nP = (nP + GD_GROUP - 1) / GD_GROUP * GD_GROUP;
  ptile = (P + nP - 1) / nP;
}

// Tiling of a job inside shared launches (batches, serving): 4 atoms per lane
// (one kernel template for every job of a launch) and the bucket's tile size,
// 64 points where the table has none.
int shared_ptile(int L, int P) {
  if (const GdTuned *t = tuned_entry(GD_TUNE_SHARED, L, P, 0)) return std::min(P, t->value);
  return std::min(P, 64);
}

// Resident waves per CU of the persistent pair kernel for lc atoms per lane:
// the tuned value for 4 atoms, else as many 8-wave groups as the registers
// allow (4 atoms: ~60 VGPRs, 8 waves per SIMD).
int pair_waves_per_cu(int lc) {
  if (lc == 4)
    if (const GdTuned *t = tuned_entry(GD_TUNE_WAVES, 0, 0, 0)) return t->value;
  return lc == 4 ? 32 : lc == 8 ? 20 : 8;
}

static gd_status alloc_partials(gd_job *j, GdJob &g, int cap_rp) {
  // partials depend on the tiling; they live in their own allocation
  if (j->d_part) {
    hipFree(j->d_part);
    j->d_part = nullptr;
  }
  Arena a;
  const size_t nS = (size_t)g.nL * g.nG;
  a.add(&g.part_lin, (size_t)GD_NLIN * nS * cap_rp);
  a.add(&g.part_hpc, (size_t)g.L * g.nG * cap_rp);
  a.add(&g.part_mcs, (size_t)std::max(1, g.M) * g.nL * cap_rp);
  a.add(&g.fin_part, (size_t)(cap_rp / 64) * GD_RK * 8 * 64);
  gd_status st = a.commit(&j->d_part);
  j->part_bytes = st == GD_OK ? a.off : 0;
  return st;
}

// Staging memory for an upload on the job's stream, held until sync_job_struct
// has waited for it.
static gd_status stage(gd_job *j, size_t bytes, HostBuf **out) {
  std::unique_ptr<HostBuf> b(new HostBuf);
  const gd_status st = b->acquire(bytes, true);
  if (st != GD_OK) return st;
  *out = b.get();
  j->staged.push_back(std::move(b));
  return GD_OK;
}

// Device order of the protein points for the job's tile count: class by
// class, tile b of nP reads points pcls[c] + b, + nP, ... (strided, see the
// pair kernel).  The class's points sorted by (type, spread) are dealt out so
// that each tile's points are one contiguous piece of that list: few type
// changes per tile (the pair kernel keeps a chunk's force-field rows across a
// type), and, by the spread order, a representative mix of distances.  The
// order changes only summation order.
static gd_status layout_points(gd_job *j) {
  GdJob &g = j->h;
  const int P = g.P, nP = g.nP, np = g.n_prt;
  const std::vector<int> &ord = j->src_order;
  std::vector<int> porder(P);
  for (int c = 0; c < 4; ++c) {
    const int lo = g.pcls[c], n = g.pcls[c + 1] - lo, q = n / nP, r = n % nP;
    for (int i = 0; i < n; ++i) {
      int b, k;  // column (tile) and row of list element i: columns are filled in turn
      if (i < r * (q + 1)) {
        b = i / (q + 1), k = i % (q + 1);
      } else {
        const int i2 = i - r * (q + 1);
        b = r + i2 / q, k = i2 % q;
      }
      porder[lo + k * nP + b] = ord[lo + i];
    }
  }
  const size_t nty1 = j->src_pspv.size() / (size_t)P;
  // gathered into staging memory in the device's layout (pcoord, pattr and pspv
  // follow each other) and sent in one copy; sync_job_struct waits for it
  HostBuf *buf;
  gd_status st = stage(j, (size_t)((const char *)g.pspv - (const char *)g.pcoord) + j->src_pspv.size() * sizeof(float),
                       &buf);
  if (st != GD_OK) return st;
  char *h = (char *)buf->p;
  float4 *pco = (float4 *)h, *pattr = (float4 *)(h + ((const char *)g.pattr - (const char *)g.pcoord));
  float *pspv = (float *)(h + ((const char *)g.pspv - (const char *)g.pcoord));
  for (int i = 0; i < np; ++i)
    for (int q2 = 0; q2 < P; ++q2) pco[(size_t)i * P + q2] = j->src_pco[(size_t)i * P + porder[q2]];
  for (int q2 = 0; q2 < P; ++q2) pattr[q2] = j->src_pattr[porder[q2]];
  for (size_t t = 0; t < nty1; ++t)
    for (int q2 = 0; q2 < P; ++q2) pspv[t * P + q2] = j->src_pspv[t * P + porder[q2]];
  const size_t bytes = (size_t)((const char *)(g.pspv + j->src_pspv.size()) - (const char *)g.pcoord);
  hipError_t e;
  if ((e = hipStreamSynchronize(j->stream)) != hipSuccess ||
      (e = hipMemcpyAsync((void *)g.pcoord, h, bytes, hipMemcpyHostToDevice, j->stream)) != hipSuccess)
    return hip_fail(e, "point layout upload");
  j->laid_nP = nP;
  return GD_OK;
}

gd_status apply_tiling(gd_job *j, int lc, int ptile) {
  GdJob &g = j->h;
  if (lc != 4 && lc != 8 && lc != 16) return GD_ERR_ARG;
  ptile = std::max(1, std::min(ptile, g.P));
  g.lc = lc;
  g.nL = (g.L + lc - 1) / lc;
  g.ptile = ptile;
  // protein tiles (tile b takes the points b, b + nP, ... of each class): a
  // multiple of GD_GROUP so that a work group's waves take tiles 8g .. 8g + 7
  const int nP = (g.P + ptile - 1) / ptile;
  g.nP = (nP + GD_GROUP - 1) / GD_GROUP * GD_GROUP;
  g.nG = g.nP / GD_GROUP;
  gd_status st = alloc_partials(j, g, g.Rp);
  if (st != GD_OK) return st;
  if (g.nP != j->laid_nP && (st = layout_points(j)) != GD_OK) return st;
  // One item per work group: (replica block, chunk, tile group).  Chunks go in
  // order of decreasing KDE work (anchors of their atoms' bins), the only part
  // of an item's cost that differs between chunks, so the launch ends with its
  // cheapest items; within a chunk, tile groups, then replica blocks, so items
  // dispatched together read the same force-field rows and KDE anchors.  The
  // order changes no result: every item writes its own partial-sum slot.
  // (Measured on a 3,000-point, 1,760-replica job: 117.3 us against 119.8 us for
  // replica-block-major order, and 121.0 us for the reverse chunk order.)
  std::vector<int> chunk(g.nL), wkde(g.nL, 0);
  for (int a = 0; a < g.nL; ++a) {
    chunk[a] = a;
    for (int l = a * lc; l < std::min((a + 1) * lc, g.L); ++l) wkde[a] += j->atom_kde[l];
  }
  std::stable_sort(chunk.begin(), chunk.end(), [&](int x, int y) { return wkde[x] > wkde[y]; });
  j->items.clear();
  for (int a : chunk)
    for (int gi = 0; gi < g.nG; ++gi)
      for (int rb = 0; rb < g.Rp; rb += 64) j->items.push_back({0, rb, a, gi});
  return GD_OK;
}

// ---------------------------------------------------------------------------
// pmf1 summed over every (atom, point) pair, atom by atom, in double.  By the
// counts of the types where that is the same number: if the magnitudes sum to
// less than 2^53 units in the last place of the smallest value, every partial sum
// in any order is exact.
static double pmf_sum(const gd_job_desc *d) {
  const gd_enepara *e = d->ene;
  std::vector<int> nl(GD_NLT, 0), np(GD_NPT, 0);
  for (int l = 0; l < d->lig_natom; ++l) ++nl[d->lig_t[l]];
  for (int p = 0; p < d->prt_npoint; ++p) ++np[d->prt_t[p]];
  double sum = 0.0, mag = 0.0, ulp = INFINITY;
  for (int a = 0; a < GD_NLT; ++a)
    for (int b = 0; b < GD_NPT; ++b) {
      const float v = e->pmf1[a][b];
      const double n = (double)nl[a] * np[b];
      if (n == 0.0 || v == 0.0f) continue;
      int ex;
      std::frexp(v, &ex);
      ulp = std::min(ulp, std::ldexp(1.0, ex - 24));
      mag += std::fabs((double)v) * n;
      sum += v * n;
    }
  if (mag < 4503599627370496.0 * ulp) return sum;  // 2^52: one bit to spare for mag's own rounding
  double sp = 0.0;
  for (int l = 0; l < d->lig_natom; ++l)
    for (int p = 0; p < d->prt_npoint; ++p) sp += e->pmf1[d->lig_t[l]][d->prt_t[p]];
  return sp;
}

// Pack a complex into the device layout.
static gd_status pack_job(const gd_job_desc *d, gd_job *j) {
  const int L = d->lig_natom, P = d->prt_npoint, K = d->kde_npoint, M = d->mcs_nrow;
  const int nl = d->n_lig, np = d->n_prt, nt = d->n_tmp;
  if (L < 1 || P < 1 || K < 0 || M < 0 || nl < 1 || np < 1 || nt < 1) return GD_ERR_ARG;
  if (!d->lig_x || !d->lig_y || !d->lig_z || !d->lig_t || !d->lig_c || !d->prt_x || !d->prt_y ||
      !d->prt_z || !d->prt_t || !d->prt_c || !d->prt_cdc || !d->prt_seq3r || !d->prt_hpp ||
      !d->prt_ele || !d->ene || !d->minus_beta || (K > 0 && (!d->kde_t || !d->kde_x)) ||
      (M > 0 && (!d->mcs_x || !d->mcs_tcc)) || (d->psp_ncol > 0 && !d->psp))
    return GD_ERR_ARG;
  const long long R64 = (long long)nl * np * nt;
  if (R64 > (1 << 26) || L > 4096 || P > (1 << 22)) return GD_ERR_SIZE;
  // the pair kernel addresses a protein conformer's points by a 32-bit byte offset
  if ((long long)np * P * 16 > 0xFFFFFFFFLL) {
    set_error("protein conformers x points over 2^28");
    return GD_ERR_SIZE;
  }
  for (int l = 0; l < L; ++l)
    if (d->lig_t[l] < 0 || d->lig_t[l] >= GD_NLT) {
      set_error("ligand atom type outside 0..23 (BADKDE)");
      return GD_ERR_TYPE;
    }
  for (int p = 0; p < P; ++p)
    if (d->prt_t[p] < 0 || d->prt_t[p] >= GD_NPT) {
      set_error("protein point type outside 0..30");
      return GD_ERR_TYPE;
    }
  const int R = (int)R64, Rp = (R + 63) / 64 * 64;
  const gd_enepara *e = d->ene;
  GdJob g;
  std::memset(&g, 0, sizeof g);
  g.L = L, g.P = P, g.K = K, g.M = M, g.n_lig = nl, g.n_prt = np, g.n_tmp = nt, g.R = R, g.Rp = Rp;

  // distinct ligand types of the job -> parameter-table rows
  std::vector<int> types;
  std::vector<int> trow(GD_NLT, -1);
  for (int l = 0; l < L; ++l)
    if (trow[d->lig_t[l]] < 0) {
      trow[d->lig_t[l]] = (int)types.size();
      types.push_back(d->lig_t[l]);
    }
  const int nty = (int)types.size();
  g.n_types = nty;
  // atom stride padded to 16 (the widest ligand chunk): the pair kernel runs whole
  // chunks; padding atoms use row block nty, all zero with a NaN psp threshold
  // (no psp, no H-bond), charge 0, no KDE bins and no MCS entries
  const int Ls = (L + 15) / 16 * 16;
  g.Ls = Ls;
  std::vector<float> ptab((size_t)(nty + 1) * GD_PTAB_PT * GD_PTAB_W, 0.0f);
  for (int pt = 0; pt < GD_PTAB_PT; ++pt) {
    ptab[((size_t)nty * GD_PTAB_PT + pt) * GD_PTAB_W + 0] = std::numeric_limits<float>::infinity();
    ptab[((size_t)nty * GD_PTAB_PT + pt) * GD_PTAB_W + 5] = std::numeric_limits<float>::quiet_NaN();
  }
  const double log2e = 1.44269504088896340736;
  const double hdb_c = std::sqrt(0.5 * log2e);
  for (int ti = 0; ti < nty; ++ti) {
    const int lt = types[ti];
    for (int pt = 0; pt < GD_NPT; ++pt) {
      float *o = &ptab[((size_t)ti * GD_PTAB_PT + pt) * GD_PTAB_W];
      const double pmf0 = e->pmf0[lt][pt];
      // LJ over p1a: w = 1 / p1a and -q = -p2a / p1a; a row without LJ
      // (p1a = p2a = 0) has w = inf, which makes the term 0
      const double p1a = e->p1a[lt][pt], p2a = e->p2a[lt][pt];
      if (p1a == 0.0 && p2a != 0.0) {
        set_error("LJ parameters with p1a = 0 and p2a != 0 are not supported");
        return GD_ERR_ARG;
      }
      o[0] = p1a != 0.0 ? (float)(1.0 / p1a) : std::numeric_limits<float>::infinity();
      o[1] = p1a != 0.0 ? (float)(-p2a / p1a) : 0.0f;
      // negated PMF exponent -(6 - r/2)(r - pmf0) log2(e) = log2(e)/2 r^2 + B r + C
      o[2] = (float)(-log2e * (6.0 + 0.5 * pmf0));
      o[3] = (float)(6.0 * log2e * pmf0);
      o[4] = e->pmf1[lt][pt];
      // psp cutoff on r^2 (compared against |o[5]|; NaN: never); the sign bit
      // marks the pairs whose H-bond term is on
      const float thr = sqrt_threshold(e->pmf0[lt][pt]);
      const bool hb = e->hdb0[lt][pt] > 0.1f;
      o[5] = std::copysign(thr >= 0.0f ? thr : std::numeric_limits<float>::quiet_NaN(), hb ? -1.0f : 1.0f);
      // H-bond: hdb1 exp(-(r - hdb0)^2 hdb1^2 / 2), the raw parameters (the
      // kernel forms the exponent in FP64); rows with hdb0 <= 0.1 are off.  The
      // near threshold covers q = ((r - hdb0) c)^2 < 160, c = hdb1 sqrt(log2(e)/2)
      const double c = (double)e->hdb1[lt][pt] * hdb_c;
      o[6] = hb ? e->hdb1[lt][pt] : 0.0f;
      o[7] = hb ? e->hdb0[lt][pt] : 0.0f;
      o[8] = near_r2_threshold(pmf0, e->el1, thr, hb, e->hdb0[lt][pt], hb ? c : 0.0);
    }
  }
  // Protein points, kept in source order: the device order depends on the tile
  // count and is laid out by layout_points (called from apply_tiling).
  // Classes: cdc flag + 2 x class-2 flag.
  {
    int nc[4] = {0, 0, 0, 0};
    auto cls = [&](int p) { return (d->prt_cdc[p] == 1 ? 1 : 0) + (d->prt_c[p] == 2 ? 2 : 0); };
    for (int p = 0; p < P; ++p) ++nc[cls(p)];
    g.pcls[0] = 0;
    for (int c = 0; c < 4; ++c) g.pcls[c + 1] = g.pcls[c] + nc[c];
    j->src_key.resize(P);
    for (int p = 0; p < P; ++p) j->src_key[p] = cls(p) * GD_PTAB_PT + d->prt_t[p];
    // within a (class, type) group: by the bit-reversed rank of the distance to the
    // pocket centre (protein conformer 0), a low-discrepancy order in which any
    // run of consecutive points spans near and far points evenly
    std::vector<uint64_t> rec(P), tmp(P);  // distance bits, point
    for (int p = 0; p < P; ++p) {
      const float dx = d->prt_x[p] - d->pocket_center[0], dy = d->prt_y[p] - d->pocket_center[1],
                  dz = d->prt_z[p] - d->pocket_center[2];
      const float dist = dx * dx + dy * dy + dz * dz;  // >= 0: ordered as its bits
      uint32_t u;
      std::memcpy(&u, &dist, 4);
      rec[p] = (uint64_t)u << 32 | (uint32_t)p;
    }
    // stable radix passes over the distance, then the key
    const auto pass = [&](const auto &digit, int n) {
      std::vector<int> at(n + 1, 0);
      for (int p = 0; p < P; ++p) ++at[digit(rec[p]) + 1];
      for (int k = 0; k < n; ++k) at[k + 1] += at[k];
      for (int p = 0; p < P; ++p) tmp[at[digit(rec[p])]++] = rec[p];
      rec.swap(tmp);
    };
    for (int sh = 32; sh < 64; sh += 11) pass([&](uint64_t v) { return (int)(v >> sh & 2047); }, 2048);
    pass([&](uint64_t v) { return j->src_key[(uint32_t)v]; }, 4 * GD_PTAB_PT);
    std::vector<int> ord(P);
    for (int p = 0; p < P; ++p) ord[p] = (int)(uint32_t)rec[p];
    j->src_order.resize(P);
    for (int i = 0; i < P;) {
      int e = i;
      while (e < P && j->src_key[ord[e]] == j->src_key[ord[i]]) ++e;
      int bits = 0;
      while ((1 << bits) < e - i) ++bits;
      // in the order of the bit-reversed rank
      int o = i;
      for (unsigned rv = 0; rv < (1u << bits); ++rv) {
        unsigned v = 0;
        for (int t = 0; t < bits; ++t) v |= ((rv >> t) & 1u) << (bits - 1 - t);
        if ((int)v < e - i) j->src_order[o++] = ord[i + (int)v];
      }
      i = e;
    }
  }
  j->src_pspv.assign((size_t)(nty + 1) * P, 0.0f);  // last row: padding atoms (zero)
  j->src_pattr.resize(P);
  for (int p = 0; p < P; ++p) {
    const int c = d->prt_c[p];
    int fl = d->prt_t[p] | (d->prt_cdc[p] == 1 ? GD_PF_CDC : 0) | (c == 2 ? GD_PF_CLS2 : 0);
    float flf;
    std::memcpy(&flf, &fl, 4);
    j->src_pattr[p] = make_float4(d->prt_ele[p], d->prt_hpp[p], flf, 0.0f);
    if (c == 2) {
      const int res = d->prt_seq3r[p];
      for (int ti = 0; ti < nty; ++ti)
        j->src_pspv[(size_t)ti * P + p] =
            (res >= 0 && res < d->psp_ncol) ? d->psp[(size_t)types[ti] * d->psp_ncol + res] : 0.0f;
    }
  }
  // KDE bins (anchors sorted by type)
  std::vector<float4> kde(std::max(1, K));
  for (int k = 0; k < K; ++k) {
    if (k > 0 && d->kde_t[k] < d->kde_t[k - 1]) {
      set_error("KDE points must be sorted by type");
      return GD_ERR_ARG;
    }
    kde[k] = make_float4(d->kde_x[k], d->kde_y[k], d->kde_z[k], 0.0f);
  }
  std::vector<GdAtom> atoms(Ls);
  for (int l = L; l < Ls; ++l) {
    GdAtom &a = atoms[l];
    std::memset(&a, 0, sizeof a);
    a.tidx = nty;
    a.hpl1 = 1.0f;
  }
  j->atom_kde.assign(L, 0);
  for (int l = 0; l < L; ++l) {
    const int lt = d->lig_t[l];
    GdAtom &a = atoms[l];
    a.tidx = trow[lt];
    a.q = d->lig_c[l];
    const int b = K ? (int)(std::lower_bound(d->kde_t, d->kde_t + K, lt) - d->kde_t) : 0;
    const int en = K ? (int)(std::upper_bound(d->kde_t, d->kde_t + K, lt) - d->kde_t) : 0;
    a.kde_b = b;
    a.kde_e = en;
    j->atom_kde[l] = en - b;
    a.kde_inv_n = en > b ? 1.0f / (float)(en - b) : 0.0f;
    a.hpl0 = e->hpl0[lt];
    a.hpl1 = e->hpl1[lt];
    a.hpl2 = e->hpl2[lt];
  }
  std::vector<float4> mcs((size_t)std::max(1, M) * Ls, make_float4(0.0f, 0.0f, 0.0f, 0.0f));
  std::vector<float2> mcsrow(std::max(1, M));
  for (int m = 0; m < M; ++m) {
    int n = 0;
    for (int l = 0; l < L; ++l) {
      const size_t i = (size_t)m * L + l;
      const bool v = d->mcs_x[i] != GD_MCS_INVALID;
      n += v;
      if (v) mcs[(size_t)m * Ls + l] = make_float4(d->mcs_x[i], d->mcs_y[i], d->mcs_z[i], 1.0f);
    }
    mcsrow[m] = make_float2(d->mcs_tcc[m], (float)n);
  }
  std::vector<float4> lig0((size_t)nl * L);
  for (int i = 0; i < nl; ++i)
    for (int l = 0; l < L; ++l) {
      const size_t q = (size_t)i * L + l;
      lig0[q] = make_float4(d->lig_x[q], d->lig_y[q], d->lig_z[q], 0.0f);
    }
  j->src_pco.resize((size_t)np * P);
  for (size_t q = 0; q < (size_t)np * P; ++q)
    j->src_pco[q] = make_float4(d->prt_x[q], d->prt_y[q], d->prt_z[q], 0.0f);
  // pmf1 summed over every (atom, point) pair: the PMF term of a pose is this
  // constant minus the pair kernel's corrections
  {
    g.pmf_all = (float)pmf_sum(d);
  }
  // scalars
  g.lj0 = e->lj0, g.lj1 = e->lj1, g.el0 = e->el0, g.el1 = e->el1, g.a1 = e->a1, g.b1 = e->b1;
  g.inv_el1 = 1.0f / e->el1;
  g.kde2l = e->kde2 * 1.44269504088896340736f;
  g.kde3_inv = 1.0f / e->kde3;
  g.inv_L = 1.0f / (float)L;
  for (int i = 0; i < 3; ++i) {
    g.center[i] = d->lig_center[i];
    g.pocket[i] = d->pocket_center[i];
    g.cp[i] = (float)((double)d->lig_center[i] - (double)d->pocket_center[i]);
  }
  for (int i = 0; i < 10; ++i) g.a_para[i] = e->a_para[i], g.b_para[i] = e->b_para[i], g.w[i] = e->w[i];

  // device memory: constant tables + replica state
  Arena a;
  float4 *d_lig0, *d_pco, *d_pattr, *d_kde, *d_mcs;
  GdAtom *d_atoms;
  float *d_ptab, *d_pspv, *d_mb;
  float2 *d_mcsrow;
  a.add(&d_lig0, lig0.size());  // the tables, to d_mb: one upload
  a.add(&d_atoms, atoms.size());
  a.add(&d_ptab, ptab.size());
  a.add(&d_kde, kde.size());
  a.add(&d_mcs, mcs.size());
  a.add(&d_mcsrow, mcsrow.size());
  a.add(&d_mb, (size_t)nt);
  a.add(&d_pco, j->src_pco.size());  // the points: another (layout_points)
  a.add(&d_pattr, j->src_pattr.size());
  a.add(&d_pspv, j->src_pspv.size());
  a.add(&g.mm, (size_t)6 * Rp);
  a.add(&g.prop, (size_t)6 * Rp);
  a.add(&g.en, (size_t)10 * Rp);
  a.add(&g.ligi, (size_t)Rp);
  a.add(&g.prti, (size_t)Rp);
  a.add(&g.tmpi, (size_t)Rp);
  a.add(&g.acc, (size_t)Rp);
  a.add(&g.nacc, (size_t)Rp);
  a.add(&g.nexc, (size_t)Rp);
  a.add(&g.nswp, (size_t)2 * Rp);
  a.add(&g.swp_e, (size_t)Rp);
  a.add(&g.best, (size_t)Rp);
  a.add(&g.own, (size_t)nl * np * nt);
  a.add(&g.coords, (size_t)3 * L * Rp);
  a.add(&g.rec_n, (size_t)2 * Rp);
  a.add(&g.ev_terms, (size_t)10 * Rp);
  a.add(&g.ev_raw, (size_t)9 * Rp);
  a.add(&g.wq, 64);
  a.add(&j->ev.job, 1);
  a.add(&j->ev.ligi, (size_t)Rp);
  a.add(&j->ev.prti, (size_t)Rp);
  a.add(&j->ev.prop, (size_t)6 * Rp);
  gd_status st = a.commit(&j->d_base);
  if (st != GD_OK) return st;
  j->bytes = a.off;
  g.lig0 = d_lig0, g.atoms = d_atoms, g.pcoord = d_pco, g.pattr = d_pattr, g.ptab = d_ptab;
  g.pspv = d_pspv, g.kde = d_kde, g.mcs = d_mcs, g.mcsrow = d_mcsrow, g.minus_beta = d_mb;
  const size_t bytes = (size_t)((char *)(d_mb + nt) - (char *)d_lig0);
  HostBuf *buf;
  if ((st = stage(j, bytes, &buf)) != GD_OK) return st;
  const auto put = [&](const void *dst, const void *src, size_t n) {
    std::memcpy((char *)buf->p + ((const char *)dst - (const char *)d_lig0), src, n);
  };
  put(d_lig0, lig0.data(), lig0.size() * sizeof(float4));
  put(d_atoms, atoms.data(), atoms.size() * sizeof(GdAtom));
  put(d_ptab, ptab.data(), ptab.size() * sizeof(float));
  put(d_kde, kde.data(), kde.size() * sizeof(float4));
  put(d_mcs, mcs.data(), mcs.size() * sizeof(float4));
  put(d_mcsrow, mcsrow.data(), mcsrow.size() * sizeof(float2));
  put(d_mb, d->minus_beta, (size_t)nt * sizeof(float));
  const hipError_t e2 = hipMemcpyAsync(d_lig0, buf->p, bytes, hipMemcpyHostToDevice, j->stream);
  if (e2 != hipSuccess) return hip_fail(e2, "table upload");
  j->h = g;
  return GD_OK;
}

// Device bytes gd_job_create allocates for a descriptor (tables, replica
// state, partial sums under the default tiling, work lists).
// Device bytes of a complex under the plain tiling, or (shared) under the
// tiling of shared launches.
size_t footprint(const gd_job_desc *d, bool shared) {
  if (!d || d->lig_natom < 1 || d->prt_npoint < 1 || d->n_lig < 1 || d->n_prt < 1 || d->n_tmp < 1)
    return 0;
  const size_t L = d->lig_natom, P = d->prt_npoint, K = d->kde_npoint, M = d->mcs_nrow;
  const size_t nl = d->n_lig, np = d->n_prt, nt = d->n_tmp;
  const size_t R = nl * np * nt, Rp = (R + 63) / 64 * 64;
  auto a = [](size_t bytes) { return (bytes + 255) / 256 * 256; };
  std::vector<int> seen(GD_NLT, 0);
  size_t nty = 0;
  for (size_t l = 0; l < L; ++l)
    if (d->lig_t[l] >= 0 && d->lig_t[l] < GD_NLT && !seen[d->lig_t[l]]++) ++nty;
  const size_t Ls = (L + 15) / 16 * 16;
  size_t b = a(nl * L * 16) + a(Ls * sizeof(GdAtom)) + a(np * P * 16) + a(P * 16) +
             a((nty + 1) * GD_PTAB_PT * GD_PTAB_W * 4) + a((nty + 1) * P * 4) +
             a(std::max<size_t>(1, K) * 16) + a(std::max<size_t>(1, M) * Ls * 16) +
             a(std::max<size_t>(1, M) * 8) + a(nt * 4);
  b += a(6 * Rp * 4) * 2 + a(10 * Rp * 4) + a(Rp * 4) * 6 + a(2 * Rp * 4) + a(Rp * 4) +
       a(Rp * 4) + a(nl * np * nt * 4) +
       a(3 * L * Rp * 4) + a(2 * Rp * 4) + a(10 * Rp * 4) + a(9 * Rp * 4) + a(64 * 4) + a(sizeof(GdJob)) +
       a(Rp * 4) * 2 + a(6 * Rp * 4);
  int lc, ptile;
  if (shared) {
    lc = 4;
    ptile = shared_ptile((int)L, (int)P);
  } else {
    default_tiling((int)L, (int)P, (int)R, lc, ptile);
  }
  const size_t nL = (L + lc - 1) / lc, nP0 = (P + ptile - 1) / ptile;
  const size_t nG = (nP0 + GD_GROUP - 1) / GD_GROUP;
  b += a(GD_NLIN * nL * nG * Rp * 4) + a(L * nG * Rp * 4) + a(std::max<size_t>(1, M) * nL * Rp * 4) +
       a((Rp / 64) * GD_RK * 8 * 64 * 4);
  b += (Rp / 64) * nL * nG * sizeof(GdItem) + (Rp / 64) * sizeof(GdBlock) + 512;
  return b;
}

// The stepping kernel's lists, made at the first run that steps by it and given
// back with the job's other lists.
static void chain_drop(gd_job *j) {
  if (j->d_chain) hipFree(j->d_chain);
  j->d_chain = nullptr;
  j->chain_bytes = 0;
}

static gd_status chain_make(gd_job *j) {
  if (j->d_chain) return GD_OK;
  ChainList &cl = j->chain;
  std::vector<GdItem> items;
  for (const GdItem &it : j->items)
    if (it.rb == 0) items.push_back(it);
  std::vector<GdChainBlock> blocks;
  for (int rb = 0; rb < j->h.Rp; rb += 64) blocks.push_back({0, rb, 0, (int)items.size()});
  auto up = [](size_t b) { return (b + 255) / 256 * 256; };
  const size_t bi = items.size() * sizeof(GdItem), bb = blocks.size() * sizeof(GdChainBlock),
               bs = chain_sync_bytes(cl.n_blocks), bq = cl.queue_bytes(), bk = keep_bytes(cl.n_blocks);
  const size_t all = up(bi) + up(bb) + up(bs) + up(bq) + up(bk);
  hipError_t e = hipMalloc(&j->d_chain, all);
  if (e != hipSuccess) return hip_fail(e, "hipMalloc stepping lists");
  j->chain_bytes = all;
  char *base = (char *)j->d_chain;
  cl.d_items = (GdItem *)base;
  cl.d_blocks = (GdChainBlock *)(base + up(bi));
  cl.d_sync = (unsigned *)(base + up(bi) + up(bb));
  cl.d_queue = (unsigned long long *)(base + up(bi) + up(bb) + up(bs));
  j->d_keep = (unsigned *)(base + up(bi) + up(bb) + up(bs) + up(bq));
  j->keep_used = false;
  cl.epoch = cl.steps = 0;
  cl.stale = false;
  if ((e = hipMemcpyAsync(base, items.data(), bi, hipMemcpyHostToDevice, j->stream)) != hipSuccess ||
      (e = hipMemcpyAsync(base + up(bi), blocks.data(), bb, hipMemcpyHostToDevice, j->stream)) != hipSuccess ||
      (e = hipMemsetAsync(cl.d_sync, 0, up(bs) + up(bq) + GD_KEEP_HEAD * sizeof(unsigned), j->stream)) != hipSuccess ||
      (e = hipStreamSynchronize(j->stream)) != hipSuccess) {
    chain_drop(j);
    return hip_fail(e, "stepping list upload");
  }
  return GD_OK;
}

gd_status sync_job_struct(gd_job *j) {
  std::vector<GdBlock> blocks;
  for (int rb = 0; rb < j->h.Rp; rb += 64) blocks.push_back({0, rb});
  j->n_blocks = (int)blocks.size();
  j->n_items = (int)j->items.size();
  // the plain path's stepping parts: n_streams contiguous ranges of the
  // blocks, as even as the block count allows, each with the job's items of
  // its blocks (in the job's order)
  const int np = std::max(1, std::min(j->n_streams, j->n_blocks));
  j->n_parts = np;
  std::vector<GdItem> part_items;
  for (int k = 0; k < np; ++k) {
    j->b0_part[k] = (int)((long)j->n_blocks * k / np);
    j->nb_part[k] = (int)((long)j->n_blocks * (k + 1) / np) - j->b0_part[k];
    const int lo = j->b0_part[k] * 64, hi = (j->b0_part[k] + j->nb_part[k]) * 64;
    j->n_items_part[k] = 0;
    for (const GdItem &it : j->items)
      if (it.rb >= lo && it.rb < hi) {
        part_items.push_back(it);
        ++j->n_items_part[k];
      }
  }
  chain_drop(j);
  if (j->d_lists) hipFree(j->d_lists);
  j->d_lists = nullptr;
  auto up = [](size_t b) { return (b + 255) / 256 * 256; };
  const size_t bi = (size_t)j->n_items * sizeof(GdItem), bb = (size_t)j->n_blocks * sizeof(GdBlock),
               bh = part_items.size() * sizeof(GdItem);
  j->lists_bytes = 0;
  hipError_t e = hipMalloc(&j->d_lists, up(bi) + up(bb) + up(bh) + 256);
  if (e != hipSuccess) return hip_fail(e, "hipMalloc lists");
  j->lists_bytes = up(bi) + up(bb) + up(bh) + 256;
  j->d_items = (GdItem *)j->d_lists;
  j->d_blocks = (GdBlock *)((char *)j->d_lists + up(bi));
  j->d_items_part[0] = (GdItem *)((char *)j->d_lists + up(bi) + up(bb));
  for (int k = 1; k < np; ++k) j->d_items_part[k] = j->d_items_part[k - 1] + j->n_items_part[k - 1];
  HostBuf *buf;
  const gd_status st = stage(j, up(bi) + up(bb) + bh, &buf);
  if (st != GD_OK) return st;
  std::memcpy(buf->p, j->items.data(), bi);
  std::memcpy((char *)buf->p + up(bi), blocks.data(), bb);
  if (bh) std::memcpy((char *)buf->p + up(bi) + up(bb), part_items.data(), bh);
  e = hipMemcpyAsync(j->d_lists, buf->p, up(bi) + up(bb) + bh, hipMemcpyHostToDevice, j->stream);
  const hipError_t e2 = hipStreamSynchronize(j->stream);
  j->staged.clear();
  if (e == hipSuccess) e = e2;
  return e == hipSuccess ? GD_OK : hip_fail(e, "list upload");
}

// ---- launches ---------------------------------------------------------------
gd_status launch_pair(int lc, const GdJob *d_jobs, const GdItem *d_items, int n_items,
                      hipStream_t s, int nb, int nb_list) {
  if (n_items <= 0) return GD_OK;
  const dim3 grid(n_items), block(64 * GD_GROUP);  // one group per item
  // At most an item to a CU: three groups to an item (gd_pair_kernel_split), which
  // run beside each other.  From about 1.3 items a CU on its repeated work costs more
  // than it gains.  An evaluation of poses with the split kernel / with one group an
  // item: 27 items 46.7 / 59.4 us, 90 items 40.0 / 42.0, 180 items 43.9 / 45.4, 240
  // items 49.0 / 49.3, 280 items 74.6 / 77.1, 420 items 99.4 / 83.3, 540 items 55.8 /
  // 53.1 (points and anchors per item differ).
  if (lc == 4 && n_items <= n_cu()) {
    hipLaunchKernelGGL(gd_pair_kernel_split, dim3(n_items, 3), block, 0, s, d_jobs, d_items, n_items, nb, nb_list);
    const hipError_t e = hipGetLastError();
    return e == hipSuccess ? GD_OK : hip_fail(e, "pair kernel launch");
  }
  switch (lc) {
    case 4:
      hipLaunchKernelGGL(gd_pair_kernel<4>, grid, block, 0, s, d_jobs, d_items, n_items, nb, nb_list);
      break;
    case 8:
      hipLaunchKernelGGL(gd_pair_kernel<8>, grid, block, 0, s, d_jobs, d_items, n_items, nb, nb_list);
      break;
    case 16:
      hipLaunchKernelGGL(gd_pair_kernel<16>, grid, block, 0, s, d_jobs, d_items, n_items, nb, nb_list);
      break;
    default:
      return GD_ERR_ARG;
  }
  hipError_t e = hipGetLastError();
  return e == hipSuccess ? GD_OK : hip_fail(e, "pair kernel launch");
}

gd_status launch_finish(const GdJob *d_jobs, const GdBlock *d_blocks, int n_blocks, int mode,
                        int step, hipStream_t s) {
  if (n_blocks <= 0) return GD_OK;
  hipLaunchKernelGGL(gd_reduce_kernel, dim3(n_blocks * GD_RK), dim3(256), 0, s, d_jobs, d_blocks);
  hipLaunchKernelGGL(gd_finish_kernel, dim3(n_blocks), dim3(1024), 0, s, d_jobs, d_blocks, mode, step,
                     (const int *)nullptr, (int *)nullptr);
  hipError_t e = hipGetLastError();
  return e == hipSuccess ? GD_OK : hip_fail(e, "finish kernel launch");
}

gd_status launch_exchange(const GdJob *d_jobs, int round, hipStream_t s) {
  hipLaunchKernelGGL(gd_exchange_kernel, dim3(1), dim3(256), 0, s, d_jobs, (const GdExch *)nullptr, round);
  hipError_t e = hipGetLastError();
  return e == hipSuccess ? GD_OK : hip_fail(e, "exchange kernel launch");
}

// ---- stepping kernel ----------------------------------------------------------
size_t chain_sync_bytes(int n_blocks) {
  return (GD_SY_HEAD + (size_t)n_blocks * GD_SY_BLOCK) * sizeof(unsigned);
}

// Finishers: a block's reduction is a chain of latencies, which a team of groups
// shortens: 8 groups for two blocks, 4 where there are few blocks or a step's items
// leave slots free (220 replicas, 46 atoms, 4,001 points: 39.0 us a step, with 1
// group 54.8, with 8 42.2; 1,760 replicas, 24 atoms, 1,200 points: 39.5, with 1
// 49.2), then one, whose time the other blocks' items cover (1,760 replicas, 40
// atoms, 3,000 points: 104.8 us, with 4 groups 108.2).  At most 64 teams, each then
// with several blocks.  Finishers hold their slots for a whole launch, and while some
// of them wait for one no worker of the launch runs: they are at most a quarter of
// what the device holds (256 of 1,024 groups on 256 CUs), so that the finishers of
// three processes leave room for workers.
// Groups of a CU: where the items of a step are fewer than the slots, added LDS
// keeps a CU from taking four groups while others have none, and keeps groups
// that only wait from being resident: 128 replicas, 40 atoms, 9,000 points (400
// items): 50.2 us a step with one group to a CU, 62.9 with four; 440 replicas, 20
// atoms, 9,000 points (420): 65.9 with two, 70.4 with four.  Less is added where
// the finishers would be over their quarter.
// Queue entries: blocks of one job are eight entries each, on lines of their own
// where there are few blocks (waiting workers then poll different lines); in
// longer lists an entry is 8 items.  The queue holds up to 1 MB of them.
void ChainList::shape(const std::vector<const GdJob *> &jobs, int cu) {
  n_blocks = n_items = n_entries = 0;
  step_pairs = 0.0;
  int most = 1;
  for (const GdJob *g : jobs) {
    n_blocks += g->Rp / 64;
    n_items += g->Rp / 64 * g->nL * g->nG;
    step_pairs += (double)g->Rp * g->L * g->P;
    most = std::max(most, g->nL * g->nG);
  }
  per_entry = std::max(jobs.size() == 1 ? (most + 7) / 8 : 8, (most + 255) / 256);
  for (const GdJob *g : jobs) n_entries += g->Rp / 64 * ((g->nL * g->nG + per_entry - 1) / per_entry);
  stride = n_blocks <= 8 ? 16 : 1;
  cap_steps = (int)std::max(2.0, std::min(1024.0, (double)(1 << 17) / ((double)n_entries * stride)));
  n_teams = std::min(n_blocks, 64);
  if (cu <= 0) cu = g_cu > 0 ? g_cu : 256;
  team = n_blocks <= 2 ? 8 : n_blocks <= 8 || n_items <= 6 * cu ? 4 : 1;
  const int groups = n_items + 2 * n_teams * team;
  static const int added[] = {60 << 10, 28 << 10, 14 << 10, 0};  // 1, 2, 3 and 4 groups to a CU
  int k = groups <= 7 * cu / 4 ? 0 : groups <= 4 * cu ? 1 : groups <= 6 * cu ? 2 : 3;
  while (k < 3 && 4 * n_teams * team > (k + 1) * cu) ++k;
  lds = added[k];
  slots = (k + 1) * cu;
  static_assert((160 << 10) / (GD_CHAIN_LDS + (60 << 10)) == 1 && (160 << 10) / (GD_CHAIN_LDS + (28 << 10)) == 2 &&
                    (160 << 10) / (GD_CHAIN_LDS + (14 << 10)) == 3 && (160 << 10) / GD_CHAIN_LDS >= 4,
                "groups of a CU");
  team = std::min(team, std::max(1, slots / 4 / n_teams));
  n_teams = std::min(n_teams, std::max(1, slots / 4));
}

// One launch stays under about a second and 2^22 groups (2^32 work items is the
// most): jobs whose single step is a sizeable part of that (10^11 pairs, 50 ms)
// gain nothing from it and are stepped by launches.  So are jobs of one block,
// where a step is one chain of latencies and the launches are the shorter one
// (25 replicas, 24 atoms, 1,200 points: 19.1 us a step against 21.6), and of two
// blocks with many items, which the 8 finishers of a block read more slowly than
// the reduce launch's 16 groups (105 replicas, 80 atoms, 9,000 points, 2,840 items:
// 91 against 111).
int chain_max_steps(const ChainList &c) {
  if (c.n_blocks < 2 || (c.n_blocks == 2 && c.n_items > 2048) || c.step_pairs > 1e11) return 0;
  const double by_time = 1e12 / std::max(1.0, c.step_pairs);
  const double by_count = (double)(1 << 22) / ((double)c.n_entries * c.per_entry);
  const int n = (int)std::min({(double)c.cap_steps, by_time, by_count});
  return n >= 2 ? n : 0;  // the first launch takes the initial pass and a step
}

// A plain run of few items is stepped by launches on one stream: a stream of its own
// for each half of the blocks leaves too little in a launch, and where the process's
// streams share a hardware queue costs twice the launches.  The line lies where the
// stepping kernel becomes the shorter (us a step, one stream / stepping kernel): two
// blocks 19.3 / 24.4 (120 items), 29.9 / 35.2 (480), 46.3 / 55.4 (1,110), 53.4 / 64.1
// (1,650); four blocks 23.7 / 27.4 (96), 24.1 / 24.8 (360), 30.0 / 31.5 (512), 34.4 /
// 34.3 (720); seven blocks 20.9 / 24.5 (224), 30.5 / 29.1 (420).  An item is the
// pairs of 64 replicas, 4 atoms and 8 tiles of 10 to 60 points here.
static bool step_by_one_stream(const ChainList &c) {
  const int cu = g_cu > 0 ? g_cu : 256;
  return c.n_items <= (c.n_blocks <= 2 ? 8 * cu : c.n_blocks <= 4 ? 2 * cu : cu);
}

// One run at a time uses the stepping kernel: groups of two such launches that
// wait for each other's slots could fill the device between them.  Runs that
// overlap it step by launches, as does a run repeated because a wait ran out of
// time (another process's launch can hold slots too): the same bits either way.
// A run takes the turn once its lists suit the kernel, so that runs which do not use
// it leave it to the others.
static std::atomic<int> g_stepping{0};
bool Stepping::take() {
  if (!mine) mine = g_stepping.exchange(1) == 0;
  return mine;
}
Stepping::~Stepping() {
  if (mine) g_stepping.store(0);
}

gd_status launch_chain(ChainList &c, const GdJob *d_jobs, int step0, int n_steps, bool init,
                       hipStream_t s) {
  if (n_steps <= 0) return GD_OK;
  GdChain a;
  a.jobs = d_jobs;
  a.items = c.d_items;
  a.blocks = c.d_blocks;
  a.sync = c.d_sync;
  a.queue = c.d_queue;
  a.stride = c.stride;
  a.per_entry = c.per_entry;
  a.epoch = ++c.epoch;
  a.n_entries = c.n_entries;
  a.steps_before = c.steps;
  a.n_teams = c.n_teams;
  a.team = c.team;
  a.n_steps = n_steps;
  a.step0 = step0;
  a.init = init ? 1 : 0;
  a.n_blocks = c.n_blocks;
  a.wait_ticks = (long long)(c.wait_s * 1e3 * g_wall_khz);
  // the finishers, then a worker group for each item of every step
  const int grid = c.n_teams * c.team + c.n_entries * c.per_entry * n_steps;
  void *args[] = {&a};
  // by the launch's own status: an error that some earlier call left would have the
  // counters miss a launch that runs
  const hipError_t e =
      hipLaunchKernel((const void *)gd_chain_kernel<4>, dim3(grid), dim3(64 * GD_GROUP), args, c.lds, s);
  if (e != hipSuccess) return hip_fail(e, "stepping kernel launch");
  c.steps += (unsigned)n_steps;  // the counters hold what was launched
  return GD_OK;
}

gd_status launch_keep(bool back, const GdJob *d_jobs, const GdBlock *d_blocks, int n_blocks, unsigned *area,
                      const unsigned *failed, int step, hipStream_t s) {
  if (n_blocks <= 0) return GD_OK;
  if (back)
    hipLaunchKernelGGL(gd_keep_kernel<true>, dim3(n_blocks), dim3(256), 0, s, d_jobs, d_blocks, area, failed,
                       (unsigned)step);
  else
    hipLaunchKernelGGL(gd_keep_kernel<false>, dim3(n_blocks), dim3(256), 0, s, d_jobs, d_blocks, area, failed,
                       (unsigned)step);
  const hipError_t e = hipGetLastError();
  return e == hipSuccess ? GD_OK : hip_fail(e, "keep kernel launch");
}

gd_status launch_swap(int axis, const GdJob *d_jobs, const GdBlock *d_blocks, int n_blocks,
                      const int *d_swr, int round, int launch_step, const int *step_base, int *wq,
                      const std::function<gd_status()> &pair, hipStream_t s) {
  if (n_blocks <= 0) return GD_OK;
  hipLaunchKernelGGL(gd_swap_propose_kernel, dim3(n_blocks), dim3(256), 0, s, d_jobs, d_blocks, axis,
                     d_swr, round);
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return hip_fail(e, "swap propose kernel launch");
  gd_status st = pair();
  if (st != GD_OK) return st;
  hipLaunchKernelGGL(gd_reduce_kernel, dim3(n_blocks * GD_RK), dim3(256), 0, s, d_jobs, d_blocks);
  hipLaunchKernelGGL(gd_finish_kernel, dim3(n_blocks), dim3(1024), 0, s, d_jobs, d_blocks, GD_MODE_EVAL,
                     0, (const int *)nullptr, wq);
  hipLaunchKernelGGL(gd_swap_accept_kernel, dim3(n_blocks), dim3(256), 0, s, d_jobs, d_blocks, axis,
                     d_swr, round, launch_step, step_base);
  e = hipGetLastError();
  return e == hipSuccess ? GD_OK : hip_fail(e, "swap kernel launch");
}

void set_mc(GdJob &g, const gd_mc_param *mc) {
  for (int i = 0; i < 6; ++i) g.move_scale[i] = mc->move_scale[i];
  g.move_mode = mc->move_mode;
  g.seed_lo = (uint32_t)mc->seed;
  g.seed_hi = (uint32_t)(mc->seed >> 32);
  g.job_id = mc->job_id;
  g.record = mc->record;
  g.xaxes = mc->exchange_axes ? mc->exchange_axes : GD_EXCH_TEMP;
  g.steps_total = mc->steps_total;
  g.step0 = 0;
}

// ---- host memory of results ---------------------------------------------------
namespace {
struct Pool {
  std::mutex mu;
  std::vector<std::pair<void *, size_t>> idle;
  size_t bytes = 0;  // of idle
  int users = 0;
};
Pool &pool() {
  static Pool *p = new Pool;  // outlives every caller
  return *p;
}
}  // namespace

void host_pool_users(int change) {
  Pool &P = pool();
  std::vector<std::pair<void *, size_t>> gone;
  {
    std::lock_guard<std::mutex> lk(P.mu);
    P.users += change;
    if (P.users > 0) return;
    gone.swap(P.idle);
    P.bytes = 0;
  }
  for (auto &b : gone) hipHostFree(b.first);
}

static std::atomic<float *> g_noalloc_host[64];
void noalloc_host_make() {
  static std::mutex mu;
  if (g_device < 0 || g_device >= 64 || g_noalloc_host[g_device].load()) return;
  std::lock_guard<std::mutex> lk(mu);
  if (g_noalloc_host[g_device].load()) return;
  void *p = nullptr;
  if (hipHostMalloc(&p, kNoallocHostBytes, hipHostMallocPortable) != hipSuccess) {
    (void)hipGetLastError();
    return;
  }
  g_noalloc_host[g_device].store((float *)p);
}
float *noalloc_host() { return g_device < 0 || g_device >= 64 ? nullptr : g_noalloc_host[g_device].load(); }

gd_status HostBuf::acquire(size_t n, bool copies_only) {
  release();
  if (copies_only && n > kHostPoolBytes) return plain(n);  // not worth pinning for one copy
  size_t want = 64 << 10;
  while (want < n) want *= 2;
  Pool &P = pool();
  {
    std::lock_guard<std::mutex> lk(P.mu);
    int best = -1;
    for (int k = 0; k < (int)P.idle.size(); ++k)
      if (P.idle[k].second >= want && (best < 0 || P.idle[k].second < P.idle[best].second)) best = k;
    if (best >= 0) {
      p = P.idle[best].first, bytes = P.idle[best].second;
      P.bytes -= bytes;
      P.idle.erase(P.idle.begin() + best);
      return GD_OK;
    }
  }
  const hipError_t e = hipHostMalloc(&p, want, hipHostMallocPortable);
  if (e != hipSuccess) {
    p = nullptr;
    if (copies_only) {
      (void)hipGetLastError();
      return plain(n);
    }
    return hip_fail(e, "hipHostMalloc");
  }
  bytes = want;
  return GD_OK;
}

gd_status HostBuf::plain(size_t n) {
  p = std::malloc(n);
  if (!p) {
    set_error("out of host memory");
    return GD_ERR_HIP;
  }
  pinned = false;
  bytes = n;
  return GD_OK;
}

void HostBuf::release() {
  if (!p) return;
  if (!pinned) {
    std::free(p);
    p = nullptr, bytes = 0, pinned = true;
    return;
  }
  Pool &P = pool();
  {
    std::lock_guard<std::mutex> lk(P.mu);
    if (P.users > 0 && P.bytes + bytes <= kHostPoolBytes) {
      P.idle.push_back({p, bytes});
      P.bytes += bytes;
      p = nullptr;
    }
  }
  if (p) hipHostFree(p);
  p = nullptr, bytes = 0;
}

gd_status out_launch(gd_job *const *jobs, gd_replica_out *const *out, int n, const unsigned *d_fail, hipStream_t s,
                     OutStage &o) {
  size_t words = 16;  // the failure word, on its own
  o.at.assign(n, 0);
  o.fail = nullptr;
  for (int k = 0; k < n; ++k)
    if (out[k]) {
      o.at[k] = words;
      words += ((size_t)jobs[k]->h.R * GD_PACK_W + 15) / 16 * 16;
    }
  if (words == 16 && !d_fail) return GD_OK;
  gd_status st = GD_OK;
  o.by_copies = words * sizeof(float) > kHostPoolBytes || o.buf.acquire(words * sizeof(float)) != GD_OK;
  if (o.by_copies) {
    if (!d_fail) return GD_OK;
    o.fail = &o.fail_word;
    const hipError_t e = hipMemcpyAsync(&o.fail_word, d_fail, sizeof(unsigned), hipMemcpyDeviceToHost, s);
    return e == hipSuccess ? GD_OK : hip_fail(e, "stepping kernel status");
  }
  float *base = (float *)o.buf.p;
  if (d_fail) o.fail = (unsigned *)base;
  GdPackList list;
  std::memset(&list, 0, sizeof list);
  list.fail = d_fail;
  list.fail_out = (unsigned *)base;
  int blocks = 1;
  const auto send = [&]() -> gd_status {
    hipLaunchKernelGGL(gd_pack_kernel, dim3(blocks, std::max(1, list.n)), dim3(256), 0, s, list);
    const hipError_t e = hipGetLastError();
    list.fail = nullptr;
    list.n = 0;
    blocks = 1;
    return e == hipSuccess ? GD_OK : hip_fail(e, "pack kernel launch");
  };
  for (int k = 0; k < n; ++k) {
    if (!out[k]) continue;
    const GdJob &g = jobs[k]->h;
    list.job[list.n++] = {g.mm, g.en, g.best, g.tmpi, g.nacc, g.nexc, g.acc, g.nswp, base + o.at[k], g.R, g.Rp};
    blocks = std::max(blocks, g.Rp / 64);
    if (list.n == GD_PACK_JOBS && (st = send()) != GD_OK) return st;
  }
  return list.n > 0 || list.fail ? send() : GD_OK;
}

// ---- energy evaluation --------------------------------------------------------
constexpr size_t kEvalWorkspace = 64 << 20;

size_t eval_carve(const GdJob &g, int nb, char *base, EvalBufs *b) {
  const size_t Rp = (size_t)nb * 64;
  size_t o = 0;
  const auto take = [&](size_t bytes) {
    char *at = base ? base + o : nullptr;
    o += (bytes + 255) / 256 * 256;
    return at;
  };
  EvalBufs c;
  c.job = (GdJob *)take(sizeof(GdJob));
  c.ligi = (int *)take(Rp * sizeof(int));
  c.prti = (int *)take(Rp * sizeof(int));
  c.prop = (float *)take(6 * Rp * sizeof(float));
  c.coords = (float *)take((size_t)3 * g.L * Rp * sizeof(float));
  c.plin = (float *)take((size_t)GD_NLIN * g.nL * g.nG * Rp * sizeof(float));
  c.phpc = (float *)take((size_t)g.L * g.nG * Rp * sizeof(float));
  c.pmcs = (float *)take((size_t)std::max(1, g.M) * g.nL * Rp * sizeof(float));
  c.fin = (float *)take((size_t)nb * GD_RK * 8 * 64 * sizeof(float));
  if (b) *b = c;
  return o;
}

gd_status eval_pass(gd_job *j, const EvalBufs &b, int cnt, const int *conf, const float *pose, float *terms,
                    float *raw, float *host, float *dev) {
  const int nb = (cnt + 63) / 64;
  float *const io = host ? host : dev;
  hipStream_t s = j->stream;
  GdJob x = j->h;  // the job's tables, the evaluation's lanes and buffers
  x.R = cnt;
  x.Rp = nb * 64;
  x.ligi = b.ligi, x.prti = b.prti, x.prop = b.prop, x.coords = b.coords;
  x.part_lin = b.plin, x.part_hpc = b.phpc, x.part_mcs = b.pmcs, x.fin_part = b.fin;
  int *h_conf = (int *)io;
  float *h_pose = io + 2 * (size_t)cnt;
  x.ev_terms = io + 8 * (size_t)cnt;  // written over the link by the finish kernel
  x.ev_raw = io + 18 * (size_t)cnt;
  x.rec = nullptr;
  x.rec_cap = 0;
  x.record = 0;
  hipError_t e = hipSuccess;
  if (host) {
    std::memcpy(h_conf, conf, (size_t)cnt * 2 * sizeof(int));
    std::memcpy(h_pose, pose, (size_t)cnt * 6 * sizeof(float));
  } else if ((e = hipMemcpyAsync(h_conf, conf, (size_t)cnt * 2 * sizeof(int), hipMemcpyHostToDevice, s)) !=
                 hipSuccess ||
             (e = hipMemcpyAsync(h_pose, pose, (size_t)cnt * 6 * sizeof(float), hipMemcpyHostToDevice, s)) !=
                 hipSuccess) {
    return hip_fail(e, "evaluation inputs");
  }
  hipLaunchKernelGGL(gd_eval_setup_kernel, dim3(nb), dim3(1024), 0, s, x, b.job, (const int *)h_conf,
                     (const float *)h_pose, cnt);
  e = hipGetLastError();
  gd_status st = e == hipSuccess ? GD_OK : hip_fail(e, "eval setup kernel launch");
  if (st == GD_OK) st = launch_pair(x.lc, b.job, j->d_items, x.nL * x.nG * nb, s, nb, j->h.Rp / 64);
  if (st == GD_OK) st = launch_finish(b.job, nullptr, nb, GD_MODE_EVAL, 0, s);
  if (!host && st == GD_OK &&
      ((e = hipMemcpyAsync(terms, x.ev_terms, (size_t)cnt * 10 * sizeof(float), hipMemcpyDeviceToHost, s)) !=
           hipSuccess ||
       (raw && (e = hipMemcpyAsync(raw, x.ev_raw, (size_t)cnt * 9 * sizeof(float), hipMemcpyDeviceToHost, s)) !=
                   hipSuccess)))
    st = hip_fail(e, "evaluation results");
  e = hipStreamSynchronize(s);
  if (st == GD_OK && e != hipSuccess) st = hip_fail(e, "energy evaluation");
  if (st != GD_OK || !host) return st;
  std::memcpy(terms, x.ev_terms, (size_t)cnt * 10 * sizeof(float));
  if (raw) std::memcpy(raw, x.ev_raw, (size_t)cnt * 9 * sizeof(float));
  return GD_OK;
}

// Results of a job row by row of the device's arrays.
static gd_status out_rows(const GdJob &g, const gd_replica_out &q, hipStream_t s) {
  const size_t R = g.R, Rp = g.Rp;
  std::vector<float> row(R);
  const auto down = [&](void *to, const void *from) -> gd_status {
    hipError_t e = hipMemcpyAsync(to, from, R * 4, hipMemcpyDeviceToHost, s);
    if (e == hipSuccess) e = hipStreamSynchronize(s);
    return e == hipSuccess ? GD_OK : hip_fail(e, "results");
  };
  gd_status st = GD_OK;
  const auto turned = [&](float *to, const float *from, int n) {  // [n][Rp] to [R][n]
    for (int i = 0; to && i < n && st == GD_OK; ++i)
      if ((st = down(row.data(), from + (size_t)i * Rp)) == GD_OK)
        for (size_t r = 0; r < R; ++r) to[r * n + i] = row[r];
  };
  turned(q.movematrix, g.mm, 6);
  turned(q.energy, g.en, 10);
  const struct {
    void *to;
    const void *from;
  } rows[] = {{q.best_energy, g.best}, {q.idx_tmp, g.tmpi},   {q.n_accept, g.nacc},  {q.n_exchange, g.nexc},
              {q.is_accept, g.acc},    {q.n_swap_lig, g.nswp}, {q.n_swap_prt, g.nswp + Rp}};
  for (const auto &x : rows)
    if (x.to && st == GD_OK) st = down(x.to, x.from);
  return st;
}

gd_status out_copy(gd_job *const *jobs, gd_replica_out *const *out, int n, const OutStage &o, hipStream_t s) {
  for (int k = 0; k < n; ++k) {
    if (!out[k]) continue;
    if (o.by_copies) {
      const gd_status st = out_rows(jobs[k]->h, *out[k], s);
      if (st != GD_OK) return st;
      continue;
    }
    const size_t R = jobs[k]->h.R;
    const float *p = (const float *)o.buf.p + o.at[k];
    const gd_replica_out &q = *out[k];
    const auto cp = [](void *dst, const float *src, size_t words) {
      if (dst) std::memcpy(dst, src, words * 4);
    };
    cp(q.movematrix, p, 6 * R);
    cp(q.energy, p + 6 * R, 10 * R);
    cp(q.best_energy, p + 16 * R, R);
    cp(q.idx_tmp, p + 17 * R, R);
    cp(q.n_accept, p + 18 * R, R);
    cp(q.n_exchange, p + 19 * R, R);
    cp(q.is_accept, p + 20 * R, R);
    cp(q.n_swap_lig, p + 21 * R, R);
    cp(q.n_swap_prt, p + 22 * R, R);
  }
  return GD_OK;
}

// A job of its own (plain tiling, its own stream), or, with a stream, one that
// runs in shared launches on that stream.
gd_status job_create(const gd_job_desc *desc, hipStream_t shared, gd_job **out) {
  if (!desc || !out) return GD_ERR_ARG;
  *out = nullptr;
  gd_status st = ensure_device();
  if (st != GD_OK) return st;
  gd_job *j = new gd_job();
  host_pool_users(1);
  noalloc_host_make();
  hipError_t e = hipSuccess;
  j->own_stream = shared == nullptr;
  j->stream = shared;
  if (!shared) e = hipStreamCreateWithFlags(&j->stream, hipStreamNonBlocking);
  if (e != hipSuccess) {
    host_pool_users(-1);
    delete j;
    return hip_fail(e, "hipStreamCreate");
  }
  st = pack_job(desc, j);
  if (st == GD_OK) {
    e = hipMalloc(&j->d_job, sizeof(GdJob));
    if (e != hipSuccess) st = hip_fail(e, "hipMalloc job");
  }
  if (st == GD_OK) {
    int lc = 4, ptile;
    if (shared)
      ptile = shared_ptile(j->h.L, j->h.P);
    else
      default_tiling(j->h.L, j->h.P, j->h.R, lc, ptile);
    st = apply_tiling(j, lc, ptile);
  }
  if (st == GD_OK) st = sync_job_struct(j);
  if (st != GD_OK) {
    gd_job_destroy(j);
    return st;
  }
  *out = j;
  return GD_OK;
}

}  // namespace gdr

using namespace gdr;

// ---------------------------------------------------------------------------
extern "C" {

gd_status gd_init(int dev) {
  std::lock_guard<std::mutex> lk(g_mu);
  int n = 0;
  hipError_t e = hipGetDeviceCount(&n);
  if (e != hipSuccess || n == 0) {
    set_error("no HIP device visible");
    return GD_ERR_NODEV;
  }
  if (dev < 0 || dev >= n) return GD_ERR_ARG;
  hipDeviceProp_t prop;
  if ((e = hipGetDeviceProperties(&prop, dev)) != hipSuccess) return hip_fail(e, "hipGetDeviceProperties");
  if (std::strncmp(prop.gcnArchName, "gfx950", 6) != 0) {
    set_error(std::string("device is ") + prop.gcnArchName + ", this library is built for gfx950");
    return GD_ERR_NODEV;
  }
  if ((e = hipSetDevice(dev)) != hipSuccess) return hip_fail(e, "hipSetDevice");
  g_device = dev;
  g_cu = prop.multiProcessorCount;
  int khz = 0;
  if (hipDeviceGetAttribute(&khz, hipDeviceAttributeWallClockRate, dev) == hipSuccess && khz > 0)
    g_wall_khz = khz;
  return GD_OK;
}

gd_status gd_device_info(char *name, int name_len, int *n_cu_out, int *clock_khz, size_t *hbm) {
  gd_status st = ensure_device();
  if (st != GD_OK) return st;
  hipDeviceProp_t prop;
  hipError_t e = hipGetDeviceProperties(&prop, g_device);
  if (e != hipSuccess) return hip_fail(e, "hipGetDeviceProperties");
  if (name && name_len > 0) {
    if (prop.name[0])
      std::snprintf(name, name_len, "%s (%s)", prop.name, prop.gcnArchName);
    else  // the runtime reports no marketing name: the architecture alone
      std::snprintf(name, name_len, "%s, %d CUs", prop.gcnArchName, prop.multiProcessorCount);
  }
  if (n_cu_out) *n_cu_out = prop.multiProcessorCount;
  if (clock_khz) *clock_khz = prop.clockRate;
  if (hbm) *hbm = prop.totalGlobalMem;
  return GD_OK;
}

const char *gd_last_error(void) { return last_error(); }
const char *gd_version(void) { return "geauxdock_amd 0.1 (gfx950)"; }

// The pair kernel's far-field r^2 threshold for (pmf0, el1) (diagnostics, tests).
float gd_far_r2(float pmf0, float el1) { return gdr::far_r2_threshold(pmf0, el1); }

// The row threshold of the pair loop's near branch for a (ligand type, point
// type) pair of the force field (diagnostics, tests): as the device row holds it.
float gd_near_r2(float pmf0, float el1, float hdb0, float hdb1) {
  const bool hb = hdb0 > 0.1f;
  const double c = (double)hdb1 * std::sqrt(0.5 * 1.44269504088896340736);
  return gdr::near_r2_threshold(pmf0, el1, gdr::sqrt_threshold(pmf0), hb, hdb0, hb ? c : 0.0);
}

void gd_philox(const uint32_t ctr[4], const uint32_t key[2], int rounds, uint32_t out[4]) {
  const gd_u32x4 r = gd_philox4x32(ctr[0], ctr[1], ctr[2], ctr[3], key[0], key[1], rounds);
  for (int i = 0; i < 4; ++i) out[i] = r.v[i];
}

gd_status gd_job_create(const gd_job_desc *desc, gd_job **out) { return gdr::job_create(desc, nullptr, out); }

gd_status gd_job_destroy(gd_job *j) {
  if (!j) return GD_OK;
  if (!j->staged.empty()) {  // uploads of a creation that failed
    hipStreamSynchronize(j->stream);
    j->staged.clear();
  }
  if (j->d_base) hipFree(j->d_base);
  if (j->d_part) hipFree(j->d_part);
  if (j->d_job) hipFree(j->d_job);
  if (j->d_lists) hipFree(j->d_lists);
  gdr::chain_drop(j);
  if (j->d_eval) hipFree(j->d_eval);
  if (j->d_rec) hipFree(j->d_rec);
  if (j->h_rec) hipHostFree(j->h_rec);
  if (j->copy_stream) hipStreamDestroy(j->copy_stream);
  for (hipStream_t ps : j->part_stream)
    if (ps) hipStreamDestroy(ps);
  if (j->stream && j->own_stream) hipStreamDestroy(j->stream);
  delete j;
  gdr::host_pool_users(-1);
  return GD_OK;
}

gd_status gd_job_sizes(const gd_job *j, int *n_rep, int *L, int *P, int *K, int *M) {
  if (!j) return GD_ERR_ARG;
  if (n_rep) *n_rep = j->h.R;
  if (L) *L = j->h.L;
  if (P) *P = j->h.P;
  if (K) *K = j->h.K;
  if (M) *M = j->h.M;
  return GD_OK;
}

size_t gd_job_footprint(const gd_job_desc *d) { return footprint(d, false); }

// Device memory the job holds: tables and replica state, partial sums, work
// lists, the record ring (when a run recorded) and the device job struct.
size_t gd_job_device_bytes(const gd_job *j) {
  if (!j) return 0;
  return j->bytes + j->part_bytes + j->lists_bytes + j->chain_bytes + j->eval_bytes + j->rec_bytes + sizeof(GdJob);
}

gd_status gd_stepping_shape(int n_cu, int n_jobs, int n_rep, int lig_chunks, int tile_groups, int *finishers,
                            int *slots) {
  if (n_cu < 1 || n_jobs < 1 || n_rep < 1 || lig_chunks < 1 || tile_groups < 1 || !finishers || !slots)
    return GD_ERR_ARG;
  if (n_cu > (1 << 20) || n_jobs > (1 << 20) || n_rep > (1 << 26) || (double)n_jobs * (n_rep + 63) / 64 * lig_chunks * tile_groups > 1e9)
    return GD_ERR_SIZE;
  GdJob g;
  std::memset(&g, 0, sizeof g);
  g.Rp = (n_rep + 63) / 64 * 64;
  g.nL = lig_chunks, g.nG = tile_groups;
  gdr::ChainList c;
  c.shape(std::vector<const GdJob *>(n_jobs, &g), n_cu);
  *finishers = c.n_teams * c.team;
  *slots = c.slots;
  return GD_OK;
}

gd_status gd_tiling_get(const gd_job *j, gd_tiling *t) {
  if (!j || !t) return GD_ERR_ARG;
  t->atoms_per_lane = j->h.lc;
  t->tile_points = j->h.ptile;
  t->waves_per_cu = 0;
  return GD_OK;
}

gd_status gd_job_set_step_wait(gd_job *j, double seconds) {
  if (!j || !(seconds >= 0.0) || seconds > 60.0) return GD_ERR_ARG;
  j->chain.wait_s = seconds;
  return GD_OK;
}

gd_status gd_job_set_streams(gd_job *j, int n_streams) {
  if (!j || n_streams < 1 || n_streams > gd_job::kMaxParts) return GD_ERR_ARG;
  j->by_launches = n_streams != gd_job::kDefaultStreams;
  if (n_streams == j->n_streams) return GD_OK;
  const gd_status st = ensure_device();
  if (st != GD_OK) return st;
  j->n_streams = n_streams;
  return sync_job_struct(j);  // the parts' item lists
}

gd_status gd_tiling_set(gd_job *j, const gd_tiling *t) {
  if (!j || !t) return GD_ERR_ARG;
  gd_status st = apply_tiling(j, t->atoms_per_lane, t->tile_points);
  if (st != GD_OK) return st;
  return sync_job_struct(j);
}

// Energies of arbitrary poses through the same pair/finish kernels, on lanes of
// their own (eval_pass); the job's replica state is not touched.
gd_status gd_energy_eval(gd_job *j, int n, const int *conf, const float *pose, float *terms,
                         float *raw, float *coords) {
  if (!j || n < 0 || (n > 0 && (!conf || !pose || !terms))) return GD_ERR_ARG;
  if (n == 0) return GD_OK;
  gd_status st = ensure_device();
  if (st != GD_OK) return st;
  GdJob &g = j->h;
  for (int i = 0; i < n; ++i)
    if (conf[2 * i] < 0 || conf[2 * i] >= g.n_lig || conf[2 * i + 1] < 0 || conf[2 * i + 1] >= g.n_prt)
      return GD_ERR_ARG;
  const int Rp = g.Rp, L = g.L;
  // Poses of a pass: the job's lanes where they suffice or fill the device (1,024
  // or more); smaller jobs with more poses take a workspace for up to 2,048, so
  // that a pass of theirs fills it too (500 poses of a 25-replica complex: one
  // pass in place of eight; 880 poses of a 220-replica one: one in place of four).
  EvalBufs b = {j->ev.job, j->ev.ligi, j->ev.prti, j->ev.prop, g.coords, g.part_lin, g.part_hpc, g.part_mcs,
                g.fin_part};
  int lanes = Rp;
  if (n > Rp && Rp < 1024) {
    int nb = std::min((n + 63) / 64, 2048 / 64);
    while (nb > Rp / 64 && eval_carve(g, nb, nullptr, nullptr) > kEvalWorkspace) --nb;
    const size_t need = eval_carve(g, nb, nullptr, nullptr);
    if (nb > Rp / 64) {
      if (need > j->eval_bytes) {
        if (j->d_eval) hipFree(j->d_eval);
        j->d_eval = nullptr;
        j->eval_bytes = 0;
        if (hipMalloc(&j->d_eval, need) == hipSuccess) j->eval_bytes = need;
        else j->d_eval = nullptr, (void)hipGetLastError();
      }
      if (j->d_eval) {
        eval_carve(g, nb, (char *)j->d_eval, &b);
        lanes = nb * 64;
      }
    }
  }
  // inputs and results: at most the pool's bytes a pass; without pinned memory, through
  // a device buffer
  lanes = std::min(lanes, (int)(kHostPoolBytes / (64 * kEvalHostWords * sizeof(float))) * 64);
  const size_t io_bytes = (size_t)std::min(n, lanes) * kEvalHostWords * sizeof(float);
  HostBuf host;
  struct DevBuf {
    void *p = nullptr;
    ~DevBuf() {
      if (p) hipFree(p);
    }
  } dev;
  if (host.acquire(io_bytes) != GD_OK) {
    const hipError_t e = hipMalloc(&dev.p, io_bytes);
    if (e != hipSuccess) {
      dev.p = nullptr;
      return hip_fail(e, "evaluation buffers");
    }
  }
  std::vector<float> oc;
  for (int base = 0; base < n && st == GD_OK; base += lanes) {
    const int cnt = std::min(lanes, n - base);
    st = eval_pass(j, b, cnt, conf + 2 * (size_t)base, pose + 6 * (size_t)base, terms + 10 * (size_t)base,
                   raw ? raw + 9 * (size_t)base : nullptr, (float *)host.p, (float *)dev.p);
    if (st != GD_OK || !coords) continue;
    const int W = (cnt + 63) / 64 * 64;  // lanes of the pass
    oc.resize((size_t)3 * L * W);
    const hipError_t e = hipMemcpy(oc.data(), b.coords, oc.size() * sizeof(float), hipMemcpyDeviceToHost);
    if (e != hipSuccess) return hip_fail(e, "eval coordinates");
    for (int i = 0; i < cnt; ++i)
      for (int l = 0; l < L; ++l)
        for (int d = 0; d < 3; ++d)
          coords[((size_t)(base + i) * L + l) * 3 + d] = oc[(size_t)(3 * l + d) * W + i];
  }
  return st;
}

// Plain one-job docking (the reference Dock shape, backend_gpu.cu:64-133):
// initial-energy pass, then steps_total steps in dump segments; temperature
// exchange every steps_per_exchange steps; with mc->record the accept records
// of the last segment stay on the device for gd_dock_records.
// Receiver of the per-dump accept records (gd_dock_stream); null: the records
// stay on the device (gd_dock_records reads the last dump).
struct RecSink {
  gd_record_fn fn;
  void *user;
  bool blocking;
};

// The plain driver: initial-energy pass, then steps_total MC steps in dumps of
// steps_per_dump (Dock, backend_gpu.cu:64-133), exchange points every
// steps_per_exchange steps.  With a sink, dump k's accept records (ring half
// k mod 2) go to the host after the dump's kernels: blocking, as the
// reference's cudaMemcpy after each dump (backend_gpu.cu:110-116), or on the
// copy stream while the device runs dump k + 1, handed to the sink once
// copied; dump k + 2 reuses the half only after the host has taken it.
// chain: the stepping kernel may be used.  *again: one of its waits ran out of
// time, nothing was handed over of this dump or later ones (*handed dumps were,
// or had been before), and the run is to go on without it from MC step *from, the
// last one whose state was kept (0: from the start).
static gd_status dock_run(gd_job *j, const gd_mc_param *mc, const RecSink *sink,
                          gd_replica_out *out, gd_stats *stats, const bool chain, int *from, int *handed,
                          bool *again) {
  if (!j || !mc || mc->steps_total < 0 || mc->steps_per_exchange < 0) return GD_ERR_ARG;
  gd_status st = ensure_device();
  if (st != GD_OK) return st;
  GdJob &g = j->h;
  hipStream_t s = j->stream;
  set_mc(g, mc);
  const bool record = mc->record || sink;
  g.record = record ? 1 : 0;
  const int spd = mc->steps_per_dump > 0 ? mc->steps_per_dump : std::max(1, mc->steps_total);
  const size_t half_floats = (size_t)g.Rp * spd * GD_REC_W;
  j->last_half = -1;
  if (record) {
    const size_t need = 2 * half_floats * sizeof(float);
    if (need > j->rec_bytes) {
      if (j->d_rec) hipFree(j->d_rec);
      j->d_rec = nullptr;
      j->rec_bytes = 0;
      hipError_t e = hipMalloc(&j->d_rec, need);
      if (e != hipSuccess) return hip_fail(e, "hipMalloc records");
      j->rec_bytes = need;
    }
    g.rec = (float *)j->d_rec;
    g.rec_cap = spd;
  } else {
    g.rec = nullptr;
    g.rec_cap = 0;
  }
  // host side of a streamed run: pinned halves (records, then counts) and the copy stream
  float *h_half[2] = {nullptr, nullptr};
  int *h_cnt[2] = {nullptr, nullptr};
  unsigned *h_fail[2] = {nullptr, nullptr};
  hipEvent_t ev_done[2] = {nullptr, nullptr}, ev_copied[2] = {nullptr, nullptr};
  if (sink) {
    const size_t hb = 2 * (half_floats * sizeof(float) + (size_t)g.Rp * sizeof(int) + sizeof(unsigned));
    if (hb > j->h_rec_bytes) {
      if (j->h_rec) hipHostFree(j->h_rec);
      j->h_rec = nullptr;
      j->h_rec_bytes = 0;
      hipError_t e = hipHostMalloc(&j->h_rec, hb, hipHostMallocDefault);
      if (e != hipSuccess) return hip_fail(e, "hipHostMalloc records");
      j->h_rec_bytes = hb;
    }
    for (int b = 0; b < 2; ++b) {
      h_half[b] = (float *)j->h_rec + b * half_floats;
      h_cnt[b] = (int *)((float *)j->h_rec + 2 * half_floats) + (size_t)b * g.Rp;
      h_fail[b] = (unsigned *)((float *)j->h_rec + 2 * half_floats) + 2 * (size_t)g.Rp + b;
    }
    if (!sink->blocking) {
      hipError_t e = hipSuccess;
      if (!j->copy_stream) e = hipStreamCreateWithFlags(&j->copy_stream, hipStreamNonBlocking);
      for (int b = 0; b < 2 && e == hipSuccess; ++b) {
        e = hipEventCreateWithFlags(&ev_done[b], hipEventDisableTiming);
        if (e == hipSuccess) e = hipEventCreateWithFlags(&ev_copied[b], hipEventDisableTiming);
      }
      if (e != hipSuccess) {
        for (int b = 0; b < 2; ++b) {
          if (ev_done[b]) hipEventDestroy(ev_done[b]);
          if (ev_copied[b]) hipEventDestroy(ev_copied[b]);
        }
        return hip_fail(e, "record stream set-up");
      }
    }
  }
  struct EvGuard {
    hipEvent_t *a, *b;
    ~EvGuard() {
      for (int k = 0; k < 2; ++k) {
        if (a[k]) hipEventDestroy(a[k]);
        if (b[k]) hipEventDestroy(b[k]);
      }
    }
  } ev_guard{ev_done, ev_copied};
  hipError_t e = hipSuccess;
  // exchange points: after MC steps spe-1, 2spe-1, ...; round k uses table entry k
  const int spe = mc->steps_per_exchange;
  const bool tx = spe > 0 && (g.xaxes & GD_EXCH_TEMP) && g.n_tmp > 1;
  const bool lx = spe > 0 && (g.xaxes & GD_EXCH_LIG) && g.n_lig > 1;
  const bool px = spe > 0 && (g.xaxes & GD_EXCH_PRT) && g.n_prt > 1;
  const int n_rounds = (tx || lx || px) ? mc->steps_total / spe : 0;
  const std::function<gd_status()> pair = [&]() {
    return launch_pair(g.lc, j->d_job, j->d_items, j->n_items, s);
  };
  // the stepping kernel takes the steps between exchange points and dump ends
  // in one launch; a job whose streams were set, with wide ligand chunks, or of few
  // items is stepped by launches
  int chain_max = 0;
  bool few = false;
  Stepping turn;
  if (!j->by_launches && g.lc == 4) {
    j->chain.shape({&g});
    few = step_by_one_stream(j->chain);
    chain_max = chain && !few ? chain_max_steps(j->chain) : 0;
    if (chain_max > 0 && !turn.take()) chain_max = 0;
    if (chain_max > 0 && chain_make(j) != GD_OK) {  // no memory for its lists
      (void)hipGetLastError();
      chain_max = 0;
    }
  }
  // hand dump k (ring half b, copied to the host) to the sink, each dump once
  const auto hand = [&](int k, int b) {
    if (k < *handed) return;
    sink->fn(sink->user, k, k * spd, g.R, spd, h_half[b], h_cnt[b]);
    *handed = k + 1;
  };
  // false: the stepping kernel failed, in it or before or since
  const auto deliver = [&](int k, int b) {
    if (chain_max > 0 && *h_fail[b]) return false;
    hand(k, b);
    return true;
  };
  const unsigned *d_fail = j->chain.d_sync + GD_SY_FAILED;
  KTimer tp;
  SpanTimer tspan;
  const bool timing = stats != nullptr;
  // Several streams, each stepping one contiguous part of the replica blocks:
  // one part's reduce and finish kernels and its launch tail overlap the other
  // parts' pair work.  Between exchange points the parts share nothing; they
  // join for every exchange point (which spans the whole job) and at dump ends.
  const int np = j->n_parts;
  bool multi = chain_max == 0 && np >= 2 && !few;
  for (int k = 0; k < np; ++k) multi = multi && j->nb_part[k] > 0;
  hipStream_t ps[gd_job::kMaxParts] = {s};
  hipEvent_t ev_fork = nullptr, ev_join[gd_job::kMaxParts] = {};
  struct ForkGuard {
    hipEvent_t *f, *jn;
    ~ForkGuard() {
      if (*f) hipEventDestroy(*f);
      for (int k = 0; k < gd_job::kMaxParts; ++k)
        if (jn[k]) hipEventDestroy(jn[k]);
    }
  } fork_guard{&ev_fork, ev_join};
  if (multi) {
    e = hipSuccess;
    for (int k = 1; k < np && e == hipSuccess; ++k) {
      if (!j->part_stream[k]) e = hipStreamCreateWithFlags(&j->part_stream[k], hipStreamNonBlocking);
      ps[k] = j->part_stream[k];
    }
    if (e == hipSuccess) e = hipEventCreateWithFlags(&ev_fork, hipEventDisableTiming);
    for (int k = 1; k < np && e == hipSuccess; ++k)
      e = hipEventCreateWithFlags(&ev_join[k], hipEventDisableTiming);
    if (e != hipSuccess) {
      return hip_fail(e, "part streams");
    }
  }
  // the other parts' streams continue after everything queued on s so far /
  // s continues after everything queued on the other parts' streams
  const auto fork = [&]() {
    hipError_t r = hipEventRecord(ev_fork, s);
    for (int k = 1; k < np && r == hipSuccess; ++k) r = hipStreamWaitEvent(ps[k], ev_fork, 0);
    return r == hipSuccess ? GD_OK : hip_fail(r, "stream fork");
  };
  const auto join = [&]() {
    hipError_t r = hipSuccess;
    for (int k = 1; k < np && r == hipSuccess; ++k) {
      r = hipEventRecord(ev_join[k], ps[k]);
      if (r == hipSuccess) r = hipStreamWaitEvent(s, ev_join[k], 0);
    }
    return r == hipSuccess ? GD_OK : hip_fail(r, "stream join");
  };
  const auto t0 = std::chrono::steady_clock::now();
  if (chain_max > 0) {
    ChainList &c = j->chain;
    if (c.stale) {
      if ((e = hipMemsetAsync(c.d_sync, 0, chain_sync_bytes(c.n_blocks), s)) != hipSuccess)
        return hip_fail(e, "stepping kernel counters");
      c.steps = 0;
    }
    c.stale = true;  // until this run has ended well
    if (j->keep_used && (e = hipMemsetAsync(j->d_keep, 0, sizeof(unsigned), s)) != hipSuccess)
      return hip_fail(e, "kept state");
    j->keep_used = false;
  }
  // initial energies (MonteCarlo_d with s2max = 1)
  hipLaunchKernelGGL(gd_start_job_kernel, dim3(j->n_blocks), dim3(256), 0, s, g, j->d_job);
  if ((e = hipGetLastError()) != hipSuccess) st = hip_fail(e, "start kernel launch");
  if (*from > 0) {
    if (st == GD_OK)
      st = launch_keep(true, j->d_job, j->d_blocks, j->n_blocks, j->d_keep, nullptr, *from, s);
  } else if (chain_max > 0) {
    if (st == GD_OK && mc->steps_total == 0) st = launch_chain(j->chain, j->d_job, 0, 1, true, s);
  } else {
    if (st == GD_OK) st = launch_pair(g.lc, j->d_job, j->d_items, j->n_items, s);
    if (st == GD_OK) st = launch_finish(j->d_job, j->d_blocks, j->n_blocks, GD_MODE_INIT, 0, s);
  }
  if (st == GD_OK && multi && timing) st = tspan.mark_ref(s);
  int pending = -1;  // streamed dump whose copy is in flight
  int chain_steps = 0;  // MC steps (and initial pass) taken by the stepping kernel
  double since = 0.0;   // work since the state was kept
  for (int k = *from / spd, s1 = k * spd; s1 < mc->steps_total && st == GD_OK; s1 += spd, ++k) {
    const int b = k & 1;
    if (record) {
      e = hipMemsetAsync(g.rec_n + (size_t)b * g.Rp, 0, (size_t)g.Rp * sizeof(int), s);
      if (e != hipSuccess) {
        st = hip_fail(e, "hipMemsetAsync");
        break;
      }
    }
    if (multi && (st = fork()) != GD_OK) break;
    const int s_end = std::min(mc->steps_total, s1 + spd);
    for (int step = std::max(s1, *from); step < s_end; ++step) {
      const bool timed = timing && step % kTimedEvery == 0;
      if (chain_max > 0) {
        // up to the next exchange point or the dump's end; the initial pass
        // goes with the first steps
        const bool init = step == 0;
        int n = std::min(s_end - step, chain_max - (init ? 1 : 0));
        if (n_rounds > 0) n = std::min(n, spe - step % spe);
        // kept where a dump of records starts, whose counts are zero
        if (since >= kKeepWork && (!record || step == s1)) {
          if ((st = launch_keep(false, j->d_job, j->d_blocks, j->n_blocks, j->d_keep, d_fail, step, s)) != GD_OK) break;
          j->keep_used = true;
          since = 0.0;
        }
        since += j->chain.work(n);
        if (timing && (st = tp.begin(s)) != GD_OK) break;
        if ((st = launch_chain(j->chain, j->d_job, step, n + (init ? 1 : 0), init, s)) != GD_OK) break;
        if (timing && (st = tp.end(s)) != GD_OK) break;
        step += n - 1;
        chain_steps += n + (init ? 1 : 0);
      } else if (multi) {
        for (int k = 0; k < np && st == GD_OK; ++k) {
          if (timed && (st = tspan.record(ps[k])) != GD_OK) break;
          if ((st = launch_pair(g.lc, j->d_job, j->d_items_part[k], j->n_items_part[k], ps[k])) != GD_OK) break;
          if (timed) st = tspan.record(ps[k]);
        }
        for (int k = 0; k < np && st == GD_OK; ++k)
          st = launch_finish(j->d_job, j->d_blocks + j->b0_part[k], j->nb_part[k], GD_MODE_STEP, step, ps[k]);
        if (st != GD_OK) break;
      } else {
        if (timed && (st = tp.begin(s)) != GD_OK) break;
        if ((st = launch_pair(g.lc, j->d_job, j->d_items, j->n_items, s)) != GD_OK) break;
        if (timed && (st = tp.end(s)) != GD_OK) break;
        if ((st = launch_finish(j->d_job, j->d_blocks, j->n_blocks, GD_MODE_STEP, step, s)) != GD_OK) break;
      }
      if (n_rounds > 0 && (step + 1) % spe == 0 && (step + 1) / spe <= n_rounds) {
        const int r = (step + 1) / spe - 1;
        if (multi && (st = join()) != GD_OK) break;
        if (tx && (st = launch_exchange(j->d_job, r, s)) != GD_OK) break;
        for (int axis = 0; axis < 2; ++axis)
          if ((axis ? px : lx) &&
              (st = launch_swap(axis, j->d_job, j->d_blocks, j->n_blocks, nullptr, r, step, nullptr,
                                nullptr, pair, s)) != GD_OK)
            break;
        if (st != GD_OK) break;
        if (multi && (st = fork()) != GD_OK) break;
      }
    }
    if (st != GD_OK) break;
    if (multi && (st = join()) != GD_OK) break;
    j->last_half = record ? b : -1;
    if (!sink) continue;
    const float *d_half = g.rec + (size_t)b * half_floats;
    const int *d_cnt = g.rec_n + (size_t)b * g.Rp;
    if (sink->blocking) {  // the reference's shape: wait, copy, hand over
      if ((e = hipStreamSynchronize(s)) != hipSuccess ||
          (e = hipMemcpy(h_half[b], d_half, half_floats * sizeof(float), hipMemcpyDeviceToHost)) !=
              hipSuccess ||
          (e = hipMemcpy(h_cnt[b], d_cnt, (size_t)g.Rp * sizeof(int), hipMemcpyDeviceToHost)) != hipSuccess ||
          (chain_max > 0 &&
           (e = hipMemcpy(h_fail[b], d_fail, sizeof(unsigned), hipMemcpyDeviceToHost)) != hipSuccess)) {
        st = hip_fail(e, "record copy");
        break;
      }
      if (!deliver(k, b)) break;
      continue;
    }
    if ((e = hipEventRecord(ev_done[b], s)) != hipSuccess ||
        (e = hipStreamWaitEvent(j->copy_stream, ev_done[b], 0)) != hipSuccess ||
        (e = hipMemcpyAsync(h_half[b], d_half, half_floats * sizeof(float), hipMemcpyDeviceToHost,
                            j->copy_stream)) != hipSuccess ||
        (e = hipMemcpyAsync(h_cnt[b], d_cnt, (size_t)g.Rp * sizeof(int), hipMemcpyDeviceToHost,
                            j->copy_stream)) != hipSuccess ||
        (chain_max > 0 && (e = hipMemcpyAsync(h_fail[b], d_fail, sizeof(unsigned), hipMemcpyDeviceToHost,
                                              j->copy_stream)) != hipSuccess) ||
        (e = hipEventRecord(ev_copied[b], j->copy_stream)) != hipSuccess) {
      st = hip_fail(e, "record stream");
      break;
    }
    if (pending >= 0) {  // the previous dump, copied while this one ran
      if ((e = hipEventSynchronize(ev_copied[pending & 1])) != hipSuccess) {
        st = hip_fail(e, "record copy");
        break;
      }
      if (!deliver(pending, pending & 1)) break;
    }
    pending = k;
  }
  OutStage res;
  if (st == GD_OK) st = out_launch(&j, &out, 1, chain_max > 0 ? d_fail : nullptr, s, res);
  {
    hipError_t e2 = hipStreamSynchronize(s);  // also covers steps_total == 0
    if (st == GD_OK && e2 != hipSuccess) st = hip_fail(e2, "hipStreamSynchronize");
    for (int k = 1; multi && k < np; ++k) {
      e2 = hipStreamSynchronize(ps[k]);
      if (st == GD_OK && e2 != hipSuccess) st = hip_fail(e2, "hipStreamSynchronize");
    }
    if (j->copy_stream) {
      e2 = hipStreamSynchronize(j->copy_stream);
      if (st == GD_OK && e2 != hipSuccess) st = hip_fail(e2, "record copy");
    }
  }
  if (st == GD_OK && chain_max > 0) {
    *again = *res.fail != 0;
    j->chain.stale = *again;
    unsigned kept = 0;
    if (*again && j->keep_used && (e = hipMemcpy(&kept, j->d_keep, sizeof kept, hipMemcpyDeviceToHost)) != hipSuccess)
      st = hip_fail(e, "kept state");
    *from = (int)kept;
  }
  // the last dump; of a run that goes on from a kept state, one that ended before it
  if (st == GD_OK && sink && !sink->blocking && pending >= 0 && (!*again || (pending + 1) * (long long)spd <= *from))
    hand(pending, pending & 1);
  if (st == GD_OK && timing) st = multi ? tspan.collect(np) : tp.collect();
  const auto t1 = std::chrono::steady_clock::now();
  if (st != GD_OK || *again) return st;
  if (stats) {
    stats->ms_total = std::chrono::duration<double, std::milli>(t1 - t0).count();
    stats->ms_pair_kernel = multi ? tspan.parts_ms : tp.ms;
    stats->ms_finish_kernel = 0.0;
    stats->n_pair_launch = multi ? tspan.n_part_launches : tp.n;
    stats->pair_evals = (double)g.R * g.L * g.P * (mc->steps_total + 1);
    stats->replica_steps = (double)g.R * mc->steps_total;
    // timed steps are 0, kTimedEvery, ...: first to last start over the steps between
    const int n_samples = multi ? tspan.n : tp.n;
    const double span_first_last = multi ? tspan.last_a - tspan.first_a : tp.first_to_last_ms;
    stats->ms_step_period =
        n_samples >= 2 ? span_first_last / ((double)(n_samples - 1) * kTimedEvery) : 0.0;
    stats->ms_pair_span = multi ? (tspan.n ? tspan.ms / tspan.n : 0.0) : (tp.n ? tp.ms / tp.n : 0.0);
    if (chain_max > 0 && chain_steps > 0) {
      // whole MC steps, pair work to next proposal, in the stepping kernel's launches
      stats->n_pair_launch = chain_steps;
      stats->ms_step_period = stats->ms_pair_span = tp.ms / chain_steps;
    }
  }
  return out_copy(&j, &out, 1, res, s);
}

static gd_status dock_impl(gd_job *j, const gd_mc_param *mc, const RecSink *sink,
                           gd_replica_out *out, gd_stats *stats) {
  int from = 0, handed = 0;
  bool again = false;
  gd_status st = dock_run(j, mc, sink, out, stats, true, &from, &handed, &again);
  if (st == GD_OK && again) {
    again = false;
    st = dock_run(j, mc, sink, out, stats, false, &from, &handed, &again);
  }
  return st;
}

gd_status gd_dock(gd_job *j, const gd_mc_param *mc, gd_replica_out *out, gd_stats *stats) {
  return dock_impl(j, mc, nullptr, out, stats);
}

gd_status gd_dock_stream(gd_job *j, const gd_mc_param *mc, gd_record_fn fn, void *user, int flags,
                         gd_replica_out *out, gd_stats *stats) {
  if (!fn || (flags & ~GD_STREAM_BLOCKING)) return GD_ERR_ARG;
  const RecSink sink = {fn, user, (flags & GD_STREAM_BLOCKING) != 0};
  return dock_impl(j, mc, &sink, out, stats);
}

gd_status gd_job_replicas(gd_job *j, gd_replica_out *out) {
  if (!j || !out) return GD_ERR_ARG;
  OutStage res;
  gd_status st = out_launch(&j, &out, 1, nullptr, j->stream, res);
  const hipError_t e = hipStreamSynchronize(j->stream);
  if (st == GD_OK && e != hipSuccess) st = hip_fail(e, "results");
  return st == GD_OK ? out_copy(&j, &out, 1, res, j->stream) : st;
}

gd_status gd_dock_records(gd_job *j, int cap, float *rec, int *count) {
  if (!j || cap < 0 || !count || (cap > 0 && !rec)) return GD_ERR_ARG;
  const GdJob &g = j->h;
  if (!g.rec || j->last_half < 0) return GD_ERR_STATE;
  const int R = g.R, Rp = g.Rp, rc = g.rec_cap;
  const size_t half = (size_t)j->last_half;
  std::vector<int> n(Rp);
  hipError_t e = hipStreamSynchronize(j->stream);
  if (e == hipSuccess)
    e = hipMemcpy(n.data(), g.rec_n + half * Rp, (size_t)Rp * sizeof(int), hipMemcpyDeviceToHost);
  if (e != hipSuccess) return hip_fail(e, "hipMemcpy rec_n");
  std::vector<float> buf((size_t)Rp * rc * GD_REC_W);
  if (!buf.empty()) {
    e = hipMemcpy(buf.data(), g.rec + half * buf.size(), buf.size() * sizeof(float),
                  hipMemcpyDeviceToHost);
    if (e != hipSuccess) return hip_fail(e, "hipMemcpy records");
  }
  for (int r = 0; r < R; ++r) {
    const int m = std::min(n[r], cap);
    count[r] = n[r];
    for (int k = 0; k < m; ++k)
      for (int w = 0; w < GD_REC_W; ++w)
        rec[((size_t)r * cap + k) * GD_REC_W + w] = buf[((size_t)r * rc + k) * GD_REC_W + w];
  }
  return GD_OK;
}

// Move increments as gd_dock draws them (statistical tests of the move
// generator): inc[s][r][6] for replicas r < n_rep at steps step0 + s,
// s < n_steps, computed on the device (on_device != 0, the kernels' own code)
// or on the host (the same source compiled for the host).
gd_status gd_move_draws(uint64_t seed, uint32_t job_id, int move_mode, const float move_scale[6],
                        int n_rep, uint32_t step0, int n_steps, int on_device, float *inc) {
  if (!move_scale || !inc || n_rep <= 0 || n_steps <= 0 ||
      (move_mode != GD_MOVE_REF_UNIFORM && move_mode != GD_MOVE_GAUSSIAN))
    return GD_ERR_ARG;
  const long long n = (long long)n_rep * n_steps;
  if (n > (1ll << 28)) return GD_ERR_SIZE;
  if (!on_device) {
    for (long long i = 0; i < n; ++i) {
      uint32_t w[8];
      gd_step_draws(seed, job_id, (uint32_t)(i % n_rep), step0 + (uint32_t)(i / n_rep), w);
      gd_move_incr(move_mode, move_scale, w, inc + i * 6);
    }
    return GD_OK;
  }
  gd_status st = ensure_device();
  if (st != GD_OK) return st;
  GdScale6 sc;
  for (int k = 0; k < 6; ++k) sc.v[k] = move_scale[k];
  float *d = nullptr;
  hipError_t e = hipMalloc(&d, (size_t)n * 6 * sizeof(float));
  if (e != hipSuccess) return hip_fail(e, "hipMalloc draws");
  hipLaunchKernelGGL(gd_move_draws_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, 0, seed,
                     job_id, move_mode, sc, n_rep, step0, (int)n, d);
  e = hipGetLastError();
  if (e == hipSuccess) e = hipMemcpy(inc, d, (size_t)n * 6 * sizeof(float), hipMemcpyDeviceToHost);
  hipFree(d);
  return e == hipSuccess ? GD_OK : hip_fail(e, "gd_move_draws_kernel");
}

// Increments from given draw words: w[n][8] -> inc[n][6] (host code path).
gd_status gd_move_incr_words(int move_mode, const float move_scale[6], int n, const uint32_t *w,
                             float *inc) {
  if (!move_scale || !w || !inc || n < 0 ||
      (move_mode != GD_MOVE_REF_UNIFORM && move_mode != GD_MOVE_GAUSSIAN))
    return GD_ERR_ARG;
  for (int i = 0; i < n; ++i) gd_move_incr(move_mode, move_scale, w + (size_t)i * 8, inc + (size_t)i * 6);
  return GD_OK;
}

// Engine clock under load: every SIMD of every CU runs dependent FMAs for
// about `ms` milliseconds; the shader-clock counter's rate against the
// constant-rate counter (hipDeviceAttributeWallClockRate) is the clock.
gd_status gd_measure_sclk(int ms, double *sclk_mhz) {
  if (!sclk_mhz || ms <= 0 || ms > 2000) return GD_ERR_ARG;
  gd_status st = ensure_device();
  if (st != GD_OK) return st;
  int wall_khz = 0;
  hipError_t e = hipDeviceGetAttribute(&wall_khz, hipDeviceAttributeWallClockRate, g_device);
  if (e != hipSuccess || wall_khz <= 0) return hip_fail(e, "hipDeviceAttributeWallClockRate");
  long long *d = nullptr;
  e = hipMalloc(&d, 2 * sizeof(long long) + sizeof(float));
  if (e != hipSuccess) return hip_fail(e, "hipMalloc clock");
  const long long ticks = (long long)wall_khz * ms;
  hipLaunchKernelGGL(gd_clock_kernel, dim3(4 * (g_cu > 0 ? g_cu : 256)), dim3(64), 0, 0, ticks, 1.0f, d,
                     (float *)(d + 2));
  long long h[2] = {0, 0};
  e = hipGetLastError();
  if (e == hipSuccess) e = hipMemcpy(h, d, sizeof h, hipMemcpyDeviceToHost);
  hipFree(d);
  if (e != hipSuccess) return hip_fail(e, "gd_clock_kernel");
  if (h[1] <= 0) return GD_ERR_STATE;
  *sclk_mhz = (double)h[0] / (double)h[1] * (double)wall_khz / 1000.0;
  return GD_OK;
}

// A plain device-to-device copy of `bytes` (a multiple of 16), `reps` times:
// the calibration for HBM traffic counters (each dispatch reads and writes
// exactly `bytes`).  *ms: mean time per copy.
gd_status gd_device_copy(size_t bytes, int reps, double *ms) {
  if (bytes == 0 || bytes % 16 != 0 || reps <= 0) return GD_ERR_ARG;
  gd_status st = ensure_device();
  if (st != GD_OK) return st;
  void *a = nullptr, *b = nullptr;
  hipError_t e = hipMalloc(&a, bytes);
  if (e == hipSuccess) e = hipMalloc(&b, bytes);
  if (e == hipSuccess) e = hipMemset(a, 0, bytes);
  if (e != hipSuccess) {
    if (a) hipFree(a);
    return hip_fail(e, "gd_device_copy buffers");
  }
  const size_t n16 = bytes / 16;
  const int grid = 4 * 8 * (g_cu > 0 ? g_cu : 256);
  e = hipDeviceSynchronize();
  const auto t0 = std::chrono::steady_clock::now();
  for (int r = 0; r < reps && e == hipSuccess; ++r) {
    hipLaunchKernelGGL(gd_copy_kernel, dim3(grid), dim3(256), 0, 0, (const float4 *)a, (float4 *)b, n16);
    e = hipGetLastError();
  }
  if (e == hipSuccess) e = hipDeviceSynchronize();
  const auto t1 = std::chrono::steady_clock::now();
  hipFree(a);
  hipFree(b);
  if (e != hipSuccess) return hip_fail(e, "gd_copy_kernel");
  if (ms) *ms = std::chrono::duration<double, std::milli>(t1 - t0).count() / reps;
  return GD_OK;
}

// PrintRecord-format text sink of gd_dock_stream (util_print.C:70-151).
struct gd_record_csv {
  FILE *f = nullptr;
  int lo = 0, hi = -1;
  bool failed = false;
};

gd_status gd_record_csv_open(const char *path, int rep_lo, int rep_hi, int header,
                             gd_record_csv **out) {
  if (!path || !out || rep_lo < 0 || rep_hi < rep_lo) return GD_ERR_ARG;
  *out = nullptr;
  FILE *f = std::fopen(path, "w");
  if (!f) {
    set_error(std::string("cannot open ") + path);
    return GD_ERR_IO;
  }
  gd_record_csv *w = new gd_record_csv();
  w->f = f;
  w->lo = rep_lo;
  w->hi = rep_hi;
  if (header) {
    static const char *names[10] = {"vdw", "ele", "pmf", "psp", "hdb", "hpc", "kde", "lhm", "dst", "total"};
    std::fprintf(f, "rep step");
    for (int i = 0; i < 10; ++i) std::fprintf(f, " %s", names[i]);
    std::fprintf(f, "\n");
  }
  *out = w;
  return GD_OK;
}

void gd_record_csv_write(void *writer, int dump, int step_begin, int n_rep, int cap,
                         const float *rec, const int *count) {
  (void)dump;
  (void)step_begin;
  gd_record_csv *w = (gd_record_csv *)writer;
  if (!w || !w->f || !rec || !count) return;
  for (int r = w->lo; r <= w->hi && r < n_rep; ++r) {
    const int n = std::min(count[r], cap);
    for (int k = 0; k < n; ++k) {
      const float *o = rec + ((size_t)r * cap + k) * GD_REC_W;
      if (std::fprintf(w->f, "%3d %d", r, (int)o[0]) < 0) w->failed = true;
      for (int i = 0; i < 10; ++i)
        if (std::fprintf(w->f, " %.4f", o[7 + i]) < 0) w->failed = true;
      if (std::fprintf(w->f, "\n") < 0) w->failed = true;
    }
  }
}

gd_status gd_record_csv_close(gd_record_csv *w) {
  if (!w) return GD_ERR_ARG;
  bool bad = w->failed;
  if (w->f && std::fclose(w->f) != 0) bad = true;
  delete w;
  if (bad) {
    set_error("record file write failed");
    return GD_ERR_IO;
  }
  return GD_OK;
}

}  // extern "C"
