// gd_internal.h -- host-side job object and runtime helpers shared by the
// runtime translation units (not part of the C ABI).
#pragma once
#include <hip/hip_runtime.h>

#include <atomic>
#include <functional>
#include <memory>
#include <string>
#include <vector>

#include "../../include/geauxdock_amd.h"
#include "gd_device.h"
#include "gd_rng.h"

namespace gdr {
// Work lists, queue and counters of the stepping kernel for a list of jobs.
struct ChainList {
  const GdItem *d_items = nullptr;
  const GdChainBlock *d_blocks = nullptr;
  unsigned *d_sync = nullptr;
  unsigned long long *d_queue = nullptr;
  int n_blocks = 0, n_items = 0;        // pair items of a step
  int n_entries = 0, per_entry = 1;     // queue entries of a step
  int stride = 1;
  int cap_steps = 0;                    // steps the queue holds
  int n_teams = 0, team = 0;            // finisher teams, groups of a team
  unsigned epoch = 0, steps = 0;        // launches and their steps since the counters were zero
  bool stale = false;                   // a run did not end well: its counters are zeroed before they are used
  int lds = 0;                          // LDS added to a group's, which bounds the groups of a CU
  std::atomic<double> wait_s{GD_CHAIN_WAIT_S};  // bound of one wait in the kernel
  double step_pairs = 0;                // (atom, point) pairs of one step
  // The host lists (items of each job, blocks) and the launch shape on a device of
  // `cu` CUs (0: this one).
  void shape(const std::vector<const GdJob *> &jobs, int cu = 0);
  int slots = 0;                        // groups that such a device holds at a time
  size_t queue_bytes() const { return (size_t)n_entries * stride * cap_steps * sizeof(unsigned long long); }
  // Work of n steps on the scale of kKeepWork.
  double work(int n) const { return n * (step_pairs > 5e7 ? step_pairs : 5e7); }
};

// A run keeps its state (gd_keep_kernel) once in that many pairs, about 0.2 s; a step of
// few pairs, whose time is its latency, counts as 25 us of them.
constexpr double kKeepWork = 4e11;
inline size_t keep_bytes(int n_blocks) {
  return (GD_KEEP_HEAD + (size_t)n_blocks * GD_KEEP_ROWS * 64) * sizeof(unsigned);
}
// The state of the jobs of a list of blocks, before MC step `step`: kept in `area`
// unless *failed, or (back) brought back from it.
gd_status launch_keep(bool back, const GdJob *d_jobs, const GdBlock *d_blocks, int n_blocks, unsigned *area,
                      const unsigned *failed, int step, hipStream_t s);
}  // namespace gdr

namespace gdr {
// Host memory that kernels read and write directly, from a pool shared by all
// threads: it keeps at most kHostPoolBytes of unused buffers, and none once the
// last job and server are gone (host_pool_users).  A buffer is given back only
// when no kernel uses it any more.
constexpr size_t kHostPoolBytes = 16u << 20;
struct HostBuf {
  void *p = nullptr;
  size_t bytes = 0;
  bool pinned = true;
  HostBuf() = default;
  HostBuf(const HostBuf &) = delete;
  HostBuf &operator=(const HostBuf &) = delete;
  ~HostBuf() { release(); }
  // copies_only: no kernel will use it, so large buffers may be ordinary memory
  gd_status acquire(size_t n, bool copies_only = false);
  void release();

 private:
  gd_status plain(size_t n);
};
struct EvalLanes {
  GdJob *job;
  int *ligi, *prti;
  float *prop;
};
}  // namespace gdr

struct gd_job {
  GdJob h{};                 // host mirror of the device struct
  GdJob *d_job = nullptr;    // device copy
  void *d_base = nullptr;    // tables + replica state
  void *d_part = nullptr;    // partial sums (tiling-dependent)
  size_t part_bytes = 0;
  void *d_lists = nullptr;   // work items + blocks
  size_t lists_bytes = 0;
  void *d_rec = nullptr;     // accept records: a two-half ring, one half per dump
  size_t rec_bytes = 0;
  void *h_rec = nullptr;     // pinned host copies of both halves (record streaming)
  size_t h_rec_bytes = 0;
  hipStream_t copy_stream = nullptr;  // D2H of finished dumps beside the MC stream
  int last_half = -1;        // ring half of the last completed dump (-1: none)
  size_t bytes = 0;          // d_base size
  std::vector<GdItem> items; // job-local work items (job index 0)
  GdItem *d_items = nullptr;
  GdBlock *d_blocks = nullptr;
  int n_items = 0, n_blocks = 0;
  // the plain path's stepping parts: n_parts contiguous ranges of the blocks,
  // [b0_part[k], b0_part[k] + nb_part[k]), each with its items (the job's items
  // of those blocks, in the job's order) and a stream (part 0: the job's own)
  static constexpr int kMaxParts = 4, kDefaultStreams = 2;
  bool by_launches = false;  // step by launches on n_streams streams (gd_job_set_streams)
  GdItem *d_items_part[kMaxParts] = {};
  int n_items_part[kMaxParts] = {}, nb_part[kMaxParts] = {}, b0_part[kMaxParts] = {};
  int n_parts = 0;
  int n_streams = kDefaultStreams;  // streams the plain path steps on (1 .. kMaxParts)
  hipStream_t part_stream[kMaxParts] = {};
  gdr::ChainList chain;      // the stepping kernel's list, its queue and its counters
  unsigned *d_keep = nullptr;  // state kept of a run by it
  bool keep_used = false;      // d_keep names a step of an earlier run
  // buffers of energy evaluations: a part of the arena for the lanes of up to Rp
  // poses (their other buffers are the job's own), and a workspace for more
  gdr::EvalLanes ev{};
  void *d_eval = nullptr;
  size_t eval_bytes = 0;
  void *d_chain = nullptr;
  size_t chain_bytes = 0;
  // protein points in source order, laid out on the device per tile count
  std::vector<float4> src_pco;     // [n_prt][P]
  std::vector<float4> src_pattr;   // [P]
  std::vector<float> src_pspv;     // [n_types + 1][P]
  std::vector<int> src_key;        // [P] class * GD_PTAB_PT + point type
  std::vector<int> src_order;      // [P] points by class, type and spread
  std::vector<int> atom_kde;       // [L] KDE anchors of each device atom (item order)
  int laid_nP = 0;                 // tile count of the device order (0: none yet)
  hipStream_t stream = nullptr;
  bool own_stream = true;
  std::vector<std::unique_ptr<gdr::HostBuf>> staged;  // uploads in flight on stream
};

namespace gdr {
void set_error(const std::string &s);
gd_status hip_fail(hipError_t e, const char *what);
gd_status ensure_device();
int device();   // the device the library runs on (-1 before initialisation)
int n_cu();
void default_tiling(int L, int P, int R, int &lc, int &ptile);  // one job per launch
int shared_ptile(int L, int P);      // tile points in shared launches (4 atoms per lane)
int pair_waves_per_cu(int lc);       // persistent pair kernel residency
int lg2_floor(int x);
gd_status apply_tiling(gd_job *j, int lc, int ptile);
gd_status sync_job_struct(gd_job *j);
gd_status job_create(const gd_job_desc *desc, hipStream_t shared, gd_job **out);
void set_mc(GdJob &g, const gd_mc_param *mc);
void host_pool_users(int change);
// Host words for gd_energy_eval_noalloc, one buffer per device, made with the
// device's first job and held until the process ends (null if there was no memory).
constexpr size_t kNoallocHostBytes = 512 << 10;
void noalloc_host_make();
float *noalloc_host();
// Results of jobs whose runs are done in stream order: out_launch queues the
// kernel that gathers them (and the word *d_fail, if given), out_copy hands them
// over once the stream was waited for.  Results of more than kHostPoolBytes, or for
// which there is no pinned memory, are copied row by row.  out[k] may be null.
struct OutStage {
  HostBuf buf;
  std::vector<size_t> at;    // word offset of each job
  const unsigned *fail = nullptr;
  unsigned fail_word = 0;
  bool by_copies = false;
};
gd_status out_launch(gd_job *const *jobs, gd_replica_out *const *out, int n, const unsigned *d_fail, hipStream_t s,
                     OutStage &o);
gd_status out_copy(gd_job *const *jobs, gd_replica_out *const *out, int n, const OutStage &o, hipStream_t s);
float far_r2_threshold(double pmf0, double el1);
// nb, nb_list: see gd_pair_kernel.
gd_status launch_pair(int lc, const GdJob *d_jobs, const GdItem *d_items, int n_items, hipStream_t s, int nb = 0,
                      int nb_list = 0);
gd_status launch_finish(const GdJob *d_jobs, const GdBlock *d_blocks, int n_blocks, int mode,
                        int step, hipStream_t s);
// Device buffers of one evaluation pass over nb 64-lane blocks.
struct EvalBufs {
  GdJob *job;
  int *ligi, *prti;
  float *prop, *coords, *plin, *phpc, *pmcs, *fin;
};
// The buffers laid out from base on; returns their bytes (base may be null).
size_t eval_carve(const GdJob &g, int nb, char *base, EvalBufs *b);
constexpr size_t kEvalHostWords = 2 + 6 + 10 + 9;  // host words of a pose: inputs, results
// One pass over cnt poses on the job's stream, waited for: setup, pair, reduce
// and finish kernels.  host: kEvalHostWords words a pose that kernels read and write;
// without, dev: as many on the device, to and from which the caller's arrays are copied.
gd_status eval_pass(gd_job *j, const EvalBufs &b, int cnt, const int *conf, const float *pose, float *terms,
                    float *raw, float *host, float *dev);
gd_status launch_exchange(const GdJob *d_jobs, int round, hipStream_t s);  // of one job
size_t chain_sync_bytes(int n_blocks);
// Steps that one launch may take (0: this list is stepped by launches).
int chain_max_steps(const ChainList &c);
// The right to launch the stepping kernel, from take() on for as long as the object
// lives: one run of the process at a time has it.
struct Stepping {
  bool mine = false;
  Stepping() = default;
  ~Stepping();
  bool take();  // whether it is this run's
  Stepping(const Stepping &) = delete;
  Stepping &operator=(const Stepping &) = delete;
};
gd_status launch_chain(ChainList &c, const GdJob *d_jobs, int step0, int n_steps, bool init,
                       hipStream_t s);
// One conformer swap sub-step along `axis` (0 ligand, 1 protein) for the jobs
// of the lists whose swr[job] round is >= 0 (d_swr null: one job, `round`): propose, pair (the caller's
// launcher), reduce, finish(EVAL), accept.  launch_step / step_base as for the
// finish kernel of the step just completed; wq is reset for the next pair
// launch when given.
gd_status launch_swap(int axis, const GdJob *d_jobs, const GdBlock *d_blocks, int n_blocks,
                      const int *d_swr, int round, int launch_step, const int *step_base, int *wq,
                      const std::function<gd_status()> &pair, hipStream_t s);

// HIP-event timer for one kernel over many launches: events are recorded
// around the timed launches and summed at synchronisation points, so timing
// never stalls the launch queue.  Each record still costs the queue about
// 4 us between the kernels around it, so an MC loop times the pair launch of
// one step in kTimedEvery (step 0, kTimedEvery, ...): the mean launch time
// comes from that sample at well under 1% of the loop's time.
constexpr int kTimedEvery = 16;
struct KTimer {
  std::vector<hipEvent_t> ev;
  int used = 0;
  double ms = 0.0;
  int n = 0;
  double first_to_last_ms = 0.0;  // first to last timed launch start (collect)
  ~KTimer();
  gd_status begin(hipStream_t s);   // records start event
  gd_status end(hipStream_t s);     // records stop event
  gd_status collect();              // after a stream sync
};
}  // namespace gdr
