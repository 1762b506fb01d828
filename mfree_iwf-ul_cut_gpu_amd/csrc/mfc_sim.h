// mfc_sim.h — the simulation handle behind the C ABI (internal to the library).
#pragma once

#include <cmath>
#include <memory>
#include <mutex>
#include <hip/hip_runtime.h>

#include <string>
#include <vector>

#include "../../include/mfc.h"
#include "mfc_kernels.h"
#include "mfc_setup.h"

namespace mfc {

// records the message of the last failing call of this thread; returns code
int fail(int code, const std::string &msg);

}  // namespace mfc

#define HIP_TRY(expr)                                                                         \
  do {                                                                                        \
    hipError_t e_ = (expr);                                                                   \
    if (e_ != hipSuccess) return mfc::fail(MFC_E_HIP, std::string(#expr) + ": " + hipGetErrorString(e_)); \
  } while (0)

constexpr int64_t HIST_CAP = 1 << 20;

struct mfc_sim;

namespace mfc {
struct adj_work;  // reverse-mode workspace (mfc_adjoint.hip)
void adj_free(adj_work *w);
// taped forward in three parts, so that a batch can interleave its instances: validate and
// allocate, keep the state at the start of step t when t is a checkpoint, and mean the window
int adj_begin(mfc_sim *s, int nsteps, int checkpoint_every, int w0, int w1);
void adj_keep_returns(mfc_sim *const *sims, int n);  // after adj_begin of every instance of the group
int adj_checkpoint(mfc_sim *s, int t);
int adj_segment(const mfc_sim *s);  // steps between its checkpoints
int adj_finish(mfc_sim *s, double Fmean[2]);
// the backward pass of a group of instances that recorded the same run (steps, checkpoint
// interval, window): one handle, or the instances of a batch, reversed together with one launch
// per phase over the group's work tables (fw: tile and chunk tables, launch variant);
// cot: 2 per instance, grad: 6 per instance
int adj_backward(mfc_sim *const *sims, int n, const batch_work &fw, hipStream_t st, const double *cot, double *grad);
}  // namespace mfc

// the patches of the grid for a number of threads per particle
constexpr int PLAN_LANES[3] = {1, 4, 8};
struct patch_plan {
  int lanes;
  int s, w, slots;  // rows and columns of cells, particles a work-group takes at a time
  int items;        // work items of the interaction launch
  int list;         // entries the list of patches can have
  int64_t entries;  // entries of the list of patches, for the initial particles
  int64_t patches;  // patches the grid can have
};

// pinned memory that results pass through on their way to the caller: two pieces of `half` bytes,
// allocated at the first read; readers take turns
struct read_stage {
  std::mutex m;
  char *p = nullptr;
  size_t half = 0;
  hipEvent_t done[2] = {nullptr, nullptr};
  ~read_stage() {
    if (p) (void)hipHostFree(p);
    for (hipEvent_t e : done)
      if (e) (void)hipEventDestroy(e);
  }
};

namespace mfc {
// Whether the cells hold so many lattice points that a patch's copy of whole records does not do: with one
// thread per particle where a column of a window (5 h by h) has more than 32 (from hdx 2.1 on),
// with several where the window of a single cell has more than the copy (from 3.2 on)
inline bool dense_cells(double hdx, bool f32, int lanes) {
  const auto lines = [](double cells) { return std::ceil(cells - 1e-6); };
  return lanes == 1 ? lines(5 * hdx) * lines(hdx) > 32 : lines(5 * hdx) * lines(5 * hdx) > patch_cap(f32, lanes, false);
}
}  // namespace mfc

struct mfc_sim {
  mfc_config cfg;      // the configuration the handle was created from (checkpoints keep it)
  mfc::scenario sc;
  mfc::dev_consts k;
  int ntiles = 0;
  hipStream_t stream = nullptr;
  std::vector<void *> allocs;
  mfc::dstate set[2];
  mfc::dbins bins = {};
  mfc::dpositional pos;
  mfc::drecords recs[2] = {};  // records of the start state of a step of parity 0 / 1
  int *chunk_sums[2] = {nullptr, nullptr};  // bins.bsum of parity 0 / 1
  int *plen = nullptr;                      // bins.plen of parity 0 / 1
  int precision = MFC_PREC_FP64;
  mfc_tool_state *tool = nullptr;  // two states, alternating each step
  mfc::return_tape *tape = nullptr;  // two, alternating each step
  double *partials = nullptr, *force_last = nullptr, *hist = nullptr;
  int64_t *hist_ctr = nullptr;
  int *force_pending = nullptr;  // per parity: the force of the step that produced it is not yet reduced
  int *force_groups = nullptr;   // mfc::dforce::gflag
  mfc::dforce force(int c) const {
    return {partials, force_groups, force_last, hist, HIST_CAP, hist_ctr, force_pending + c, force_pending + 1 - c};
  }
  int64_t hist_base = 0;           // steps recorded before the last history reset
  int cur = 0;                     // set holding the current state, and index of the current tool state
  int64_t step = 0;
  hipGraphExec_t graph[2] = {nullptr, nullptr};  // GRAPH_STEPS steps starting from parity 0 / 1
  bool graph_general = false;                    // of the variant they were captured with
  void drop_graphs();
  bool use_graphs = true;
  mfc::adj_work *adj = nullptr;    // reverse-mode tape of the last mfc_vjp_forward
  bool batched = false;            // instance of a batch: stepped by mfc_batch_step only
  // bins.key/clist, the chunk sums and the records hold the binning and the neighbour records of
  // the current state (computed by the last step's interaction); false after creation and after anything else wrote the state or the bins
  bool keys_fresh = false;
  std::shared_ptr<read_stage> reads = std::make_shared<read_stage>();  // one for the instances of a batch
  double *wear_part = nullptr;     // tool wear: 4 doubles per tile, then the 4 results
  double wear_accum = 0.;          // accumulated wear, sum of dt * mean rate (tool_wear.cu:59)
  mfc_tuning tuning = {};
  int lanes = 1;  // threads per particle of the interaction (set_patches)
  // Whether its interaction takes the general variant of the kernel (patch_mem's GEN): for an h of its
  // own for each particle, or for dense cells. us per step of 197k particles by tiles of the sorted
  // order (what there was before the patches) / from the records in memory (interact_rest) / with this: FP64
  // an uneven h 135 / 229 / 116, hdx 2.3 260 / 547 / 222, 3.0 372 / 955 / 287; FP32C 81 / 154 / 65, 138 / 325
  // / 118, 188 / - / 148; hdx 3.5 536 / - / 569 and 267 / - / 281. Where whole records fit it costs: FP64
  // an even h 102, FP32C 57.
  bool general() const {
    return !k.uniform_h || mfc::dense_cells(cfg.hdx, recs[0].f32, lanes);
  }
  mfc::variant variant() const { return {lanes, tuning.xcd_chunk ? tuning.xcd_chunk : mfc::XCD_CHUNK}; }
  // the step runs the batched kernels on a batch of one: descriptors of this handle for start
  // parity 0 and 1, and its (instance, block) work tables
  mfc::inst_args *dargs = nullptr;
  mfc::inst_args *slot[2] = {nullptr, nullptr};  // where its descriptors are read from (a batch's for its instances)
  int2 *dtiles = nullptr, *dchunks = nullptr, *dpatches = nullptr;
  int nchunks = 0, npatches = 0;
  int npatch_items = 0;            // patch work items (mfc::inst_args)
  int npatch_items_max = 0;        // the most for any number of lanes
  int npatch_max = 0;              // patches the buffers hold
  patch_plan plans[3] = {};        // for PLAN_LANES, from the initial particles
  mfc::grid_geo *geo = nullptr;    // adaptive grid: the geometry of the last step (device)
  mfc::batch_work work(int c) const {
    return {dargs + c, 1, dtiles, ntiles, dchunks, nchunks, dpatches, npatches, recs[0].f32, variant(),
            k.adaptive != 0, k.pse != 0, general(), k.rothlin != 0};
  }

  template <class T>
  int alloc(T **p, size_t n) {
    void *q = nullptr;
    if (n == 0) n = 1;
    hipError_t e = hipMalloc(&q, n * sizeof(T));
    if (e != hipSuccess) return mfc::fail(MFC_E_NOMEM, std::string("hipMalloc: ") + hipGetErrorString(e));
    allocs.push_back(q);
    *p = (T *)q;
    return MFC_OK;
  }
};

// the state arrays of one set, carved from one allocation in the order of dstate
// (DSTATE_DOUBLES doubles, then flags and id), so that a set is one contiguous block
size_t state_block_bytes(int N);
void carve_state(void *base, int N, mfc::dstate &d);
// the positional arrays (nx, ny, p, rxx, rxy, ryy), one contiguous block
size_t positional_block_bytes(int N);
void carve_positional(void *base, int N, mfc::dpositional &p);
// queue one step: set[c] -> set[1-c]
// steps per captured hipGraph (even: a graph starts and ends on the same buffer parity)
constexpr int GRAPH_STEPS = 8;
void enqueue_step(mfc_sim *s, int c);
// the binning and the records of the current state, recomputed when keys_fresh is false
int ensure_keys(mfc_sim *s);
// the work tables of the sort launch and of the interaction launch over a group of instances
void sort_items(std::vector<int2> &items, mfc_sim *const *sims, int n);
void patch_items(std::vector<int2> &items, mfc_sim *const *sims, int n);
// threads per particle of the interaction for n handles stepped together, and a handle's patches
// for that
int interaction_lanes(const mfc_sim *const *sims, int n);
const patch_plan &patches_for(const mfc_sim *s, int lanes);
void set_patches(mfc_sim *s, int lanes);
// copies the handle's descriptors to where the kernels read them (synchronises its stream)
int upload_descriptors(mfc_sim *s);
// whether the current state's h is the same for every particle (host copy of the field)
void check_uniform_h(mfc_sim *s, const double *h);
void finish_steps(mfc_sim *s);
// nsteps steps of a handle whose binning is fresh (hipGraph replays where there are enough)
int queue_steps(mfc_sim *s, int nsteps);
int check_tuning(const mfc_tuning *t);
// the batched kernels' view of a handle for start parity c
mfc::inst_args instance_args(const mfc_sim *s, int c);
// the grid of the last step: the creation geometry for a locked grid, the device's record for
// an adaptive one (synchronises the handle's stream)
int current_geometry(const mfc_sim *s, mfc::grid_geo &g);
