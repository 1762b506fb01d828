// mfc_kernels.h — launch interface of the gfx950 kernels of one SPH cutting step.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "mfc_device.h"

namespace mfc {

// one set of the permuted persistent particle fields, structure of arrays in storage order
struct dstate {
  double *px, *py, *vx, *vy;
  double *sxx, *sxy, *syy, *szz;
  double *rho, *T, *eps, *epsd, *h;
  double *fcx, *fcy, *ftx, *fty;
  double *ptx, *pty, *vtx, *vty, *rhot, *stxx, *stxy, *styy, *stzz, *Tt;
  int *flags, *id;
};
constexpr int DSTATE_DOUBLES = 27;

// binning scratch and cell table
struct dbins {
  int *key;          // cell id per particle in the current (unsorted) order
  int *key_sorted;   // cell id per particle in sorted order (= reference's sorted hash)
  int *offsets;      // num_cell + 1 exclusive prefix sums: cell c = [offsets[c], offsets[c+1])
  int *bucket;       // particle indices grouped by cell, unordered inside a cell
  int *tags;         // sorted position -> current position and flags of the record there (make_tag)
  int *spos;         // current position -> sorted position (the reverse mode's replay; else null)
  int *bsum;         // particles counted in each scan chunk of cells (the start state's)
  int *bsum_next;    // the same for the next step: cleared by the sort, counted by the interaction
  int2 *clist;       // per scan chunk, (current position, cell id) of the particles counted in
                     // its cells, in arrival order (ccap entries per chunk; a chunk that counts
                     // more finds them by a pass over all particles)
  int ccap;
  int *pcnt;         // per patch of cells: particles of the next step's start state in it
  int2 *plist;       // the interaction's work: (patch, part) for every patch_slots particles of a
                     // patch, in ascending order (written by the sort launch, which clears pcnt)
  int *plen;         // its length
  int *plen_next;    // the next step's, cleared by the sort launch
  int *offsets_r;    // MFC_GRID_ROTHLIN: the ranges rebuilt from the sorted ids (the step reads these)
  unsigned long long *clamped;  // binned particles whose position lay outside the grid on an axis
};

// positional (not permuted) arrays, as particle_gpu::{n,p,R} (particle_gpu.h:39-47)
struct dpositional {
  double *nx, *ny, *p, *rxx, *rxy, *ryy;
  double *nx_out, *ny_out;  // where the step's normals go: nx and ny, or (the reverse mode's replay,
                            // which keeps the normals each step starts from) arrays of their own
};

constexpr int REC = 16;    // doubles per neighbour record (FP64; FP32C: floats)
constexpr int ACC_N = 14;  // neighbour sums per particle

// neighbour records in the storage order of the start state (sorted index j is particle
// tag_index(tags[j])): rec (FP64 path, 128 bytes: x y flags h u v rho vol Axx Axy Ayy Rxx Rxy Ryy c T) or
// rec32 (FP32C path, 64 bytes: x y in FP64, then u v rho vol Axx Axy Ayy c Rxx Rxy Ryy T), and the
// flags of the record, vfl. h is the state's (it does not change). The interaction writes those
// of the next step into the other of two sets
struct drecords {
  bool f32;
  double *rec;
  float4 *rec32;
  int *vfl;
};
constexpr int REC32_PIECES = 4;  // float4 per FP32C record

// The interaction runs over patches: rectangles of cells whose particles one work-group of TILE
// threads takes, `lanes` threads per particle. The records of every window candidate of a patch
// (its cells and two more on each side) are staged in LDS: up to patch_cap of them; a patch with
// more candidates reads them from memory. The FP64 kernel with
// one thread per particle gets three work-groups to a CU only up to 53,760 bytes (LDS is given out
// in pieces of 1,280): with 484 candidates, 54,256 bytes, there were two, and a step of 197k particles
// took 109 us instead of 102, of 500k with PSE 350 instead of 299.
constexpr int PATCH_TABLE = 256;  // cell starts a patch holds in LDS: (patch_w + 4) (patch_s + 5) at most
constexpr int PATCH_COLS = 24;    // patch_w + 4 at most
// The general variant (gen) copies less of each (of 128 bytes 64, of 64 32, with several threads per
// particle 16 of both, and the tag), so that as many work-groups run at once.
__host__ __device__ constexpr int patch_cap(bool f32, int lanes, bool gen) {
  return gen ? (f32 ? 1080 : lanes > 1 ? 1408 : 760) : lanes > 1 ? 256 : f32 ? 576 : 479;
}
// What the patches of a full lattice may have of that: a body in compression has more particles in a
// cell, and a few patches over the copy's room make the launch twice as long (in FP32C, planned up to
// 512 of 512, steps of the impact of 131k particles went from 65 to 128 us behind the shock and of
// the rings of 171k from 63 to 113, now 81 and 63)
__host__ __device__ constexpr int patch_plan_cap(bool f32, int lanes, bool gen) {
  return patch_cap(f32, lanes, gen) * 12 / 13;
}

// tool-force reduction: the interaction flags the groups of 64 particles (storage order) in which
// some contact or friction force is not zero; the next step's sort launch sums those groups from
// the state (the others' sums are zero) and its interaction launch adds the group sums up, or one
// kernel does both after the last step. F is appended to the history
struct dforce {
  double *partials;      // 4 per group of 64 particles: sum fc.x, fc.y, ft.x, ft.y
  int *gflag;            // per group: 1 when it has a force
  double *force_last;    // F of the last step
  double *hist;          // force history, 2 per step, cap entries
  int64_t cap;
  int64_t *ctr;          // steps recorded
  int *pending;          // 1: the force of the step that produced the start state is not yet reduced
  int *pending_next;     // the same for the state this step produces
};

// the particle flags of the state (FIXED, BLANKED, TOOL)
constexpr int FLAG_MASK = MFC_FLAG_FIXED | MFC_FLAG_BLANKED | MFC_FLAG_TOOL;

// internal flag: some value of the particle's neighbour record is NaN or Inf
constexpr int FLAG_NONFINITE = 8;

// launch variant of the interaction (results are identical for every variant)
struct variant {
  int lanes;  // threads per particle: 1, 4 or 8
  int chunk;  // work items per XCD chunk of the interaction's map (1..XCD_CHUNK_MAX)
};

// The secant results of a run that the reverse mode recorded: the next step's place (a double per
// particle in sorted order, written where the particle returns: dl, or -dl where its last update
// folded) and how many steps have one. Passed on from step to step on the device as the tool is,
// since a captured step cannot be told its number.
struct return_tape {
  double *at;
  long long left;
};

// one instance of a batch as the batched kernels see it (an array of these lives in device
// memory, one per instance and step parity)
struct inst_args {
  dev_consts k;
  dstate cur, nxt;  // state at the start of the step, and the sorted copy updated by the step
  dbins b;
  dpositional pos;
  drecords r, rn;   // records of the start state, and of the next step's
  const mfc_tool_state *tool_in;
  mfc_tool_state *tool_out;
  dforce f;
  double *acc_out;  // when set, the interaction also stores its neighbour sums there (ACC_N
                    // arrays of N doubles), then each particle's secant result (N doubles,
                    // end_update); the reverse mode's replay keeps them, and takes the secant
                    // results from the tape where it has some instead of iterating again
  grid_geo *geo;  // adaptive grid: the geometry of the current step (written by the device)
  int ntiles;   // particle tiles of TILE
  int nscan;    // scan chunks of the cell table
  int npatch_items;  // patch work items of the instance: item q takes the entries q, q + npatch_items, ... of plist
  const return_tape *tape_in;
  return_tape *tape_out;
};

// the work of one batched step: instance descriptors and (instance, block) work tables
struct batch_work {
  const inst_args *args;  // n descriptors, device memory
  int n;
  const int2 *tiles;      // (instance, particle tile) for every tile of every instance
  int ntiles;
  const int2 *chunks;     // (instance, scan chunk) for every chunk of every cell table, and each
                          // instance's SORT_ITEM_* (push_sort_items)
  int nchunks;
  const int2 *patches;    // (instance, patch item), and each instance's SORT_ITEM_FORCE first
  int npatches;
  bool f32;
  variant v;
  bool adaptive;          // some instance has an adaptive grid (a geometry pass starts the step)
  bool pse;               // some instance conducts heat by PSE
  bool general;           // some instance needs the general variant of the interaction
  bool rothlin;           // some instance uses grid_gpu_rothlin's cell ranges (a pass after the sort)
};

// one step of every instance of a batch: 2 launches, and its phases. The
// cell ids, chunk lists, chunk sums and neighbour records of a step's start state are computed by
// the previous step's interaction; launch_batch_hash and launch_batch_records compute them from
// the state itself (chunk sums zeroed before); launch_batch_patch_counts counts its patches again
// (counts zeroed before), for another number of lanes
void launch_batch_step(const batch_work &w, hipStream_t s);
void launch_batch_hash(const batch_work &w, hipStream_t s);
void launch_batch_patch_counts(const batch_work &w, hipStream_t s);
void launch_batch_binning(const batch_work &w, hipStream_t s);
void launch_batch_records(const batch_work &w, hipStream_t s);
// with events t0 and t1 the launch records the kernel's own start and end in them
// (hipExtLaunchKernelGGL), which times the kernel without the gap before it
void launch_batch_interact(const batch_work &w, hipStream_t s, hipEvent_t t0 = nullptr, hipEvent_t t1 = nullptr);
void launch_batch_force(const batch_work &w, hipStream_t s);
// work items of the sort launch beside the chunks (negative, where a chunk's index stands)
constexpr int SORT_ITEM_TOOL = -1;     // the tool's move
constexpr int SORT_ITEM_FORCE = -2;    // and below: the group sums of a block of FORCE_GROUPS groups
constexpr int FORCE_GROUPS = 64;
constexpr int SORT_ITEM_PATCHES = -(1 << 30);  // and below: the interaction's work from a section of patches
constexpr int PLIST_SECTION = 1024;
constexpr int PATCH_ITEM_FORCE = -1;   // of the interaction launch: the sum of the group sums
int scan_chunk_cells();
// entries of a scan chunk's particle list: 4 particles per cell of the chunk (a cell holds
// about 2.25 at the lattice spacing), at most N
int chunk_list_cap(int N);

// Usui wear rate of state st: out = {min, max, sum, count} over the particles in contact
// (part: 4 doubles per tile of scratch)
void launch_tool_wear(const dev_consts &k, const dstate &st, const dpositional &pos, double K, double alpha,
                      double tvx, double tvy, double *part, double *out, hipStream_t s);
int scan_blocks(int num_cell);
// out[i nc + c] = src[c][first + i], i < count (out may be pinned host memory)
void launch_interleave(int nc, const double *const *src, int64_t first, int64_t count, double *out, hipStream_t s);
void launch_device_math(int fn, const double *x, const double *y, double *out, int64_t n, hipStream_t s);

}  // namespace mfc
