// mfc_adjoint.hip — reverse mode of the SPH cutting step on gfx950: gradients of the mean tool
// force over a window of steps with respect to the Johnson-Cook constants and the friction
// coefficient, theta = (A, B, n, C, m, mu).
//
// Tape: the state at the start of every K-th step (state block, positional block, stale cell
// ids of blanked particles, tool) is copied into a checkpoint. The backward pass walks the
// checkpoint segments from last to first. Each segment is replayed forward with the step kernels,
// whose descriptors (one per step of the segment) point each step's output at a slot of its own:
// the next slot's start state and normals, this slot's sort (sorted cell ids, cell ranges,
// permutation and its inverse, list of patches), its neighbour sums and secant results and the tool.
// So the replay is two launches per step and nothing is computed or copied again for the reverse
// steps, which take two each:
//   kb_adj_tail     the VJP of the record and predictor of the step after (record_vjp) and the
//                   gather of its result through the inverse of its sort, then the VJP of
//                   everything after the neighbour sums of this step (tail_vjp), per particle, its
//                   record for the pull, and the per-tile theta partials
//   kb_adj_pull     VJP of the neighbour sums with respect to the records: each particle pulls the
//                   contributions of the pairs it takes part in over its symmetric 5 x 5 cell
//                   window, in a fixed order (no atomics); one more work-group per instance adds up
//                   the theta partials
// and kb_adj_record takes the segment's first step back to the storage order of its start state.
// (With a copy of each replayed state, and the binning, sort, sorted state and records of the
// reversed step computed again, a replayed and reversed step took 12 launches, and launching them
// took longer than running them.)
// The positional contact normal (read by the friction heat of the next step at the same sorted
// index) carries its adjoint from step to step without permutation, like its forward value.
//
// A group of instances that ran the same taped forward (one handle, or the instances of a
// batch) is reversed together: every phase, the checkpoint copies included, is one launch over
// the group's work tables, with per-instance descriptors in device memory, as the batched forward
// step runs. Each instance computes exactly what it computes alone.
//
// Derivatives follow the smooth map of promote_fp64 = 1 with a tight secant tolerance; the
// handle must use FP64 records.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstring>
#include <memory>
#include <vector>

#include "mfc_adjoint.h"
#include "mfc_pairs.h"
#include "mfc_sim.h"

namespace mfc {

namespace {

using namespace adj;

}  // namespace

// a checkpoint of one instance: state block, positional block, cell ids, tool
struct snapshot {
  char *state;            // state block (state_block_bytes)
  char *pos;              // positional block
  int *keys;              // cell ids of the previous step (kept by blanked particles)
  mfc_tool_state *tool;
};

namespace {

int padded(int ntiles) { return ((ntiles + 7) / 8) * 8; }

static_assert(L_N == ACC_N, "a replay slot holds the interaction's neighbour sums in the tail's order");

constexpr int LAM = 16;  // doubles per particle of lam_acc (ACC_N, padded to whole 16-byte pieces)

// one instance of the backward pass as its kernels see it (device memory, one per instance). The
// slots of the segment's steps follow each other in each array; state has one more, for the
// last step's end state, as have normal and tool
struct adj_args {
  dev_consts k;
  int ntiles;
  char *state;                      // start states in storage order (state_block_bytes each)
  size_t state_bytes;
  double *normal;                   // normals before the step, nx then ny (2 N)
  int *tags, *spos, *key_sorted;    // N each
  int *offsets;                     // num_cell + 1 each
  int2 *plist;                      // list of patches (list_len each) and its length
  int *plen;
  int list_len, ncell1;
  mfc_tool_state *tool;             // before the step's move
  return_tape *tape;                // of the step's secant results
  double *returns;                  // those of the whole run (N a step), or null
  int K;                            // steps of a segment
  double *acc;                      // neighbour sums and secant results, (ACC_N + 1) N each
  double *lam;                      // adjoint of a segment's end state, in the storage order of the next one's start
  double *lam_n;                    // adjoint of the positional normals
  double *g_s[2];                   // adjoint of the sorted start state by parity of the slot
  double *lam_acc, *rec, *g_rec;    // LAM, REC_DOUBLES and REC_DOUBLES per particle, sorted order
  double *theta_part, *theta_acc;
  double Fb[2];                     // cotangent over the window length
  const snapshot *ckpt;
  int *chunk_sums[2], *pcnt;        // the handle's binning scratch
  int nscan, npatch;
};

// an instance's descriptor read through the constant address space: the pointers loaded from it
// are then known to point to global memory, and the kernels use global instead of flat loads
// (a flat load also holds up every wait for an LDS or scalar load)
#define MFC_ADJ_ARGS(d, q) const __attribute__((address_space(4))) adj_args &d = \
    *(const __attribute__((address_space(4))) adj_args *)(D + (q))

// ------------------------------------------------------------------ checkpoint copies
// the checkpoint of segment sg into slot 0, and the binning scratch cleared for the
// binning of that state. Grid (copy_blocks, instances).
__global__ __launch_bounds__(256) void kb_adj_restore(const adj_args *__restrict__ D, int sg) {
  MFC_ADJ_ARGS(d, blockIdx.y);
  const snapshot sn = d.ckpt[sg];
  const size_t stride = (size_t)gridDim.x * blockDim.x;
  const size_t i0 = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  const size_t N = d.k.N;
  uint64_t *st = (uint64_t *)d.state;
  const uint64_t *src = (const uint64_t *)sn.state;
  for (size_t q = i0; q < d.state_bytes / sizeof(uint64_t); q += stride) st[q] = src[q];
  const double *pos = (const double *)sn.pos;  // nx, ny first
  for (size_t q = i0; q < 2 * N; q += stride) d.normal[q] = pos[q];
  for (size_t q = i0; q < N; q += stride) d.key_sorted[q] = sn.keys[q];
  for (size_t q = i0; q < (size_t)d.nscan; q += stride) d.chunk_sums[0][q] = d.chunk_sums[1][q] = 0;
  for (size_t q = i0; q < (size_t)d.npatch; q += stride) d.pcnt[q] = 0;
  if (i0 == 0) {
    d.tool[0] = *sn.tool;
    d.plen[0] = 0;
    const return_tape t = {d.returns ? d.returns + (size_t)sg * d.K * N : nullptr, d.returns ? d.K : 0};
    d.tape[0] = t;
  }
}

// a checkpoint of the current state (the sources of one handle), and where the following steps
// record their secant results
__global__ __launch_bounds__(256) void k_adj_save(snapshot sn, const uint64_t *__restrict__ state, size_t state_words,
                                                  const uint64_t *__restrict__ pos, size_t pos_words,
                                                  const int *__restrict__ keys, int N,
                                                  const mfc_tool_state *__restrict__ tool, return_tape *tape,
                                                  return_tape t) {
  const size_t stride = (size_t)gridDim.x * blockDim.x;
  const size_t i0 = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  for (size_t q = i0; q < state_words; q += stride) ((uint64_t *)sn.state)[q] = state[q];
  for (size_t q = i0; q < pos_words; q += stride) ((uint64_t *)sn.pos)[q] = pos[q];
  for (size_t q = i0; q < (size_t)N; q += stride) sn.keys[q] = keys[q];
  if (i0 == 0) {
    *sn.tool = *tool;
    *tape = t;
  }
}

// ------------------------------------------------------------------ B1: per-particle tail
__device__ inline const double *slot_state(const __attribute__((address_space(4))) adj_args &d, int slot) {
  return (const double *)(d.state + (size_t)slot * d.state_bytes);
}
__device__ inline const int *slot_flags(const __attribute__((address_space(4))) adj_args &d, int slot) {
  return (const int *)(slot_state(d, slot) + (size_t)DSTATE_DOUBLES * d.k.N);
}
// EOS pressure of the predicted density (0 for a tool particle: no sum reads it)
__device__ inline double eos_pressure(adj_consts &k, const double *s, int flags) {
  if (flags & MFC_FLAG_TOOL) return 0.;
  const double rho = flags & MFC_FLAG_BLANKED ? s[TS_RHO] : s[TS_RHO] + 0.5 * k.dt * s[TS_RHOT];
  return k.c0 * k.c0 * (rho - k.rho0);
}

// step `slot` of the segment; last: the segment's last step, whose end state's adjoint is in lam
// (else it comes from step slot + 1); in_win: its force is in the loss window. lam_n: adjoint of the positional normal written by this step
// (in) and of the one read by it (out)
__global__ __launch_bounds__(TILE) void kb_adj_tail(const adj_args *__restrict__ D, const int2 *__restrict__ work,
                                                    int nwork, int slot, int last, int in_win) {
  const int w = xcd_tile(blockIdx.x, nwork);
  if (w < 0) return;
  const int2 it = work[w];
  MFC_ADJ_ARGS(d, it.x);
  adj_consts &k = d.k;
  const int t = it.y;
  const int i = t * TILE + threadIdx.x;
  const size_t N = k.N;
  double th[6] = {0., 0., 0., 0., 0., 0.};
  if (i < k.N) {
    double ob[TS_N];
    if (last) {
#pragma unroll
      for (int q = 0; q < TS_N; q++) ob[q] = d.lam[q * N + i];
    } else {  // particle i of this step's end state is at a in the next step's sorted order
      const int a = d.spos[(size_t)(slot + 1) * N + i];
      const double *__restrict__ st = slot_state(d, slot + 1);
      const double *__restrict__ gs = d.g_s[(slot + 1) & 1];
      double s[TS_N], br[REC_DOUBLES];
#pragma unroll
      for (int q = 0; q < TS_N; q++) { s[q] = st[q * N + i]; ob[q] = gs[q * N + a]; }
      const double2 *__restrict__ g2 = reinterpret_cast<const double2 *>(d.g_rec + (size_t)REC_DOUBLES * a);
#pragma unroll
      for (int q = 0; q < REC_DOUBLES / 2; q++) { const double2 v = g2[q]; br[2 * q] = v.x; br[2 * q + 1] = v.y; }
      const int fl = slot_flags(d, slot + 1)[i] & FLAG_MASK;
      record_vjp(k, s, fl, eos_pressure(k, s, fl), br, ob);
    }
    const unsigned sidx = tag_index(d.tags[(size_t)slot * N + i]);
    const double *__restrict__ st = slot_state(d, slot);
    tail_in in;
#pragma unroll
    for (int q = 0; q < TS_N; q++) in.s[q] = st[q * N + sidx];
    in.flags = slot_flags(d, slot)[sidx] & FLAG_MASK;
    in.p = eos_pressure(k, in.s, in.flags);
    const double *__restrict__ nn = d.normal + (size_t)slot * 2 * N;
    in.nx = nn[i];
    in.ny = nn[N + i];
    in.pse_flag_zero = k.pse_quirk && i >= k.N / 2;
    const double *__restrict__ acc = d.acc + (size_t)slot * (L_N + 1) * N;
#pragma unroll
    for (int q = 0; q < L_N; q++) in.acc[q] = acc[q * N + i];
    in.dl_rec = acc[L_N * N + i];
    double p = in.p, R3[3] = {0., 0., 0.}, rec[REC_DOUBLES];
    record_fwd(k, in.s, in.flags, p, R3, rec);
    rec[R_FLAGS] = bits_to_double(in.flags);
    double2 *__restrict__ rdst = reinterpret_cast<double2 *>(d.rec + (size_t)REC_DOUBLES * i);
#pragma unroll
    for (int q = 0; q < REC_DOUBLES / 2; q++) rdst[q] = make_double2(rec[2 * q], rec[2 * q + 1]);
    const double nbx = d.lam_n[i], nby = d.lam_n[N + i];
    tail_grad g;
    tail_vjp(k, d.tool[slot + 1], in, ob, nbx, nby, in_win ? d.Fb[0] : 0., in_win ? d.Fb[1] : 0., g, nullptr);
    double *__restrict__ gs = d.g_s[slot & 1];
#pragma unroll
    for (int q = 0; q < TS_N; q++) gs[q * N + i] = g.s[q];
    double2 *__restrict__ ldst = reinterpret_cast<double2 *>(d.lam_acc + (size_t)LAM * i);
#pragma unroll
    for (int q = 0; q < L_N / 2; q++) ldst[q] = make_double2(g.acc[2 * q], g.acc[2 * q + 1]);
    d.lam_n[i] = g.nx;
    d.lam_n[N + i] = g.ny;
#pragma unroll
    for (int q = 0; q < 6; q++) th[q] = g.theta[q];
  }
  // theta partials: halving-stride tree per tile
  __shared__ double red[6][TILE];
#pragma unroll
  for (int q = 0; q < 6; q++) red[q][threadIdx.x] = th[q];
  for (int s = TILE / 2; s > 0; s >>= 1) {
    __syncthreads();
    if (threadIdx.x < s) {
#pragma unroll
      for (int q = 0; q < 6; q++) red[q][threadIdx.x] = red[q][threadIdx.x] + red[q][threadIdx.x + s];
    }
  }
  if (threadIdx.x == 0) {
#pragma unroll
    for (int q = 0; q < 6; q++) d.theta_part[6 * t + q] = red[q][0];
  }
}

// adds the step's theta partials of an instance to its running totals: lane l sums the tiles l,
// l + TILE, ... in ascending order, lane sums reduced by halving strides; red: 6 TILE doubles of LDS
__device__ inline void add_theta(const __attribute__((address_space(4))) adj_args &d, double (*red)[TILE]) {
  double a[6] = {0., 0., 0., 0., 0., 0.};
  for (int u = threadIdx.x; u < d.ntiles; u += TILE)
#pragma unroll
    for (int q = 0; q < 6; q++) a[q] = a[q] + d.theta_part[6 * u + q];
#pragma unroll
  for (int q = 0; q < 6; q++) red[q][threadIdx.x] = a[q];
  for (int s = TILE / 2; s > 0; s >>= 1) {
    __syncthreads();
    if (threadIdx.x < s) {
#pragma unroll
      for (int q = 0; q < 6; q++) red[q][threadIdx.x] = red[q][threadIdx.x] + red[q][threadIdx.x + s];
    }
  }
  if (threadIdx.x < 6) d.theta_acc[threadIdx.x] = d.theta_acc[threadIdx.x] + red[threadIdx.x][0];
}

// ------------------------------------------------------------------ B2: pull over pairs
// For each window member a of particle b, both kinds of pair that link them: the pairs (a, b) of
// a's sums that include b, with the adjoint of a's sums, and the pairs (b, a) of b's own sums,
// with b's adjoint, in one evaluation (pair_vjp_sym). PULL_LANES neighbouring lanes share a
// particle: they list its pairs in the window's order, lane r takes the pairs r, r + PULL_LANES,
// ..., and the lanes' partial sums are added by a butterfly of shuffles, which gives every lane the
// same bits (((g0 + g1) + (g2 + g3)) + ...). The count is fixed, and so is the lanes' split of a
// window, so that an instance's gradient has the same bits alone and in a batch, whatever the patches.
// A work-group takes a part of a patch of cells, as the interaction does, with the records and the
// adjoints of the sums of its window candidates staged in LDS (240 bytes each; three work-groups to a
// CU): read from memory per pair, by one work-group per 32 particles of the sorted order, they were 30
// gathers of 64 scattered lines, and the pass took 95 us at 37.5k particles, now 41.
constexpr int PULL_LANES = 8;
constexpr int PULL_AT_ONCE = TILE / PULL_LANES;  // particles a work-group takes at once
constexpr int PULL_CAP = 208;  // window candidates a work-group stages: 5 x 5 cells at hdx 1.5 have 196 at most
constexpr int PULL_PIECES = REC_DOUBLES / 2 + ACC_N / 2;  // 16-byte pieces: the record, then the adjoints

struct pull_mem {
  double2 piece[PULL_PIECES][PULL_CAP + 1];
  int table[PATCH_TABLE];
  int col_first[PATCH_COLS + 1], col_shift[PATCH_COLS], own_first[PATCH_COLS + 1];
  unsigned char list[TILE / PULL_LANES][64];
};

// a pair of window members by their flags: whether the sums of a take b when it is in a's support
// (and not at the same place), and those of b take a
struct pull_pair {
  bool of_a, of_b;
};
__device__ inline pull_pair pull_flags(adj_consts &k, int fa, int fb) {
  const bool blank = (fa | fb) & MFC_FLAG_BLANKED, pse = k.pse != 0;
  return {!blank && (!pse || !(fa & MFC_FLAG_TOOL)), !blank && (!pse || !(fb & MFC_FLAG_TOOL))};
}

// the lanes' sums of a particle added and written (every lane of the particle calls it)
__device__ inline void pull_store(double *gb, int r, double *__restrict__ dst) {
#pragma unroll
  for (int st = 1; st < PULL_LANES; st <<= 1)
#pragma unroll
    for (int q = 0; q < REC_DOUBLES; q++) gb[q] = gb[q] + __shfl_xor(gb[q], st, PULL_LANES);
  if (r == 0) {
#pragma unroll
    for (int q = 0; q < REC_DOUBLES / 2; q++)
      reinterpret_cast<double2 *>(dst)[q] = make_double2(gb[2 * q], gb[2 * q + 1]);
  }
}

// where the pull reads the window members from (piece p, 16 bytes, of member j): the patch's copy in
// LDS, by index in the copy, or memory, by sorted index
struct pull_lds {
  const pull_mem &m;
  __device__ inline double2 piece(int p, int j) const { return m.piece[p][j]; }
};
struct pull_memory {
  const double2 *rec, *lam;
  __device__ inline double2 piece(int p, int j) const {
    return p < REC_DOUBLES / 2 ? rec[(size_t)j * (REC_DOUBLES / 2) + p] : lam[(size_t)j * (LAM / 2) + p - REC_DOUBLES / 2];
  }
};

// the pairs of particle b (index in src; all h equal) over its window, lane r of its lanes; gl: its
// first lane in the wave, list: 64 bytes of LDS of its own
template <class SRC>
__device__ inline void pull_particle(adj_consts &k, const SRC &src, int b, const window &w, int r, int gl,
                                     unsigned char *list, double *gb) {
  auto value = [&](int j, int q) { const double2 v = src.piece(q / 2, j); return q % 2 ? v.y : v.x; };
  auto load = [&](int j, double *rec, double *la) {
#pragma unroll
    for (int q = 0; q < REC_DOUBLES; q++) rec[q] = value(j, q);
#pragma unroll
    for (int q = 0; q < L_N; q++) la[q] = value(j, REC_DOUBLES + q);
  };
#pragma unroll
  for (int q = 0; q < REC_DOUBLES; q++) gb[q] = 0.;
  const double2 pb = src.piece(0, b);
  const int fb = double_to_bits(value(b, R_FLAGS));
  const bool pse = k.pse != 0, tool_b = fb & MFC_FLAG_TOOL;
  const bool pse_b = !(fb & MFC_FLAG_BLANKED) && pse && k.thermal_wp;
  const double ta_b = pse ? 0. : (tool_b ? k.alpha_tool : k.alpha_wp);
  for (int b0 = 0; b0 < w.total; b0 += 64) {
    const int nb = w.total - b0 < 64 ? w.total - b0 : 64;
    int cnt = 0;
    for (int u0 = 0; u0 < nb; u0 += PULL_LANES) {
      const bool in = u0 + r < nb;
      const int t = in ? u0 + r : nb - 1, a = w.at(b0 + t);
      const double2 pa = src.piece(0, a);
      const int fa = double_to_bits(value(a, R_FLAGS));
      const double dx = pa.x - pb.x, dy = pa.y - pb.y, rr2 = dx * dx + dy * dy;
      const pull_pair pm = pull_flags(k, fa, fb);
      const bool hit = in && a != b && pm.of_a && pm.of_b && rr2 < 4 * k.h0 * k.h0 && rr2 >= 1e-8;
      const unsigned bits = (unsigned)(__ballot(hit) >> gl) & ((1u << PULL_LANES) - 1u);
      if (hit) list[cnt + __popc(bits & ((1u << r) - 1u))] = (unsigned char)t;
      cnt += __popc(bits);
      if (pse && in && a != b) {
        const bool pse_a = !(fa & MFC_FLAG_BLANKED) && k.thermal_wp;
        if (pse_a || pse_b) {
          double ra[REC_DOUBLES], la[LAM], rb[REC_DOUBLES], lb[LAM], dummy[REC_DOUBLES];
          load(a, ra, la);
          load(b, rb, lb);
          if (pse_a) pse_vjp(k, ra, rb, la[L_TPSE], false, true, dummy, gb);
          if (pse_b) pse_vjp(k, rb, ra, lb[L_TPSE], true, false, gb, dummy);
        }
      }
    }
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");  // the list, by lanes of the same wave
    __builtin_amdgcn_wave_barrier();
    for (int p = r; p < cnt; p += PULL_LANES) {
      // both records are read where a value is used: held in registers across the pair (the
      // particle's own across the pairs) they spill
      const int a = w.at(b0 + list[p]);
      const bool tool_a = double_to_bits(value(a, R_FLAGS)) & MFC_FLAG_TOOL;
      // the mechanical sums of both take a pair without a tool particle; each conduction sum
      // counts where its particle conducts
      const double ta_a = pse ? 0. : (tool_a ? k.alpha_tool : k.alpha_wp);
      auto adj = [&](int j, double ta, int q) { return q == L_TL && ta == 0. ? 0. : value(j, REC_DOUBLES + q); };
      asm volatile("" ::: "memory");
      pair_vjp_sym(
          k, [&](int q) { return value(b, q); }, [&](int q) { return value(a, q); }, !tool_a && !tool_b,
          ta_a != 0. || ta_b != 0., [&](int q) { return adj(b, ta_b, q); }, [&](int q) { return adj(a, ta_a, q); }, gb);
    }
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
  }
}

// one entry of the list from the records in memory: what the staged path does not take (more
// candidates than the stage holds, an h that is not uniform, entries past the work items). With a
// uniform h the same bits; else each pair's two terms one after the other, with the h of each
__device__ inline void pull_rest(pull_mem &m, const adj_args *__restrict__ D, int inst, int slot, int patch, int part) {
  MFC_ADJ_ARGS(d, inst);
  adj_consts &k = d.k;
  const size_t N = k.N;
  const int *__restrict__ offsets = d.offsets + (size_t)slot * d.ncell1, *__restrict__ keys = d.key_sorted + (size_t)slot * N;
  const int nrb = patch_rows(k), pc = patch / nrb, pr = patch - pc * nrb;
  const int r0 = pr * k.patch_s, r1 = r0 + k.patch_s < k.gny ? r0 + k.patch_s : k.gny;
  const int c0 = pc * k.patch_w, c1 = c0 + k.patch_w < k.gnx ? c0 + k.patch_w : k.gnx;
  const int lane = threadIdx.x & 63, r = lane % PULL_LANES, gl = lane - r;
  const double *__restrict__ rec = d.rec, *__restrict__ lam = d.lam_acc;
  for (int s0 = 0; s0 < k.patch_slots; s0 += PULL_AT_ONCE) {
    int n = part * k.patch_slots + s0 + (int)threadIdx.x / PULL_LANES, b = -1;
    for (int c = c0; c < c1 && b < 0; c++) {
      const int first = offsets[c * k.gny + r0], count = offsets[c * k.gny + r1] - first;
      if (n < count) b = first + n;
      n -= count;
    }
    if (b < 0) return;  // whole groups of lanes
    double gb[REC_DOUBLES];
    const window w = make_window(k, offsets, keys[b]);
    if (k.uniform_h) {
      const pull_memory src = {reinterpret_cast<const double2 *>(rec), reinterpret_cast<const double2 *>(lam)};
      pull_particle(k, src, b, w, r, gl, m.list[threadIdx.x / PULL_LANES], gb);
    } else {
      const double *rb = rec + (size_t)REC_DOUBLES * b, *lb = lam + (size_t)LAM * b;
      double dummy[REC_DOUBLES];
#pragma unroll
      for (int q = 0; q < REC_DOUBLES; q++) gb[q] = 0.;
      const int fb = double_to_bits(rb[R_FLAGS]);
      const bool pse = k.pse != 0, tool_b = fb & MFC_FLAG_TOOL;
      const double ta_b = pse ? 0. : (tool_b ? k.alpha_tool : k.alpha_wp);
      const bool pse_b = !(fb & MFC_FLAG_BLANKED) && pse && k.thermal_wp;
      for (int t = r; t < w.total; t += PULL_LANES) {
        const int a = w.at(t);
        if (a == b) continue;
        asm volatile("" ::: "memory");  // b's record is read again for each pair: kept, it spills
        const double *ra = rec + (size_t)REC_DOUBLES * a, *la = lam + (size_t)LAM * a;
        const int fa = double_to_bits(ra[R_FLAGS]);
        const bool tool_a = fa & MFC_FLAG_TOOL;
        const double dx = ra[R_X] - rb[R_X], dy = ra[R_Y] - rb[R_Y], rr2 = dx * dx + dy * dy;
        const pull_pair pm = pull_flags(k, fa, fb);
        const double ha = ra[R_H], hb = rb[R_H];
        const bool of_a = pm.of_a && rr2 < 4 * ha * ha && rr2 >= 1e-8, of_b = pm.of_b && rr2 < 4 * hb * hb && rr2 >= 1e-8;
        const bool pse_a = !(fa & MFC_FLAG_BLANKED) && pse && k.thermal_wp;
        const double ta_a = pse ? 0. : (tool_a ? k.alpha_tool : k.alpha_wp);
        if (of_a) pair_vjp(k, ra, rb, tool_a, tool_b, ta_a, la, false, true, dummy, gb);
        if (pse_a) pse_vjp(k, ra, rb, la[L_TPSE], false, true, dummy, gb);
        asm volatile("" ::: "memory");
        if (of_b) pair_vjp(k, rb, ra, tool_b, tool_a, ta_b, lb, true, false, gb, dummy);
        if (pse_b) pse_vjp(k, rb, ra, lb[L_TPSE], true, false, gb, dummy);
      }
    }
    pull_store(gb, r, d.g_rec + (size_t)REC_DOUBLES * b);
  }
}

// returns false, with nothing done, for an entry that pull_rest takes
__device__ inline bool pull_patch(pull_mem &m, const adj_args *__restrict__ D, int inst, int slot, int patch, int part) {
  MFC_ADJ_ARGS(d, inst);
  adj_consts &k = d.k;
  const size_t N = k.N;
  const int *__restrict__ offsets = d.offsets + (size_t)slot * d.ncell1;
  const int tid = threadIdx.x;
  const int nrb = patch_rows(k), pc = patch / nrb, pr = patch - pc * nrb;
  const int r0 = pr * k.patch_s, r1 = r0 + k.patch_s < k.gny ? r0 + k.patch_s : k.gny;
  const int g0 = pc * k.patch_w, g1 = g0 + k.patch_w < k.gnx ? g0 + k.patch_w : k.gnx;
  const int s0 = r0 < 2 ? 0 : r0 - 2, s1 = r1 + 2 < k.gny ? r1 + 2 : k.gny;
  const int q0 = g0 < 2 ? 0 : g0 - 2, q1 = g1 + 2 < k.gnx ? g1 + 2 : k.gnx;
  const int ncol = q1 - q0, nrow = s1 - s0 + 1;
  const int te = tid / nrow;
  if (tid < ncol * nrow) m.table[tid] = offsets[(q0 + te) * k.gny + s0 + (tid - te * nrow)];
  __syncthreads();
  if (tid < 64) {
    int first = 0, c = 0, o = 0;
    if (tid < ncol) {
      first = m.table[tid * nrow];
      c = m.table[tid * nrow + nrow - 1] - first;
      if (q0 + tid >= g0 && q0 + tid < g1) o = m.table[tid * nrow + r1 - s0] - m.table[tid * nrow + r0 - s0];
    }
    int xc = c, xo = o;
#pragma unroll
    for (int s = 1; s < 32; s <<= 1) {
      const int yc = __shfl_up(xc, s, 64), yo = __shfl_up(xo, s, 64);
      if (tid >= s) { xc += yc; xo += yo; }
    }
    if (tid <= ncol) {
      m.col_first[tid] = xc - c;
      m.own_first[tid] = xo - o;
      if (tid < ncol) m.col_shift[tid] = xc - c - first;
    }
  }
  __syncthreads();
  const int ncand = m.col_first[ncol], nown = m.own_first[ncol];
  const int cap = k.stage_limit > 0 && k.stage_limit < PULL_CAP ? k.stage_limit : PULL_CAP;
  if (ncand > cap || !k.uniform_h) return false;  // the same in every thread
  // the pieces of a candidate's record and adjoints by neighbouring lanes (15 of each 16)
  const int pl = tid % 16;
  for (int q = tid / 16; q < ncand; q += TILE / 16) {
    int c = 0;
    for (int e = 1; e < ncol; e++) c += q >= m.col_first[e];
    const size_t j = q - m.col_shift[c];
    if (pl < REC_DOUBLES / 2) m.piece[pl][q] = reinterpret_cast<const double2 *>(d.rec)[j * (REC_DOUBLES / 2) + pl];
    else if (pl < PULL_PIECES)
      m.piece[pl][q] = reinterpret_cast<const double2 *>(d.lam_acc)[j * (LAM / 2) + pl - REC_DOUBLES / 2];
  }
  if (tid < ncol * nrow) m.table[tid] += m.col_shift[te];
  __syncthreads();
  const int lane = tid & 63, r = lane % PULL_LANES, gl = lane - r;
  const pull_lds src = {m};
  for (int t0 = 0; t0 < k.patch_slots; t0 += PULL_AT_ONCE) {
    const int n = part * k.patch_slots + t0 + tid / PULL_LANES;
    if (n >= nown) return true;  // whole groups of lanes
    int col = 0;
    for (int e = 1; e < ncol; e++) col += n >= m.own_first[e];
    const int li = m.table[col * nrow + r0 - s0] + (n - m.own_first[col]);
    const int b = li - m.col_shift[col];
    const int gi = q0 + col, gj = d.key_sorted[(size_t)slot * N + b] - gi * k.gny;
    const window w = make_window_at(k, gi, gj, [&](int c, int row) { return m.table[(c - q0) * nrow + row - s0]; });
    double gb[REC_DOUBLES];
    pull_particle(k, src, li, w, r, gl, m.list[tid / PULL_LANES], gb);
    pull_store(gb, r, d.g_rec + (size_t)REC_DOUBLES * b);
  }
  return true;
}

__global__ __launch_bounds__(TILE) __attribute__((amdgpu_waves_per_eu(3))) void kb_adj_pull(
    const adj_args *__restrict__ D, const inst_args *__restrict__ rep, const int2 *__restrict__ work, int nwork, int slot) {
  const int u = xcd_chunk_tile(blockIdx.x, nwork);
  if (u < 0) return;
  const int2 it = work[u];
  MFC_ADJ_ARGS(d, it.x);
  __shared__ pull_mem m;
  if (it.y == PATCH_ITEM_FORCE) {  // the work table's other item, in the pull the theta partials
    add_theta(d, reinterpret_cast<double(*)[TILE]>(&m));
    return;
  }
  const int count = d.plen[slot], step = rep[it.x].npatch_items;
  if (it.y >= count) return;
  const int2 *__restrict__ plist = d.plist + (size_t)slot * d.list_len;
  const int2 p = plist[it.y];
  const bool staged = pull_patch(m, D, it.x, slot, p.x, p.y);
  for (int q = staged ? it.y + step : it.y; q < count; q += step) pull_rest(m, D, it.x, slot, plist[q].x, plist[q].y);
}

// ------------------------------------------------------------------ B3: record VJP + unsort
// the segment's first step: the adjoint of its start state into storage order
__global__ __launch_bounds__(TILE) void kb_adj_record(const adj_args *__restrict__ D, const int2 *__restrict__ work,
                                                      int nwork) {
  const int w = xcd_tile(blockIdx.x, nwork);
  if (w < 0) return;
  const int2 it = work[w];
  MFC_ADJ_ARGS(d, it.x);
  adj_consts &k = d.k;
  const int a = it.y * TILE + threadIdx.x;
  if (a >= k.N) return;
  const size_t N = k.N;
  const unsigned dst = tag_index(d.tags[a]);
  const double *__restrict__ st = slot_state(d, 0);
  double s[TS_N], gs[TS_N], br[REC_DOUBLES];
#pragma unroll
  for (int q = 0; q < TS_N; q++) { s[q] = st[q * N + dst]; gs[q] = d.g_s[0][q * N + a]; }
#pragma unroll
  for (int q = 0; q < REC_DOUBLES; q++) br[q] = d.g_rec[(size_t)REC_DOUBLES * a + q];
  const int fl = slot_flags(d, 0)[dst] & FLAG_MASK;
  record_vjp(k, s, fl, eos_pressure(k, s, fl), br, gs);
#pragma unroll
  for (int q = 0; q < TS_N; q++) d.lam[q * N + dst] = gs[q];
}

}  // namespace

// ------------------------------------------------------------------ workspace
// threads per particle of the replayed interaction, whose patches the pull takes too: those of the
// forward steps, or 4 where they have one (whose patches' windows do not fit the pull's stage)
int replay_lanes(mfc_sim *const *sims, int n) {
  const int lanes = interaction_lanes(sims, n);
  return lanes > 4 ? lanes : 4;
}

// device memory of the backward pass of a group of instances, kept between calls with the first
// instance's workspace; the descriptors are written at every call
struct adj_group {
  int lanes = 0;                // replay_lanes
  std::vector<int> items;       // work items of each instance's patches
  int nck = 0;
  char *mem = nullptr;
  inst_args *rep = nullptr;     // K x n replay descriptors
  adj_args *adj = nullptr;      // n
  snapshot *snaps = nullptr;    // n x nck
  int2 *patches = nullptr;
  int npatches = 0;
  ~adj_group() {
    if (mem) (void)hipFree(mem);
  }
};

struct adj_work {
  int N = 0, nsteps = 0, K = 0, w0 = 0, w1 = 0;  // K set when everything is allocated
  bool valid = false;
  int64_t hist0 = 0;  // force-history index of the first step of the run
  double Fmean[2] = {0., 0.};
  std::vector<void *> allocs;
  std::vector<snapshot> ckpt;
  // the slots of a segment's steps (adj_args)
  char *state = nullptr;
  double *normal = nullptr;
  int *tags = nullptr, *spos = nullptr, *key_sorted = nullptr, *offsets = nullptr, *plen = nullptr;
  int2 *plist = nullptr;
  mfc_tool_state *tool = nullptr;
  return_tape *tape = nullptr;
  double *acc = nullptr;
  double *returns = nullptr;            // secant results of the run's steps, N each, or null (adj_keep_returns)
  bool returns_decided = false;
  size_t held = 0;                      // bytes of all the other allocations
  int uniform_h = 0;  // of the recorded run's states
  double h0 = 0.;
  char *posw = nullptr;                 // replay positional block (pressure and artificial stress)
  double *partials = nullptr, *force_last = nullptr, *hist = nullptr;
  int64_t *ctr = nullptr;
  int *pending = nullptr, *gflag = nullptr;
  double *lam = nullptr, *lam_n = nullptr, *g_s[2] = {nullptr, nullptr}, *lam_acc = nullptr, *rec = nullptr,
         *g_rec = nullptr, *theta_part = nullptr, *theta_acc = nullptr;
  std::unique_ptr<adj_group> group;     // of the group that this instance is the first of

  template <class T>
  int alloc(T **p, size_t n) {
    void *q = nullptr;
    if (n == 0) n = 1;
    hipError_t e = hipMalloc(&q, n * sizeof(T));
    if (e != hipSuccess) return fail(MFC_E_NOMEM, std::string("hipMalloc (adjoint): ") + hipGetErrorString(e));
    allocs.push_back(q);
    held += n * sizeof(T);
    *p = (T *)q;
    return MFC_OK;
  }
  int alloc_snapshot(snapshot &sn) {
    int rc;
    if ((rc = alloc(&sn.state, state_block_bytes(N))) || (rc = alloc(&sn.pos, positional_block_bytes(N))) ||
        (rc = alloc(&sn.keys, (size_t)N)) || (rc = alloc(&sn.tool, 1)))
      return rc;
    return MFC_OK;
  }
  ~adj_work() {
    for (void *q : allocs) (void)hipFree(q);
  }
};

void adj_free(adj_work *w) { delete w; }

namespace {

int setup_work(mfc_sim *s, int nsteps, int K, int w0, int w1) {
  const int N = s->k.N;
  adj_work *w = s->adj;
  const int nck = (nsteps + K - 1) / K;
  const bool reuse = w && w->N == N && w->K == K && (int)w->ckpt.size() >= nck;
  if (!reuse) {
    HIP_TRY(hipStreamSynchronize(s->stream));  // nothing queued uses the old one
    HIP_TRY(hipMemsetAsync(s->tape, 0, 2 * sizeof(return_tape), s->stream));  // nor do later steps, if a run broke off
    adj_free(w);
    w = s->adj = new adj_work();
    w->N = N;
    int rc;
    w->ckpt.resize(nck);
    for (auto &c : w->ckpt)
      if ((rc = w->alloc_snapshot(c))) return rc;
    const size_t n = (size_t)N, k = (size_t)K;
    const size_t list = std::max(patches_for(s, 4).list, patches_for(s, 8).list);
    if ((rc = w->alloc(&w->state, (k + 1) * state_block_bytes(N))) || (rc = w->alloc(&w->normal, (k + 1) * 2 * n)) ||
        (rc = w->alloc(&w->tags, k * n)) || (rc = w->alloc(&w->spos, k * n)) || (rc = w->alloc(&w->key_sorted, k * n)) ||
        (rc = w->alloc(&w->offsets, k * ((size_t)s->k.ncell_table + 1))) || (rc = w->alloc(&w->plen, k + 1)) ||
        (rc = w->alloc(&w->plist, k * list)) || (rc = w->alloc(&w->tool, k + 1)) || (rc = w->alloc(&w->tape, k + 1)) ||
        (rc = w->alloc(&w->acc, k * (L_N + 1) * n)) ||
        (rc = w->alloc(&w->posw, positional_block_bytes(N))) ||
        (rc = w->alloc(&w->partials, 16 * (size_t)s->ntiles)) || (rc = w->alloc(&w->force_last, 2)) ||
        (rc = w->alloc(&w->hist, 2)) || (rc = w->alloc(&w->ctr, 1)) || (rc = w->alloc(&w->pending, 2)) ||
        (rc = w->alloc(&w->gflag, 4 * (size_t)s->ntiles)) || (rc = w->alloc(&w->lam, TS_N * n)) ||
        (rc = w->alloc(&w->lam_n, 2 * n)) || (rc = w->alloc(&w->g_s[0], TS_N * n)) ||
        (rc = w->alloc(&w->g_s[1], TS_N * n)) || (rc = w->alloc(&w->lam_acc, LAM * n)) ||
        (rc = w->alloc(&w->rec, REC_DOUBLES * n)) || (rc = w->alloc(&w->g_rec, REC_DOUBLES * n)) ||
        (rc = w->alloc(&w->theta_part, 6 * (size_t)s->ntiles)) || (rc = w->alloc(&w->theta_acc, 6)))
      return rc;
    // the replay's force reduction keeps no history (cap 0) but counts steps
    HIP_TRY(hipMemsetAsync(w->ctr, 0, sizeof(int64_t), s->stream));
    HIP_TRY(hipMemsetAsync(w->pending, 0, 2 * sizeof(int), s->stream));
    HIP_TRY(hipMemsetAsync(w->gflag, 0, 4 * sizeof(int) * (size_t)s->ntiles, s->stream));
    w->K = K;
  }
  w->nsteps = nsteps;
  w->w0 = w0;
  w->w1 = w1;
  w->valid = false;
  return MFC_OK;
}

// the group's device memory and work table, kept while a call's instances have the same work items
int setup_group(mfc_sim *const *sims, int n, hipStream_t st) {
  adj_work *w0 = sims[0]->adj;
  const int K = w0->K, nck = (w0->nsteps + K - 1) / K;
  const int lanes = replay_lanes(sims, n);
  std::vector<int> per(n);
  for (int i = 0; i < n; i++) per[i] = patches_for(sims[i], lanes).items;
  adj_group *g = w0->group.get();
  if (g && g->lanes == lanes && g->items == per && g->nck >= nck) return MFC_OK;
  HIP_TRY(hipStreamSynchronize(st));  // nothing queued uses the old one
  w0->group.reset(new adj_group());
  g = w0->group.get();
  g->lanes = lanes;
  g->items = per;
  g->nck = nck;
  std::vector<int2> items;
  for (int i = 0; i < n; i++) items.push_back(make_int2(i, PATCH_ITEM_FORCE));
  for (int i = 0; i < n; i++)
    for (int q = 0; q < per[i]; q++) items.push_back(make_int2(i, q));
  g->npatches = (int)items.size();
  auto up = [](size_t b) { return (b + 255) & ~(size_t)255; };
  const size_t b_rep = up(sizeof(inst_args) * (size_t)K * n), b_adj = up(sizeof(adj_args) * n);
  const size_t b_sn = up(sizeof(snapshot) * (size_t)n * nck), b_pt = up(sizeof(int2) * items.size());
  const hipError_t e = hipMalloc(&g->mem, b_rep + b_adj + b_sn + b_pt);
  if (e != hipSuccess) {
    g->mem = nullptr;
    w0->group.reset();
    return fail(MFC_E_NOMEM, std::string("hipMalloc (adjoint group): ") + hipGetErrorString(e));
  }
  char *p = g->mem;
  g->rep = (inst_args *)p; p += b_rep;
  g->adj = (adj_args *)p; p += b_adj;
  g->snaps = (snapshot *)p; p += b_sn;
  g->patches = (int2 *)p;
  if (hipMemcpy(g->patches, items.data(), sizeof(int2) * items.size(), hipMemcpyHostToDevice) != hipSuccess) {
    w0->group.reset();
    return fail(MFC_E_HIP, "upload of the adjoint's work table");
  }
  return MFC_OK;
}

// segment sg of len steps: the replay, then the reverse steps
void enqueue_segment(const adj_group &g, const adj_work &w, const batch_work &fw, int sg, int len, int copy_blocks,
                     hipStream_t st) {
  const int n = (int)g.items.size();
  batch_work rw = fw;
  rw.patches = g.patches;
  rw.npatches = g.npatches;
  rw.v.lanes = g.lanes;
  rw.args = g.rep;
  const dim3 gt(padded(fw.ntiles)), gp(chunked_blocks(g.npatches));
  hipLaunchKernelGGL(kb_adj_restore, dim3(copy_blocks, n), dim3(256), 0, st, g.adj, sg);
  launch_batch_hash(rw, st);
  launch_batch_records(rw, st);
  for (int j = 0; j < len; j++) {
    rw.args = g.rep + (size_t)j * n;
    launch_batch_step(rw, st);
  }
  for (int j = len - 1; j >= 0; j--) {
    const int t = sg * w.K + j;
    hipLaunchKernelGGL(kb_adj_tail, gt, dim3(TILE), 0, st, g.adj, fw.tiles, fw.ntiles, j, (int)(j == len - 1),
                       (int)(t >= w.w0 && t < w.w1));
    hipLaunchKernelGGL(kb_adj_pull, gp, dim3(TILE), 0, st, g.adj, g.rep, g.patches, g.npatches, j);
  }
  hipLaunchKernelGGL(kb_adj_record, gt, dim3(TILE), 0, st, g.adj, fw.tiles, fw.ntiles);
}

// about 8 words of a state block per thread
int copy_blocks_of(int N) {
  const size_t want = (state_block_bytes(N) / sizeof(uint64_t) + 2047) / 2048;
  return want < 16 ? 16 : (want > 1024 ? 1024 : (int)want);
}

}  // namespace

int adj_begin(mfc_sim *s, int nsteps, int checkpoint_every, int w0, int w1) {
  if (nsteps < 1 || checkpoint_every < 1 || w0 < 0 || w1 <= w0 || w1 > nsteps)
    return fail(MFC_E_INVALID, "need nsteps >= 1, checkpoint_every >= 1 and 0 <= w0 < w1 <= nsteps");
  if (s->precision != MFC_PREC_FP64 || !s->k.promote)
    return fail(MFC_E_INVALID, "the adjoint needs precision FP64 and promote_fp64 = 1");
  if (s->sc.tool.num_seg == 0 || !s->k.plastic)
    return fail(MFC_E_INVALID, "the adjoint differentiates the cutting scenario (tool and plasticity present)");
  if (s->k.jc_tanh) return fail(MFC_E_INVALID, "the adjoint differentiates the plain Johnson-Cook model (jc_model = 0)");
  if (s->k.adaptive) return fail(MFC_E_INVALID, "the adjoint runs on a locked grid (grid_adaptive = 0)");
  if (s->k.rothlin) return fail(MFC_E_INVALID, "the adjoint runs on the green grid (grid_kind = 0)");
  int64_t base = 0;
  int rc = mfc_force_history(s, nullptr, 0, &base);
  if (rc) return rc;
  if (base + nsteps > HIST_CAP) return fail(MFC_E_INVALID, "force history full: reset it before the run");
  if ((rc = setup_work(s, nsteps, checkpoint_every, w0, w1))) return rc;
  s->adj->hist0 = base;
  s->adj->uniform_h = s->k.uniform_h;
  s->adj->h0 = s->k.h0;
  return MFC_OK;
}

// Whether the runs' secant results are recorded for their replay: they take 8 bytes per particle and step,
// and a tape that would be larger than its instance's checkpoints and slots of a segment (`held`) isn't kept,
// nor are tapes of a group that together take more than a quarter of the memory that is free once every
// instance has all it needs (the replay then iterates again). Runs of up to about 9,000 steps with a
// checkpoint every sqrt(steps) keep one. It makes a pass 21 to 24 % shorter (the figures stand at
// on_tape), whatever the length: the line is drawn by memory alone.
void adj_keep_returns(mfc_sim *const *sims, int n) {
  bool decided = true;
  for (int i = 0; i < n; i++) decided = decided && sims[i]->adj->returns_decided;
  if (decided) return;  // asking for the free memory takes 0.1 ms
  size_t avail = 0, total = 0;
  if (hipMemGetInfo(&avail, &total) != hipSuccess) {
    (void)hipGetLastError();
    return;
  }
  size_t left = avail / 4;
  for (int i = 0; i < n; i++) {
    adj_work *w = sims[i]->adj;
    if (w->returns_decided) continue;
    w->returns_decided = true;
    const size_t tape = w->ckpt.size() * (size_t)w->K * w->N * sizeof(double);
    void *q = nullptr;
    if (tape > w->held || tape > left) continue;
    if (hipMalloc(&q, tape) != hipSuccess) {
      (void)hipGetLastError();  // none kept
      continue;
    }
    w->allocs.push_back(q);
    w->returns = (double *)q;
    left -= tape;
  }
}

int adj_segment(const mfc_sim *s) { return s->adj->K; }

int adj_checkpoint(mfc_sim *s, int t) {
  adj_work *w = s->adj;
  if (t % w->K) return MFC_OK;
  const int c = s->cur, N = s->k.N, left = w->nsteps - t < w->K ? w->nsteps - t : w->K;
  const return_tape first = {w->returns ? w->returns + (size_t)t * N : nullptr, w->returns ? left : 0};
  hipLaunchKernelGGL(k_adj_save, dim3(copy_blocks_of(N)), dim3(256), 0, s->stream, w->ckpt[t / w->K],
                     (const uint64_t *)s->set[c].px, state_block_bytes(N) / sizeof(uint64_t),
                     (const uint64_t *)s->pos.nx, positional_block_bytes(N) / sizeof(uint64_t),
                     (const int *)s->bins.key_sorted, N, (const mfc_tool_state *)(s->tool + c), s->tape + c, first);
  return MFC_OK;
}

int adj_finish(mfc_sim *s, double Fmean[2]) {
  adj_work *w = s->adj;
  const int n = w->w1 - w->w0;
  std::vector<double> F((size_t)2 * n);
  HIP_TRY(hipMemcpyAsync(F.data(), s->hist + 2 * (w->hist0 + w->w0), sizeof(double) * F.size(),
                         hipMemcpyDeviceToHost, s->stream));
  HIP_TRY(hipStreamSynchronize(s->stream));
  double sx = 0., sy = 0.;
  for (int t = 0; t < n; t++) {
    sx += F[2 * t];
    sy += F[2 * t + 1];
  }
  w->Fmean[0] = Fmean[0] = sx / n;
  w->Fmean[1] = Fmean[1] = sy / n;
  w->valid = true;
  return MFC_OK;
}

int adj_backward(mfc_sim *const *sims, int n, const batch_work &handle_work, hipStream_t st, const double *cot, double *grad) {
  if (n < 1) return fail(MFC_E_INVALID, "empty group");
  const adj_work *w0 = sims[0]->adj;
  for (int i = 0; i < n; i++) {
    const adj_work *w = sims[i]->adj;
    if (!w || !w->valid) return fail(MFC_E_INVALID, "no recorded run: call mfc_vjp_forward first");
    if (w->nsteps != w0->nsteps || w->K != w0->K || w->w0 != w0->w0 || w->w1 != w0->w1)
      return fail(MFC_E_INVALID, "the instances recorded different runs");
  }
  int rc = setup_group(sims, n, st);
  if (rc) return rc;
  adj_group &g = *w0->group;
  batch_work fw = handle_work;
  for (int i = 0; i < n; i++) fw.general = fw.general || !sims[i]->adj->uniform_h;  // of the recorded states
  const int nsteps = w0->nsteps, K = w0->K, nseg = (nsteps + K - 1) / K;
  const int slots = K < nsteps ? K : nsteps;
  // the descriptors: a replay step each (inst_args, the step kernels' view of a slot), the reverse
  // kernels' view of the instance, and its checkpoints
  std::vector<inst_args> rep((size_t)slots * n);
  std::vector<adj_args> da(n);
  std::vector<snapshot> snaps((size_t)n * nseg);
  int maxN = 0;
  for (int i = 0; i < n; i++) {
    mfc_sim *s = sims[i];
    adj_work *w = s->adj;
    const int N = s->k.N;
    const size_t sb = state_block_bytes(N), nc1 = (size_t)s->k.ncell_table + 1;
    maxN = N > maxN ? N : maxN;
    dev_consts k = s->k;
    const patch_plan &plan = patches_for(s, g.lanes);
    k.patch_s = plan.s;
    k.patch_w = plan.w;
    k.patch_slots = plan.slots;
    k.uniform_h = w->uniform_h;
    k.h0 = w->h0;
    for (int j = 0; j < slots; j++) {
      inst_args &a = rep[(size_t)j * n + i];
      std::memset(&a, 0, sizeof(a));
      const int p = j & 1;
      a.k = k;
      carve_state(w->state + j * sb, N, a.cur);
      carve_state(w->state + (j + 1) * sb, N, a.nxt);
      a.b = s->bins;
      a.b.key_sorted = w->key_sorted + (size_t)j * N;
      a.b.tags = w->tags + (size_t)j * N;
      a.b.spos = w->spos + (size_t)j * N;
      a.b.offsets = w->offsets + j * nc1;
      a.b.plist = w->plist + (size_t)j * plan.list;
      a.b.plen = w->plen + j;
      a.b.plen_next = w->plen + j + 1;
      a.b.bsum = s->chunk_sums[p];
      a.b.bsum_next = s->chunk_sums[1 - p];
      carve_positional(w->posw, N, a.pos);
      a.pos.nx = w->normal + (size_t)j * 2 * N;
      a.pos.ny = a.pos.nx + N;
      a.pos.nx_out = a.pos.nx + 2 * (size_t)N;
      a.pos.ny_out = a.pos.nx + 3 * (size_t)N;
      a.r = s->recs[p];
      a.rn = s->recs[1 - p];
      a.tool_in = w->tool + j;
      a.tool_out = w->tool + j + 1;
      a.tape_in = w->tape + j;
      a.tape_out = w->tape + j + 1;
      a.f = {w->partials, w->gflag, w->force_last, w->hist, 0, w->ctr, w->pending + p, w->pending + 1 - p};  // no history, counted
      a.acc_out = w->acc + (size_t)j * (L_N + 1) * N;
      a.ntiles = s->ntiles;
      a.nscan = scan_blocks(s->k.ncell_table);
      a.npatch_items = plan.items;
    }
    adj_args &d = da[i];
    std::memset(&d, 0, sizeof(d));
    d.k = k;
    d.ntiles = s->ntiles;
    d.state = w->state;
    d.state_bytes = sb;
    d.normal = w->normal;
    d.tags = w->tags; d.spos = w->spos; d.key_sorted = w->key_sorted;
    d.offsets = w->offsets;
    d.plist = w->plist; d.plen = w->plen;
    d.list_len = plan.list; d.ncell1 = (int)nc1;
    d.tool = w->tool;
    d.tape = w->tape;
    d.returns = w->returns;
    d.K = K;
    d.acc = w->acc;
    d.lam = w->lam; d.lam_n = w->lam_n;
    d.g_s[0] = w->g_s[0]; d.g_s[1] = w->g_s[1];
    d.lam_acc = w->lam_acc; d.rec = w->rec; d.g_rec = w->g_rec;
    d.theta_part = w->theta_part; d.theta_acc = w->theta_acc;
    d.Fb[0] = cot[2 * i] / (w->w1 - w->w0);
    d.Fb[1] = cot[2 * i + 1] / (w->w1 - w->w0);
    d.ckpt = g.snaps + (size_t)i * nseg;
    d.chunk_sums[0] = s->chunk_sums[0]; d.chunk_sums[1] = s->chunk_sums[1];
    d.pcnt = s->bins.pcnt;
    d.nscan = scan_blocks(s->k.ncell_table);
    d.npatch = s->npatch_max;
    for (int c = 0; c < nseg; c++) snaps[(size_t)i * nseg + c] = w->ckpt[c];
  }
  const int copy_blocks = copy_blocks_of(maxN);
  auto run = [&]() -> int {
    HIP_TRY(hipMemcpyAsync(g.rep, rep.data(), sizeof(inst_args) * rep.size(), hipMemcpyHostToDevice, st));
    HIP_TRY(hipMemcpyAsync(g.adj, da.data(), sizeof(adj_args) * da.size(), hipMemcpyHostToDevice, st));
    HIP_TRY(hipMemcpyAsync(g.snaps, snaps.data(), sizeof(snapshot) * snaps.size(), hipMemcpyHostToDevice, st));
    for (int i = 0; i < n; i++) {
      mfc_sim *s = sims[i];
      adj_work *w = s->adj;
      const size_t N = (size_t)s->k.N;
      HIP_TRY(hipMemsetAsync(w->lam, 0, sizeof(double) * TS_N * N, st));
      HIP_TRY(hipMemsetAsync(w->lam_n, 0, sizeof(double) * 2 * N, st));
      HIP_TRY(hipMemsetAsync(w->theta_acc, 0, sizeof(double) * 6, st));
      // the pass bins its states with the handle's scratch and overwrites its records: both are
      // computed again at the handle's next step
      s->keys_fresh = false;
    }
    for (int sg = nseg - 1; sg >= 0; sg--) {
      const int len = sg == nseg - 1 ? nsteps - sg * K : K;
      enqueue_segment(g, *w0, fw, sg, len, copy_blocks, st);
    }
    HIP_TRY(hipGetLastError());
    for (int i = 0; i < n; i++)
      HIP_TRY(hipMemcpyAsync(grad + 6 * i, sims[i]->adj->theta_acc, sizeof(double) * 6, hipMemcpyDeviceToHost, st));
    HIP_TRY(hipStreamSynchronize(st));
    return MFC_OK;
  };
  rc = run();
  if (rc) (void)hipStreamSynchronize(st);  // nothing queued may still read the descriptors' host copies
  return rc;
}

}  // namespace mfc

using namespace mfc;

extern "C" {

int mfc_vjp_forward(mfc_sim *s, int nsteps, int checkpoint_every, int w0, int w1, double Fmean[2]) {
  if (!s || !Fmean) return fail(MFC_E_INVALID, "null argument");
  if (s->batched) return fail(MFC_E_INVALID, "instance of a batch: use mfc_batch_vjp_forward");
  int rc = adj_begin(s, nsteps, checkpoint_every, w0, w1);
  if (rc) return rc;
  mfc::adj_keep_returns(&s, 1);
  if ((rc = ensure_keys(s))) return rc;
  const int K = mfc::adj_segment(s);
  for (int t = 0; t < nsteps; t += K) {
    if ((rc = adj_checkpoint(s, t)) || (rc = queue_steps(s, nsteps - t < K ? nsteps - t : K))) return rc;
  }
  finish_steps(s);
  HIP_TRY(hipGetLastError());
  return adj_finish(s, Fmean);
}

int mfc_vjp_backward(mfc_sim *s, const double cot[2], double grad[6]) {
  if (!s || !cot || !grad) return fail(MFC_E_INVALID, "null argument");
  if (s->batched) return fail(MFC_E_INVALID, "instance of a batch: use mfc_batch_vjp_backward");
  return adj_backward(&s, 1, s->work(s->cur), s->stream, cot, grad);
}

int mfc_vjp(mfc_sim *s, mfc_vjp_req *req, double grad[6]) {
  if (!s || !req || !grad) return fail(MFC_E_INVALID, "null argument");
  int rc = mfc_vjp_forward(s, req->nsteps, req->checkpoint_every, req->w0, req->w1, req->Fmean);
  if (rc) return rc;
  return mfc_vjp_backward(s, req->cot, grad);
}

}  // extern "C"
