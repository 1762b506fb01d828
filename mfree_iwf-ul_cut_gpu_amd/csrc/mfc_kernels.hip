// mfc_kernels.hip — gfx950 kernels of one SPH cutting step (FP64 and FP32C).
//
// Per step (the reference's ~20 launches of leap_frog::step, leap_frog.cu:94-155, become 2):
//   sort         one work-group per chunk of cells: the cells' offsets, buckets and the rank of
//                every particle in its cell, a stable counting sort by cell
//                (thrust::sort_by_key + reorder_data_and_find_cell_start,
//                grid_gpu_green.cu:22-116,177-201) from the cell ids (grid.cu:34-51), per-cell
//                and per-chunk counts and the chunks' particle lists that the previous step's
//                interaction computed for the updated state (hash_count computes them when the
//                state was written from outside, for every state the reverse mode restores, and
//                behind an adaptive grid's geometry pass); a few more work-groups of the launch move the tool, list the patches of
//                cells that hold particles and sum the previous step's tool force
//                (output.cu:30-39) over groups of 64 particles
//   interact     neighbour sums (interactions_gpu.cu:88-345) fused with every per-particle action
//                that follows them in the step: Jaumann, continuity, momentum, advection, correct,
//                friction heat, Johnson-Cook return, tool-particle move, contact, boundary
//                conditions, NaN blanking and the gather into sorted order; then, for the next step,
//                the cell ids and counts and each particle's neighbour record: leap-frog predict
//                (leap_frog.cu:30-66), EOS (actions_gpu.cu:41-51) and artificial stress (:53-97)
//                (records computes them when the state was written from outside). A work-group
//                takes a patch of cells with its window candidates staged in LDS, with 1, 4 or 8
//                threads per particle; one more adds up the previous step's force sums
// After the last step of a call, force_final reduces the last step's tool force. The record of a
// step could not be written by a kernel of the same step that also reads it (every particle's sums
// need all its neighbours' records), but the previous interaction holds all it is made of in
// registers: with a launch of its own, which read 19 of the 27 state fields again, the step took
// 80 us instead of 72 (FP32C, 197k particles) and 63 instead of 53 (FP64, 6k).
// Each body is a device function of its work index; the kb_* kernels run it over an
// (instance, tile) work table for any number of instances (a single handle is a batch of one).
//
// Memory layout: the persistent particle state is a structure of arrays in cell-sorted order,
// double-buffered across the step. Neighbour data are packed per particle into one 128-byte
// record (FP64) or one of 64 bytes (FP32C, the position in FP64); the records stay where
// the interaction wrote them (the storage order of the next step's start state) and are found
// through the sort permutation. Work-group to tile
// mapping is XCD-aware.
#include <hip/hip_ext.h>

#include <cfloat>
#include <type_traits>

#include "mfc_kernels.h"
#include "mfc_pairs.h"

namespace mfc {

namespace {

constexpr int SCAN_THREADS = 256;
constexpr int SCAN_ITEMS = 2;                         // cells per thread of the sort
constexpr int SCAN_CHUNK = SCAN_THREADS * SCAN_ITEMS;  // cells per chunk of the sort
constexpr int SORT_BATCH = 6;            // particles per thread the sort holds in registers
static_assert(SCAN_THREADS * SORT_BATCH == MFC_SORT_FAST_MAX, "the sort's register path bound of the header");
constexpr int CARRY_BATCH = 4;            // 16-byte loads of chunk sums per thread the sort
                                          // has in flight at once


// exclusive scan of one int per thread over a 256-thread block; total receives the block sum
__device__ inline int block_exclusive_scan(int v, int &total) {
  __shared__ int wsum[SCAN_THREADS / 64];
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  int x = v;
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    int y = __shfl_up(x, o, 64);
    if (lane >= o) x += y;
  }
  if (lane == 63) wsum[w] = x;
  __syncthreads();
  int pre = 0, tot = 0;
#pragma unroll
  for (int q = 0; q < SCAN_THREADS / 64; q++) {
    if (q < w) pre += wsum[q];
    tot += wsum[q];
  }
  total = tot;
  __syncthreads();
  return pre + x - v;
}

// ------------------------------------------------------------------------------- binning
// Each kernel body is a device function of its work index, called by the batched kernel with
// the index of an (instance, block) item of its work table.

// cell id of a particle for the binning (grid.cu:34-51; blanked particles keep their last
// sorted id, grid.cu:39-41); positions outside the grid are counted
template <class K>  // dev_consts or kconst
__device__ inline int particle_cell(K &k, double x, double y, int fl, int sorted_id,
                                    unsigned long long *__restrict__ clamped) {
  if (fl & MFC_FLAG_BLANKED) return sorted_id;
  bool cl;
  const int h = cell_of(k, x, y, cl);
  if (cl) atomicAdd(clamped, 1ull);
  return h;
}

// records cell id h of particle i (storage order) and appends (i, h) to the particle list of
// its chunk of SCAN_CHUNK cells (bsum counts the chunk's particles; the list keeps the first ccap
// of them). All 64 lanes of the wave take part (lanes past N carry h = -1). The storage order is
// the previous step's cell order, so neighbouring lanes mostly share a chunk: each run of equal
// chunks in the wave takes its list places with one atomic.
__device__ inline void count_cell(int i, int h, int *__restrict__ key, int *__restrict__ bsum,
                                  int2 *__restrict__ clist, int ccap) {
  if (h >= 0) key[i] = h;
  const int lane = threadIdx.x & 63;
  const unsigned long long upto = (lane == 63) ? ~0ull : ((2ull << lane) - 1ull);
  const int c = h >= 0 ? h / SCAN_CHUNK : -1;
  const int cprev = __shfl_up(c, 1, 64);
  const bool chead = lane == 0 || cprev != c;
  const unsigned long long cheads = __ballot(chead);
  const int my_chead = 63 - __clzll(cheads & upto);
  const unsigned long long cafter = (lane == 63) ? 0ull : (cheads & ~upto);
  const int cnext = cafter ? __ffsll((long long)cafter) - 1 : 64;
  int cbase = 0;
  if (chead && c >= 0) cbase = atomicAdd(&bsum[c], cnext - lane);
  cbase = __shfl(cbase, my_chead, 64);
  const int place = cbase + (lane - my_chead);
  if (c >= 0 && place < ccap) clist[(size_t)c * ccap + place] = make_int2(i, h);
}

// the patch of a cell of the grid
template <class K>  // dev_consts or kconst
__device__ inline int patch_of(K &k, int h) {
  const int gi = h / k.gny, gj = h - gi * k.gny;
  return (gi / k.patch_w) * patch_rows(k) + gj / k.patch_s;
}

// counts a particle in its patch p (all 64 lanes of the wave; p = -1: no particle): one atomic per
// run of equal patches in the wave
__device__ inline void count_patch(int p, int *__restrict__ pcnt) {
  const int lane = threadIdx.x & 63, prev = __shfl_up(p, 1, 64);
  const bool head = lane == 0 || prev != p;
  const unsigned long long after = lane == 63 ? 0ull : __ballot(head) & ~((2ull << lane) - 1ull);
  if (head && p >= 0) atomicAdd(&pcnt[p], (after ? __ffsll((long long)after) - 1 : 64) - lane);
}

// cell id of every particle of the start state, counted in its chunk
template <class K>
__device__ inline void hash_count(K &k, int i, const double *__restrict__ px,
                                  const double *__restrict__ py, const int *__restrict__ flags,
                                  const dbins &b) {
  const int h = i < k.N ? particle_cell(k, px[i], py[i], flags[i], b.key_sorted[i], b.clamped) : -1;
  count_cell(i, h, b.key, b.bsum, b.clist, b.ccap);
  // a blanked particle keeps its cell id, which an adaptive grid can shrink below: such particles
  // are sorted past the grid's cells and make a patch of their own behind the grid's
  count_patch(h < 0 ? -1 : h >= k.num_cell ? patch_total(k) : patch_of(k, h), b.pcnt);
}

// The counting sort of one chunk of SCAN_CHUNK cells (SCAN_ITEMS per thread), by one work-group,
// from the chunk's particle list:
// 1. the particles counted per cell (LDS atomics, which also give each its arrival slot);
// 2. the cells' offsets (the chunk's offset is the sum of the chunk sums before it, added up
//    here, so no separate scan of the chunk sums);
// 3. every particle into its cell's bucket at its arrival slot;
// 4. each one ranked in its cell by current position, the order thrust::sort_by_key gives on
//    (cell id, 0..N-1): its sorted position, its tag and the sorted cell id there. (The tag joins
//    the flags to the position here, where their load hides behind the counting, so that the
//    interaction's staging has one load fewer before the records'.)
// The chunks' cells, bucket ranges and particles are disjoint, so the work-groups share nothing
// but the chunk sums they read. A chunk of at most SCAN_THREADS * SORT_BATCH particles (a dense
// chunk holds about 2.25 per cell at the lattice spacing) keeps them in registers and their
// buckets in LDS, and its list, chunk sum and preceding chunk sums are loaded at once: the
// only global loads of the work-group. A larger chunk walks its list (or, when the list
// overflowed, every particle's cell id) three times and uses the global bucket. Two cells per
// thread keep most work-groups of a large table resident at once (a 500k-particle cut has 1.18
// million cells: 2,310 work-groups). sort_fast and sort_list (launch settings, 0: none) lower
// the two bounds, so that the other paths can be run on any cut.
__device__ inline void sort_chunk(int blk, int N, int n, const dbins &b, const int *__restrict__ vfl, int sort_fast,
                                  int sort_list) {
  __shared__ int off_l[SCAN_CHUNK], cnt_l[SCAN_CHUNK], fill_l[SCAN_CHUNK];
  __shared__ int bk_l[SCAN_THREADS * SORT_BATCH];
  const int c0 = blk * SCAN_CHUNK;
  const int2 *__restrict__ list = b.clist + (size_t)blk * b.ccap;
  const int list_cap = sort_list > 0 && sort_list < b.ccap ? sort_list : b.ccap;
  int fast_cap = list_cap < SCAN_THREADS * SORT_BATCH ? list_cap : SCAN_THREADS * SORT_BATCH;
  if (sort_fast > 0 && sort_fast < fast_cap) fast_cap = sort_fast;
  // the list's first entries, loaded before the chunk sum says how many are valid
  int2 e[SORT_BATCH];
#pragma unroll
  for (int u = 0; u < SORT_BATCH; u++) {
    const int p = u * SCAN_THREADS + threadIdx.x;
    e[u] = p < fast_cap ? list[p] : make_int2(-1, -1);
  }
  const int members = b.bsum[blk];
  // the chunk sums before this chunk, four per load (the sums are allocated in whole
  // 16-byte words), CARRY_BATCH loads per thread in flight at once
  const int4 *__restrict__ bsum4 = reinterpret_cast<const int4 *>(b.bsum);
  int carry_part = 0;
  for (int q0 = 0; q0 < blk; q0 += 4 * SCAN_THREADS * CARRY_BATCH) {
    int4 t[CARRY_BATCH];
#pragma unroll
    for (int u = 0; u < CARRY_BATCH; u++) {
      const int q = q0 + 4 * (u * SCAN_THREADS + (int)threadIdx.x);
      t[u] = q < blk ? bsum4[q >> 2] : make_int4(0, 0, 0, 0);
    }
#pragma unroll
    for (int u = 0; u < CARRY_BATCH; u++) {
      const int q = q0 + 4 * (u * SCAN_THREADS + (int)threadIdx.x);
      carry_part += (q < blk ? t[u].x : 0) + (q + 1 < blk ? t[u].y : 0) + (q + 2 < blk ? t[u].z : 0) +
                    (q + 3 < blk ? t[u].w : 0);
    }
  }
#pragma unroll
  for (int q = 0; q < SCAN_ITEMS; q++) {
    cnt_l[q * SCAN_THREADS + threadIdx.x] = 0;
    fill_l[q * SCAN_THREADS + threadIdx.x] = 0;
  }
  const bool fast = members <= fast_cap;  // the same in every thread
  const bool listed = members <= list_cap;
  const int lim = listed ? members : N;
  __syncthreads();
  int ls[SORT_BATCH], fl[SORT_BATCH];
  if (fast) {
#pragma unroll
    for (int u = 0; u < SORT_BATCH; u++) {
      const int p = u * SCAN_THREADS + threadIdx.x;
      if (p >= members) e[u].x = -1;
      fl[u] = e[u].x >= 0 ? vfl[e[u].x] : 0;
      ls[u] = e[u].x >= 0 ? atomicAdd(&cnt_l[e[u].y - c0], 1) : 0;
    }
  } else {
    for (int p = threadIdx.x; p < lim; p += SCAN_THREADS) {
      const int h = (listed ? list[p].y : b.key[p]) - c0;
      if (h >= 0 && h < SCAN_CHUNK) atomicAdd(&cnt_l[h], 1);
    }
  }
  int carry;
  block_exclusive_scan(carry_part, carry);  // its barriers also complete the counts
  // the thread's SCAN_ITEMS consecutive cells
  const int l0 = threadIdx.x * SCAN_ITEMS;
  int v[SCAN_ITEMS], sv = 0;
#pragma unroll
  for (int q = 0; q < SCAN_ITEMS; q++) {
    v[q] = cnt_l[l0 + q];
    sv += v[q];
  }
  if (threadIdx.x == 0) b.bsum_next[blk] = 0;  // the interaction counts the next step's there
  int total;
  int o = block_exclusive_scan(sv, total) + carry;
#pragma unroll
  for (int q = 0; q < SCAN_ITEMS; q++) {
    const int cell = c0 + l0 + q;
    off_l[l0 + q] = o;
    if (cell < n) {
      b.offsets[cell] = o;
      if (cell == n - 1) b.offsets[n] = o + v[q];
    }
    o += v[q];
  }
  __syncthreads();  // off_l
  const int base = off_l[0];
  // the sorted position of particle i (cell h of the chunk): its rank among the entries of the
  // cell's bucket (bk, indexed from offset bbase)
  auto rank = [&](int i, int h, int flags, const int *bk, int bbase) {
    const int cb = off_l[h], ce = cb + cnt_l[h];
    int rnk = 0;
    for (int q = cb; q < ce; q++) rnk += bk[q - bbase] < i;
    const int j = cb + rnk;
    if (b.spos) b.spos[i] = j;  // the same in every thread
    b.tags[j] = make_tag(i, flags);
    b.key_sorted[j] = h + c0;
  };
  if (fast) {
#pragma unroll
    for (int u = 0; u < SORT_BATCH; u++)
      if (e[u].x >= 0) bk_l[off_l[e[u].y - c0] - base + ls[u]] = e[u].x;
    __syncthreads();  // the chunk's buckets
#pragma unroll
    for (int u = 0; u < SORT_BATCH; u++)
      if (e[u].x >= 0) rank(e[u].x, e[u].y - c0, fl[u], bk_l, base);
  } else {
    int *__restrict__ bucket = b.bucket;
    for (int p = threadIdx.x; p < lim; p += SCAN_THREADS) {
      const int2 q = listed ? list[p] : make_int2(p, b.key[p]);
      const int h = q.y - c0;
      if (h >= 0 && h < SCAN_CHUNK) bucket[off_l[h] + atomicAdd(&fill_l[h], 1)] = q.x;
    }
    __syncthreads();  // the chunk's buckets
    for (int p = threadIdx.x; p < lim; p += SCAN_THREADS) {
      const int2 q = listed ? list[p] : make_int2(p, b.key[p]);
      const int h = q.y - c0;
      if (h >= 0 && h < SCAN_CHUNK) rank(q.x, h, vfl[q.x], bucket, 0);
    }
  }
}

// the work of the interaction from the patches [PLIST_SECTION sec, + PLIST_SECTION), by one
// work-group: for every patch that holds particles an entry (patch, part) per patch_slots of them.
// A section's entries follow each other in ascending order, the sections in any (the results do
// not depend on the order of the list). Clears the patches' counts
constexpr int PLIST_BATCH = PLIST_SECTION / SCAN_THREADS;  // patches per thread
__device__ inline void list_patches(kconst &k, int sec, const dbins &b) {
  const int np = patch_total(k) + (k.adaptive ? 1 : 0);  // and that past the grid (hash_count)
  const int p0 = sec * PLIST_SECTION + threadIdx.x * PLIST_BATCH;
  if (sec == 0 && threadIdx.x == 0) *b.plen_next = 0;
  if (sec * PLIST_SECTION >= np) return;
  int f[PLIST_BATCH], cnt = 0;
#pragma unroll
  for (int u = 0; u < PLIST_BATCH; u++) f[u] = p0 + u < np ? b.pcnt[p0 + u] : 0;
#pragma unroll
  for (int u = 0; u < PLIST_BATCH; u++)
    if (f[u]) {
      b.pcnt[p0 + u] = 0;
      f[u] = (f[u] + k.patch_slots - 1) / k.patch_slots;
      cnt += f[u];
    }
  __shared__ int first;
  int total;
  int o = block_exclusive_scan(cnt, total);
  if (total == 0) return;  // the same in every thread
  if (threadIdx.x == 0) first = atomicAdd(b.plen, total);
  __syncthreads();
  o += first;
#pragma unroll
  for (int u = 0; u < PLIST_BATCH; u++)
    for (int q = 0; q < f[u]; q++) b.plist[o++] = make_int2(p0 + u, q);
}

// sums of (fc.x, fc.y, ft.x, ft.y) over group g of 64 particles (storage order) of state st by one
// wave: the halving-stride tree over the lanes (lane l adds lane l + s for s = 32, 16, ..., 1, so
// lane 0 ends with the tree's root); lanes past N add zeros
__device__ inline void force_group(int N, int g, const dstate &st, double *__restrict__ partials) {
  const int lane = threadIdx.x & 63, i = 64 * g + lane;
  double v0 = 0., v1 = 0., v2 = 0., v3 = 0.;
  if (i < N) { v0 = st.fcx[i]; v1 = st.fcy[i]; v2 = st.ftx[i]; v3 = st.fty[i]; }
#pragma unroll
  for (int s = 32; s > 0; s >>= 1) {
    v0 = v0 + __shfl_down(v0, s, 64);
    v1 = v1 + __shfl_down(v1, s, 64);
    v2 = v2 + __shfl_down(v2, s, 64);
    v3 = v3 + __shfl_down(v3, s, 64);
  }
  if (lane == 0) { partials[4 * g] = v0; partials[4 * g + 1] = v1; partials[4 * g + 2] = v2; partials[4 * g + 3] = v3; }
}

// the group sums of the groups [g0, g0 + n) (n <= 64) by one wave: zeros for the groups without a
// force; clears the groups' flags
__device__ inline void force_groups(int N, int g0, int n, const dstate &st, const dforce &fo) {
  const int lane = threadIdx.x & 63, g = g0 + lane;
  const bool in = lane < n && g < (N + TILE - 1) / TILE * (TILE / 64);  // the groups of whole tiles
  const bool some = in && fo.gflag[g] != 0;
  if (some) fo.gflag[g] = 0;
  else if (in) reinterpret_cast<double4 *>(fo.partials)[g] = make_double4(0., 0., 0., 0.);
  for (unsigned long long m = __ballot(some); m; m &= m - 1ull)
    force_group(N, g0 + __builtin_ctzll(m), st, fo.partials);
}

// ------------------------------------------------------------------------------- predict
// artificial stress in single precision without trigonometry: with d = sqrt((sxx-syy)^2 + 4 sxy^2),
// cos 2theta = (sxx-syy)/d and sin 2theta = 2 sxy/d for theta = atan2(2 sxy, sxx-syy)/2, and the
// rotated normal stresses are the principal stresses (sxx+syy)/2 +- d/2 (actions_gpu.cu:53-97)
__device__ inline void artificial_stress_f32(float rho, float p, float Sxx, float Sxy, float Syy, float eps, float &Rxx,
                                             float &Rxy, float &Ryy) {
  const float sxx = Sxx - p, syy = Syy - p, sxy = Sxy;
  const float r21 = 1.0f / (rho * rho);
  const float a = sxx - syy, b = 2.0f * sxy;
  const float d = sqrtf(a * a + b * b);
  float c2 = 1.0f, s2 = 0.0f;
  if (d > 0.0f) { c2 = a / d; s2 = b / d; }
  const float ct2 = 0.5f * (1.0f + c2), st2 = 0.5f * (1.0f - c2), cs = 0.5f * s2;
  const float mid = 0.5f * (sxx + syy);
  const float r1 = mid + 0.5f * d, r2 = mid - 0.5f * d;
  const float q1 = r1 > 0.0f ? -eps * r1 * r21 : 0.0f;
  const float q2 = r2 > 0.0f ? -eps * r2 * r21 : 0.0f;
  Rxx = ct2 * q1 + st2 * q2;
  Rxy = cs * (q1 - q2);
  Ryy = st2 * q1 + ct2 * q2;
}

// the fields a neighbour record is made of: a particle's state and the rates of the predictor
struct rec_input {
  double x, y, u, v, sxx, sxy, syy, rho, T, h;
  double ptx, pty, vtx, vty, rhot, stxx, stxy, styy, Tt;
  int fl;
};

__device__ inline rec_input load_rec_input(const dstate &c, int s) {
  rec_input q;
  q.x = c.px[s]; q.y = c.py[s]; q.u = c.vx[s]; q.v = c.vy[s];
  q.sxx = c.sxx[s]; q.sxy = c.sxy[s]; q.syy = c.syy[s];
  q.rho = c.rho[s]; q.T = c.T[s];
  q.ptx = c.ptx[s]; q.pty = c.pty[s]; q.vtx = c.vtx[s]; q.vty = c.vty[s];
  q.rhot = c.rhot[s]; q.stxx = c.stxx[s]; q.stxy = c.stxy[s]; q.styy = c.styy[s];
  q.Tt = c.Tt[s];
  q.fl = c.flags[s] & FLAG_MASK;
  q.h = c.h[s];
  return q;
}

// leap-frog init + predict (in place)
__device__ inline void predict_input(kconst &k, rec_input &q) {
  if (q.fl & MFC_FLAG_BLANKED) return;  // leap_frog.cu:42-66
  const double hdt = 0.5 * k.dt;
  q.x = q.x + hdt * q.ptx; q.y = q.y + hdt * q.pty;
  q.u = q.u + hdt * q.vtx; q.v = q.v + hdt * q.vty;
  q.sxx = q.sxx + hdt * q.stxx; q.sxy = q.sxy + hdt * q.stxy; q.syy = q.syy + hdt * q.styy;
  q.rho = q.rho + hdt * q.rhot;
  q.T = q.T + hdt * q.Tt;
}

// the FP64 record of predicted input q with pressure p and artificial stress R, written at i
__device__ inline void store_record(kconst &k, const rec_input &q, double p, double rxx, double rxy,
                                    double ryy, int i, const drecords &recs) {
  const double r21 = 1. / (q.rho * q.rho);
  double r[REC];
  r[0] = q.x; r[1] = q.y;
  r[3] = q.h;
  r[4] = q.u; r[5] = q.v;
  r[6] = q.rho;
  r[7] = k.mass / q.rho;
  r[8] = (q.sxx - p) * r21;
  r[9] = q.sxy * r21;
  r[10] = (q.syy - p) * r21;
  r[11] = rxx; r[12] = rxy; r[13] = ryy;
  r[14] = tsqrt(k, k.K / q.rho);
  r[15] = q.T;
  bool fin = true;
#pragma unroll
  for (int c = 0; c < REC; c++)
    if (c != 2) fin = fin && finite_d(r[c]);
  const int rfl = q.fl | (fin ? 0 : FLAG_NONFINITE);
  r[2] = bits_to_double(rfl);
  double2 *dst = reinterpret_cast<double2 *>(recs.rec + (size_t)REC * i);
#pragma unroll
  for (int c = 0; c < REC / 2; c++) dst[c] = make_double2(r[2 * c], r[2 * c + 1]);
  recs.vfl[i] = rfl;
}

// leap-frog predict, EOS, artificial stress and the neighbour record of a particle in state q,
// written at its storage index i. The pressure and artificial stress of a tool particle enter no sum (every term that
// reads them skips pairs with one) and are 0 in its record.
template <bool F32>
__device__ inline void write_record(kconst &k, rec_input q, int i, const drecords &recs) {
  predict_input(k, q);
  const bool tool = q.fl & MFC_FLAG_TOOL;
  const double p = tool ? 0. : k.c0 * k.c0 * (q.rho - k.rho0);
  if constexpr (F32) {
    float fxx = 0.0f, fxy = 0.0f, fyy = 0.0f;
    if (!tool)
      artificial_stress_f32((float)q.rho, (float)p, (float)q.sxx, (float)q.sxy, (float)q.syy, (float)k.stress_eps, fxx,
                            fxy, fyy);
    const float rf = (float)q.rho, pf = (float)p;
    const float r21 = 1.0f / (rf * rf);
    float4 *dst = recs.rec32 + (size_t)REC32_PIECES * i;
    *reinterpret_cast<double2 *>(dst) = make_double2(q.x, q.y);
    dst[1] = make_float4((float)q.u, (float)q.v, rf, (float)(k.mass / q.rho));
    dst[2] = make_float4(((float)q.sxx - pf) * r21, (float)q.sxy * r21, ((float)q.syy - pf) * r21,
                         sqrtf((float)(k.K / q.rho)));
    dst[3] = make_float4(fxx, fxy, fyy, (float)q.T);
    recs.vfl[i] = q.fl;
  } else {
    double rxx = 0., rxy = 0., ryy = 0.;
    if (!tool) artificial_stress(q.rho, p, q.sxx, q.sxy, q.syy, k.stress_eps, rxx, rxy, ryy, k.promote != 0);
    store_record(k, q, p, rxx, rxy, ryy, i, recs);
  }
}

// the positional pressure and artificial stress of the step at sorted index i (the reference's
// arrays p and R, which its sort does not permute: a tool particle leaves what the slot holds),
// from the particle's record at storage index s
template <bool F32>
__device__ inline void store_positional(const dpositional &pos, int i, int s, double p, const drecords &recs) {
  pos.p[i] = p;
  if constexpr (F32) {
    const float4 a3 = recs.rec32[(size_t)REC32_PIECES * s + 3];
    pos.rxx[i] = a3.x; pos.rxy[i] = a3.y; pos.ryy[i] = a3.z;
  } else {
    const double *r = recs.rec + (size_t)REC * s;
    pos.rxx[i] = r[11]; pos.rxy[i] = r[12]; pos.ryy[i] = r[13];
  }
}

// ------------------------------------------------------------------------------- descriptors
// Fields of the instance descriptors read through the constant address space: the compiler
// then takes the pointers loaded from them for global pointers and emits global loads, which
// count only against the vector-memory wait counter, instead of flat loads, which also hold up
// every wait for an LDS or scalar load. (A whole-struct copy loses that, hence the field lists.)
// The descriptors do not change while a kernel runs.
#define MFC_CONST(T) const __attribute__((address_space(4))) T
#define MFC_F(f) o.f = c->f
__device__ inline dstate load_state(MFC_CONST(dstate) * c) {
  dstate o;
  MFC_F(px); MFC_F(py); MFC_F(vx); MFC_F(vy); MFC_F(sxx); MFC_F(sxy); MFC_F(syy); MFC_F(szz); MFC_F(rho);
  MFC_F(T); MFC_F(eps); MFC_F(epsd); MFC_F(h); MFC_F(fcx); MFC_F(fcy); MFC_F(ftx); MFC_F(fty); MFC_F(ptx);
  MFC_F(pty); MFC_F(vtx); MFC_F(vty); MFC_F(rhot); MFC_F(stxx); MFC_F(stxy); MFC_F(styy); MFC_F(stzz); MFC_F(Tt);
  MFC_F(flags); MFC_F(id);
  return o;
}
__device__ inline dbins load_bins(MFC_CONST(dbins) * c) {
  dbins o;
  MFC_F(key); MFC_F(key_sorted); MFC_F(offsets); MFC_F(bucket); MFC_F(tags);
  MFC_F(spos); MFC_F(bsum); MFC_F(bsum_next); MFC_F(pcnt); MFC_F(plist); MFC_F(plen); MFC_F(plen_next); MFC_F(clist); MFC_F(ccap); MFC_F(offsets_r); MFC_F(clamped);
  return o;
}
__device__ inline dpositional load_pos(MFC_CONST(dpositional) * c) {
  dpositional o;
  MFC_F(nx); MFC_F(ny); MFC_F(p); MFC_F(rxx); MFC_F(rxy); MFC_F(ryy); MFC_F(nx_out); MFC_F(ny_out);
  return o;
}
__device__ inline drecords load_recs(MFC_CONST(drecords) * c) {
  drecords o;
  MFC_F(f32); MFC_F(rec); MFC_F(rec32); MFC_F(vfl);
  return o;
}
__device__ inline dforce load_force(MFC_CONST(dforce) * c) {
  dforce o;
  MFC_F(partials); MFC_F(gflag); MFC_F(pending_next); MFC_F(force_last); MFC_F(hist); MFC_F(cap); MFC_F(ctr); MFC_F(pending);
  return o;
}
__device__ inline MFC_CONST(inst_args) * const_args(const inst_args *A, int q) {
  return (MFC_CONST(inst_args) *)(A + q);
}
#undef MFC_F

// ------------------------------------------------------------------------------- interact
// compensated (Kahan) accumulation in single precision
struct kahan {
  float s = 0.0f, c = 0.0f;
  __device__ inline void add(float x) {
    const float y = x - c;
    const float t = s + y;
    c = (t - s) - y;
    s = t;
  }
  __device__ inline double value() const { return (double)s - (double)c; }
};

// a particle's FP32C record as the pair terms read it
struct rec32 {
  double x, y;
  float u, v, rho, vol, Axx, Axy, Ayy, c, Rxx, Rxy, Ryy, T, h;
};
template <bool F32>
using rec_t = std::conditional_t<F32, rec32, rec64>;

// LDS of a work-group of the interaction (patch_cap, PATCH_TABLE and PATCH_COLS above). The records
// lie in arrays of 16-byte pieces (FP64: xy uv rho/vol A A/R R c/T; FP32C: xy u v rho vol | A c |
// R T), each one 16 bytes longer than a multiple of the banks, so that the lanes that stage the
// pieces of a record write different banks. FP64 with one thread per particle has no room for both c
// and T beside six pieces, the flags and the record's index, if three work-groups are to fit a
// CU (53.9 of 160 KB). Where c is a float's value (promote = 0) it takes the index's place once the
// record is staged; else one of the two (X) is there and c or T, whichever the sums read less, in
// memory. (With the c of each pair gathered from memory, through a pointer that could be to either memory,
// and full quotients and roots in the pair's terms the interaction of 197k particles took 116 us, now 104.)
//
// GEN: the variant of the kernel for states that do not suit that copy (mfc_sim::general): an h of its
// own for each particle, or so many particles per cell that few cells' windows fit. Only some pieces
// of a record are staged, and the others are read from memory for each pair (with positions and tags alone
// staged, a step of 197k particles took 287 us at hdx 2.3 instead of 222, 141 instead of 116 with an uneven h, FP64;
// with whole records and the h's for two work-groups to a CU 257 and 115).
constexpr int WALK_U = 4;  // candidates of a window whose loads are issued together
template <bool F32, int G, bool GEN>
struct patch_mem {
  static constexpr int CAP = patch_cap(F32, G, GEN);
  static constexpr bool ALL_IN_LDS = F32 || G > 1 || GEN;
  static constexpr int PIECES = GEN ? (G > 1 ? 1 : F32 ? 2 : 4) : F32 ? 4 : ALL_IN_LDS ? 7 : 6;
  // the terms of one pair per thread, exchanged between the threads of a particle: FP32C all nine,
  // FP64 in two halves (an odd stride keeps the rows on different banks)
  static constexpr int TERM_BYTES = G == 1 ? 0 : TILE * (F32 ? 9 * (int)sizeof(float) : 7 * (int)sizeof(double));
  float4 pieces[PIECES * (CAP + 1) + (PIECES == 1 ? WALK_U : 0)];  // sums_lds reads up to WALK_U - 1 past a candidate
  __device__ inline float4 *piece(int p) { return pieces + p * (CAP + 1); }
  __device__ inline const float4 *piece(int p) const { return pieces + p * (CAP + 1); }
  double X[ALL_IN_LDS ? 1 : CAP];
  int tag[CAP + WALK_U - 1];            // or, without ALL_IN_LDS and promote, c
  unsigned char fl[ALL_IN_LDS ? 1 : CAP + WALK_U - 1];  // the flags of the tag
  int flags;               // of all the candidates, PATCH_DENSE, PATCH_DENSER and PATCH_HEAPED
  int table[PATCH_TABLE];  // LDS index of the first candidate of each cell (row-major in a column)
  int col_first[PATCH_COLS + 1];  // of each staged column
  int col_shift[PATCH_COLS];      // LDS index minus sorted index in each staged column
  int own_first[PATCH_COLS + 1];  // number of the first particle of each own column
  using place = std::conditional_t<GEN, unsigned short, unsigned char>;  // holds an LDS index
  place list[G == 1 ? 1 : TILE / G][64];  // the pairs of a particle
  alignas(16) char terms[TERM_BYTES ? TERM_BYTES : 16];
  return_tape tape;  // G > 1
};

// a column range of some window of the patch holds more candidates than a mask of sums_lds (G == 1) has
// bits, than two of them have, or than five (without GEN: than one)
constexpr int PATCH_DENSE = 16, PATCH_DENSER = 32, PATCH_HEAPED = 64;

// where a sum reads the window candidates from: a patch's copy in LDS (index: place in the copy)
template <bool F32, int G, bool GEN>
struct lds_source {
  using mem = patch_mem<F32, G, GEN>;
  const mem *m;
  template <class T>
  using global = const __attribute__((address_space(1))) T *;  // no load of either memory
  global<double> rec;
  using float4v = float __attribute__((ext_vector_type(4)));
  using double2v = double __attribute__((ext_vector_type(2)));
  global<float4v> rec32;
  global<double> h;  // the start state's
  bool uniform_h;
  double h0;
  bool c_in_tag;  // mem::X holds T and mem::tag c
  bool t_in_lds;  // else mem::X holds T (some particle conducts heat), or c
  // GEN: piece Q of a record (without that of its flags and h), from the copy or from storage index s
  template <int Q>
  __device__ inline float4v part32(int j, size_t s) const {
    if constexpr (Q < mem::PIECES) return reinterpret_cast<const float4v *>(m->piece(Q))[j];
    else return rec32[REC32_PIECES * s + Q];
  }
  template <int Q>
  __device__ inline double2v part64(int j, size_t s) const {
    if constexpr (Q < mem::PIECES) return reinterpret_cast<const double2v *>(m->piece(Q))[j];
    else return ((global<double2v>)rec)[REC / 2 * s + Q + 1];
  }
  __device__ inline double2 pos(int j) const { return reinterpret_cast<const double2 *>(m->piece(0))[j]; }
  __device__ inline int tag(int j) const {  // its flags
    if constexpr (mem::ALL_IN_LDS) return m->tag[j];
    else return m->fl[j];
  }
  __device__ inline void cand(int j, double2 &p, int &t) const {
    p = pos(j);
    t = tag(j);
  }
  __device__ inline void heat(int j, int t, rec_t<F32> &q) const {  // T and rho
    if constexpr (GEN) {
      const size_t s = tag_index(t);
      if constexpr (F32) {
        q.rho = part32<1>(j, s).z; q.T = part32<3>(j, s).w;
      } else {
        q.rho = part64<2>(j, s).x; q.T = part64<6>(j, s).y;
      }
    } else if constexpr (F32) {
      q.rho = m->piece(1)[j].z; q.T = m->piece(3)[j].w;
    } else {
      q.rho = reinterpret_cast<const double2 *>(m->piece(2))[j].x;
      if constexpr (mem::ALL_IN_LDS) q.T = reinterpret_cast<const double2 *>(m->piece(6))[j].y;
      else if (c_in_tag || t_in_lds) q.T = m->X[j];
      else q.T = rec[(size_t)REC * tag_index(m->tag[j]) + 15];
    }
  }
  __device__ inline void record(int j, rec_t<F32> &q) const {
    if constexpr (GEN) {
      const size_t s = tag_index(m->tag[j]);
      if constexpr (F32) {
        const float4v a = part32<1>(j, s), b = part32<2>(j, s), c = part32<3>(j, s);
        q.u = a.x; q.v = a.y; q.rho = a.z; q.vol = a.w;
        q.Axx = b.x; q.Axy = b.y; q.Ayy = b.z; q.c = b.w;
        q.Rxx = c.x; q.Rxy = c.y; q.Ryy = c.z; q.T = c.w;
        q.h = (float)(uniform_h ? h0 : h[s]);
      } else {
        const double2v a = part64<1>(j, s), b = part64<2>(j, s), c = part64<3>(j, s), d = part64<4>(j, s),
                       e = part64<5>(j, s), f = part64<6>(j, s);
        q.u = a.x; q.v = a.y; q.rho = b.x; q.vol = b.y;
        q.Axx = c.x; q.Axy = c.y; q.Ayy = d.x; q.Rxx = d.y; q.Rxy = e.x; q.Ryy = e.y; q.c = f.x; q.T = f.y;
        q.h = uniform_h ? h0 : rec[REC * s + 3];
      }
    } else if constexpr (F32) {
      const float4 a = m->piece(1)[j], b = m->piece(2)[j], c = m->piece(3)[j];
      q.u = a.x; q.v = a.y; q.rho = a.z; q.vol = a.w;
      q.Axx = b.x; q.Axy = b.y; q.Ayy = b.z; q.c = b.w;
      q.Rxx = c.x; q.Rxy = c.y; q.Ryy = c.z; q.T = c.w;
      q.h = (float)h0;
    } else {
      if constexpr (mem::ALL_IN_LDS) {
        const double2 f = reinterpret_cast<const double2 *>(m->piece(6))[j];
        q.c = f.x; q.T = f.y;
      } else if (c_in_tag) {
        q.c = __int_as_float(m->tag[j]);
        q.T = m->X[j];
      } else if (t_in_lds) {
        q.c = rec[(size_t)REC * tag_index(m->tag[j]) + 14];
        q.T = m->X[j];
      } else {
        q.c = m->X[j];
        q.T = 0.;  // not read
      }
      const double2 a = reinterpret_cast<const double2 *>(m->piece(1))[j];
      const double2 b = reinterpret_cast<const double2 *>(m->piece(2))[j];
      const double2 c = reinterpret_cast<const double2 *>(m->piece(3))[j];
      const double2 d = reinterpret_cast<const double2 *>(m->piece(4))[j];
      const double2 e = reinterpret_cast<const double2 *>(m->piece(5))[j];
      q.u = a.x; q.v = a.y; q.rho = b.x; q.vol = b.y;
      q.Axx = c.x; q.Axy = c.y; q.Ayy = d.x; q.Rxx = d.y; q.Rxy = e.x; q.Ryy = e.y;
      q.h = h0;
    }
  }
};

// or the records in memory, their tags and positions there too (index: sorted index) or from a copy of
// them alone in LDS (index: place in the copy)
template <bool F32>
struct mem_records {
  const drecords r;
  const double *h;  // the start state's
  __device__ inline double2 pos_of(int tag) const {
    const size_t s = tag_index(tag);
    if constexpr (F32) return *reinterpret_cast<const double2 *>(r.rec32 + REC32_PIECES * s);
    else return *reinterpret_cast<const double2 *>(r.rec + REC * s);
  }
  __device__ inline void heat(int tag, rec_t<F32> &q) const {
    if constexpr (F32) {
      const float4 *d = r.rec32 + (size_t)REC32_PIECES * tag_index(tag);
      q.rho = d[1].z; q.T = d[3].w;
    } else {
      const double *d = r.rec + (size_t)REC * tag_index(tag);
      q.rho = d[6]; q.T = d[15];
    }
  }
  __device__ inline void record(int tag, rec_t<F32> &q) const {
    if constexpr (F32) {
      const float4 *d = r.rec32 + (size_t)REC32_PIECES * tag_index(tag);
      const float4 a = d[1], b = d[2], c = d[3];
      q.u = a.x; q.v = a.y; q.rho = a.z; q.vol = a.w;
      q.Axx = b.x; q.Axy = b.y; q.Ayy = b.z; q.c = b.w;
      q.Rxx = c.x; q.Rxy = c.y; q.Ryy = c.z; q.T = c.w;
      q.h = (float)h[tag_index(tag)];
    } else {
      const double *d = r.rec + (size_t)REC * tag_index(tag);
      q.h = d[3]; q.u = d[4]; q.v = d[5]; q.rho = d[6]; q.vol = d[7];
      q.Axx = d[8]; q.Axy = d[9]; q.Ayy = d[10]; q.Rxx = d[11]; q.Rxy = d[12]; q.Ryy = d[13];
      q.c = d[14]; q.T = d[15];
    }
  }
};
template <bool F32>
struct mem_source : mem_records<F32> {
  const int *tags;
  template <int U>
  __device__ inline void cands(const int (&j)[U], double2 (&p)[U], int (&tag)[U]) const {
#pragma unroll
    for (int u = 0; u < U; u++) tag[u] = tags[j[u]];
#pragma unroll
    for (int u = 0; u < U; u++) p[u] = this->pos_of(tag[u]);
  }
};
template <class T>
using lds_ptr = __attribute__((address_space(3))) T *;
struct lds_pos {
  double x, y;
};
template <bool F32>
struct copy_source : mem_records<F32> {
  lds_ptr<lds_pos> pos;
  lds_ptr<int> tags;
  template <int U>
  __device__ inline void cands(const int (&j)[U], double2 (&p)[U], int (&tag)[U]) const {
#pragma unroll
    for (int u = 0; u < U; u++) {
      tag[u] = tags[j[u]];
      p[u] = make_double2(pos[j[u]].x, pos[j[u]].y);
    }
  }
};

// what a particle's sums need of itself beside its record
struct sum_flags {
  bool tool, nonfinite, run_mech, run_pse;
  double ta;
};

// e^x with the operations of mfcm::exp, without its special cases for x in (-700, 0]
__device__ inline double exp_neg(double x) {
  if (!(x > -700. && x <= 0.)) return mfcm::exp(x);
  const double kd = floor(x * mfcm::INV_LN2 + 0.5);
  const double r = (x - kd * mfcm::LN2_HI) - kd * mfcm::LN2_LO;
  return __builtin_ldexp(mfcm::exp_reduced(r), (int)kd);  // 2^k is exact
}

// FP64 sums of a particle: the support test and PSE term of a window candidate, and the terms of
// a pair
struct math64 {
  using rec = rec64;
  static constexpr int TERMS = 13;
  kconst &k;
  const rec64 &a;
  const sum_flags &f;
  double h1, fourh2, fac, h2, inv_h2, pse_c, inv_wd;
  __device__ inline math64(kconst &k_, const rec64 &a_, const sum_flags &f_) : k(k_), a(a_), f(f_) {
    h1 = 1 / a.h;
    fourh2 = 4 * a.h * a.h;
    fac = PI_FAC * h1 * h1;
    h2 = a.h * a.h;
    const double h4 = h2 * h2;
    pse_c = 4. / (h4 * M_PI);
    inv_h2 = 1. / h2;
    inv_wd = 1. / k.wdeltap;
  }
  // outside the support the reference adds exact zeros, unless a value is non-finite
  __device__ inline bool near(double2 p) const {
    const double dx = a.x - p.x, dy = a.y - p.y;
    const double rr2 = dx * dx + dy * dy;
    return !(rr2 >= fourh2 || rr2 < 1e-8);
  }
  __device__ inline bool support(double2 p, int tag) const {
    return !(tag & MFC_FLAG_BLANKED) && (near(p) || f.nonfinite || (tag & FLAG_NONFINITE));
  }
  template <bool FINITE>
  __device__ inline double pse(double2 p, const rec64 &b) const {  // do_interactions_heat_pse (interactions_gpu.cu:130-139)
    const double dx = a.x - p.x, dy = a.y - p.y;
    const double xx = sqrt(dx * dx + dy * dy);
    const double w2 = pse_c * (FINITE ? exp_neg(div_by(-xx * xx, h2, inv_h2)) : mfcm::exp(-xx * xx / (h2)));
    return (b.T - a.T) * w2 * k.mass / b.rho;
  }
  template <bool FINITE, class ADD>
  __device__ inline void pair(double2 p, bool tool_j, rec64 &b, ADD &add) const {
    b.x = p.x; b.y = p.y;
    pair_terms<FINITE>(k, a, f.tool, f.ta, h1, fourh2, fac, inv_wd, b, tool_j, add);
  }
};

// FP32C sums with Kahan compensation (the same pair terms, rearranged for single precision:
// hardware reciprocals and reciprocal square roots instead of divisions, the particle mass and
// the factor 2 of Brookshaw taken out of the sums, e.gradW/r of Brookshaw written as der*fac,
// which is its exact value, and the stress and viscosity terms of each acceleration component
// added before their one compensated sum). Pair distances are formed in FP64 and then rounded.
struct terms32 {
  float vd0, vd1, vd2, vd3, ax, ay, xt0, xt1, tl;
  bool mech;  // the first eight are added to the sums (tl when ta != 0)
  __device__ inline void add_mech(float a0, float a1, float a2, float a3, float a4, float a5, float a6, float a7) {
    vd0 = a0; vd1 = a1; vd2 = a2; vd3 = a3; ax = a4; ay = a5; xt0 = a6; xt1 = a7;
    mech = true;
  }
  __device__ inline void add_heat(float t) { tl = t; }
};
// the sums themselves, by one thread
struct sums32 {
  kahan s[9];
  __device__ inline void add_mech(float a0, float a1, float a2, float a3, float a4, float a5, float a6, float a7) {
    s[0].add(a0); s[1].add(a1); s[2].add(a2); s[3].add(a3); s[4].add(a4); s[5].add(a5); s[6].add(a6); s[7].add(a7);
  }
  __device__ inline void add_heat(float t) { s[8].add(t); }
};
struct math32 {
  using rec = rec32;
  kconst &k;
  const rec32 &a;
  const sum_flags &f;
  float ta, Ti, h1, fourh2, fac, inv_wd, eta2, alpha, beta, xeps, inv_h2, pse_c, massf;
  __device__ inline math32(kconst &k_, const rec32 &a_, const sum_flags &f_) : k(k_), a(a_), f(f_) {
    ta = (float)f.ta;
    Ti = ta != 0.0f ? a.T : 0.0f;
    h1 = 1.0f / a.h;
    fourh2 = 4.0f * a.h * a.h;
    fac = (float)PI_FAC * h1 * h1;
    inv_wd = (float)(1.0 / k.wdeltap);
    eta2 = (float)(k.av_eta * k.av_eta);
    alpha = (float)k.av_alpha; beta = (float)k.av_beta; xeps = (float)k.xsph_eps;
    inv_h2 = h1 * h1;
    pse_c = (float)(4. / M_PI) * inv_h2 * inv_h2;
    massf = (float)k.mass;
  }
  __device__ inline void distance(double2 p, float &dx, float &dy, float &rr2) const {
    dx = (float)(a.x - p.x);
    dy = (float)(a.y - p.y);
    rr2 = __builtin_fmaf(dx, dx, dy * dy);
  }
  __device__ inline bool near(double2 p) const {
    float dx, dy, rr2;
    distance(p, dx, dy, rr2);
    return !(rr2 >= fourh2 || rr2 < 1e-8f);
  }
  __device__ inline bool support(double2 p, int tag) const { return near(p) && !(tag & MFC_FLAG_BLANKED); }
  template <bool>
  __device__ inline float pse(double2 p, const rec32 &b) const {
    float dx, dy, rr2;
    distance(p, dx, dy, rr2);
    const float w2 = pse_c * __expf(-rr2 * inv_h2);
    return (b.T - a.T) * w2 * (massf * __builtin_amdgcn_rcpf(b.rho));
  }
  template <class SINK>
  __device__ inline void pair(double2 p, bool tool_j, const rec32 &b, SINK &sink) const {
    float dx, dy, rr2;
    distance(p, dx, dy, rr2);
    const float inv_r = __builtin_amdgcn_rsqf(rr2);
    const float q = rr2 * inv_r * h1;
    float val, der;  // der = dW/dr / r without the factor fac
    if (q > 1.0f) {
      const float m = 2.0f - q, m2 = m * m;
      val = 0.25f * m2 * m2 * m2;
      der = -0.75f * m2 * h1 * inv_r;
    } else {
      val = 1.0f - 1.5f * q * q * (1.0f - 0.5f * q);
      der = -3.0f * q * (1.0f - 0.75f * q) * h1 * inv_r;
    }
    const float w = val * fac, gr = der * fac;
    const float w_x = gr * dx, w_y = gr * dy;
    if (!f.tool && !tool_j) {
      const float tx = w_x * b.vol, ty = w_y * b.vol;
      const float du = b.u - a.u, dv = b.v - a.v;
      float fab = w * inv_wd;
      fab *= fab;
      fab *= fab;
      const float sx = a.Axx + b.Axx + fab * (a.Rxx + b.Rxx);
      const float sy = a.Axy + b.Axy + fab * (a.Rxy + b.Rxy);
      const float sz = a.Ayy + b.Ayy + fab * (a.Ryy + b.Ryy);
      float fx = __builtin_fmaf(sx, w_x, sy * w_y), fy = __builtin_fmaf(sy, w_x, sz * w_y);
      const float vijx = -du, vijy = -dv;
      const float vdx = __builtin_fmaf(vijx, dx, vijy * dy);
      const float inv_rhoij = 2.0f * __builtin_amdgcn_rcpf(a.rho + b.rho);
      if (vdx < 0.0f) {
        const float cij = 0.5f * (a.c + b.c);
        const float hij = 0.5f * (a.h + b.h);
        const float muij = hij * vdx * __builtin_amdgcn_rcpf(__builtin_fmaf(eta2 * hij, hij, rr2));
        const float piij = (-alpha * cij * muij + beta * muij * muij) * inv_rhoij;
        fx = __builtin_fmaf(-piij, w_x, fx);
        fy = __builtin_fmaf(-piij, w_y, fy);
      }
      const float xs = -xeps * w * inv_rhoij;
      sink.add_mech(du * tx, du * ty, dv * tx, dv * ty, fx, fy, xs * vijx, xs * vijy);
    }
    if (ta != 0.0f) sink.add_heat(b.vol * (Ti - b.T) * gr);
  }
};
template <bool F32>
using math_t = std::conditional_t<F32, math32, math64>;

// the sums as update_particle takes them, from the FP32C sums s (in the order of terms32; the
// stress and viscosity sums enter the acceleration only as sd0 + sd1 + vt0 and sd2 + sd3 + vt1
// (actions_gpu.cu momentum), so they are accumulated as those two)
__device__ inline pair_acc acc_of_sums32(kconst &k, const double *s) {
  return {s[0], s[1], s[2], s[3], k.mass * s[4], 0., k.mass * s[5], 0., 0., 0., k.mass * s[6], k.mass * s[7], 2.0 * s[8]};
}

__device__ inline pair_acc acc_of(kconst &k, const sums32 &q) {
  double s[9];
#pragma unroll
  for (int c = 0; c < 9; c++) s[c] = q.s[c].value();
  return acc_of_sums32(k, s);
}
__device__ inline double value_of(const kahan &s) { return s.value(); }
__device__ inline double value_of(double s) { return s; }

// The neighbour sums of a particle by one thread from the records in memory: the window's
// candidates in order, which is the reference's (interactions_gpu.cu:219-331), 64 at a time: first the
// support tests, whose loads are issued together for WALK_U candidates, then the pairs
template <bool F32, bool FINITE, class SRC>
__device__ inline void sums_mem(kconst &k, const SRC &src, const window &w, const rec_t<F32> &a, const sum_flags &f,
                                pair_acc &acc, double &tpse) {
  const math_t<F32> mt(k, a, f);
  std::conditional_t<F32, sums32, pair_sums> sum = {};
  std::conditional_t<F32, kahan, double> tp = {};
  for (int c0 = 0; c0 < w.total; c0 += 64) {
    const int n = w.total - c0 < 64 ? w.total - c0 : 64;
    unsigned long long mask = 0ull;
    for (int q = 0; q < n; q += WALK_U) {
      int j[WALK_U], tag[WALK_U];
      double2 p[WALK_U];
#pragma unroll
      for (int u = 0; u < WALK_U; u++) j[u] = w.at(c0 + (q + u < n ? q + u : n - 1));
      src.cands(j, p, tag);
#pragma unroll
      for (int u = 0; u < WALK_U; u++) {
        if (q + u >= n) continue;
        if (f.run_pse) {  // all members of the window
          rec_t<F32> b;
          src.heat(tag[u], b);
          if constexpr (F32) tp.add(mt.template pse<FINITE>(p[u], b));
          else tp += mt.template pse<FINITE>(p[u], b);
        }
        if (f.run_mech && mt.support(p[u], tag[u])) mask |= 1ull << (q + u);
      }
    }
    for (; mask; mask &= mask - 1ull) {
      const int j[1] = {w.at(c0 + __builtin_ctzll(mask))};
      double2 p[1];
      int tag[1];
      rec_t<F32> b;
      src.cands(j, p, tag);
      src.record(tag[0], b);
      if constexpr (F32) mt.pair(p[0], (tag[0] & MFC_FLAG_TOOL) != 0, b, sum);
      else mt.template pair<FINITE>(p[0], (tag[0] & MFC_FLAG_TOOL) != 0, b, sum);
    }
  }
  if constexpr (F32) acc = acc_of(k, sum);
  else acc = sum;
  tpse = value_of(tp);
}

// The same by one thread from a patch's LDS copy, the window as 5 column ranges [b, e) of it. First
// the support tests of every candidate set the bits of a mask per column, then the pairs of the
// set bits are evaluated in order: the wave runs the pair body about as often as its busiest lane
// has pairs instead of once per candidate. The test loops run column by column (about 80 rounds of
// a wave for windows of 56 candidates, whose columns hold 8 or 16 by turns), because a candidate
// numbered through the columns costs 11 instructions to find and one of a column none; in the
// loop over the pairs a lane moves its next column's mask up when its current one is used up.
// flags: what the patch's candidates have of TOOL and BLANKED (without PSE, the copy holds both
// coordinates of a blanked particle at infinity, whatever they are: one that is not a number would
// pass the test of near).
// Where a column has more candidates than a mask has bits (GEN), two columns are taken at a time, each in two
// masks, or one in five.
template <bool F32, int G, bool PSE, bool GEN>
__device__ inline void sums_lds(kconst &k, const lds_source<F32, G, GEN> &src, int flags, const int b[5],
                                const int e[5], const rec_t<F32> &a, const sum_flags &f, pair_acc &acc, double &tpse) {
  const math_t<F32> mt(k, a, f);
  std::conditional_t<F32, sums32, pair_sums> sum = {};
  std::conditional_t<F32, kahan, double> tp = {};
  if constexpr (PSE) {
    if (f.run_pse) {  // all members of the window, two at a time
      const window w = window_of(b, e);
      for (int t = 0; t < w.total; t += 2) {
        const bool two = t + 1 < w.total;
        const int j0 = w.at(t), j1 = w.at(two ? t + 1 : t);
        rec_t<F32> c0, c1;
        src.heat(j0, src.tag(j0), c0);
        src.heat(j1, src.tag(j1), c1);
        const auto v0 = mt.template pse<true>(src.pos(j0), c0), v1 = mt.template pse<true>(src.pos(j1), c1);
        if constexpr (F32) {
          tp.add(v0);
          if (two) tp.add(v1);
        } else {
          tp += v0;
          if (two) tp += v1;
        }
      }
    }
  }
  const bool dense = GEN && (flags & PATCH_DENSE), denser = GEN && (flags & PATCH_DENSER);
  for (int pass = 0; pass < (denser ? 5 : dense ? 3 : 1); pass++) {
    unsigned m[5];
    int at[5];
#pragma unroll
    for (int r = 0; r < 5; r++) {
      int first = b[r], n = e[r] - b[r];
      if (denser) {
        first = (pass == 0 ? b[0] : pass == 1 ? b[1] : pass == 2 ? b[2] : pass == 3 ? b[3] : b[4]) + 32 * r;
        n = (pass == 0 ? e[0] : pass == 1 ? e[1] : pass == 2 ? e[2] : pass == 3 ? e[3] : e[4]) - first;
      } else if (dense) {
        first = (r < 2 ? (pass == 0 ? b[0] : pass == 1 ? b[2] : b[4]) : pass == 0 ? b[1] : b[3]) + (r & 1 ? 32 : 0);
        n = (r < 2 ? (pass == 0 ? e[0] : pass == 1 ? e[2] : e[4]) : pass == 0 ? e[1] : e[3]) - first;
        if (r == 4 || (pass == 2 && r >= 2)) n = 0;
      }
      if (GEN) n = n < 32 ? n : 32;
      if (!f.run_mech) n = 0;
      unsigned mr = 0u;
      for (int q = 0; q < n; q += WALK_U) {
        double2 p[WALK_U];
#pragma unroll
        for (int u = 0; u < WALK_U; u++) p[u] = src.pos(first + q + u);  // past the range: some other piece of the copy
        unsigned hits = 0u;
#pragma unroll
        for (int u = 0; u < WALK_U; u++) {
          bool hit = q + u < n;
          if (PSE && (flags & MFC_FLAG_BLANKED)) hit = hit && !(src.tag(first + q + u) & MFC_FLAG_BLANKED);
          const bool in = mt.near(p[u]);
          hits |= (hit & in) ? 1u << u : 0u;
        }
        mr |= hits << q;
      }
      m[r] = mr;
      at[r] = first;
    }
#pragma unroll
    for (int r = 3; r >= 0; r--)  // columns without a pair to the end
      if (m[r] == 0u) {
#pragma unroll
        for (int q = r; q < 4; q++) { m[q] = m[q + 1]; at[q] = at[q + 1]; }
        m[4] = 0u;
      }
    while (m[0]) {
      const int j = at[0] + __builtin_ctz(m[0]);
      m[0] &= m[0] - 1u;
      const double2 p = src.pos(j);
      rec_t<F32> c;
      src.record(j, c);
      bool tool_j = false;
      if (flags & MFC_FLAG_TOOL) tool_j = src.tag(j) & MFC_FLAG_TOOL;  // the same branch in every lane
      const bool used = m[0] == 0u;  // selects: under a branch every mask is moved twice
#pragma unroll
      for (int q = 0; q < 4; q++) { m[q] = used ? m[q + 1] : m[q]; at[q] = used ? at[q + 1] : at[q]; }
      m[4] = used ? 0u : m[4];
      if constexpr (F32) mt.pair(p, tool_j, c, sum);
      else mt.template pair<true>(p, tool_j, c, sum);
    }
  }
  if constexpr (F32) acc = acc_of(k, sum);
  else acc = sum;
  tpse = value_of(tp);
}

// LDS written by lanes of a wave and read by others of the same wave: DS operations of a wave
// complete in order, so only the compiler has to keep theirs
__device__ inline void wave_lds_fence() {
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  __builtin_amdgcn_wave_barrier();
}

// The same sums by G neighbouring threads, for a state too small to fill the chip with one thread
// per particle, where the length of a thread's chain of dependent operations is what a step takes.
// The threads test G candidates at a time and list the pairs in order; then each evaluates one
// pair, and every sum belongs to one of them, which adds the G pairs' terms in order through LDS:
// the order of every sum, and so its bits, are sums_lds's. The sums end in out[0..ACC_N) (LDS).
template <bool F32, int G, bool GEN>
__device__ inline void sums_group(kconst &k, const lds_source<F32, G, GEN> &src, const window &w,
                                  const rec_t<F32> &a, const sum_flags &f, typename patch_mem<F32, G, GEN>::place *list, char *terms,
                                  double *out) {
  const math_t<F32> mt(k, a, f);
  const int lane = threadIdx.x & 63, r = lane % G, g0 = lane - r;
  constexpr int ROW = F32 ? 9 : 7;                  // terms per row
  constexpr int PARTS = F32 ? 1 : 2;                // rows a pair's terms take, one after the other
  constexpr int OWN = (ROW + G - 1) / G;            // sums per thread and part
  using T = std::conditional_t<F32, float, double>;
  T *row = reinterpret_cast<T *>(terms) + (size_t)lane * ROW;
  const T *rows = reinterpret_cast<const T *>(terms) + (size_t)g0 * ROW;
  std::conditional_t<F32, kahan, double> sum[PARTS][OWN] = {};
  std::conditional_t<F32, kahan, double> tp = {};
  for (int c0 = 0; c0 < w.total; c0 += 64) {
    const int n = w.total - c0 < 64 ? w.total - c0 : 64;
    int cnt = 0;
    for (int u0 = 0; u0 < n; u0 += G) {
      const bool in = u0 + r < n;
      const int j = w.at(c0 + (in ? u0 + r : n - 1));
      double2 p;
      int tag;
      src.cand(j, p, tag);
      if (f.run_pse) {
        rec_t<F32> b;
        src.heat(j, tag, b);
        const T v = mt.template pse<true>(p, b);
#pragma unroll
        for (int q = 0; q < G; q++) {
          const T vq = __shfl(v, q, G);
          if (u0 + q < n) {
            if constexpr (F32) tp.add(vq);
            else tp += vq;
          }
        }
      }
      const bool hit = f.run_mech && in && mt.support(p, tag);
      const unsigned bits = (unsigned)(__ballot(hit) >> g0) & ((1u << G) - 1u);
      if (hit) list[cnt + __popc(bits & ((1u << r) - 1u))] = (typename patch_mem<F32, G, GEN>::place)j;
      cnt += __popc(bits);
    }
    wave_lds_fence();
    for (int p0 = 0; p0 < cnt; p0 += G) {
      const bool in = p0 + r < cnt;
      const int j = list[in ? p0 + r : p0];
      double2 p;
      int tag;
      rec_t<F32> b;
      src.cand(j, p, tag);
      src.record(j, b);
      if constexpr (F32) {
        terms32 t = {0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, false};
        mt.pair(p, (tag & MFC_FLAG_TOOL) != 0, b, t);
        row[0] = t.vd0; row[1] = t.vd1; row[2] = t.vd2; row[3] = t.vd3;
        row[4] = t.ax; row[5] = t.ay; row[6] = t.xt0; row[7] = t.xt1; row[8] = t.tl;
        const unsigned mech = (unsigned)(__ballot(in && t.mech) >> g0);
        wave_lds_fence();
#pragma unroll
        for (int q = 0; q < G; q++) {
#pragma unroll
          for (int o = 0; o < OWN; o++) {
            const int c = r + G * o;
            const float v = rows[q * ROW + (c < ROW ? c : 0)];
            if (c < 8 ? (mech >> q) & 1u : p0 + q < cnt && mt.ta != 0.0f) sum[0][o].add(v);
          }
        }
        wave_lds_fence();
      } else {
        pair_row terms_of;
        mt.template pair<true>(p, (tag & MFC_FLAG_TOOL) != 0, b, terms_of);
        const double *tv = terms_of.t;
#pragma unroll
        for (int h = 0; h < PARTS; h++) {
#pragma unroll
          for (int c = 0; c < ROW; c++) row[c] = tv[h * ROW + c];
          wave_lds_fence();
#pragma unroll
          for (int q = 0; q < G; q++) {
#pragma unroll
            for (int o = 0; o < OWN; o++) {
              const int c = r + G * o;
              const double v = rows[q * ROW + (c < ROW ? c : 0)];
              if (p0 + q < cnt) sum[h][o] += v;
            }
          }
          wave_lds_fence();
        }
      }
    }
  }
  wave_lds_fence();
#pragma unroll
  for (int h = 0; h < PARTS; h++)
#pragma unroll
    for (int o = 0; o < OWN; o++) {
      const int c = r + G * o;
      if constexpr (F32) {
        if (c < ROW) out[c] = sum[h][o].value();
      } else {
        if (c < ROW && h * ROW + c < ACC_N - 1) out[h * ROW + c] = sum[h][o];
      }
    }
  if (r == 0) {
    if constexpr (F32) out[ACC_N - 1] = tp.value();
    else out[ACC_N - 1] = tp;
  }
}

// a particle's Johnson-Cook return, left for the secant after update_particle: the
// yield test's inputs and the state the return starts from (the stress, plastic strain and rate
// and temperature that update_particle stored are replaced once the return is done)
struct deferred_return {
  bool need;   // the particle returns this step
  bool fixed;  // the thermal boundary condition resets its temperature after the return
  rr_input in;
  double rho, sxx, sxy, syy, szz, eps, epsd, T;
};

// everything after the neighbour sums for particle i (sorted index), in the reference's order;
// returns the particle's fc and ft for the tool force. The secant of a Johnson-Cook return runs
// after this call (finish_return); the other results do not depend on it
// reads particle s of the unsorted start state src (tags[i]) and writes the updated
// particle to position i of dst: the gather into sorted order happens here, once. Also writes the
// step's positional values and, with the state before a return, the next step's record (rn)
template <bool F32>
__device__ inline void update_particle(kconst &k, int i, int s, const pair_acc &acc, double tpse,
                                       const dstate &src, const dstate &dst, const dpositional &pos,
                                       const drecords &r, const drecords &rn, const mfc_tool_state &tool_now, double fsum[4], double &x_out, double &y_out,
                                       int &fl_out, deferred_return &dr) {
  const bool pse = k.pse != 0;
  int fl = src.flags[s] & FLAG_MASK;
  const bool blank = fl & MFC_FLAG_BLANKED, tool = fl & MFC_FLAG_TOOL, fixed = fl & MFC_FLAG_FIXED;
  const double ta = pse ? 0. : (tool ? k.alpha_tool : k.alpha_wp);
  const bool run_mech = !blank && (!pse || !tool);
  const bool run_pse = !blank && pse && k.thermal_wp;
  // state at the start of the step (sorted) and previous derivatives
  const double x0 = src.px[s], y0 = src.py[s], u0 = src.vx[s], v0 = src.vy[s];
  const double sxx0 = src.sxx[s], sxy0 = src.sxy[s], syy0 = src.syy[s], szz0 = src.szz[s];
  const double rho0 = src.rho[s], T0 = src.T[s];
  double ptx = src.ptx[s], pty = src.pty[s], vtx = src.vtx[s], vty = src.vty[s];
  double rhot = src.rhot[s], stxx = src.stxx[s], stxy = src.stxy[s], styy = src.styy[s], stzz = src.stzz[s];
  double Tt = src.Tt[s];
  // grid_gpu_rothlin's sort leaves ft in place: the contact reads the history at the sorted index
  const int sft = k.rothlin ? i : s;
  double fcx = src.fcx[s], fcy = src.fcy[s], ftx = src.ftx[sft], fty = src.fty[sft];
  double eps = src.eps[s], epsd = src.epsd[s];
  // predicted state (same expressions as predict)
  double pu = u0, pv = v0, psxx = sxx0, psxy = sxy0, psyy = syy0, pszz = szz0, prho = rho0;
  if (!blank) {
    const double hdt = 0.5 * k.dt;
    pu = u0 + hdt * vtx; pv = v0 + hdt * vty;
    psxx = sxx0 + hdt * stxx; psxy = sxy0 + hdt * stxy; psyy = syy0 + hdt * styy; pszz = szz0 + hdt * stzz;
    prho = rho0 + hdt * rhot;
  }
  const double p = k.c0 * k.c0 * (prho - k.rho0);  // EOS of the predicted density
  if (!tool) store_positional<F32>(pos, i, s, p, r);
  // interaction outputs (interactions_gpu.cu:334-344, :143)
  if (run_mech) {
    ptx = acc.xt0; pty = acc.xt1; vtx = acc.vt0; vty = acc.vt1;
    if (ta != 0.) Tt = ta * acc.tl;
  }
  if (run_pse) {
    double tflag = tool ? 1. : 0.;
    if (k.pse_quirk && i >= k.N / 2) tflag = 0.;
    Tt = ((tflag == 1.) ? k.alpha_tool : k.alpha_wp) * tpse;
  }
  if (!tool) {
    // Jaumann rate, continuity, momentum, advection (actions_gpu.cu:99-224)
    jaumann(k.G, acc.vd0, acc.vd1, acc.vd2, acc.vd3, psxx, psxy, psyy, pszz, stxx, stxy, styy, stzz);
    rhot = -prho * (acc.vd0 + acc.vd3);
    vtx += acc.sd0 + acc.sd1 + fcx / k.mass + ftx / k.mass;
    vty += acc.sd2 + acc.sd3 + fcy / k.mass + fty / k.mass;
    ptx = ptx + pu;
    pty = pty + pv;
  }
  // leap-frog corrector (leap_frog.cu:68-92)
  double x = x0, y = y0, u = u0, v = v0, sxx = sxx0, sxy = sxy0, syy = syy0, szz = szz0, rho = rho0, T = T0;
  if (!blank) {
    x = x0 + k.dt * ptx; y = y0 + k.dt * pty;
    u = u0 + k.dt * vtx; v = v0 + k.dt * vty;
    sxx = sxx0 + k.dt * stxx; sxy = sxy0 + k.dt * stxy; syy = syy0 + k.dt * styy; szz = szz0 + k.dt * stzz;
    rho = rho0 + k.dt * rhot;
    T = T0 + k.dt * Tt;
  }
  // frictional heating with the positional normal of the previous step (actions_gpu.cu:135-162)
  if (k.fric_heat && !tool) {
    const double fmag = tsqrt(k, ftx * ftx + fty * fty);
    if (fmag != 0.) {
      const double nx = pos.nx[i], ny = pos.ny[i];
      const double dvx = u - k.tool_vx, dvy = v - k.tool_vy;
      const double dvn = dvx * nx + dvy * ny;
      const double rx = dvx - dvn, ry = dvy - dvn;
      const double vmag = tsqrt(k, rx * rx + ry * ry);
      T += k.eta_heat * k.dt * fmag * vmag / (k.cp * k.mass);
    }
  }
  if (!tool && k.plastic) {
    dr.need = plasticity_test(k, p, sxx, sxy, syy, szz, eps, epsd, T, dr.in);
    if (dr.need) {
      dr.fixed = fixed;
      dr.rho = rho; dr.sxx = sxx; dr.sxy = sxy; dr.syy = syy; dr.szz = szz;
      dr.eps = eps; dr.epsd = epsd; dr.T = T;
    }
  }
  if (tool) {  // update_tool_particles (tool_gpu.cu:210-221)
    x += k.dt * k.tool_vx;
    y += k.dt * k.tool_vy;
    if (pos.nx_out != pos.nx) {  // the same in every thread; a tool particle leaves what the slot holds
      pos.nx_out[i] = pos.nx[i];
      pos.ny_out[i] = pos.ny[i];
    }
  }
  if (!tool) {
    double nx, ny;
    contact_force(k, tool_now, x, y, u, v, fcx, fcy, ftx, fty, nx, ny);
    pos.nx_out[i] = nx; pos.ny_out[i] = ny;
    if (fixed) {  // actions_gpu.cu:296-311
      u = 0.; v = 0.; fcx = 0.; fcy = 0.; ptx = 0.; pty = 0.; vtx = 0.; vty = 0.;
    }
  }
  if (k.thermal_bc && fixed) T = k.T_init;  // actions_gpu.cu:287-294
  if (!blank) {  // actions_gpu.cu:317-349
    bool bad = !finite_d(ptx) || !finite_d(pty) || !finite_d(vtx) || !finite_d(vty) || !finite_d(stxx) ||
               !finite_d(stxy) || !finite_d(styy) || !finite_d(stzz) || !finite_d(rhot) || !finite_d(Tt);
    if (bad) fl |= MFC_FLAG_BLANKED;
  }
  dst.px[i] = x; dst.py[i] = y; dst.vx[i] = u; dst.vy[i] = v;
  dst.sxx[i] = sxx; dst.sxy[i] = sxy; dst.syy[i] = syy; dst.szz[i] = szz;
  const double h = src.h[s];
  dst.rho[i] = rho; dst.T[i] = T; dst.eps[i] = eps; dst.epsd[i] = epsd; dst.h[i] = h;
  dst.fcx[i] = fcx; dst.fcy[i] = fcy; dst.ftx[i] = ftx; dst.fty[i] = fty;
  dst.ptx[i] = ptx; dst.pty[i] = pty; dst.vtx[i] = vtx; dst.vty[i] = vty;
  dst.rhot[i] = rhot; dst.stxx[i] = stxx; dst.stxy[i] = stxy; dst.styy[i] = styy; dst.stzz[i] = stzz;
  dst.Tt[i] = Tt;
  dst.flags[i] = fl;
  dst.id[i] = src.id[s];
  fsum[0] = fcx; fsum[1] = fcy; fsum[2] = ftx; fsum[3] = fty;
  x_out = x; y_out = y; fl_out = fl;
  write_record<F32>(k, {x, y, u, v, sxx, sxy, syy, rho, T, h, ptx, pty, vtx, vty, rhot, stxx, stxy, styy, Tt, fl}, i,
                    rn);
}

// the return of a particle that needed one, with the secant's dl: the stress, plastic strain and
// rate and temperature at sorted index i (the thermal boundary condition after the return, as in
// update_particle), and its record again with them
template <bool F32>
__device__ inline void finish_return(kconst &k, int i, double dl, deferred_return &dr, const dstate &dst,
                                     const drecords &rn) {
  plasticity_finish(k, dr.rho, dl, dr.in, dr.sxx, dr.sxy, dr.syy, dr.szz, dr.eps, dr.epsd, dr.T);
  if (k.thermal_bc && dr.fixed) dr.T = k.T_init;  // actions_gpu.cu:287-294
  dst.sxx[i] = dr.sxx; dst.sxy[i] = dr.sxy; dst.syy[i] = dr.syy; dst.szz[i] = dr.szz;
  dst.eps[i] = dr.eps; dst.epsd[i] = dr.epsd; dst.T[i] = dr.T;
  // the other fields as update_particle stored them: few particles return, so reading them back
  // costs less than keeping them in registers through the secant
  rec_input q = load_rec_input(dst, i);
  q.sxx = dr.sxx; q.sxy = dr.sxy; q.syy = dr.syy; q.T = dr.T;
  write_record<F32>(k, q, i, rn);
}

// the next step's first binning pass for the updated particle i (its storage position in the
// next step): cell id, arrival slot and patch, as hash_count would take them from the updated
// state (the bins are passed by value so that they stay in registers). An adaptive grid bins the
// next step's start state after its geometry pass instead.
__device__ inline void next_cell(kconst &k, int i, bool live, double x, double y, int fl, const dbins next) {
  if (k.adaptive) return;  // the same in every thread
  const int h = live ? particle_cell(k, x, y, fl, next.key_sorted[i], next.clamped) : -1;
  count_cell(i, h, next.key, next.bsum_next, next.clist, next.ccap);
  count_patch(h < 0 ? -1 : patch_of(k, h), next.pcnt);
}

__device__ inline sum_flags flags_of(kconst &k, int tag) {
  const bool pse = k.pse != 0, blank = tag & MFC_FLAG_BLANKED, tool = tag & MFC_FLAG_TOOL;
  sum_flags f;
  f.tool = tool;
  f.nonfinite = tag & FLAG_NONFINITE;
  f.ta = pse ? 0. : (tool ? k.alpha_tool : k.alpha_wp);
  f.run_mech = !blank && (!pse || !tool);
  f.run_pse = !blank && pse && k.thermal_wp;
  return f;
}

// What follows the sums for the particle at sorted index i, index s of the start state, up to its
// return: the particle's next cell is left in the struct
struct after_update {
  deferred_return dr;
  double x, y;
  int fl;
};
template <bool F32>
__device__ inline void begin_update(const inst_args *ap, int i, unsigned s, bool live, const pair_acc &acc, double tpse,
                                    after_update &u) {
  MFC_CONST(inst_args) *c = const_args(ap, 0);
  kconst &k = c->k;
  u.dr.need = false;
  u.x = u.y = 0.;
  u.fl = 0;
  if (!live) return;
  double fsum[4] = {0., 0., 0., 0.};
  if (c->acc_out) store_acc(c->acc_out, k.N, i, acc, tpse);  // the same in every thread
  update_particle<F32>(k, i, s, acc, tpse, load_state(&c->cur), load_state(&c->nxt), load_pos(&c->pos), load_recs(&c->r), load_recs(&c->rn), *c->tool_out, fsum,
                       u.x, u.y, u.fl, u.dr);
  if (fsum[0] != 0. || fsum[1] != 0. || fsum[2] != 0. || fsum[3] != 0.) c->f.gflag[i >> 6] = 1;
}

// The step's tape of secant results, written by the launch before, which makes it a load from memory.
// A work-group with several threads per particle takes it into LDS while the records are on their way
// (loaded with the update, a step of 37.5k particles takes 0.8 % more than without a tape, so 0.3).
__device__ inline return_tape load_tape(MFC_CONST(inst_args) * c) {
  const __attribute__((address_space(1))) return_tape *t = (const __attribute__((address_space(1))) return_tape *)c->tape_in;
  return {t->at, t->left};
}

// Whether the wave's returns are on the tape: the replay of a recorded run takes the secant's result
// from there. The run's own iteration made it from the same state, so it is the same to the last bit,
// and the longest return of a step (up to 101 iterations of 0.6 us) isn't waited for again: ms per
// forward and backward pass of 60 steps of 6k particles 14.2 -> 10.8, of 100 steps of 37.5k 31.1 -> 24.5.
template <bool F32>
__device__ inline bool on_tape(MFC_CONST(inst_args) * c, const return_tape &t, bool need) {
  return !F32 && __ballot(need) && c->acc_out && __builtin_amdgcn_readfirstlane((int)(t.left > 0));
}
__device__ inline double from_tape(const return_tape &t, int i, bool &folded) {
  const double v = t.at[i];
  folded = v < 0.;
  return fabs(v);
}

// The rest (all 64 lanes of the wave): the return with the secant's dl, kept for the reverse mode's
// replay (-dl where its last update folded, 0 for no return), and the next step's binning
template <bool F32>
__device__ inline void end_update(const inst_args *ap, int i, bool live, double dl, bool folded, const return_tape &t,
                                  after_update &u) {
  MFC_CONST(inst_args) *c = const_args(ap, 0);
  kconst &k = c->k;
  if (u.dr.need) {
    finish_return<F32>(k, i, dl, u.dr, load_state(&c->nxt), load_recs(&c->rn));
    if (!F32 && t.left > 0 && !c->acc_out) t.at[i] = folded ? -dl : dl;
  }
  if (c->acc_out && live) c->acc_out[(size_t)ACC_N * k.N + i] = u.dr.need ? (folded ? -dl : dl) : 0.;
  next_cell(k, i, live, u.x, u.y, u.fl, load_bins(&c->b));
}

// both, each wave by itself
template <bool F32>
__device__ inline void finish_particle(const inst_args *ap, int i, unsigned s, bool live, const pair_acc &acc,
                                       double tpse) {
  after_update u;
  begin_update<F32>(ap, i, s, live, acc, tpse, u);
  return_tape t = {nullptr, 0};
  if (!F32 && __ballot(u.dr.need)) t = load_tape(const_args(ap, 0));
  const bool taped = on_tape<F32>(const_args(ap, 0), t, u.dr.need);
  bool folded;
  double dl = rr_secant_wave<F32>(const_args(ap, 0)->k, u.dr.need && !taped, u.dr.in, u.dr.eps, u.dr.T, folded);
  if (taped && u.dr.need) dl = from_tape(t, i, folded);
  end_update<F32>(ap, i, live, dl, folded, t, u);
}

// The state of the particle at index s of the start state on its way into L2 while the sums are
// formed: a load of a word of each field to LDS that nothing reads (no registers), `wave` 256 bytes.
// For the kernels with several threads per particle, where the update waits for its loads: us per
// step of 6k particles 31.7 -> 29.5 (FP64), of 37.5k 51 -> 46.5. With one thread per particle the
// loads of all work-groups together are bound by bandwidth, and it costs (197k FP32C 56 -> 60).
__device__ inline void fetch_state(const dstate &src, size_t N, unsigned s, unsigned *wave) {
  typedef const __attribute__((address_space(1))) unsigned *global_word;
  typedef __attribute__((address_space(3))) unsigned *lds_word;
  const double *p = src.px + s;
#pragma unroll
  for (int c = 0; c < DSTATE_DOUBLES; c++, p += N)
    __builtin_amdgcn_global_load_lds((global_word)(const unsigned *)p, (lds_word)wave, 4, 0, 0);
  __builtin_amdgcn_global_load_lds((global_word)(const unsigned *)(src.flags + s), (lds_word)wave, 4, 0, 0);
}

// One patch of cells by one work-group, G threads per particle: the cell starts and the records of
// the window candidates staged in LDS, the neighbour sums of its particles, and everything that
// follows them in the step. Why patches: a tile of consecutive particles of the sorted order is a
// strip along one grid column, whose windows hold about 1,500 candidates at 150k particles; the
// 10 x 10 cells of a patch have about 440, so that whole records fit LDS and a pair reads no
// memory (each gather of 16 bytes by 64 lanes from scattered records kept the address and data
// path of the vector caches busy for about 50 cycles, 60-70 % of the kernel). What bounds it: with
// one thread per particle a work-group of the 197k cut lives 42 us (FP32C; FP64 50), of which the
// staging takes 8, the sums 17 (29), the update and the next record 13 (9) and the next binning 3;
// its loads and stores move in a burst, since one round of work-groups fills the chip (FP32C four,
// FP64 three to a CU). With 4 or 8 threads per particle the sums of 6k particles take 13 or 8 us
// instead of 21 (FP64). Measured, us per step (tiles of the sorted order with candidate positions
// in LDS and a launch for the records, then this): FP32C 6k 55 -> 26, 27k 68 -> 35, 71k 63 -> 45,
// 197k 80 -> 56, 500k PSE 276 -> 169; FP64 6k 63 -> 29, 27k 77 -> 46, 71k 93 -> 61, 197k 137 -> 102,
// 500k PSE 403 -> 299.
// returns false, with nothing done, for a patch whose window candidates do not fit the stage or the masks
// and for the particles past the grid (interact_rest takes them)
template <bool F32, int G, bool PSE, bool GEN>
__device__ inline bool interact_patch(patch_mem<F32, G, GEN> &m, unsigned *unread, const inst_args *A, int inst, int patch, int part) {
  const inst_args &a_ = A[inst];
  MFC_CONST(inst_args) *c_ = const_args(&a_, 0);
  kconst &k = c_->k;
  const drecords r = load_recs(&c_->r);
  const int *__restrict__ offsets = k.rothlin ? c_->b.offsets_r : c_->b.offsets;
  const int *__restrict__ tags = c_->b.tags;
  const int *__restrict__ key_sorted = c_->b.key_sorted;
  constexpr int SLOTS = TILE / G;  // particles at a time
  const int tid = threadIdx.x;
  const int nrb = patch_rows(k);
  const int pc = patch / nrb, pr = patch - pc * nrb;
  // own cells: rows [r0, r1), columns [g0, g1); staged: rows [s0, s1), columns [q0, q1)
  const int r0 = pr * k.patch_s, r1 = r0 + k.patch_s < k.gny ? r0 + k.patch_s : k.gny;
  const int g0 = pc * k.patch_w, g1 = g0 + k.patch_w < k.gnx ? g0 + k.patch_w : k.gnx;
  if (g0 >= k.gnx) return false;  // the particles past the grid
  const int s0 = r0 < 2 ? 0 : r0 - 2, s1 = r1 + 2 < k.gny ? r1 + 2 : k.gny;
  const int q0 = g0 < 2 ? 0 : g0 - 2, q1 = g1 + 2 < k.gnx ? g1 + 2 : k.gnx;
  const int ncol = q1 - q0, nrow = s1 - s0 + 1;  // cell starts per column, with the end of the last
  const int te = tid / nrow;                     // the column of this thread's table entry
  if (tid < ncol * nrow) m.table[tid] = offsets[(q0 + te) * k.gny + s0 + (tid - te * nrow)];
  if (tid == 0) m.flags = 0;
  __syncthreads();
  if (tid < 64) {  // the first wave: where each column's candidates and own particles start
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
  using mem = patch_mem<F32, G, GEN>;
  constexpr int CAP = mem::CAP;
  const int cap = k.stage_limit > 0 && k.stage_limit < CAP ? k.stage_limit : CAP;
  if (ncand > cap || (!GEN && !k.uniform_h)) return false;  // the same in every thread
  if (G == 1 && tid < ncol * nrow) {
    const int last = (te + 1) * nrow - 1, n = m.table[tid + 5 < last ? tid + 5 : last] - m.table[tid];
    if (n > 32) atomicOr(&m.flags, !GEN || n > 5 * 32 ? PATCH_HEAPED : n > 2 * 32 ? PATCH_DENSER : PATCH_DENSE);
  }
  for (int q = tid; q < ncand; q += TILE) {
    int c = 0;
    for (int e = 1; e < ncol; e++) c += q >= m.col_first[e];
    const int tag = tags[q - m.col_shift[c]], fl = tag & ((1 << TAG_BITS) - 1);
    m.tag[q] = tag;
    if constexpr (!mem::ALL_IN_LDS) m.fl[q] = (unsigned char)fl;
    if (fl & ~MFC_FLAG_FIXED) {
      int set = fl & ~MFC_FLAG_FIXED;
      // a blanked particle enters no sum but those of PSE, so its record may hold anything
      if ((set & MFC_FLAG_BLANKED) && !k.pse) set &= ~FLAG_NONFINITE;
      atomicOr(&m.flags, set);
    }
  }
  __syncthreads();
  const int flags = m.flags;
  if (flags & (PATCH_HEAPED | FLAG_NONFINITE)) return false;  // the same in every thread
  const bool t_in_lds = k.alpha_wp != 0. || k.alpha_tool != 0., c_in_tag = k.promote == 0;
  {
    return_tape tape = {nullptr, 0};
    if (G > 1 && !F32 && tid == 0) tape = load_tape(c_);
    // the lanes take the 16-byte pieces of the records in turn, so that a load of a wave covers
    // whole records
    constexpr int LPR = F32 ? 4 : 8;  // lanes per record
    const int pl = tid % LPR;
    constexpr int STAGE_U = 4;
    if constexpr (GEN) {
      constexpr int P = mem::PIECES;
      const int p = tid % P;
      for (int q = tid / P; q < ncand; q += TILE / P) {
        const size_t s = tag_index(m.tag[q]);
        m.piece(p)[q] = F32 ? r.rec32[s * REC32_PIECES + p] : reinterpret_cast<const float4 *>(r.rec)[s * (REC / 2) + (p ? p + 1 : 0)];
      }
    } else for (int q = tid / LPR; q < ncand; q += STAGE_U * (TILE / LPR)) {
      float4 v[STAGE_U];
#pragma unroll
      for (int u = 0; u < STAGE_U; u++) {
        const int c = q + u * (TILE / LPR);
        const size_t s = tag_index(m.tag[c < ncand ? c : q]);
        if constexpr (F32) v[u] = r.rec32[s * REC32_PIECES + pl];
        else v[u] = reinterpret_cast<const float4 *>(r.rec)[s * (REC / 2) + pl];
      }
#pragma unroll
      for (int u = 0; u < STAGE_U; u++) {
        const int c = q + u * (TILE / LPR);
        if (c >= ncand) break;
        if (!PSE && (flags & MFC_FLAG_BLANKED) && pl == 0 &&
            ((mem::ALL_IN_LDS ? m.tag[c] : (int)m.fl[mem::ALL_IN_LDS ? 0 : c]) & MFC_FLAG_BLANKED))
          reinterpret_cast<double2 &>(v[u]) = make_double2(__builtin_huge_val(), __builtin_huge_val());
        if constexpr (F32) {
          m.piece(pl)[c] = v[u];
        } else if (pl != 1) {  // piece 1 of a record: flags (in the tag) and h (uniform)
          const int p = pl == 0 ? 0 : pl - 1;
          if (mem::ALL_IN_LDS || p < 6) m.piece(p)[c] = v[u];
          else {
            const double2 ct = reinterpret_cast<const double2 &>(v[u]);
            m.X[c] = c_in_tag || t_in_lds ? ct.y : ct.x;
            if (c_in_tag) m.tag[c] = __float_as_int((float)ct.x);  // read by the lanes of this wave only, before
          }
        }
      }
    }
    if (tid < ncol * nrow) m.table[tid] += m.col_shift[te];
    if (G > 1 && !F32 && tid == 0) m.tape = tape;
  }
  __syncthreads();
  // the sorted index, column and staged index of own particle number n
  auto locate = [&](int n, int &col, int &li) -> int {
    col = 0;
    for (int e = 1; e < ncol; e++) col += n >= m.own_first[e];
    li = m.table[col * nrow + r0 - s0] + (n - m.own_first[col]);
    return li - m.col_shift[col];
  };
  const int base = part * SLOTS;
  {
    [[maybe_unused]] pair_acc acc;
    [[maybe_unused]] double tpse = 0.;
    const int n = base + tid / G;  // the particle whose sums this thread takes part in
    const bool mine = n < nown;
    [[maybe_unused]] int i_mine = 0;
    unsigned s_mine = 0;  // loaded before the sums, which hide its latency
    // the exchange area of the wave; the sums of its particles end there too
    constexpr int WAVE_BYTES = mem::TERM_BYTES / (TILE / 64);
    static_assert(G == 1 || WAVE_BYTES >= 64 / G * ACC_N * (int)sizeof(double), "a wave's sums fit its exchange area");
    [[maybe_unused]] char *terms = m.terms + (size_t)(tid >> 6) * WAVE_BYTES;
    [[maybe_unused]] double *out = reinterpret_cast<double *>(terms) + (size_t)((tid & 63) / G) * ACC_N;
    int i_own = 0;  // of the particle this thread updates (G > 1)
    if constexpr (G > 1)
      if (tid < SLOTS && base + tid < nown) {
        int col, li;
        i_own = locate(base + tid, col, li);
        s_mine = tag_index(m.tag[li]);
        fetch_state(load_state(&c_->cur), k.N, s_mine, unread);
      }
    if (mine) {
      int col, li;
      const int i = locate(n, col, li);
      i_mine = i;
      const int key = key_sorted[i];
      if constexpr (G == 1) s_mine = tag_index(tags[i]);
      double2 p;
      int tag;
      rec_t<F32> a;
      using src = lds_source<F32, G, GEN>;
      const src lds = {&m, (typename src::template global<double>)r.rec, (typename src::template global<typename src::float4v>)r.rec32,
                       (typename src::template global<double>)(GEN ? load_state(&c_->cur).h : nullptr), k.uniform_h != 0, k.h0, c_in_tag, t_in_lds};
      lds.cand(li, p, tag);
      lds.record(li, a);
      a.x = p.x; a.y = p.y;
      const sum_flags f = flags_of(k, tag);
      auto at = [&](int c, int row) { return m.table[(c - q0) * nrow + row - s0]; };
      const int gi = q0 + col, gj = key - gi * k.gny;
      if constexpr (G == 1) {
        int b[5], e[5];
        window_ranges(k, gi, gj, at, b, e);
        if (!f.run_mech && !f.run_pse)
#pragma unroll
          for (int q = 0; q < 5; q++) e[q] = b[q];
        sums_lds<F32, G, PSE, GEN>(k, lds, flags, b, e, a, f, acc, tpse);
      } else {
        window w = make_window_at(k, gi, gj, at);
        if (!f.run_mech && !f.run_pse) w.total = 0;
        sums_group<F32, G, GEN>(k, lds, w, a, f, m.list[tid / G], terms, out);
      }
    }
    // fetch_state's words have arrived before the LDS is given back
    if constexpr (G > 1) asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    // the update, one thread per particle: with G > 1 the first SLOTS threads
    int i = i_mine;
    bool live = mine;
    if constexpr (G > 1) {
      __syncthreads();
      live = tid < SLOTS && base + tid < nown;
      if (live) {
        i = i_own;
        // summed by wave tid / (64 / G)
        const double *o = reinterpret_cast<const double *>(m.terms + (size_t)(tid / (64 / G)) * WAVE_BYTES) +
                          (size_t)(tid % (64 / G)) * ACC_N;
        if constexpr (F32) acc = acc_of_sums32(k, o);
        else load_acc(o, 1, 0, acc, tpse);
        tpse = o[ACC_N - 1];
      }
    }
    if constexpr (G == 1) {
      finish_particle<F32>(A + inst, i, s_mine, live, acc, tpse);
    } else {  // by the first wave, the returns by all
      static_assert(SLOTS <= 64 && sizeof(return_slots) <= sizeof(m.pieces), "one wave's particles");
      after_update u;
      u.dr.need = false;
      if (tid < 64) begin_update<F32>(A + inst, i, s_mine, live, acc, tpse, u);
      const return_tape t = m.tape;
      const bool taped = on_tape<F32>(c_, t, u.dr.need);
      bool folded;
      double dl = rr_secant_group<F32>(k, reinterpret_cast<return_slots &>(m.pieces), u.dr.need && !taped, u.dr.in,
                                       u.dr.eps, u.dr.T, folded);
      if (taped && u.dr.need) dl = from_tape(t, i, folded);
      if (tid < 64) end_update<F32>(A + inst, i, live, dl, folded, t, u);
    }
  }
  return true;
}

// Positions and tags of the window candidates of a patch copied to `lds` (of `bytes`; 20 bytes each, four
// times as many as whole records): the columns [q0, q0 + ncol) of cells, rows [s0, s1). False where they
// do not fit or a record of some sum is not finite; shift: a column's places minus its sorted indices
template <bool F32>
__device__ inline bool copy_window(kconst &k, const mem_records<F32> &rec, const int *offsets, const int *tags, int q0,
                                   int ncol, int s0, int s1, lds_ptr<char> lds, int bytes, lds_ptr<int> &shift,
                                   copy_source<F32> &copy) {
  lds_ptr<int> first = (lds_ptr<int>)lds, nonfinite = first + 63;
  shift = first + 32;  // PATCH_COLS at most of each
  constexpr int HEAD = 64 * sizeof(int);
  const int cap = (bytes - HEAD) / (int)(sizeof(lds_pos) + sizeof(int)), tid = threadIdx.x;
  copy.pos = (lds_ptr<lds_pos>)(lds + HEAD);
  copy.tags = (lds_ptr<int>)(copy.pos + cap);
  __syncthreads();  // what was in the LDS before is no longer read
  if (tid < 64) {
    int j0 = 0, c = 0;
    if (tid < ncol) {
      j0 = offsets[(q0 + tid) * k.gny + s0];
      c = offsets[(q0 + tid) * k.gny + s1] - j0;
    }
    int x = c;
#pragma unroll
    for (int s = 1; s < 32; s <<= 1) {
      const int y = __shfl_up(x, s, 64);
      if (tid >= s) x += y;
    }
    if (tid <= ncol) {
      first[tid] = x - c;
      shift[tid] = x - c - j0;
    }
    if (tid == 63) *nonfinite = 0;
  }
  __syncthreads();
  const int ncand = first[ncol];
  if (ncand > cap) return false;  // the same in every thread
  for (int q = tid; q < ncand; q += TILE) {
    int c = 0;
    for (int e = 1; e < ncol; e++) c += q >= first[e];
    const int tag = tags[q - shift[c]];
    const double2 p = rec.pos_of(tag);
    copy.tags[q] = tag;
    copy.pos[q].x = p.x; copy.pos[q].y = p.y;
    if ((tag & FLAG_NONFINITE) && (k.pse || !(tag & MFC_FLAG_BLANKED))) *nonfinite = 1;
  }
  __syncthreads();
  return *nonfinite == 0;
}

// What interact_patch leaves, one thread per particle over the records in memory: a patch that it does not
// take, an entry past the end of the launch's work items, the particles past the grid, or (patch < 0) tile
// `part` of the sorted order. A launch waits for its last work-group, so what counts is how long one takes.
// us per step with every patch sent here: 6k particles FP64 60, 197k 167, FP32C 84 (one candidate
// after the other from memory, with the pair terms for any value, 81, 234 and 158).
template <bool F32>
__device__ __attribute__((always_inline)) inline void interact_rest(const inst_args *ap, int patch, int part,
                                                                    lds_ptr<char> lds, int bytes) {
  MFC_CONST(inst_args) *c_ = const_args(ap, 0);
  kconst &k = c_->k;
  const dbins b = load_bins(&c_->b);
  const int *offsets = k.rothlin ? b.offsets_r : b.offsets;
  const mem_records<F32> rec = {load_recs(&c_->r), load_state(&c_->cur).h};
  copy_source<F32> copy = {rec, nullptr, nullptr};
  lds_ptr<int> shift = nullptr;
  int i = -1, q0 = 0;   // the thread's particle; the first column of the copy
  bool copied = false;  // the same in every thread
  if (patch < 0) {
    const int j = part * TILE + (int)threadIdx.x;
    if (j < k.N) i = j;
  } else {
    const int nrb = patch_rows(k);
    const int pc = patch / nrb, pr = patch - pc * nrb;
    const int r0 = pr * k.patch_s, r1 = r0 + k.patch_s < k.gny ? r0 + k.patch_s : k.gny;
    const int g0 = pc * k.patch_w, g1 = g0 + k.patch_w < k.gnx ? g0 + k.patch_w : k.gnx;
    int n = (int)threadIdx.x < k.patch_slots ? part * k.patch_slots + (int)threadIdx.x : 0x7fffffff;
    for (int c = g0; c < g1; c++) {
      const int first = offsets[c * k.gny + r0], count = offsets[c * k.gny + r1] - first;
      if (i < 0 && n < count) i = first + n;
      if (n != 0x7fffffff) n -= count;
    }
    if (g0 >= k.gnx) {  // the particles past the grid: blanked ones, which have no sums
      const int first = offsets[k.num_cell];
      if (n < k.N - first) i = first + n;
    } else {
      q0 = g0 < 2 ? 0 : g0 - 2;
      copied = copy_window(k, rec, offsets, b.tags, q0, (g1 + 2 < k.gnx ? g1 + 2 : k.gnx) - q0, r0 < 2 ? 0 : r0 - 2,
                           r1 + 2 < k.gny ? r1 + 2 : k.gny, lds, bytes, shift, copy);
    }
  }
  pair_acc acc = {};
  double tpse = 0.;
  unsigned s = 0u;
  if (i >= 0) {
    const int tag = b.tags[i], key = b.key_sorted[i];
    s = tag_index(tag);
    const double2 p = rec.pos_of(tag);
    rec_t<F32> a;
    rec.record(tag, a);
    a.x = p.x; a.y = p.y;
    const sum_flags f = flags_of(k, tag);
    const int gi = key / k.gny, gj = key - gi * k.gny;
    window w = make_window_at(k, gi, gj, [&](int col, int row) {
      return offsets[col * k.gny + row] + (copied ? shift[col - q0] : 0);
    });
    if (!f.run_mech && !f.run_pse) w.total = 0;
    if (copied) sums_mem<F32, true>(k, copy, w, a, f, acc, tpse);
    else sums_mem<F32, false>(k, mem_source<F32>{rec, b.tags}, w, a, f, acc, tpse);
  }
  finish_particle<F32>(ap, i, s, i >= 0, acc, tpse);
}

// As a call it takes no registers from the kernel, but saves up to 600 bytes of them per thread. In line it makes
// every patch sent here 197k FP64 214 -> 167 us, FP32C 134 -> 84; but in FP64 with several threads per particle, where it
// gives less (6k 60 -> 56), the registers it takes cost the kernel 1 % (150 steps of 37.5k 7.85 -> 7.95 ms).
template <bool F32>
__device__ __attribute__((noinline)) void call_interact_rest(const inst_args *ap, int patch, int part, lds_ptr<char> lds,
                                                             int bytes) {
  interact_rest<F32>(ap, patch, part, lds, bytes);
}

constexpr int FF_BATCH = 8;  // group sums a thread of force_final loads at a time

// tool force of a step from its group sums: lane l of TILE adds the sums of the groups l,
// l + TILE, ... in ascending order, then the lane sums are reduced by halving strides;
// F = sum(fc) + sum(ft). The first TILE threads of the work-group do the adding, all of its
// threads call it; red: 4 TILE doubles of LDS.
__device__ inline void force_final(int ntiles, const dforce &fo, double (*red)[TILE]) {
  double a0 = 0., a1 = 0., a2 = 0., a3 = 0.;
  // each thread adds the group sums q = threadIdx.x, + TILE, + 2 TILE, ... in that order (4
  // per tile), eight loads in flight at a time: one load at a time made this work-group the last
  // of its launch
  const double4 *__restrict__ p4 = reinterpret_cast<const double4 *>(fo.partials);
  const int nq = threadIdx.x < TILE ? 4 * ntiles : 0;
  for (int q0 = threadIdx.x; q0 < nq; q0 += TILE * FF_BATCH) {
    double4 v[FF_BATCH];
#pragma unroll
    for (int u = 0; u < FF_BATCH; u++) v[u] = q0 + u * TILE < nq ? p4[q0 + u * TILE] : make_double4(0., 0., 0., 0.);
#pragma unroll
    for (int u = 0; u < FF_BATCH; u++)
      if (q0 + u * TILE < nq) {
        a0 = a0 + v[u].x; a1 = a1 + v[u].y; a2 = a2 + v[u].z; a3 = a3 + v[u].w;
      }
  }
  if (threadIdx.x < TILE) {
    red[0][threadIdx.x] = a0; red[1][threadIdx.x] = a1;
    red[2][threadIdx.x] = a2; red[3][threadIdx.x] = a3;
  }
  for (int s = TILE / 2; s > 0; s >>= 1) {
    __syncthreads();
    if (threadIdx.x < s) {
#pragma unroll
      for (int c = 0; c < 4; c++) red[c][threadIdx.x] = red[c][threadIdx.x] + red[c][threadIdx.x + s];
    }
  }
  if (threadIdx.x == 0) {
    const double F0 = red[0][0] + red[2][0], F1 = red[1][0] + red[3][0];
    fo.force_last[0] = F0;
    fo.force_last[1] = F1;
    const int64_t n = *fo.ctr;
    if (n >= 0 && n < fo.cap) { fo.hist[2 * n] = F0; fo.hist[2 * n + 1] = F1; }
    *fo.ctr = n + 1;
    *fo.pending = 0;
  }
}

// ------------------------------------------------------------------------------- tool wear
// Usui wear rate (tool_wear.cu:20-60) of the current state: particles count as in contact when
// |fc.x|, |fc.y| or |ft.x| is non-zero (the reference tests fc.y twice and never ft.y); the
// relative velocity is v - v*n with the component-wise product of its glm code, the pressure
// |fc| / (2 pi h), the rate K exp(alpha / T) p |v_r|. Per tile: min (from FLT_MAX, as the
// reference), max (from 0), sum and count over the tile's particles in contact, then one
// work-group folds the tiles in a fixed order. Min, max and count do not depend on the order;
// the sum is the fixed-order tree instead of the reference's sequential loop.
__device__ inline void wear_tree(double (*red)[TILE]) {
  for (int st = TILE / 2; st > 0; st >>= 1) {
    __syncthreads();
    if (threadIdx.x < st) {
      red[0][threadIdx.x] = fmin(red[0][threadIdx.x], red[0][threadIdx.x + st]);
      red[1][threadIdx.x] = fmax(red[1][threadIdx.x], red[1][threadIdx.x + st]);
      red[2][threadIdx.x] = red[2][threadIdx.x] + red[2][threadIdx.x + st];
      red[3][threadIdx.x] = red[3][threadIdx.x] + red[3][threadIdx.x + st];
    }
  }
}

__global__ __launch_bounds__(TILE) void k_wear_tiles(int N, int ntiles, dstate st, const double *__restrict__ nx,
                                                     const double *__restrict__ ny, double K, double alpha,
                                                     double tvx, double tvy, double *__restrict__ part) {
  const int t = xcd_tile(blockIdx.x, ntiles);
  if (t < 0) return;
  __shared__ double red[4][TILE];
  const int i = t * TILE + threadIdx.x;
  double wmin = (double)FLT_MAX, wmax = 0., wsum = 0., cnt = 0.;
  if (i < N) {
    const double fcx = st.fcx[i], fcy = st.fcy[i], ftx = st.ftx[i];
    if (fabs(fcx) > 0. || fabs(fcy) > 0. || fabs(ftx) > 0. || fabs(fcy) > 0.) {
      const double vx = st.vx[i] - tvx, vy = st.vy[i] - tvy;
      const double rx = vx - vx * nx[i], ry = vy - vy * ny[i];
      const double vmag = sqrt(rx * rx + ry * ry);
      const double fmag = sqrt(fcx * fcx + fcy * fcy);
      const double A = 2 * st.h[i] * M_PI;
      const double p = fmag / A;
      const double w = K * mfcm::exp(alpha / st.T[i]) * p * vmag;
      wmin = w; wmax = w; wsum = w; cnt = 1.;
    }
  }
  red[0][threadIdx.x] = wmin; red[1][threadIdx.x] = wmax; red[2][threadIdx.x] = wsum; red[3][threadIdx.x] = cnt;
  wear_tree(red);
  if (threadIdx.x == 0) {
#pragma unroll
    for (int c = 0; c < 4; c++) part[4 * t + c] = red[c][0];
  }
}

__global__ __launch_bounds__(TILE) void k_wear_final(int ntiles, const double *__restrict__ part,
                                                     double *__restrict__ out) {
  __shared__ double red[4][TILE];
  double wmin = (double)FLT_MAX, wmax = 0., wsum = 0., cnt = 0.;
  for (int q = threadIdx.x; q < ntiles; q += TILE) {
    wmin = fmin(wmin, part[4 * q]); wmax = fmax(wmax, part[4 * q + 1]);
    wsum = wsum + part[4 * q + 2]; cnt = cnt + part[4 * q + 3];
  }
  red[0][threadIdx.x] = wmin; red[1][threadIdx.x] = wmax; red[2][threadIdx.x] = wsum; red[3][threadIdx.x] = cnt;
  wear_tree(red);
  if (threadIdx.x == 0) {
#pragma unroll
    for (int c = 0; c < 4; c++) out[c] = red[c][0];
  }
}

// ------------------------------------------------------------------------------- batched

// One launch per phase for all instances of a batch: block b takes work item xcd_tile(b) (the
// interaction kernels: xcd_chunk_tile(b)) of the (instance, block) table, and runs the device
// body with that instance's constants and buffers, so every instance computes exactly its own
// run.
// adaptive: of the instances with an adaptive grid, whose steps bin their start state behind the geometry
// pass, else of the others
__global__ __launch_bounds__(256) void kb_hash_count(const inst_args *__restrict__ A, const int2 *__restrict__ work,
                                                     int nwork, int adaptive) {
  const int w = xcd_tile(blockIdx.x, nwork);
  if (w < 0) return;
  const int2 it = work[w];
  const inst_args &a = A[it.x];
  if (a.k.adaptive != adaptive) return;
  hash_count(a.k, it.y * 256 + threadIdx.x, a.cur.px, a.cur.py, a.cur.flags, a.b);
}

// the patches' counts of the start state again, from its cell ids: for another shape of the patches
// (an adaptive grid counts them in its geometry pass)
__global__ __launch_bounds__(256) void kb_count_patches(const inst_args *__restrict__ A, const int2 *__restrict__ work,
                                                        int nwork) {
  const int w = xcd_tile(blockIdx.x, nwork);
  if (w < 0) return;
  const int2 it = work[w];
  const inst_args &a = A[it.x];
  if (a.k.adaptive) return;
  const int i = it.y * 256 + threadIdx.x;
  count_patch(i < a.k.N ? patch_of(a.k, a.b.key[i]) : -1, a.b.pcnt);
}

// Adaptive grid (grid_base::update_geometry, grid.cu:97-136), one work-group per instance: the
// box of all positions (blanked particles included, as thrust::min_element / max_element over
// the whole array) and the largest h give this step's geometry, which the work-group writes
// into the instance's descriptor for the step's later kernels, the first of which bins the start
// state with it (by this work-group itself, a step of 131k particles took 396 us, of
// 11.6k 71, now 176 and 57). Minimum and maximum do not depend on the order they are taken in; NaN
// positions are passed over. A geometry that needs as many cells as
// the binning table holds is not taken (the reference asserts): the previous step's (kept in
// geo, which every step writes) stays and the step is counted in geo->overflow.
constexpr int GEO_THREADS = 1024;
__global__ __launch_bounds__(GEO_THREADS) void kb_geometry(inst_args *__restrict__ A) {
  // plain loads: this kernel writes the descriptor it reads (not through the constant space)
  const inst_args a = A[blockIdx.x];
  if (!a.k.adaptive) return;  // the same in every thread of the work-group
  __shared__ double red[5][GEO_THREADS / 64];
  const int N = a.k.N;
  const double inf = __builtin_huge_val();
  double x0 = inf, x1 = -inf, y0 = inf, y1 = -inf, hm = -inf;
  for (int i = threadIdx.x; i < N; i += GEO_THREADS) {
    const double x = a.cur.px[i], y = a.cur.py[i], h = a.cur.h[i];
    x0 = fmin(x0, x); x1 = fmax(x1, x);
    y0 = fmin(y0, y); y1 = fmax(y1, y);
    hm = fmax(hm, h);
  }
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) {
    x0 = fmin(x0, __shfl_xor(x0, o, 64)); x1 = fmax(x1, __shfl_xor(x1, o, 64));
    y0 = fmin(y0, __shfl_xor(y0, o, 64)); y1 = fmax(y1, __shfl_xor(y1, o, 64));
    hm = fmax(hm, __shfl_xor(hm, o, 64));
  }
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
  if (lane == 0) { red[0][wv] = x0; red[1][wv] = x1; red[2][wv] = y0; red[3][wv] = y1; red[4][wv] = hm; }
  __syncthreads();
  if (threadIdx.x == 0) {
    for (int q = 1; q < GEO_THREADS / 64; q++) {
      x0 = fmin(x0, red[0][q]); x1 = fmax(x1, red[1][q]);
      y0 = fmin(y0, red[2][q]); y1 = fmax(y1, red[3][q]);
      hm = fmax(hm, red[4][q]);
    }
    double bx = x0 - 1e-6, by = y0 - 1e-6;
    const double ex = x1 + 1e-6, ey = y1 + 1e-6;
    double cell = hm * 2. / 2.;
    const double fnx = ceil((ex - bx) / cell), fny = ceil((ey - by) / cell);
    int gnx, gny;
    if (fnx >= 1. && fny >= 1. && fnx * fny < (double)a.k.ncell_table) {
      gnx = (int)fnx; gny = (int)fny;
    } else {  // keep the previous step's geometry (the instance's record: the descriptor of
              // this buffer parity holds the one of two steps before)
      bx = a.geo->bbmin_x; by = a.geo->bbmin_y; cell = a.geo->cell; gnx = a.geo->gnx; gny = a.geo->gny;
      a.geo->overflow = a.geo->overflow + 1;
    }
    dev_consts *kd = &A[blockIdx.x].k;
    kd->bbmin_x = bx; kd->bbmin_y = by; kd->cell = cell;
    kd->gnx = gnx; kd->gny = gny; kd->num_cell = gnx * gny;
    a.geo->bbmin_x = bx; a.geo->bbmin_y = by; a.geo->cell = cell;
    a.geo->gnx = gnx; a.geo->gny = gny; a.geo->num_cell = gnx * gny;
  }
}

// the sort of a chunk of cells, and the work items of an instance beside its chunks: the tool's
// move, the list of its patches and the group sums of the previous step's tool force, if they are
// still pending (the items come first in the work table, so that their work-groups start first)
__global__ __launch_bounds__(SCAN_THREADS) void kb_sort(const inst_args *__restrict__ A, const int2 *__restrict__ work,
                                                         int nwork) {
  const int w = xcd_tile(blockIdx.x, nwork);
  if (w < 0) return;
  const int2 it = work[w];
  MFC_CONST(inst_args) *c = const_args(A, it.x);
  if (it.y <= SORT_ITEM_PATCHES) {
    list_patches(c->k, SORT_ITEM_PATCHES - it.y, load_bins(&c->b));
    return;
  }
  if (it.y <= SORT_ITEM_FORCE) {
    const dforce fo = load_force(&c->f);
    if (*fo.pending == 0) return;  // the same value in every thread
    constexpr int PER_WAVE = FORCE_GROUPS / (SCAN_THREADS / 64);
    const int g0 = (SORT_ITEM_FORCE - it.y) * FORCE_GROUPS + (threadIdx.x >> 6) * PER_WAVE;
    force_groups(A[it.x].k.N, g0, PER_WAVE, load_state(&c->cur), fo);
    return;
  }
  if (it.y == SORT_ITEM_TOOL) {
    if (threadIdx.x == 64) {  // beside the tool's move, not behind it
      const return_tape t = *c->tape_in;
      const return_tape next = {t.left > 0 ? t.at + c->k.N : nullptr, t.left > 0 ? t.left - 1 : 0};
      *c->tape_out = next;
    }
    tool_move(A[it.x].tool_in, A[it.x].tool_out, A[it.x].k.dt);
    return;
  }
  kconst &k = c->k;
  sort_chunk(it.y, k.N, k.ncell_table, load_bins(&c->b), load_recs(&c->r).vfl, k.sort_fast, k.sort_list);
}

// the records of a start state that no interaction wrote
template <bool F32>
__global__ __launch_bounds__(TILE) void kb_records(const inst_args *__restrict__ A, const int2 *__restrict__ work,
                                                   int nwork) {
  const int w = xcd_tile(blockIdx.x, nwork);
  if (w < 0) return;
  const int2 it = work[w];
  MFC_CONST(inst_args) *c = const_args(A, it.x);
  kconst &k = c->k;
  const int s = it.y * TILE + threadIdx.x;
  if (s >= k.N) return;
  write_record<F32>(k, load_rec_input(load_state(&c->cur), s), s, load_recs(&c->r));
}

// The cell ranges of grid_gpu_rothlin (grid_gpu_rothlin.cu:28-127) rebuilt from the sorted cell
// ids: the lane at the end of each run of equal ids (where unique_by_key_copy starts the next run)
// writes the run's end into the offsets of its cell's successor and of every empty cell up to the
// next run's cell, which is the scatter of the run lengths and their scan over the empty cells
// between in one pass; the first lane writes 0 up to the first id, the last run fills the table's
// end with N. Every entry of offsets_r is written by exactly one lane; the same ranges as the
// counting sort's offsets.
__global__ __launch_bounds__(256) void kb_rothlin_cells(const inst_args *__restrict__ A, const int2 *__restrict__ work,
                                                        int nwork) {
  const int w = xcd_tile(blockIdx.x, nwork);
  if (w < 0) return;
  const int2 it = work[w];
  MFC_CONST(inst_args) *c = const_args(A, it.x);
  const int rothlin = A[it.x].k.rothlin, N = A[it.x].k.N, nc = A[it.x].k.ncell_table;
  if (!rothlin) return;
  const int i = it.y * 256 + threadIdx.x;
  if (i >= N) return;
  const dbins b = load_bins(&c->b);
  const int h = b.key_sorted[i];
  if (i == 0)
    for (int q = 0; q <= h; q++) b.offsets_r[q] = 0;
  const int hn = i + 1 < N ? b.key_sorted[i + 1] : nc;
  if (hn != h)
    for (int q = h + 1; q <= hn; q++) b.offsets_r[q] = i + 1;
}

// Particles spread over so many patches that the entries of the list are more than 1.3 times the launch's
// work items: a patch then has few particles, and the work-groups take the particles as tiles of the
// sorted order instead, by interact_rest. us per step of 171k particles, by patches (what does not fit the
// work items behind the others, one entry after the other) / by tiles, FP64: scattered over the whole grid 504 / 59,
// a quarter of it 163 / 90, a sixth (1.6 times) 128 / 111; a body of which 0.5 % (1.25 times) are scattered 129 / 174,
// 1 % (1.8 times) 156 / 175, 3 % 290 / 170. Of 27k FP64: 1.5 % (1.1 times) 60 / 86, 3 % (1.6 times) 76 / 85, a sixth (1.4) 64 / 62.
__device__ inline bool sparse(int entries, int items) { return 10ll * entries > 13ll * items; }
template <bool F32, int G, bool PSE, bool GEN>
__global__ __launch_bounds__(TILE) __attribute__((amdgpu_waves_per_eu(F32 ? 4 : 3))) void kb_interact(
    const inst_args *__restrict__ A, const int2 *__restrict__ work, int nwork, int chunk) {
  const int w = xcd_chunk_tile(blockIdx.x, nwork, chunk);
  if (w < 0) return;
  const int2 it = work[w];
  MFC_CONST(inst_args) *c = const_args(A, it.x);
  __shared__ patch_mem<F32, G, GEN> m;
  __shared__ unsigned unread[G > 1 ? 64 : 1];
  if (it.y == PATCH_ITEM_FORCE) {
    const dforce fo = load_force(&c->f);
    // pending: the same value in every thread
    if (*fo.pending != 0) force_final(c->ntiles, fo, reinterpret_cast<double(*)[TILE]>(&m));
    if (threadIdx.x == 0) *fo.pending_next = 1;
    return;
  }
  const int count = *c->b.plen, step = c->npatch_items;
  const lds_ptr<char> lds = (lds_ptr<char>)(char *)&m;
  const bool tiles = sparse(count, step);
  if (!tiles && it.y >= count) return;
  int q = it.y;
  if (!tiles) {
    const int2 p = c->b.plist[q];
    if (interact_patch<F32, G, PSE, GEN>(m, unread, A, it.x, p.x, p.y)) q += step;
  }
  const int end = tiles ? c->ntiles : count;
#pragma clang loop unroll(disable)
  for (; q < end; q += step) {  // of most work-groups none
    int2 p = make_int2(-1, q);
    if (!tiles) p = c->b.plist[q];
    if constexpr (F32 || G == 1) interact_rest<F32>(A + it.x, p.x, p.y, lds, sizeof(m));
    else call_interact_rest<F32>(A + it.x, p.x, p.y, lds, sizeof(m));
  }
}

// after the last step of a call: its tool force, by one work-group per instance
constexpr int FORCE_LAST_THREADS = 1024;
__global__ __launch_bounds__(FORCE_LAST_THREADS) void kb_force_final(const inst_args *__restrict__ A) {
  MFC_CONST(inst_args) *c = const_args(A, blockIdx.x);
  const dforce fo = load_force(&c->f);
  if (*fo.pending == 0) return;  // the same value in every thread
  const int N = A[blockIdx.x].k.N, ntiles = A[blockIdx.x].ntiles;
  const dstate st = load_state(&c->cur);
  for (int g0 = (threadIdx.x >> 6) * 64; 64 * g0 < N; g0 += FORCE_LAST_THREADS) force_groups(N, g0, 64, st, fo);
  __syncthreads();  // the group sums
  __shared__ double red[4][TILE];
  force_final(ntiles, fo, red);
}

// components of a field side by side, as the caller gets them: whole 16-byte stores over the host
// link, which bounds it (55 GB/s)
template <int NC>
__global__ __launch_bounds__(256) void k_interleave(const double *__restrict__ a, const double *__restrict__ b,
                                                    const double *__restrict__ c, const double *__restrict__ d,
                                                    int64_t count, double *__restrict__ out) {
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < count; i += (int64_t)gridDim.x * blockDim.x) {
    if constexpr (NC == 3) {
      out[3 * i] = a[i]; out[3 * i + 1] = b[i]; out[3 * i + 2] = c[i];
    } else {
      double2 *o = reinterpret_cast<double2 *>(out) + (NC / 2) * i;
      o[0] = make_double2(a[i], b[i]);
      if constexpr (NC == 4) o[1] = make_double2(c[i], d[i]);
    }
  }
}

__global__ void k_device_math(int fn, const double *__restrict__ x, const double *__restrict__ y,
                              double *__restrict__ out, int64_t n) {
  int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  double a = x[i], b = y ? y[i] : 0., r = 0.;
  switch (fn) {
    case 0: r = mfcm::exp(a); break;
    case 1: r = mfcm::log(a); break;
    case 2: r = mfcm::pow(a, b); break;
    case 3: r = mfcm::atan2(a, b); break;
    case 4: r = mfcm::sin(a); break;
    case 5: r = mfcm::cos(a); break;
    case 6: r = (double)mfcm::atan2f(a, b); break;
    case 7: r = (double)mfcm::cosf(a); break;
    case 8: r = (double)mfcm::sinf(a); break;
    case 9: r = sqrt(a); break;
    case 10: r = f32sqrt(a); break;
    case 11: r = a / b; break;
    case 12: r = mfcm::tanh(a); break;
    default: r = 0.;
  }
  out[i] = r;
}

}  // namespace

int scan_blocks(int num_cell) { return (num_cell + SCAN_CHUNK - 1) / SCAN_CHUNK; }

static int padded_tiles(int ntiles) { return ((ntiles + 7) / 8) * 8; }

void launch_tool_wear(const dev_consts &k, const dstate &st, const dpositional &pos, double K, double alpha,
                      double tvx, double tvy, double *part, double *out, hipStream_t s) {
  const int nt = (k.N + TILE - 1) / TILE;
  hipLaunchKernelGGL(k_wear_tiles, dim3(padded_tiles(nt)), dim3(TILE), 0, s, k.N, nt, st, pos.nx, pos.ny, K, alpha,
                     tvx, tvy, part);
  hipLaunchKernelGGL(k_wear_final, dim3(1), dim3(TILE), 0, s, nt, part, out);
}

void launch_interleave(int nc, const double *const *src, int64_t first, int64_t count, double *out, hipStream_t s) {
  const dim3 g((unsigned)(count < 256 * 1024 ? (count + 255) / 256 : 1024)), b(256);
  const double *p[4];
  for (int c = 0; c < 4; c++) p[c] = c < nc ? src[c] + first : nullptr;
  if (nc == 2) hipLaunchKernelGGL(HIP_KERNEL_NAME(k_interleave<2>), g, b, 0, s, p[0], p[1], p[2], p[3], count, out);
  else if (nc == 3) hipLaunchKernelGGL(HIP_KERNEL_NAME(k_interleave<3>), g, b, 0, s, p[0], p[1], p[2], p[3], count, out);
  else hipLaunchKernelGGL(HIP_KERNEL_NAME(k_interleave<4>), g, b, 0, s, p[0], p[1], p[2], p[3], count, out);
}

void launch_device_math(int fn, const double *x, const double *y, double *out, int64_t n, hipStream_t s) {
  const int64_t g = (n + 255) / 256;
  hipLaunchKernelGGL(k_device_math, dim3((unsigned)g), dim3(256), 0, s, fn, x, y, out, n);
}

int scan_chunk_cells() { return SCAN_CHUNK; }
int chunk_list_cap(int N) { return N < 4 * SCAN_CHUNK ? N : 4 * SCAN_CHUNK; }

void launch_batch_hash(const batch_work &w, hipStream_t s) {
  hipLaunchKernelGGL(kb_hash_count, dim3(padded_tiles(w.ntiles)), dim3(256), 0, s, w.args, w.tiles, w.ntiles, 0);
}

void launch_batch_patch_counts(const batch_work &w, hipStream_t s) {
  hipLaunchKernelGGL(kb_count_patches, dim3(padded_tiles(w.ntiles)), dim3(256), 0, s, w.args, w.tiles, w.ntiles);
}

void launch_batch_binning(const batch_work &w, hipStream_t s) {
  const dim3 gc(padded_tiles(w.nchunks));
  if (w.adaptive) {  // the descriptors are device memory of the batch; the geometry pass updates them
    hipLaunchKernelGGL(kb_geometry, dim3(w.n), dim3(GEO_THREADS), 0, s, const_cast<inst_args *>(w.args));
    hipLaunchKernelGGL(kb_hash_count, dim3(padded_tiles(w.ntiles)), dim3(256), 0, s, w.args, w.tiles, w.ntiles, 1);
  }
  hipLaunchKernelGGL(kb_sort, gc, dim3(SCAN_THREADS), 0, s, w.args, w.chunks, w.nchunks);
  if (w.rothlin)
    hipLaunchKernelGGL(kb_rothlin_cells, dim3(padded_tiles(w.ntiles)), dim3(256), 0, s, w.args, w.tiles, w.ntiles);
}

void launch_batch_records(const batch_work &w, hipStream_t s) {
  const dim3 gt(padded_tiles(w.ntiles));
  if (w.f32) hipLaunchKernelGGL(HIP_KERNEL_NAME(kb_records<true>), gt, dim3(TILE), 0, s, w.args, w.tiles, w.ntiles);
  else hipLaunchKernelGGL(HIP_KERNEL_NAME(kb_records<false>), gt, dim3(TILE), 0, s, w.args, w.tiles, w.ntiles);
}

template <class K>
static void launch_patches(K kern, const batch_work &w, hipStream_t s, hipEvent_t t0, hipEvent_t t1) {
  const dim3 grid(chunked_blocks(w.npatches, w.v.chunk));
  if (t0)
    hipExtLaunchKernelGGL(kern, grid, dim3(TILE), 0, s, t0, t1, 0, w.args, w.patches, w.npatches, w.v.chunk);
  else
    hipLaunchKernelGGL(kern, grid, dim3(TILE), 0, s, w.args, w.patches, w.npatches, w.v.chunk);
}

void launch_batch_interact(const batch_work &w, hipStream_t s, hipEvent_t t0, hipEvent_t t1) {
#define MFC_PICK(lanes, pse, gen) (w.f32 ? kb_interact<true, lanes, pse, gen> : kb_interact<false, lanes, pse, gen>)
#define MFC_PICK_PSE(lanes) launch_patches(w.general ? MFC_PICK(lanes, true, true) : \
                                           w.pse ? MFC_PICK(lanes, true, false) : MFC_PICK(lanes, false, false), w, s, t0, t1)
  switch (w.v.lanes) {
    case 1: MFC_PICK_PSE(1); break;
    case 4: MFC_PICK_PSE(4); break;
    default: MFC_PICK_PSE(8); break;
  }
}

void launch_batch_force(const batch_work &w, hipStream_t s) {
  hipLaunchKernelGGL(kb_force_final, dim3(w.n), dim3(FORCE_LAST_THREADS), 0, s, w.args);
}

// one step; the cell ids, counts and records of its start state come from the previous step's
// interaction (or launch_batch_hash and launch_batch_records), and its own interaction computes
// those of the next step
void launch_batch_step(const batch_work &w, hipStream_t s) {
  launch_batch_binning(w, s);  // also the tool's move, the patch list, the previous step's force groups
  launch_batch_interact(w, s);
}

}  // namespace mfc
