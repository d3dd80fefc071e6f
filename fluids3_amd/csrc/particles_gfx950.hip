// particles_gfx950.hip -- the SPH step as hand-written gfx950 (CDNA4, wave64)
// kernels, built into one code object that keeps the reference's module
// contract: the same extern "C" kernel names and argument lists
// (fluids5.0/src/particles.cuh:29-42) and the same four __constant__ symbols
// (fluids5.0/src/particles.cu:17-20), so a host that loads kernels and
// globals by name can drive it.
//
// Every stage is a device function over one scene: its FParams_t and its
// particle and cell ranges.  The reference-named kernels run it for the
// single scene held in FParams; the *Batch kernels run it for many
// independent scenes concatenated in the same buffers, one launch per stage,
// each block working inside one scene (a table maps block -> scene).
//
// Arithmetic contract (shared with the CPU oracle, which evaluates the same
// expression trees): the file is compiled with -ffp-contract=off, every fused
// multiply-add is an explicit fmaf(), sqrtf and '/' are IEEE correctly
// rounded.  With the stable in-cell order produced by the counting sort the
// FP32 results are then reproducible run to run and comparable bit for bit.
#include <hip/hip_runtime.h>

#include <climits>
#include <type_traits>

#include "fluidsx_params.h"
#include "fx_near.hpp"
#include "fx_walk.hpp"
#include "fx_trig.hpp"

typedef unsigned int uint;

__constant__ FParams_t FParams;
__constant__ cuDataX FPnts;
__constant__ cuDataX FPntTmp;
__constant__ cuDataX FAccel;

#define SCAN_BLOCKSIZE 512  // threads per scan block; each covers 1024 cells

// Words of neighbour bitmask a particle may record: FX_NBR_WORDS unless the
// host lowers it while the bitmask buffer is a smaller one (a reverse-mode
// tape slot).  A particle whose stencil rows need more records only the
// first ones, which the force stage does not read: it tests that particle's
// candidates in place.
__constant__ int FNbrWords = FX_NBR_WORDS;
__device__ __forceinline__ int nbr_cap() { return min(FNbrWords, FX_NBR_WORDS); }

// FX_CAP_* bits of what the host set up beyond the reference's layout; 0 for
// a host that binds this module as Fluids 5.0 binds its own.
__constant__ int FHostCaps = 0;
__device__ __forceinline__ bool host_tail() { return (FHostCaps & FX_CAP_TAIL) != 0; }
__device__ __forceinline__ bool host_ranked() { return (FHostCaps & FX_CAP_RANKED) != 0; }

// When set (the reverse mode's rollouts), the ranked counting sort writes
// its permutation here: FSortSrc[s] = pre-sort index of the particle it puts
// in slot s.  Null otherwise.
__constant__ uint* FSortSrc = nullptr;
#define FX_RANK_CAP 65536   // cells with more members keep atomic order

// ---------------------------------------------------------------- helpers

// Buffer id -> pointer.  The table holds global-memory addresses; passing
// them through the global address space lets the compiler emit global_*
// instructions instead of flat ones (flat accesses also count against the
// LDS wait counter and force coarser waits).
template <class T>
__device__ __forceinline__ T* pbuf(const cuDataX& d, int id) {
  typedef __attribute__((address_space(1))) T gT;
  return (T*)(gT*)(d.mbuf[id]);
}

// A scene's parameters read through the constant address space, so that the
// (block-uniform) reads are scalar loads.
// Three floats of element i, loaded and stored as scalars: an fx_float3
// copied as a whole (a struct select, say) can leave the compiler an
// aggregate it places in LDS or scratch memory instead of registers.
__device__ __forceinline__ fx_float3 ld3(const fx_float3* __restrict__ p, size_t i) {
  const float* f = reinterpret_cast<const float*>(p) + 3 * i;
  return fx_float3{f[0], f[1], f[2]};
}
// ld3 with non-temporal loads, for data read once
__device__ __forceinline__ fx_float3 ld3nt(const fx_float3* __restrict__ p, size_t i) {
  const float* f = reinterpret_cast<const float*>(p) + 3 * i;
  return fx_float3{__builtin_nontemporal_load(f), __builtin_nontemporal_load(f + 1), __builtin_nontemporal_load(f + 2)};
}
__device__ __forceinline__ void st3(fx_float3* __restrict__ p, size_t i, float x, float y, float z) {
  float* f = reinterpret_cast<float*>(p) + 3 * i;
  f[0] = x;
  f[1] = y;
  f[2] = z;
}
// Nt: non-temporal stores
template <bool Nt, class T>
__device__ __forceinline__ void put(T* p, T v) {
  if (Nt)
    __builtin_nontemporal_store(v, p);
  else
    *p = v;
}
template <bool Nt>
__device__ __forceinline__ void put3(fx_float3* __restrict__ p, size_t i, float x, float y, float z) {
  float* f = reinterpret_cast<float*>(p) + 3 * i;
  put<Nt>(f, x);
  put<Nt>(f + 1, y);
  put<Nt>(f + 2, z);
}

__device__ __forceinline__ const FParams_t* cparams(const FParams_t* p) {
  typedef const __attribute__((address_space(4))) FParams_t cP;
  return (const FParams_t*)(cP*)p;
}

// One block's view of its scene: particles [p0, p1), first cell c0 of the
// scene's cell table, and the block's index inside the scene.
struct Span {
  int p0, p1, c0, blk;
};

// Batch lookup: entry b of the block table is (scene, block inside scene).
// With a queue the launch is persistent: a fixed grid pulls the nitems
// entries as work items (see batch_items).
struct BatchArgs {
  const FParams_t* params;  // one FParams_t per scene
  const int* pbase;         // first particle of each scene (nscene + 1 entries)
  const int* cbase;         // first cell of each scene's table (nscene + 1)
  const int2* btab;         // (scene, local block) per block-table entry
  uint* queue;              // FX_NUM_XCD claim counters, zero at launch; null: one block per entry
  int nitems;               // entries of btab
  int pad;
};

__device__ __forceinline__ Span batch_span(const BatchArgs& B, int b, const FParams_t*& P) {
  const int2 e = B.btab[b];
  P = cparams(B.params + e.x);
  return Span{B.pbase[e.x], B.pbase[e.x + 1], B.cbase[e.x], e.y};
}

// Inclusive scan of one uint per lane across a wave64 with DPP row shifts and
// row broadcasts (GFX9 family).  Lanes whose DPP source is outside the row
// receive 0 through the 'old' operand.
__device__ __forceinline__ uint wave_inclusive_scan(uint v) {
  uint t;
  t = __builtin_amdgcn_update_dpp(0u, v, 0x111, 0xf, 0xf, false);  // row_shr:1
  v += t;
  t = __builtin_amdgcn_update_dpp(0u, v, 0x112, 0xf, 0xf, false);  // row_shr:2
  v += t;
  t = __builtin_amdgcn_update_dpp(0u, v, 0x114, 0xf, 0xf, false);  // row_shr:4
  v += t;
  t = __builtin_amdgcn_update_dpp(0u, v, 0x118, 0xf, 0xf, false);  // row_shr:8
  v += t;
  t = __builtin_amdgcn_update_dpp(0u, v, 0x142, 0xa, 0xf, false);  // row_bcast:15
  v += t;
  t = __builtin_amdgcn_update_dpp(0u, v, 0x143, 0xc, 0xf, false);  // row_bcast:31
  v += t;
  return v;
}

// Block barrier that orders LDS accesses only: global loads and atomics
// already in flight stay in flight across it (a __syncthreads() would first
// wait for them).
__device__ __forceinline__ void lds_barrier() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
  __builtin_amdgcn_s_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

__device__ __forceinline__ uint lanes_below(unsigned long long mask) {
  return __builtin_amdgcn_mbcnt_hi((uint)(mask >> 32), __builtin_amdgcn_mbcnt_lo((uint)mask, 0u));
}

// XCD-aware block order.  MI355X hands consecutive workgroups to its eight
// XCDs round-robin, and each XCD has its own L2.  Cell-sorted particles that
// are close in index share neighbours, so runs of FX_XCD_RUN consecutive
// logical blocks are given to one XCD, and the runs rotate over the XCDs (a
// contiguous share per XCD would unbalance the load, since the work per
// particle follows the local density).  Dispatch slot b is the k-th block
// of XCD x = b % 8; it runs logical block (run * 8 + x) * FX_XCD_RUN + k % RUN
// with run = k / RUN.  Blocks past the last full round keep their index.
#define FX_NUM_XCD 8
#ifndef FX_XCD_RUN
#define FX_XCD_RUN 32
#endif
__device__ __forceinline__ int xcd_block() {
  const int nb = (int)gridDim.x, b = (int)blockIdx.x;
  const int round = FX_NUM_XCD * FX_XCD_RUN;
  if (b >= nb / round * round) return b;
  const int x = b % FX_NUM_XCD, k = b / FX_NUM_XCD;
  return ((k / FX_XCD_RUN) * FX_NUM_XCD + x) * FX_XCD_RUN + k % FX_XCD_RUN;
}

// The XCD this workgroup runs on (hardware register XCC_ID, bits 3:0).
__device__ __forceinline__ int xcc_id() { return (int)(__builtin_amdgcn_s_getreg(20 | (3 << 11)) & 7u); }

// Persistent launches.  A fixed grid of resident blocks pulls work items
// (entries of the block table) until none is left.  The items are split into
// FX_NUM_XCD contiguous ranges, one per XCD, each drained in order through
// its own counter by the blocks running on that XCD, so that the blocks an
// XCD holds at a time work on neighbouring particles, whose neighbour cells
// then stay in that XCD's L2; a block whose range is exhausted takes items
// from the following ranges in turn.  A block leaves once every range is
// exhausted, so the launch drains whatever the grid size.  Thread 0 claims,
// the block reads the item from LDS.
// The claim state (current range, ranges tried) lives in LDS beside the
// claimed item: only thread 0 uses it, and it stays out of the registers of
// the work the block runs between claims.
struct Claim {
  int item, q, tried;
};

__device__ __forceinline__ int next_item(uint* ctr, int n, Claim* c) {
  if (threadIdx.x == 0) {
    int it = -1;
    int q = c->q, tried = c->tried;
    while (tried < FX_NUM_XCD) {
      const int lo = (int)(((long long)n * q) / FX_NUM_XCD);
      const int hi = (int)(((long long)n * (q + 1)) / FX_NUM_XCD);
      const int k = (int)atomicAdd(&ctr[q], 1u);
      if (k < hi - lo) {
        it = lo + k;
        break;
      }
      q = (q + 1) % FX_NUM_XCD;
      tried++;
    }
    c->item = it;
    c->q = q;
    c->tried = tried;
  }
  __syncthreads();
  const int it = c->item;
  __syncthreads();  // every thread has read the item before thread 0 claims the next
  return it;
}

// Runs body(entry) for every block-table entry this block claims in a
// persistent launch.
template <class F>
__device__ __forceinline__ void batch_items(const BatchArgs& B, F&& body) {
  __shared__ Claim c;
  if (threadIdx.x == 0) c = Claim{-1, xcc_id(), 0};
  for (int it = next_item(B.queue, B.nitems, &c); it >= 0; it = next_item(B.queue, B.nitems, &c)) body(it);
}

// Particles per thread of the streaming stages (index: FX_STAGE_INSERT 0,
// FX_STAGE_SORT 2, FX_STAGE_ADVANCE 5): a block covers blockDim * ppt
// consecutive particles, thread t taking t, t + blockDim, ...  A host that
// does not set it runs one particle per thread, as the reference's launches
// do (particles.cpp:26-30,294-296).
#define FX_MAX_PPT 8
__constant__ int FPpt[8] = {1, 1, 1, 1, 1, 1, 1, 1};
__device__ __forceinline__ int ppt_of(int stage) { return max(1, min(FPpt[stage], FX_MAX_PPT)); }
// the k-th of a block's ppt sub-blocks of blockDim particles
__device__ __forceinline__ Span sub_span(Span S, int ppt, int k) {
  S.blk = S.blk * ppt + k;
  return S;
}

// ----------------------------------------------------------- fill (memset)

// Fill used instead of hipMemsetAsync so that a captured step graph holds
// kernel nodes only.
extern "C" __global__ void fxFillUint(uint* __restrict__ p, uint v, int n) {
  int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) p[i] = v;
}

// No work: one dispatch of it marks a point of the stream in kernel traces
// and counter runs (the benchmark brackets its timed region with two).
extern "C" __global__ void fxMark(int tag) {}

// ------------------------------------------------------------------ insert

// Cell of each particle and its count slot.  Follows particles.cu:24-54:
//   gc = int((p - gridMin) * gridDelta), gs = (gc.y*res.z + gc.z)*res.x + gc.x,
//   in range iff 1 <= gc <= gridScanMax on every axis, else GRID_UNDEF.
// The range test is done on the float before truncation (trunc(g) >= 1 iff
// g >= 1; trunc(g) <= M iff g < M+1), which is the same predicate for every
// finite input and sends NaN to GRID_UNDEF.  Out-of-range particles are
// counted in slot gridTotal of the scene (its tail bucket).  Stored cell
// indices are offsets into the concatenated cell table (c0 + local cell).
// Without a tail slot (tail = false: a table of gridTotal entries, as the
// reference allocates) out-of-range particles are not counted and keep the
// gndx the host cleared, as in particles.cu:45-52.
//
// The counting is aggregated per wave: the particles arrive sorted by cell
// from the previous step, so the 64 lanes of a wave fall into few cells;
// lanes of one cell take a single atomicAdd of their number and their slot
// is the returned base plus their rank among those lanes.  The atomics of
// all the wave's cells are issued together (no round trip per cell).  The
// tail bucket is aggregated per block instead: particles that leave the grid
// stay out of it (the advance parks them), they are sorted to the end, and
// in a long run whole blocks hold nothing else (a sixth of the particles by
// step 200 of the 4M dam break), so one count per wave would put thousands
// of atomics on that one address.  `tl` is the block's LDS (two sets of 17
// words, alternating between calls so that one call's reads cannot meet
// the next call's writes).
template <bool Nt>
__device__ __forceinline__ void insert_at(const FParams_t& P, const Span S, int i, bool active, const fx_float3 p,
                                          bool tail, uint (*tl)[17]) {
  // active: the lane has particle i, at p; below, one that takes a count slot
  int gs = 0;
  if (active) {
    const float gx = (p.x - P.gridMin.x) * P.gridDelta.x;
    const float gy = (p.y - P.gridMin.y) * P.gridDelta.y;
    const float gz = (p.z - P.gridMin.z) * P.gridDelta.z;
    const bool in = gx >= 1.0f && gx < (float)(P.gridScanMax.x + 1) && gy >= 1.0f &&
                    gy < (float)(P.gridScanMax.y + 1) && gz >= 1.0f && gz < (float)(P.gridScanMax.z + 1);
    if (in) {
      gs = S.c0 + ((int)gy * P.gridRes.z + (int)gz) * P.gridRes.x + (int)gx;
      put<Nt>(&pbuf<int>(FPnts, FGCELL)[i], gs);
    } else {
      gs = S.c0 + P.gridTotal;
      put<Nt>(&pbuf<int>(FPnts, FGCELL)[i], (int)FX_GRID_UNDEF);
      active = tail;
    }
    uint* tflag = pbuf<uint>(FAccel, ATAILFLAG);
    if (tflag != nullptr) put<Nt>(&tflag[i], in ? 0u : 1u);
  }
  uint* cnt = pbuf<uint>(FAccel, AGRIDCNT);
  const int tslot = S.c0 + P.gridTotal;
  const bool intail = active && gs == tslot;
  // group the wave's lanes by slot (register-only ballots), then every
  // group's first lane adds the group's size with one atomic; all groups'
  // atomics go out together and each lane reads its group's base from the
  // leader lane
  unsigned long long todo = __ballot(active && !intail);
  unsigned long long mine = 0ull;
  int leader_of = 0;
  while (todo != 0ull) {  // one pass per distinct slot in the wave
    const int leader = __ffsll((long long)todo) - 1;
    const int v = __builtin_amdgcn_readlane(gs, leader);
    const unsigned long long same = __ballot(active && gs == v) & todo;
    if (active && gs == v) {
      mine = same;
      leader_of = leader;
    }
    todo &= ~same;
  }
  uint base = 0, tbase = 0;
  if (active && !intail && (int)__lane_id() == leader_of) base = atomicAdd(&cnt[gs], (uint)__popcll(mine));
  unsigned long long tm = 0ull;
  if (tail) {  // uniform: the block's tail lanes, one atomic (the cell atomics stay in flight meanwhile)
    tm = __ballot(intail);
    const int wv = (int)(threadIdx.x >> 6), nw = (int)((blockDim.x + 63u) >> 6);
    uint* L = tl[S.blk & 1];
    if (__lane_id() == 0) L[wv] = (uint)__popcll(tm);
    lds_barrier();
    if (threadIdx.x == 0) {
      uint tot = 0;
      for (int w = 0; w < nw; w++) tot += L[w];
      L[16] = tot != 0u ? atomicAdd(&cnt[tslot], tot) : 0u;
    }
    lds_barrier();
    if (intail) {
      tbase = L[16];
      for (int w = 0; w < wv; w++) tbase += L[w];
    }
  }
  base = (uint)__shfl((int)base, leader_of, 64);
  if (intail) {
    base = tbase;
    mine = tm;
  }
  if (active) put<Nt>(&pbuf<int>(FPnts, FGNDX)[i], (int)(base + lanes_below(mine)));
}

__device__ __forceinline__ void insert_impl(const FParams_t& P, const Span S, bool tail, uint (*tl)[17]) {
  const int i = S.p0 + S.blk * (int)blockDim.x + (int)threadIdx.x;
  fx_float3 p = fx_float3{0.0f, 0.0f, 0.0f};
  if (i < S.p1) p = ld3(pbuf<const fx_float3>(FPnts, FPOS), (size_t)i);
  insert_at<false>(P, S, i, i < S.p1, p, tail, tl);
}

// The streaming kernels keep a straight-line body for one particle per
// thread (the reference's launches and the usual choice), the loop otherwise.
extern "C" __global__ void insertParticles(int pnum) {
  __shared__ uint tl[2][17];
  const int ppt = ppt_of(0);
  const Span S{0, pnum, 0, (int)blockIdx.x};
  if (ppt == 1) {
    insert_impl(*cparams(&FParams), S, host_tail(), tl);
    return;
  }
  for (int k = 0; k < ppt; k++) insert_impl(*cparams(&FParams), sub_span(S, ppt, k), host_tail(), tl);
}

// one block-table entry of a batch stage (the *Batch kernels run one per
// block, the *BatchP kernels claim them)
__device__ __forceinline__ void insert_entry(const BatchArgs& B, int b) {
  const int ppt = ppt_of(0);
  const FParams_t* P;
  const Span S = batch_span(B, b, P);
  __shared__ uint tl[2][17];
  for (int k = 0; k < ppt; k++) insert_impl(*P, sub_span(S, ppt, k), true, tl);
}

extern "C" __global__ void insertParticlesBatch(BatchArgs B) { insert_entry(B, blockIdx.x); }

extern "C" __global__ void insertParticlesBatchP(BatchArgs B) {
  batch_items(B, [&](int b) { insert_entry(B, b); });
}

// ------------------------------------------------------------- prefix scan

// Block-local scan of 1024 uints, reference semantics (particles.cu:333-369):
// block b covers [1024b, 1024b+1024); zeroff=1 gives the exclusive scan,
// zeroff=0 the inclusive one; aux[b] (if given) receives the block total.
// Each thread owns two adjacent elements; waves scan with DPP, the eight wave
// totals are combined through LDS.  A batch of scenes is scanned in one pass
// over the concatenated cell tables: every scene's counts (tail bucket
// included) add up to its particle count, so the running sum enters each
// scene at its first particle.
extern "C" __global__ __launch_bounds__(SCAN_BLOCKSIZE) void prefixSum(
    uint* input, uint* output, uint* aux, int len, int zeroff) {
  __shared__ uint wsum[SCAN_BLOCKSIZE / 64];
  const int t = threadIdx.x;
  const uint e0 = blockIdx.x * (2u * SCAN_BLOCKSIZE) + 2u * t;
  const uint e1 = e0 + 1;
  const uint ulen = (uint)len;
  const uint a = e0 < ulen ? input[e0] : 0u;
  const uint b = e1 < ulen ? input[e1] : 0u;
  const uint s = a + b;
  const uint inc = wave_inclusive_scan(s);
  const int lane = t & 63, wave = t >> 6;
  if (lane == 63) wsum[wave] = inc;
  __syncthreads();
  uint wpre = 0, total = 0;
#pragma unroll
  for (int w = 0; w < SCAN_BLOCKSIZE / 64; w++) {
    const uint v = wsum[w];
    wpre += (w < wave) ? v : 0u;
    total += v;
  }
  const uint excl = wpre + inc - s;
  if (zeroff) {
    if (e0 < ulen) output[e0] = excl;
    if (e1 < ulen) output[e1] = excl + a;
  } else {
    if (e0 < ulen) output[e0] = excl + a;
    if (e1 < ulen) output[e1] = excl + a + b;
  }
  if (aux != nullptr && t == 0) aux[blockIdx.x] = total;
}

// Adds aux[b] to the 1024 elements of block b (particles.cu:325-331).
extern "C" __global__ __launch_bounds__(SCAN_BLOCKSIZE) void prefixFixup(
    uint* input, uint* aux, int len) {
  const uint t = threadIdx.x;
  const uint start = t + 2u * blockIdx.x * SCAN_BLOCKSIZE;
  const uint add = aux[blockIdx.x];
  if (start < (uint)len) input[start] += add;
  if (start + SCAN_BLOCKSIZE < (uint)len) input[start + SCAN_BLOCKSIZE] += add;
}

// The step's own scans (cell counts -> offsets, out-of-range flags -> tail
// ranks) in two launches each instead of the three to five of the
// reference's prefixSum/prefixFixup levels: fxScanSums writes the total of
// every block of FXS_BLOCK elements; in fxScanApply block b adds up the
// totals of the blocks before it (a few thousand at most, read once per
// block) and scans its own elements on top.  Exclusive, uint32: the same
// results as the reference-named kernels.  Where sums is null there is no
// first launch: a block adds up the elements before its own itself.
#define FXS_THREADS 512
#define FXS_PER 4
#define FXS_BLOCK (FXS_THREADS * FXS_PER)

// elements i..i+3 (zero beyond n); one 16-byte load when all four exist
__device__ __forceinline__ uint4 fxs_load(const uint* __restrict__ in, int i, int n) {
  if (i + 3 < n) return *reinterpret_cast<const uint4*>(in + i);
  uint4 v = make_uint4(0u, 0u, 0u, 0u);
  if (i < n) v.x = in[i];
  if (i + 1 < n) v.y = in[i + 1];
  if (i + 2 < n) v.z = in[i + 2];
  return v;
}

// sum of v over the block, returned to every thread (lds: one uint per wave)
__device__ __forceinline__ uint fxs_block_sum(uint v, uint* lds) {
  const uint tot = (uint)__builtin_amdgcn_readlane((int)wave_inclusive_scan(v), 63);
  if ((threadIdx.x & 63u) == 0u) lds[threadIdx.x >> 6] = tot;
  __syncthreads();
  uint s = 0u;
  for (int w = 0; w < (int)(blockDim.x >> 6); w++) s += lds[w];
  __syncthreads();  // every thread has read lds before it is written again
  return s;
}

// One launch serves up to two independent scans (the step scans the cell
// counts and the out-of-range flags): blocks [0, j[0].nb) take the first,
// the rest the second.
struct FxScanJob {
  const uint* in;
  uint* out;
  uint* sums;  // one total per block of FXS_BLOCK elements, or null
  int n;
  int nb;  // blocks: ceil(n / FXS_BLOCK)
};
// The set exchange of the counting sort: FPnts and FPntTmp receive the two
// 128-byte tables of bank[parity] and bank[parity ^ 1] (64 threads).  In a
// captured step it also moves the step clock: clock[1] holds the time of the
// step about to run, which becomes clock[0] (read by the advance of this
// step) while clock[1] moves on by dt.  No exchange where bank is null.
struct FxExchange {
  const uint* bank;
  uint* pnts;
  uint* tmp;
  float* clock;
  float dt;
  int parity;
};

__device__ __forceinline__ void exchange_tables(const FxExchange& E) {
  const int t = (int)threadIdx.x;
  constexpr int W = (int)(sizeof(cuDataX) / sizeof(uint));
  static_assert(2 * W <= 64, "one thread per word of the two tables");
  if (t < W) E.pnts[t] = E.bank[E.parity * W + t];
  else if (t < 2 * W) E.tmp[t - W] = E.bank[(E.parity ^ 1) * W + t - W];
  if (E.clock != nullptr && t == 0) {
    const float now = E.clock[1];
    E.clock[0] = now;
    E.clock[1] = now + E.dt;
  }
}

// (fxScanApply also makes the exchange when a step runs straight through: the
// scans read neither table.)
struct FxScanJobs {
  FxScanJob j[2];
  FxExchange ex;
};

__device__ __forceinline__ const FxScanJob& fxs_job(const FxScanJobs& J, int& b) {
  b = (int)blockIdx.x;
  if (b < J.j[0].nb) return J.j[0];
  b -= J.j[0].nb;
  return J.j[1];
}

extern "C" __global__ __launch_bounds__(FXS_THREADS) void fxScanSums(FxScanJobs J) {
  __shared__ uint lds[FXS_THREADS / 64];
  int b;
  const FxScanJob& S = fxs_job(J, b);
  const uint4 v = fxs_load(S.in, b * FXS_BLOCK + (int)threadIdx.x * FXS_PER, S.n);
  const uint s = fxs_block_sum(v.x + v.y + v.z + v.w, lds);
  if (threadIdx.x == 0) S.sums[b] = s;
}

extern "C" __global__ __launch_bounds__(FXS_THREADS) void fxScanApply(FxScanJobs J) {
  __shared__ uint lds[FXS_THREADS / 64];
  if (blockIdx.x == 0 && J.ex.bank != nullptr) exchange_tables(J.ex);
  int b;
  const FxScanJob& S = fxs_job(J, b);
  const uint* __restrict__ in = S.in;
  uint* __restrict__ out = S.out;
  const int n = S.n;
  uint pre = 0u;
  if (S.sums != nullptr) {
    for (int j = (int)threadIdx.x; j < b; j += FXS_THREADS) pre += S.sums[j];
  } else {
    const uint4* __restrict__ in4 = reinterpret_cast<const uint4*>(in) + threadIdx.x;
    for (int j0 = 0; j0 < b; j0 += 16) {  // 16 loads in flight
      uint4 w[16];
#pragma unroll
      for (int k = 0; k < 16; k++) w[k] = in4[(size_t)(j0 + k < b ? j0 + k : 0) * FXS_THREADS];
#pragma unroll
      for (int k = 0; k < 16; k++) pre += j0 + k < b ? w[k].x + w[k].y + w[k].z + w[k].w : 0u;
    }
  }
  pre = fxs_block_sum(pre, lds);
  const int i = b * FXS_BLOCK + (int)threadIdx.x * FXS_PER;
  const uint4 v = fxs_load(in, i, n);
  const uint t = v.x + v.y + v.z + v.w;
  const uint inc = wave_inclusive_scan(t);
  const int wave = (int)(threadIdx.x >> 6);
  if ((threadIdx.x & 63u) == 63u) lds[wave] = inc;
  __syncthreads();
  uint wpre = 0u;
  for (int w = 0; w < wave; w++) wpre += lds[w];
  const uint e = pre + wpre + inc - t;
  if (i + 3 < n) {
    *reinterpret_cast<uint4*>(out + i) = make_uint4(e, e + v.x, e + v.x + v.y, e + v.x + v.y + v.z);
  } else {
    if (i < n) out[i] = e;
    if (i + 1 < n) out[i + 1] = e + v.x;
    if (i + 2 < n) out[i + 2] = e + v.x + v.y;
  }
}

// ------------------------------------------------------------ counting sort

// x slab of an in-range position inside its cell, from the insert's float
// cell coordinate gx: floor(frac(gx) * FX_SLABS) (gx - (int)gx is exact for
// gx >= 1, and the product by a power of two is exact).
__device__ __forceinline__ int slab_of(const FParams_t& P, float px) {
  const float gx = (px - P.gridMin.x) * P.gridDelta.x;
  const float f = gx - (float)(int)gx;
  return min((int)(f * (float)FX_SLABS), FX_SLABS - 1);
}

// Index sort: AGRID[off[cell] + gndx] = i | slab << FX_MEMBER_BITS, the
// member list of every cell in insertion (atomic) order, each entry carrying
// the member's x slab for the full sort.  Same role as fluids3.2's
// countingSortIndex (fluids3.2/fluids/fluid_system_kern.cu:139-150); reads
// the pre-sort set FPntTmp.  Out-of-range particles fill their scene's tail
// bucket (slab 0).
#define FX_MEMBER_MASK ((1u << FX_MEMBER_BITS) - 1u)
__device__ __forceinline__ void sort_index_impl(const FParams_t& P, const Span S) {
  const int i = S.p0 + S.blk * (int)blockDim.x + (int)threadIdx.x;
  if (i >= S.p1) return;
  const int c = pbuf<const int>(FPntTmp, FGCELL)[i];
  const int cell = (c == FX_GRID_UNDEF) ? S.c0 + P.gridTotal : c;
  const uint* off = pbuf<const uint>(FAccel, AGRIDOFF);
  const uint slot = off[cell] + (uint)pbuf<const int>(FPntTmp, FGNDX)[i];
  const uint slab = c == FX_GRID_UNDEF ? 0u : (uint)slab_of(P, pbuf<const fx_float3>(FPntTmp, FPOS)[i].x);
  pbuf<uint>(FAccel, AGRID)[slot] = (uint)i | (slab << FX_MEMBER_BITS);
}

// Full counting sort FPntTmp -> FPnts (particles.cu:64-95) with a fixed
// in-cell order: a particle's slot in its cell is the number of members that
// precede it by (x slab, pre-sort index) -- the cell split into FX_SLABS
// equal slabs along x (slab_of) -- read from the member list, so the sorted
// order does not depend on atomic timing, and every cell's members lie in
// ascending slabs, which lets the density stage trim each stencil row to the
// particle's x-range.  The tail bucket of out-of-range particles, which can
// hold many, is ranked by the exclusive scan of the insert stage's
// out-of-range flags instead (particle order).  Cells above FX_RANK_CAP
// members keep the atomic order.  The sort moves the state that outlives a
// step (pos, vel, veval, clr, id) and the fresh gcell and gndx; press and
// force are recomputed by the next two stages.
//
// A member entry is (slab << FX_MEMBER_BITS) | index, so "precedes" is one
// unsigned comparison of entries.  Cells of up to FX_RANK_WAVE members are
// ranked per lane that way.  Larger ones are ranked by the wave together, one
// distinct cell at a time: per 64 member entries the wave takes five ballots
// (valid, and the four slab bits) and every lane walks the slab bits from the
// top, keeping the members that agree with its slab so far and counting
// those that fall below it; the members in its own slab with an index below
// the wave's first, and the wave's own lanes below it in the same cell and
// slab, complete the rank.  The same walk with slab = lane gives where each
// slab begins, which lanes 0..FX_SLABS-1 store in ASLABSTART (when the host
// has it) for the density stage; smaller cells get no slab starts.
#ifndef FX_RANK_WAVE
#define FX_RANK_WAVE 16
#endif
#define FX_SLAB_BITS 4
static_assert((1 << FX_SLAB_BITS) == FX_SLABS, "FX_SLABS is a power of two");

__device__ __forceinline__ void sort_full_impl(const FParams_t& P, const Span S) {
  const int lane = (int)(threadIdx.x & 63u);
  const int i = S.p0 + S.blk * (int)blockDim.x + (int)threadIdx.x;
  const bool act = i < S.p1;  // active lanes are a prefix of the wave
  const uint* off = pbuf<const uint>(FAccel, AGRIDOFF);
  const uint* grid = pbuf<const uint>(FAccel, AGRID);
  const uint* tscan = pbuf<const uint>(FAccel, ATAILSCAN);
  uint* sstart = pbuf<uint>(FAccel, ASLABSTART);
  const int c = act ? __builtin_nontemporal_load(&pbuf<const int>(FPntTmp, FGCELL)[i]) : FX_GRID_UNDEF;
  const int cell = (c == FX_GRID_UNDEF) ? S.c0 + P.gridTotal : c;
  // an in-range cell ends where the next begins (the counts may be cleared)
  uint o = 0u, n = 0u;
  if (act) {
    o = off[cell];
    n = off[cell + (c != FX_GRID_UNDEF ? 1 : 0)];
  }
  n -= o;
  // Everything that moves is loaded beside the cell's bounds: the ranking
  // below waits for memory twice more by itself (sort stage 158 -> 140 us at
  // the compressed 4M dam break, 172 -> 154 at the 4M beach from step 90,
  // 17.2 -> 16.6 at 16,384 particles).  The source set is read
  // once, with non-temporal loads, so that it displaces less of the sorted
  // set that the density stage reads next (sort 0.158 -> 0.146 ms at the 4M
  // beach scene, 0.201 -> 0.192 ms over 200 dam-break steps).
  const bool has_id = FPntTmp.mbuf[FID] != 0 && FPnts.mbuf[FID] != 0;
  float px = 0.0f, py = 0.0f, pz = 0.0f;
  fx_float3 vel = {0.0f, 0.0f, 0.0f}, vev = {0.0f, 0.0f, 0.0f};
  uint clr = 0u, id = 0u;
  if (act) {
    const fx_float3 q = ld3nt(pbuf<const fx_float3>(FPntTmp, FPOS), (size_t)i);
    px = q.x;
    py = q.y;
    pz = q.z;
    vel = ld3nt(pbuf<const fx_float3>(FPntTmp, FVEL), (size_t)i);
    vev = ld3nt(pbuf<const fx_float3>(FPntTmp, FVEVAL), (size_t)i);
    clr = __builtin_nontemporal_load(&pbuf<const uint>(FPntTmp, FCLR)[i]);
    if (has_id) id = __builtin_nontemporal_load(&pbuf<const uint>(FPntTmp, FID)[i]);
  }
  const int slab = c == FX_GRID_UNDEF ? 0 : slab_of(P, px);
  const uint key = ((uint)slab << FX_MEMBER_BITS) | (uint)i;  // this particle's own member entry
  const bool wide = act && c != FX_GRID_UNDEF && n > FX_RANK_WAVE && n <= FX_RANK_CAP;
  int rank = 0;
  {
    const uint w0 = (uint)(i - lane);
    const int tq = lane & (FX_SLABS - 1);  // the slab whose start this lane counts
    const unsigned long long lower = (1ull << lane) - 1ull;
    unsigned long long pending = __ballot(wide);
    while (pending != 0ull) {  // one distinct dense cell per pass (wave-uniform)
      const int lead = __ffsll((long long)pending) - 1;
      const int cl = __shfl(cell, lead, 64);
      const uint ol = (uint)__shfl((int)o, lead, 64), nl = (uint)__shfl((int)n, lead, 64);
      int below = 0, early = 0, start = 0;
      for (uint k0 = 0; k0 < nl; k0 += 64) {
        const uint k = k0 + (uint)lane;
        const bool valid = k < nl;
        const uint e = valid ? grid[ol + k] : 0u;
        unsigned long long m1 = __ballot(valid), m2 = m1;
        const unsigned long long low = __ballot(valid && (e & FX_MEMBER_MASK) < w0);
#pragma unroll
        for (int b = FX_SLAB_BITS - 1; b >= 0; b--) {
          const unsigned long long bit = __ballot(valid && ((e >> (FX_MEMBER_BITS + b)) & 1u));
          const bool s1 = (slab >> b) & 1, s2 = (tq >> b) & 1;
          below += s1 ? __popcll(m1 & ~bit) : 0;
          m1 = s1 ? (m1 & bit) : (m1 & ~bit);
          start += s2 ? __popcll(m2 & ~bit) : 0;
          m2 = s2 ? (m2 & bit) : (m2 & ~bit);
        }
        early += __popcll(m1 & low);
      }
      const bool mine = wide && cell == cl;
      unsigned long long m3 = __ballot(mine);
#pragma unroll
      for (int b = FX_SLAB_BITS - 1; b >= 0; b--) {
        const unsigned long long bit = __ballot(mine && ((slab >> b) & 1));
        m3 = ((slab >> b) & 1) ? (m3 & bit) : (m3 & ~bit);
      }
      if (mine) rank = below + early + __popcll(m3 & lower);
      if (sstart != nullptr && lane < FX_SLABS) sstart[(size_t)cl * FX_SLABS + lane] = (uint)start;
      pending &= ~__ballot(mine);
    }
  }
  if (!act) return;
  if (wide) {
    // ranked above
  } else if (c == FX_GRID_UNDEF && tscan != nullptr) {
    // tail bucket: the number of the scene's out-of-range particles before i
    rank = (int)(tscan[i] - tscan[S.p0]);
  } else if (const uint m = c != FX_GRID_UNDEF ? n : pbuf<const uint>(FAccel, AGRIDCNT)[cell]; m <= FX_RANK_CAP) {
    // member entries below this particle's own; eight in flight per step, the
    // last of them repeated (a loop over the remainder waited for each)
    for (uint k = 0; k < m; k += 8) {
      uint e[8];
#pragma unroll
      for (uint u = 0; u < 8; u++) e[u] = grid[o + min(k + u, m - 1)];
#pragma unroll
      for (uint u = 0; u < 8; u++) rank += k + u < m && e[u] < key ? 1 : 0;
    }
  } else {
    rank = pbuf<const int>(FPntTmp, FGNDX)[i];
  }
  const uint s = o + (uint)rank;
  st3(pbuf<fx_float3>(FPnts, FPOS), s, px, py, pz);
  st3(pbuf<fx_float3>(FPnts, FVEL), s, vel.x, vel.y, vel.z);
  st3(pbuf<fx_float3>(FPnts, FVEVAL), s, vev.x, vev.y, vev.z);
  pbuf<uint>(FPnts, FCLR)[s] = clr;
  if (has_id) pbuf<uint>(FPnts, FID)[s] = id;
  pbuf<int>(FPnts, FGCELL)[s] = c;
  pbuf<int>(FPnts, FGNDX)[s] = rank;
  if (FSortSrc != nullptr) FSortSrc[s] = (uint)i;
}

// The counting sort of a host that runs no countingSortIndex (the reference's
// own, particles.cpp:832-842): every particle goes to off[cell] + gndx, its
// insert slot, so the in-cell order is the insert's atomic order; the eight
// reference buffers move (press and force included, particles.cu:80-89), the
// id when both sets have one, and AGRID[slot] = slot (particles.cu:91).
// Without a tail slot out-of-range particles are not moved (particles.cu:78),
// with one they go to the scene's tail bucket in gndx order.
__device__ __forceinline__ void sort_full_gndx(const FParams_t& P, const Span S, bool tail) {
  const int i = S.p0 + S.blk * (int)blockDim.x + (int)threadIdx.x;
  if (i >= S.p1) return;
  const int c = pbuf<const int>(FPntTmp, FGCELL)[i];
  if (c == FX_GRID_UNDEF && !tail) return;
  const int cell = (c == FX_GRID_UNDEF) ? S.c0 + P.gridTotal : c;
  const int nd = pbuf<const int>(FPntTmp, FGNDX)[i];
  const uint s = pbuf<const uint>(FAccel, AGRIDOFF)[cell] + (uint)nd;
  const bool has_id = FPntTmp.mbuf[FID] != 0 && FPnts.mbuf[FID] != 0;
  const fx_float3 pos = ld3(pbuf<const fx_float3>(FPntTmp, FPOS), (size_t)i);
  const fx_float3 vel = ld3(pbuf<const fx_float3>(FPntTmp, FVEL), (size_t)i);
  const fx_float3 vev = ld3(pbuf<const fx_float3>(FPntTmp, FVEVAL), (size_t)i);
  const fx_float3 frc = ld3(pbuf<const fx_float3>(FPntTmp, FFORCE), (size_t)i);
  const float prs = pbuf<const float>(FPntTmp, FPRESS)[i];
  const uint clr = pbuf<const uint>(FPntTmp, FCLR)[i];
  const uint id = has_id ? pbuf<const uint>(FPntTmp, FID)[i] : 0u;
  st3(pbuf<fx_float3>(FPnts, FPOS), s, pos.x, pos.y, pos.z);
  st3(pbuf<fx_float3>(FPnts, FVEL), s, vel.x, vel.y, vel.z);
  st3(pbuf<fx_float3>(FPnts, FVEVAL), s, vev.x, vev.y, vev.z);
  st3(pbuf<fx_float3>(FPnts, FFORCE), s, frc.x, frc.y, frc.z);
  pbuf<float>(FPnts, FPRESS)[s] = prs;
  pbuf<uint>(FPnts, FCLR)[s] = clr;
  if (has_id) pbuf<uint>(FPnts, FID)[s] = id;
  pbuf<int>(FPnts, FGCELL)[s] = c;
  pbuf<int>(FPnts, FGNDX)[s] = nd;
  uint* grid = pbuf<uint>(FAccel, AGRID);
  if (grid != nullptr) grid[s] = s;
}

// Clears n counts, spread over the launch, for the next step's insert, which
// the force launch of this step makes (force_end): after the scan no stage of
// a step that runs straight through reads them.  The density launch does it
// with two or four lanes to a particle, the sort's with one: there two more
// registers cost the density a wave a SIMD and 4 % of its time (beach 102.3 ->
// 101.0 ms for 100 steps), while small scenes lose by it in the sort (65,537
// particles 79.2 -> 80.5 us a step).
__device__ __forceinline__ void clear_counts(uint* __restrict__ p, int n) {
  if (p == nullptr) return;
  for (int k = (int)(blockIdx.x * blockDim.x + threadIdx.x); k < n; k += (int)(gridDim.x * blockDim.x)) p[k] = 0u;
}

extern "C" __global__ void countingSortIndex(int pnum) {
  const int ppt = ppt_of(2);
  const Span S{0, pnum, 0, (int)blockIdx.x};
  if (ppt == 1) {
    sort_index_impl(*cparams(&FParams), S);
    return;
  }
  for (int k = 0; k < ppt; k++) sort_index_impl(*cparams(&FParams), sub_span(S, ppt, k));
}

// The sort of a host that runs the index sort first (libfluidsx).  Kept apart
// from countingSortFull: compiling the insert-slot variant into the same
// kernel slows this one by half (183 vs 114 us per launch at 4M particles).
// It also clears the counts (none where clear is null), in a step whose force
// launch makes the next insert; countingSortFullRanked, at the end of this
// file, is the same without that, for hosts that launch it with pnum alone.
extern "C" __global__ void countingSortFullRankedClear(int pnum, uint* clear, int nclear) {
  const int ppt = ppt_of(2);
  const Span S{0, pnum, 0, xcd_block()};
  if (ppt == 1) {
    sort_full_impl(*cparams(&FParams), S);
  } else {
    for (int k = 0; k < ppt; k++) sort_full_impl(*cparams(&FParams), sub_span(S, ppt, k));
  }
  clear_counts(clear, nclear);
}

// The reference's kernel name (particles.cu:64-95): the insert's slots for a
// host without the index sort, the stable ranking for one that runs it
// (FX_CAP_RANKED; countingSortFullRanked is the faster entry for that case).
extern "C" __global__ void countingSortFull(int pnum) {
  const int ppt = ppt_of(2);
  if (!host_ranked()) {
    for (int k = 0; k < ppt; k++)
      sort_full_gndx(*cparams(&FParams), sub_span(Span{0, pnum, 0, (int)blockIdx.x}, ppt, k), host_tail());
    return;
  }
  for (int k = 0; k < ppt; k++) sort_full_impl(*cparams(&FParams), sub_span(Span{0, pnum, 0, xcd_block()}, ppt, k));
}

__device__ __forceinline__ void sort_index_entry(const BatchArgs& B, int b) {
  const int ppt = ppt_of(2);
  const FParams_t* P;
  const Span S = batch_span(B, b, P);
  for (int k = 0; k < ppt; k++) sort_index_impl(*P, sub_span(S, ppt, k));
}

__device__ __forceinline__ void sort_full_entry(const BatchArgs& B, int b) {
  const int ppt = ppt_of(2);
  const FParams_t* P;
  const Span S = batch_span(B, b, P);
  if (ppt == 1) {
    sort_full_impl(*P, S);
    return;
  }
  for (int k = 0; k < ppt; k++) sort_full_impl(*P, sub_span(S, ppt, k));
}

extern "C" __global__ void countingSortIndexBatch(BatchArgs B) { sort_index_entry(B, blockIdx.x); }
extern "C" __global__ void countingSortFullBatch(BatchArgs B, uint* clear, int nclear) {
  sort_full_entry(B, xcd_block());
  clear_counts(clear, nclear);
}

extern "C" __global__ void countingSortIndexBatchP(BatchArgs B) {
  batch_items(B, [&](int b) { sort_index_entry(B, b); });
}

extern "C" __global__ void countingSortFullBatchP(BatchArgs B) {
  batch_items(B, [&](int b) { sort_full_entry(B, b); });
}

// ----------------------------------------------------------------- density

// Row decomposition of the stencil: gridAdj[(y*srch + z)*srch + x] =
// (y*res.z + z)*res.x + x (particles.cpp:614-618) is contiguous in x, so the
// srch cells of one (y, z) row are one contiguous run of sorted particles,
// visited in the same order as the reference's per-cell loop.
// Row r of the stencil at base (an in-range particle's): candidates
// [jb, je).  The row ends where the cell after its last one begins -- a cell
// of the same grid row, since an in-range particle's stencil stays one cell
// inside the grid -- so two loads, not three.
__device__ __forceinline__ void row_range(const FParams_t& P, int base, int r, const uint* __restrict__ off,
                                          const uint* __restrict__ cnt, int& jb, int& je) {
  (void)cnt;
  const int srch = P.gridSrch;
  const int c0 = base + P.gridAdj[r * srch];
  jb = (int)off[c0];
  je = (int)off[c0 + srch];
}

__device__ __forceinline__ int stencil_base(const FParams_t& P, int gc) {
  return gc - (P.gridRes.z + 1) * P.gridRes.x - 1;
}

// Tiling.  A block owns the consecutive sorted particles [h0, h1) (in-range
// particles only; out-of-range ones sit in the scene's tail).  Their cells
// form one contiguous index range [cf, cl], so for every stencil row the
// candidates of all the block's particles form one contiguous run of sorted
// particles, from the row start of cf to the row end of cl.  The block stages
// that run in LDS in chunks of TILE_P with coalesced loads; each lane then
// reads the part of the chunk that falls in its own row window.  Chunks are
// visited in increasing order, so every lane still sees its candidates in the
// reference's order.
// One tile entry (a candidate's position) in LDS, 12 bytes: with a 16-byte
// stride entries 16 apart share banks, and the lanes of a wave, whose windows
// start at different entries (their x-range trims differ, and at rest density
// they lie in different cells), queued on them; with a 12-byte stride the
// entries of 21 consecutive candidates fall in distinct banks.  (Separate
// x, y and z arrays measured the same as this.)
struct TileP {
  float x, y, z;
};
#ifndef TILE_P
#define TILE_P 1024  // candidates per tile, 12 KB
#endif
#define FX_TILE_FLOATS (3 * TILE_P)
__device__ __forceinline__ void tile_put(float* t, int k, const fx_float3& q) {
  t[3 * k] = q.x;
  t[3 * k + 1] = q.y;
  t[3 * k + 2] = q.z;
}
__device__ __forceinline__ TileP tile_get(const float* t, int k) { return TileP{t[3 * k], t[3 * k + 1], t[3 * k + 2]}; }

struct BlockSpan {
  int h1;      // end of the block's in-range particles
  int cf, cl;  // first and last cell of the block
};

__device__ __forceinline__ bool block_span(const FParams_t& P, const Span S, int h0,
                                           const int* __restrict__ gcell, const uint* __restrict__ off,
                                           const uint* __restrict__ cnt, bool tail, BlockSpan& s) {
  // end of the scene's in-range particles: the start of its tail bucket, or
  // the end of its last cell when the table has no tail slot
  const int last = S.c0 + P.gridTotal - 1;
  const int nvalid = tail ? (int)off[last + 1] : (int)(off[last] + cnt[last]);
  if (h0 >= nvalid || h0 >= S.p1) return false;
  s.h1 = min(min(h0 + (int)blockDim.x, nvalid), S.p1);
  s.cf = gcell[h0];
  s.cl = gcell[s.h1 - 1];
  return true;
}

// Number of bitmask words a particle of cell gc uses: one word-aligned run of
// ceil(len/32) words per stencil row.
__device__ __forceinline__ int nbr_words(const FParams_t& P, int gc, const uint* __restrict__ off,
                                         const uint* __restrict__ cnt) {
  const int base = stencil_base(P, gc);
  int w = 0;
  for (int r = 0; r < P.gridSrch * P.gridSrch; r++) {
    int jb, je;
    row_range(P, base, r, off, cnt, jb, je);
    w += (je - jb + 31) >> 5;
  }
  return w;
}

// Density (particles.cu:120-157): rho_i = m * poly6 * sum_{0<d2<rd2}
// ((rd2 - d2) * d2s)^3 with d2 in world units, stored in FPRESS; an isolated
// particle gets 1.0.
//
// When the host provides the ANBRBITS and AFREC buffers the kernel also
// records, for the force stage, one bit per stencil candidate (set for the
// in-radius pairs; row r of particle i occupies words W_r .. W_r+ceil(len/32)-1
// at [w * N + i], N the size of the whole particle buffer) and the particle's
// (pos, rho), (veval, 0) record.  A particle whose candidates need more than
// the cap's words (FNbrWords) records only its first ones, which the force
// stage does not read: it finds the particle over the cap from its own row
// lengths and tests its candidates in place.
//
// Row trimming (when the sort ordered every cell's members by x slab and
// wrote where each slab begins, `trim`).  In grid units (the insert's
// gx = (x - gridMin.x) * gridDelta.x, cells of width 1) a member of slab k of
// a cell at x index c has gx in [c + k/16, c + (k+1)/16).  A particle at gp
// is out of radius of a whole slab of its row's first cell (x index cx - 1)
// when gp - (cx - 1) - (k+1)/16 > Rg, and of a whole slab of its row's last
// cell (x index cx + srch - 2) when (cx + srch - 2) + k/16 - gp > Rg, with
// Rg = rlim * gridDelta.x plus a margin of 2^-7 cells and gridRes.x * 2^-20
// that covers the rounding of gx (about 2^-22 of it) on both sides: every
// member of such a slab has fl(|px - x|) > rlim, so fl(dx * dx) > rd2 and it
// fails the radius test whatever its y and z.  Those slabs are a prefix of
// the first cell and a suffix of the last (the members lie in ascending
// slabs), located through the slab starts, and the lane walks only [ts, te)
// of its row.  The skipped candidates' bits are zero: the bitmask keeps its
// layout (bit s of the row for candidate s), written with the lane's phase
// ts % 32.
#define FX_TRIM_MARGIN 0.0078125f

// Slabs [0, lo) of the row's first cell and [hi, FX_SLABS) of its last cell
// lie beyond the radius of a particle at grid x coordinate gp in cell cx.
__device__ __forceinline__ void trim_slabs(float gp, int cx, int srch, float Rg, int& lo, int& hi) {
  const float fx = (float)(cx - 1), lx = (float)(cx + srch - 2);
  lo = min(max((int)ceilf((float)FX_SLABS * (gp - fx - Rg) - 1.0f), 0), FX_SLABS);
  hi = min(max((int)floorf((float)FX_SLABS * (gp - lx + Rg)) + 1, 0), FX_SLABS);
}

// Members of cell c (n of them) in slabs below k.
__device__ __forceinline__ int slab_start(const uint* __restrict__ sstart, int c, int n, int k) {
  return (n == 0 || k == 0) ? 0 : (k >= FX_SLABS ? n : (int)sstart[(size_t)c * FX_SLABS + k]);
}

__device__ __forceinline__ void pressure_impl(const FParams_t& P, const Span S, int N, float* tile, bool tail,
                                              bool trim) {
  const int t = threadIdx.x;
  const int h0 = S.p0 + S.blk * (int)blockDim.x;
  const int i = h0 + t;
  const int* __restrict__ gcell = pbuf<const int>(FPnts, FGCELL);
  const fx_float3* __restrict__ pos = pbuf<const fx_float3>(FPnts, FPOS);
  const uint* __restrict__ off = pbuf<const uint>(FAccel, AGRIDOFF);
  const uint* __restrict__ cnt = pbuf<const uint>(FAccel, AGRIDCNT);
  uint* __restrict__ bits = pbuf<uint>(FAccel, ANBRBITS);
  const bool wbits = bits != nullptr && FAccel.mbuf[AFREC] != 0;
  BlockSpan B;
  if (!block_span(P, S, h0, gcell, off, cnt, tail, B)) return;  // uniform per block
  const bool act = i < B.h1;
  const int gc = act ? gcell[i] : B.cf;
  fx_float3 p = fx_float3{0.0f, 0.0f, 0.0f};
  if (act) p = pos[i];
  const int shift = (P.gridRes.z + 1) * P.gridRes.x + 1;
  const int srch = P.gridSrch;
  const float rd2 = P.rd2, d2 = P.d2;
  const size_t NN = (size_t)N;
  // The bitmask's words are written up to the cap: a particle that needs
  // more is found so by the force stage from its own row lengths, which then
  // tests its candidates in place and reads none of them.
  const bool rec = wbits && act;
  const int cap = nbr_cap();
  auto put = [&](int w, uint v) {
    if (rec && w < cap) bits[(size_t)w * NN + i] = v;
  };
  // x-distance beyond which fl(dx * dx) > rd2: dx > rlim > sqrt(rd2) (1 + 2^-21)
  const float rlim = __fsqrt_rn(rd2) * (1.0f + 0x1p-20f);
  const float Rg = rlim * P.gridDelta.x + FX_TRIM_MARGIN + (float)P.gridRes.x * 0x1p-20f;
  const float gp = (p.x - P.gridMin.x) * P.gridDelta.x;  // the insert's cell coordinate
  const uint* __restrict__ sstart = pbuf<const uint>(FAccel, ASLABSTART);
  const bool trim_lane = trim && sstart != nullptr && act;
  int slo = 0, shi = FX_SLABS;
  if (trim_lane) trim_slabs(gp, (int)gp, srch, Rg, slo, shi);
  float sum = 0.0f;
  int W = 0;  // first word of the current row
  for (int r = 0; r < srch * srch; r++) {
    const int adj = P.gridAdj[r * srch] - shift;
    // a row ends where the cell after its last one begins (an in-range
    // particle's row is followed by a cell of the same grid row)
    const int lo = (int)off[B.cf + adj];
    const int hi = (int)off[B.cl + adj + srch];
    int jb = 0, je = 0;
    if (act) {
      jb = (int)off[gc + adj];
      je = (int)off[gc + adj + srch];
    }
    // the lane walks candidates [ts, te) of its row (relative to jb); a row
    // of at most FX_RANK_WAVE candidates has no cell with slab starts
    int ts = 0, te = je - jb;
    if (trim_lane && je - jb > FX_RANK_WAVE) {
      const int c0 = gc + adj, c2 = gc + adj + srch - 1;
      const int n0 = (int)cnt[c0], n2 = (int)cnt[c2];
      // slab starts exist for the cells the sort ranked by wave
      if (n0 > FX_RANK_WAVE && n0 <= FX_RANK_CAP) ts = slab_start(sstart, c0, n0, slo);
      if (n2 > FX_RANK_WAVE && n2 <= FX_RANK_CAP) te = max(ts, te - n2 + slab_start(sstart, c2, n2, shi));
    }
    if (hi - lo <= TILE_P) {
      // The row's run fits one tile: the lane's candidate s (0 <= s < len)
      // is tile entry a + s and bit s % 32 of the row's word s / 32, the
      // same position in every lane.  The wave walks s in lockstep, 32
      // candidates per word; candidates every lane has are unchecked, the
      // rest are masked by s < len.  Bits are shifted in (first candidate
      // highest) and the word is bit-reversed when stored.
      for (int k = t; k < hi - lo; k += blockDim.x) {
        const fx_float3 q = pos[lo + k];
        tile_put(tile, k, q);
      }
      __syncthreads();
      const int a = act ? jb - lo : 0, len = act ? je - jb : 0;
      const int L = te - ts, a0 = a + ts, ph = ts & 31, w0 = ts >> 5;
      const int lmax = wave_max(L), lmin = wave_min(act ? L : INT_MAX);
      const int last = hi - lo - 1;  // last entry of the run
      const int nw = (len + 31) >> 5;
      uint acc = 0u;
      auto cand = [&](int s, auto checked) {
        int k = a0 + s;
        if (decltype(checked)::value) k = min(k, last);
        const TileP q = tile_get(tile, k);
        const float dx = p.x - q.x, dy = p.y - q.y, dz = p.z - q.z;
        const float dsq = fmaf(dz, dz, fmaf(dy, dy, dx * dx));
        if (decltype(checked)::value) {
          const bool pair = dsq < rd2 && dsq > 0.0f && s < L;
          const float tt = pair ? (rd2 - dsq) * d2 : 0.0f;
          sum = fmaf(tt * tt, tt, sum);  // + 0 when not a pair: sum unchanged
          acc = acc + acc + (pair ? 1u : 0u);
        } else {
          // The same three steps with the wave's pair mask m used as it is:
          // the term selected by m (v_cndmask) and the bit shifted in as the
          // carry of acc + acc (v_addc), one instruction each where the
          // compiler spends two on the bit.  One ballot per compare, so that
          // m is the compares' own mask.
          const unsigned long long m = __builtin_amdgcn_ballot_w64(dsq < rd2) & __builtin_amdgcn_ballot_w64(dsq > 0.0f);
          const float t0 = (rd2 - dsq) * d2;
          float tt;
          __asm__("v_cndmask_b32_e64 %0, 0, %1, %2" : "=v"(tt) : "v"(t0), "s"(m));
          sum = fmaf(tt * tt, tt, sum);  // + 0 when not a pair: sum unchanged
          unsigned long long carry;
          uint acc2;
          __asm__("v_addc_co_u32_e64 %0, %1, %2, %2, %3" : "=v"(acc2), "=s"(carry) : "v"(acc), "s"(m));
          acc = acc2;
        }
      };
      // the block of candidates ts + s0 .. ts + s0 + 31 straddles words
      // w0 + s0/32 (bits ph..31) and the next (bits 0..ph-1): the second
      // part is carried into the next block's word
      uint carry = 0u;
      int wb = w0;
      for (int s0 = 0; s0 < lmax; s0 += 32) {
        const int n = min(32, lmax - s0);
        const int nu = max(0, min(n, lmin - s0));
        int u = 0;
        // unrolled by hand: the asm in cand keeps the compiler from unrolling
        for (; u + 4 <= nu; u += 4) {
          cand(s0 + u, std::false_type());
          cand(s0 + u + 1, std::false_type());
          cand(s0 + u + 2, std::false_type());
          cand(s0 + u + 3, std::false_type());
        }
        for (; u < nu; u++) cand(s0 + u, std::false_type());
        for (; u < n; u++) cand(s0 + u, std::true_type());
        const uint chunk = __builtin_bitreverse32(acc << (32 - n));
        if (wb < nw) put(W + wb, carry | (chunk << ph));
        carry = ph ? chunk >> (32 - ph) : 0u;
        wb++;
        acc = 0u;
      }
      if (rec) {  // the words the walk did not reach hold no pair
        for (int w = 0; w < w0; w++) put(W + w, 0u);
        if (wb < nw) put(W + wb, carry);
        for (int w = wb + 1; w < nw; w++) put(W + w, 0u);
      }
      __syncthreads();
      W += (je - jb + 31) >> 5;
      continue;
    }
    // bits of the current word and the next one's mask, from the lane's phase
    uint acc = 0, bit = 1u << (ts & 31);
    int wcur = W + (ts >> 5);  // current word
    if (rec)
      for (int w = W; w < wcur; w++) put(w, 0u);  // skipped candidates
    for (int c0 = lo; c0 < hi; c0 += TILE_P) {
      const int n = min(TILE_P, hi - c0);
      for (int k = t; k < n; k += blockDim.x) {
        const fx_float3 q = pos[c0 + k];
        tile_put(tile, k, q);
      }
      __syncthreads();
      const int a = max(jb + ts, c0) - c0, b = min(jb + te, c0 + n) - c0;
      for (int k = a; k < b; k++) {
        const TileP q = tile_get(tile, k);
        const float dx = p.x - q.x, dy = p.y - q.y, dz = p.z - q.z;
        const float dsq = fmaf(dz, dz, fmaf(dy, dy, dx * dx));
        const bool pair = dsq < rd2 && dsq > 0.0f;
        if (pair) {
          const float tt = (rd2 - dsq) * d2;
          sum = fmaf(tt * tt, tt, sum);
        }
        if (rec) {
          acc |= pair ? bit : 0u;
          if (bit == 0x80000000u) {  // word complete
            put(wcur, acc);
            acc = 0;
            wcur++;
          }
          bit = __builtin_amdgcn_alignbit(bit, bit, 31);  // rotate left by one
        }
      }
      __syncthreads();
    }
    if (rec && bit != 1u) put(wcur++, acc);  // the walk's partial last word
    if (rec)
      for (int w = wcur; w < W + ((je - jb + 31) >> 5); w++) put(w, 0u);
    W += (je - jb + 31) >> 5;
  }
  if (act) {
    sum = sum * P.pmass * P.poly6kern;
    if (sum == 0.0f) sum = 1.0f;
    pbuf<float>(FPnts, FPRESS)[i] = sum;
    if (wbits) {
      // read once here: non-temporal (density 0.305 -> 0.298 ms at the 4M beach scene)
      const fx_float3 v = ld3nt(pbuf<const fx_float3>(FPnts, FVEVAL), (size_t)i);
      float4* fr = pbuf<float4>(FAccel, AFREC);
      fr[2 * (size_t)i] = make_float4(p.x, p.y, p.z, sum);
      fr[2 * (size_t)i + 1] = make_float4(v.x, v.y, v.z, 0.0f);
    }
  }
}

extern "C" __global__ __launch_bounds__(1024) void computePressure(int pnum) {
  __shared__ __align__(16) float tile[FX_TILE_FLOATS];
  pressure_impl(*cparams(&FParams), Span{0, pnum, 0, xcd_block()}, pnum, tile, host_tail(), host_ranked());
}

extern "C" __global__ __launch_bounds__(1024) void computePressureBatch(BatchArgs B, int ntotal) {
  __shared__ __align__(16) float tile[FX_TILE_FLOATS];
  const FParams_t* P;
  const Span S = batch_span(B, xcd_block(), P);
  pressure_impl(*P, S, ntotal, tile, true, true);
}

extern "C" __global__ __launch_bounds__(1024) void computePressureBatchP(BatchArgs B, int ntotal) {
  __shared__ __align__(16) float tile[FX_TILE_FLOATS];
  batch_items(B, [&](int b) {
    const FParams_t* P;
    const Span S = batch_span(B, b, P);
    pressure_impl(*P, S, ntotal, tile, true, true);
    __syncthreads();  // the next entry's tile loads wait for this entry's last reads
  });
}

// --------------------------------------------------------- density by wave
//
// The library's own density stage (stencil rows of 2 or 3 cells): each wave
// works alone, with G lanes to a particle, on 64 / G consecutive sorted
// particles.  What the block-wide tiles above cost is waiting: two barriers
// and two dependent loads per stencil row, nine times, for rows of about 11
// candidates at rest density, and a block whose particles spread over a
// sparse layer walks the whole run between its first and last cell.  Here
// every row's bounds are loaded at once, and the wave stages a layer of the
// stencil (gridSrch rows), or all rows when they fit, in its own LDS tile
// with all loads in flight and no barrier.  A layer beyond the tile goes row
// by row, trimmed to the particle's x-range as above (dense cells), from
// memory where even one row's run is longer than the tile (sparse layers).
//
// G lanes to a particle take candidates s, s + 1, .. of one step each and add
// their terms in candidate order through DPP broadcasts, so the sums are the
// same bits for every G.  It costs more instructions per candidate (about 24
// a wave step of 4 candidates at G = 4, against 15 for one at G = 1) and
// shortens the chain of a wave, which is what a launch of few waves waits
// for.  Measured per launch, block tiles / G = 1 / 2 / 4 (us, HIP events
// around the stage): 16,384 compressed 46 / 28 / 20 / 16; at rest density
// 65,536 85 / 45 / 33 / 30, 100,000 91 / 49 / 37 / 39, 262,144
// 99 / 55 / 54 / 71, 400,000 106 / 53 / 60 / 82, 1,000,000
// 170 / 80 / 112 / 160; the 4M beach from step 20 246 / 185 / 272 / 435 and
// from step 90 394 / 325 / 475 / 721; the compressed 4M dam break from step 5
// 917 / 920 / 1500 / 2359, from step 25 1055 / 1050, from step 60
// 2055 / 1820 (G = 1).  At G = 1 in dense cells VALU issue bounds it (14
// instructions a candidate in the unchecked walk, 15 in a staged row): 0.39 to
// 0.41 a cycle and SIMD, where independent two-operand instructions reach
// 0.40, with the LDS busy for 0.7 of the cycles.  At rest density (0.26 to
// 0.33) the waves wait for row bounds and staging for a third to half of their
// cycles.
//
// Tile: FX_DENS_TILE entries a wave, and FX_DENS_PAD entries after a block's
// last tile that a lane past its row's end may read and discard: 256-thread
// blocks of 20 KB, eight to a CU.  Six blocks to a CU (384 entries, a pad of
// 384) took 207 us on the beach from step 20 and 965 on the compressed dam
// break, 512 entries 224 and 1095, 256 entries 188 and 959.  Where the lanes'
// windows lie in a run longer than the tile (compressed cells), the tile
// slides along the walk; with such rows read from memory, 40 dam-break steps
// from step 5 took 153.8 instead of 152.0 ms.

// lane K of the particle's G lanes
template <int G, int K>
__device__ __forceinline__ float lane_bcast(float v) {
  constexpr int ctrl = G == 4 ? K * 0x55 : (K == 0 ? 0xA0 : 0xF5);  // quad_perm
  return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), ctrl, 0xf, 0xf, true));
}

// OR over the particle's G lanes
template <int G>
__device__ __forceinline__ uint lanes_or(uint v) {
  if (G >= 2) v |= __builtin_amdgcn_update_dpp(0u, v, 0xB1, 0xf, 0xf, true);  // quad_perm 1,0,3,2
  if (G >= 4) v |= __builtin_amdgcn_update_dpp(0u, v, 0x4E, 0xf, 0xf, true);  // quad_perm 2,3,0,1
  return v;
}

// bit u of v to bit u * G
template <int G>
__device__ __forceinline__ uint spread_bits(uint v) {
  if constexpr (G == 2) {
    v = (v | v << 8) & 0x00ff00ffu;
    v = (v | v << 4) & 0x0f0f0f0fu;
    v = (v | v << 2) & 0x33333333u;
    v = (v | v << 1) & 0x55555555u;
  } else if constexpr (G == 4) {
    v = (v | v << 12) & 0x000f000fu;
    v = (v | v << 6) & 0x03030303u;
    v = (v | v << 3) & 0x11111111u;
  }
  return v;
}

// sum + t^3 of the particle's lanes in lane order (tt = t * t)
template <int G>
__device__ __forceinline__ float sum_lanes(float tt, float t, float sum) {
  if constexpr (G == 1) {
    return fmaf(tt, t, sum);
  } else if constexpr (G == 2) {
    sum = fmaf(lane_bcast<2, 0>(tt), lane_bcast<2, 0>(t), sum);
    return fmaf(lane_bcast<2, 1>(tt), lane_bcast<2, 1>(t), sum);
  } else {
    sum = fmaf(lane_bcast<4, 0>(tt), lane_bcast<4, 0>(t), sum);
    sum = fmaf(lane_bcast<4, 1>(tt), lane_bcast<4, 1>(t), sum);
    sum = fmaf(lane_bcast<4, 2>(tt), lane_bcast<4, 2>(t), sum);
    return fmaf(lane_bcast<4, 3>(tt), lane_bcast<4, 3>(t), sum);
  }
}

// The density sum of one lane and the bits of the walk's current word, the
// first candidate highest.
struct DensAcc {
  fx_float3 p;
  float rd2, d2, sum;
  uint acc;
};

// One candidate a lane; ok: the lanes that have one.  A lane without a pair
// adds +0 (sum unchanged).  v_cndmask and v_addc take the wave's pair mask as
// it is, as in pressure_impl.
template <int G>
__device__ __forceinline__ void dens_cand(DensAcc& D, const TileP q, unsigned long long ok) {
  const float dx = D.p.x - q.x, dy = D.p.y - q.y, dz = D.p.z - q.z;
  const float dsq = fmaf(dz, dz, fmaf(dy, dy, dx * dx));
  const unsigned long long m = __builtin_amdgcn_ballot_w64(dsq < D.rd2) & __builtin_amdgcn_ballot_w64(dsq > 0.0f) & ok;
  const float t0 = (D.rd2 - dsq) * D.d2;
  float t;
  __asm__("v_cndmask_b32_e64 %0, 0, %1, %2" : "=v"(t) : "v"(t0), "s"(m));
  unsigned long long carry;
  uint acc;
  __asm__("v_addc_co_u32_e64 %0, %1, %2, %2, %3" : "=v"(acc), "=s"(carry) : "v"(D.acc), "s"(m));
  D.acc = acc;
  D.sum = sum_lanes<G>(t * t, t, D.sum);
}

// the word of n steps: bit u * G + sub for this lane's step u, all of the
// particle's lanes
template <int G>
__device__ __forceinline__ uint dens_word(uint acc, int n, int sub) {
  return lanes_or<G>(spread_bits<G>(__builtin_bitreverse32(acc << (32 - n))) << sub);
}

template <int G, int SR>
__device__ __forceinline__ void density_wave(const FParams_t& P, const Span S, int N, uint* __restrict__ bits, int cap,
                                             float* lds) {
  constexpr int R = SR * SR;
  const int lane = (int)(threadIdx.x & 63u), sub = lane & (G - 1);
  const int i = S.p0 + (S.blk * (int)blockDim.x + (int)threadIdx.x) / G;
  float* tile = lds + (threadIdx.x >> 6) * (3 * FX_DENS_TILE);
  const fx_float3* __restrict__ pos = pbuf<const fx_float3>(FPnts, FPOS);
  const uint* __restrict__ off = pbuf<const uint>(FAccel, AGRIDOFF);
  const int gc = i < S.p1 ? pbuf<const int>(FPnts, FGCELL)[i] : FX_GRID_UNDEF;
  const bool act = gc != FX_GRID_UNDEF;  // the in-range particles are the scene's first
  const unsigned long long am = __ballot(act);
  if (am == 0ull) return;
  const int lastl = 63 - __clzll((long long)am);
  const int shift = (P.gridRes.z + 1) * P.gridRes.x + 1;
  const size_t NN = (size_t)N;
  const bool rec = act && sub == 0;  // the lane that writes the particle's words
  // Row r: the lane's candidates [jb, jb + len), the wave's run [lo, hi).  A
  // row ends where the cell after its last one begins.  Lanes past the last
  // particle load nothing and read what lane 0 reads.
  int jb[R], len[R], lo[R], hi[R];
  DensAcc D;
  D.p = fx_float3{0.0f, 0.0f, 0.0f};
  D.rd2 = P.rd2;
  D.d2 = P.d2;
  D.sum = 0.0f;
  D.acc = 0u;
#pragma unroll
  for (int r = 0; r < R; r++) jb[r] = len[r] = 0;
  fx_float3 vev = {0.0f, 0.0f, 0.0f};  // of the record written at the end; loaded there it was waited for (beach 194 -> 186 us)
  if (act) {
    D.p = ld3(pos, (size_t)i);
    if (sub == G - 1) vev = ld3nt(pbuf<const fx_float3>(FPnts, FVEVAL), (size_t)i);
#pragma unroll
    for (int r = 0; r < R; r++) {
      const int c0 = gc + P.gridAdj[r * SR] - shift;
      jb[r] = (int)off[c0];
      len[r] = (int)off[c0 + SR];
    }
  }
  int total = 0, longest = 0;
#pragma unroll
  for (int r = 0; r < R; r++) {
    lo[r] = __builtin_amdgcn_readlane(jb[r], 0);
    hi[r] = __builtin_amdgcn_readlane(len[r], lastl);
    len[r] -= jb[r];
    jb[r] = act ? jb[r] : lo[r];
    total += hi[r] - lo[r];
    longest = max(longest, len[r]);
  }
  longest = wave_max(longest);
  // n tile entries, entry k the particle at(k); four loads in flight
  auto stage = [&](int n, auto at) {
    for (int k0 = 0; k0 < n; k0 += 256) {
      fx_float3 q[4];
#pragma unroll
      for (int v = 0; v < 4; v++) q[v] = ld3(pos, (size_t)at(min(k0 + 64 * v + lane, n - 1)));
#pragma unroll
      for (int v = 0; v < 4; v++) {
        const int k = k0 + 64 * v + lane;
        if (k < n) tile_put(tile, k, q[v]);
      }
    }
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront", "local");
  };
  // entry k of the rows [r0, r1) staged one after another
  auto entry = [&](int r0, int r1, int k) {
    int q = lo[r0], e = 0;
#pragma unroll
    for (int r = r0 + 1; r < r1; r++) {
      e += hi[r - 1] - lo[r - 1];
      q = k >= e ? lo[r] - e : q;
    }
    return q + k;
  };
  // a staged row: the lane's candidate s is tile entry a + s, bit s % 32 of
  // word W + s / 32
  auto staged_row = [&](int W, int a, int L, int lm) {
    for (int s0 = 0; s0 < lm; s0 += 32) {
      const int n = (min(32, lm - s0) + G - 1) / G;  // steps
      const int left = L - s0 - sub;                 // step u is this lane's while u * G < left
      D.acc = 0u;
      int u = 0;
      for (; u + 4 <= n; u += 4) {
        TileP q[4];
#pragma unroll
        for (int v = 0; v < 4; v++) q[v] = tile_get(tile, a + s0 + (u + v) * G + sub);
#pragma unroll
        for (int v = 0; v < 4; v++) dens_cand<G>(D, q[v], __builtin_amdgcn_ballot_w64((u + v) * G < left));
      }
      for (; u < n; u++)
        dens_cand<G>(D, tile_get(tile, a + s0 + u * G + sub), __builtin_amdgcn_ballot_w64(u * G < left));
      const uint word = dens_word<G>(D.acc, n, sub);
      const int w = W + (s0 >> 5);
      if (rec && s0 < L && w < cap) bits[(size_t)w * NN + i] = word;
    }
  };
  // a row on its own: the lane walks candidates [ts, te) (see "Row trimming"),
  // those every lane has unchecked; its words carry the phase ts % 32
  const uint* __restrict__ sstart = pbuf<const uint>(FAccel, ASLABSTART);
  int slo = 0, shi = FX_SLABS;
  if (total > FX_DENS_TILE) {
    const float rlim = __fsqrt_rn(D.rd2) * (1.0f + 0x1p-20f);
    const float Rg = rlim * P.gridDelta.x + FX_TRIM_MARGIN + (float)P.gridRes.x * 0x1p-20f;
    const float gp = (D.p.x - P.gridMin.x) * P.gridDelta.x;
    if (act) trim_slabs(gp, (int)gp, SR, Rg, slo, shi);
  }
  auto long_row = [&](int W, int r, int jbr, int L0, int lor, int n) {
    const int nw = (L0 + 31) >> 5;
    int ts = 0, te = L0;
    if (act && sstart != nullptr && L0 > FX_RANK_WAVE) {
      const int c0 = gc + P.gridAdj[r * SR] - shift, c2 = c0 + SR - 1;
      const int n0 = (int)off[c0 + 1] - jbr, n2 = jbr + L0 - (int)off[c2];  // the counts, which may be cleared
      if (n0 > FX_RANK_WAVE && n0 <= FX_RANK_CAP) ts = slab_start(sstart, c0, n0, slo);
      if (n2 > FX_RANK_WAVE && n2 <= FX_RANK_CAP) te = max(ts, te - n2 + slab_start(sstart, c2, n2, shi));
    }
    auto put = [&](int w, uint v) {
      if (rec && W + w < cap) bits[(size_t)(W + w) * NN + i] = v;
    };
    const int L = te - ts, ph = ts & 31;
    const int lm = wave_max(L), lmin = wave_min(act ? L : INT_MAX);
    int a0 = jbr - lor + ts;  // the lane's first candidate in the row's run
    const int amin = wave_min(act ? a0 : INT_MAX), spread = wave_max(act ? a0 : 0) - amin;
    a0 = act ? a0 : amin;
    int w = ts >> 5;
    uint carry = 0u;
    for (int k = 0; k < w; k++) put(k, 0u);
    // steps [sb, se) of the walk, candidate s at fetch(a0 + s), which holds
    // entries up to `last`
    auto part = [&](int sb, int se, int last, auto fetch) {
      for (int s0 = sb; s0 < se; s0 += 32) {
        const int ns = (min(32, se - s0) + G - 1) / G;
        const int nu = max(0, min(ns, (lmin - s0) / G));  // steps with a candidate in every lane
        D.acc = 0u;
        int u = 0;
        for (; u + 4 <= nu; u += 4) {
          TileP q[4];
#pragma unroll
          for (int v = 0; v < 4; v++) q[v] = fetch(a0 + s0 + (u + v) * G + sub);
#pragma unroll
          for (int v = 0; v < 4; v++) dens_cand<G>(D, q[v], ~0ull);
        }
        for (; u < ns; u++) {
          const int s = s0 + u * G + sub;
          dens_cand<G>(D, fetch(min(a0 + s, last)), __builtin_amdgcn_ballot_w64(s < L));
        }
        const uint chunk = dens_word<G>(D.acc, ns, sub);
        if (w < nw) put(w, carry | (chunk << ph));
        carry = ph ? chunk >> (32 - ph) : 0u;
        w++;
      }
    };
    // The lanes' windows start within `spread` entries of each other, so a
    // tile from the first of them serves as many steps as it has entries
    // beyond that; it then slides on.
    const int steps = (FX_DENS_TILE - spread) & ~31;
    if (steps > 0) {
      for (int sb = 0; sb < lm; sb += steps) {
        const int base = amin + sb, m = min(n - base, FX_DENS_TILE);
        stage(m, [&](int k) { return lor + base + k; });
        part(sb, min(lm, sb + steps), base + m - 1, [&](int k) { return tile_get(tile, k - base); });
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront", "local");
      }
    } else {
      part(0, lm, n - 1, [&](int k) {
        const fx_float3 q = ld3(pos, (size_t)(lor + k));
        return TileP{q.x, q.y, q.z};
      });
    }
    if (w < nw) put(w, carry);
    for (int k = w + 1; k < nw; k++) put(k, 0u);
  };
  // reading past a row's end stays within the pad: rows of at most PAD - G
  const bool all = total <= FX_DENS_TILE && longest <= FX_DENS_PAD - G;
  int W = 0, t0 = 0;  // the row's first word and tile entry
#pragma unroll
  for (int r0 = 0; r0 < R; r0 += SR) {  // a layer of the stencil
    int n = 0;
#pragma unroll
    for (int r = r0; r < r0 + SR; r++) n += hi[r] - lo[r];
    if (all || (n <= FX_DENS_TILE && longest <= FX_DENS_PAD - G)) {
      if (!all) {
        t0 = 0;
        stage(n, [&](int k) { return entry(r0, r0 + SR, k); });
      } else if (r0 == 0) {
        stage(total, [&](int k) { return entry(0, R, k); });
      }
#pragma unroll
      for (int r = r0; r < r0 + SR; r++) {
        staged_row(W, t0 + jb[r] - lo[r], len[r], wave_max(len[r]));
        t0 += hi[r] - lo[r];
        W += (len[r] + 31) >> 5;
      }
      __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront", "local");
    } else {
      // one copy of the row's code: the bounds of the layer's rows move down
      int j[SR], m[SR], f[SR], e[SR];
#pragma unroll
      for (int k = 0; k < SR; k++) {
        j[k] = jb[r0 + k];
        m[k] = len[r0 + k];
        f[k] = lo[r0 + k];
        e[k] = hi[r0 + k];
      }
#pragma clang loop unroll(disable)
      for (int k = 0; k < SR; k++) {
        long_row(W, r0 + k, j[0], m[0], f[0], e[0] - f[0]);
        W += (m[0] + 31) >> 5;
#pragma unroll
        for (int q = 0; q < SR - 1; q++) {
          j[q] = j[q + 1];
          m[q] = m[q + 1];
          f[q] = f[q + 1];
          e[q] = e[q + 1];
        }
      }
    }
  }
  if (!act) return;
  float rho = D.sum * P.pmass * P.poly6kern;
  if (rho == 0.0f) rho = 1.0f;
  float4* fr = pbuf<float4>(FAccel, AFREC);
  if (sub == 0) {
    pbuf<float>(FPnts, FPRESS)[i] = rho;
    fr[2 * (size_t)i] = make_float4(D.p.x, D.p.y, D.p.z, rho);
  }
  if (sub == G - 1) {
    fr[2 * (size_t)i + 1] = make_float4(vev.x, vev.y, vev.z, 0.0f);
  }
}

extern __shared__ __align__(16) float dens_lds[];  // FX_DENS_LDS(threads) bytes

template <int G>
__device__ __forceinline__ void density_wave_any(const FParams_t& P, const Span S, int N, uint* bits, int cap) {
  if (P.gridSrch == 3)
    density_wave<G, 3>(P, S, N, bits, cap, dens_lds);
  else
    density_wave<G, 2>(P, S, N, bits, cap, dens_lds);
}

// bits: cap words of bitmask a particle (the system's buffer, or a rollout's tape)
#define FX_DENSITY_WAVE(G, BATCH)                                                                             \
  extern "C" __global__ __launch_bounds__(FX_DENS_THREADS) void computePressureWave##G(                       \
      int pnum, uint* bits, int cap, uint* clear, int nclear) {                                               \
    density_wave_any<G>(*cparams(&FParams), Span{0, pnum, 0, xcd_block()}, pnum, bits, cap);                  \
    if (G > 1) clear_counts(clear, nclear);                                                                   \
  }                                                                                                           \
  extern "C" __global__ __launch_bounds__(FX_DENS_THREADS) BATCH void computePressureWaveBatch##G(            \
      BatchArgs B, int ntotal, uint* bits, int cap, uint* clear, int nclear) {                                \
    const FParams_t* P;                                                                                       \
    const Span S = batch_span(B, xcd_block(), P);                                                             \
    density_wave_any<G>(*P, S, ntotal, bits, cap);                                                            \
    if (G > 1) clear_counts(clear, nclear);                                                                   \
  }
// In a batch the kernels take 73, 81 and 97 registers by themselves, each just
// over a step of the occupancy; they are held at seven, six and five waves a
// SIMD (the first spills two): 64 scenes of 5.3M particles 93.2 -> 92.4 ms for
// 50 steps, 24 of 208,000 101 -> 99 us a step, 16 of 73,000 64.6 -> 63.4.
FX_DENSITY_WAVE(1, __attribute__((amdgpu_waves_per_eu(7))))
FX_DENSITY_WAVE(2, __attribute__((amdgpu_waves_per_eu(6))))
FX_DENSITY_WAVE(4, __attribute__((amdgpu_waves_per_eu(5))))

// ------------------------------------------------------------------- force

// Force (particles.cu:188-225): for 0 < d2 < rd2, r = sqrt(d2 * d2s),
// c = h - r, p = (rho - rho0) * k,
// pterm = (ss * -0.5) * c * spiky * (pi + pj) / r,
// F += (pterm * dist + vterm * (veval_j - veval_i)) * c / (rho_i rho_j).
//
// With the density stage's bitmask the kernel never re-tests candidates.
// Two walks over the bitmask: the word queue further below (blocks of up to
// 256 threads, 2- and 3-cell stencil rows), and the pair ring here (any
// block size and stencil).  The ring: each lane turns the set bits of its
// words into neighbour indices in a per-lane ring in LDS; the wave then
// evaluates queued pairs in batches: a batch takes from every lane as many
// pairs as the shortest active queue holds (more only when a queue must make
// room).  Each lane adds its own pairs in candidate order.  Waves are
// independent: no block-wide barrier.
#define FQ_SLOTS 1024  // ring slots per block (16 per lane at 64 threads)

struct ForceI {
  float px, py, pz, vx, vy, vz;
  float di, pi;
  float fx, fy, fz;
};

// One pair's term, arranged around a single correctly rounded reciprocal:
// with D = rho_i rho_j and inv = 1 / (r D),
//   F += A dist + B (veval_j - veval_i),
//   A = ((ss * -0.5) * spiky) c^2 (p_i + p_j) inv,  B = vterm c r inv,
// which is the reference's (pterm dist + vterm dv) c / D with
// pterm = ss (-0.5) c spiky (p_i + p_j) / r.  The term is split from its
// accumulation so that several pairs' terms can be evaluated before they
// are added in order.
struct PairTerm {
  float A, B, dx, dy, dz, ux, uy, uz;
};

// Near: square root and reciprocal by near_sqrt and near_rcp, their arguments
// ORed into chk (the term holds when chk < FX_NEAR_SPAN).
template <bool Near>
__device__ __forceinline__ PairTerm pair_term(const FParams_t& P, const ForceI& I, const float4 a, const float4 v,
                                              uint& chk) {
  PairTerm q;
  q.dx = I.px - a.x;
  q.dy = I.py - a.y;
  q.dz = I.pz - a.z;
  const float dsq = fmaf(q.dz, q.dz, fmaf(q.dy, q.dy, q.dx * q.dx));
  const float r2 = dsq * P.d2;
  const float rr = Near ? near_sqrt(r2) : sqrtf(r2);
  const float c = P.psmoothradius - rr;
  const float dj = a.w;
  const float pj = (dj - P.prest_dens) * P.pintstiff;
  const float den = rr * (I.di * dj);
  const float inv = Near ? near_rcp(den) : 1.0f / den;
  if (Near) chk |= near_bits(r2) | near_bits(den);
  const float kp = (P.sim_scale * -0.5f) * P.spikykern;
  q.A = (kp * (c * c)) * (I.pi + pj) * inv;
  q.B = (P.vterm * c) * rr * inv;
  q.ux = v.x - I.vx;
  q.uy = v.y - I.vy;
  q.uz = v.z - I.vz;
  return q;
}

__device__ __forceinline__ void pair_add(ForceI& I, const PairTerm& q) {
  I.fx = fmaf(q.A, q.dx, fmaf(q.B, q.ux, I.fx));
  I.fy = fmaf(q.A, q.dy, fmaf(q.B, q.uy, I.fy));
  I.fz = fmaf(q.A, q.dz, fmaf(q.B, q.uz, I.fz));
}

// pair_add when ok, else nothing (a select, no branch)
__device__ __forceinline__ void pair_add_if(ForceI& I, const PairTerm& q, bool ok) {
  const float fx = fmaf(q.A, q.dx, fmaf(q.B, q.ux, I.fx));
  const float fy = fmaf(q.A, q.dy, fmaf(q.B, q.uy, I.fy));
  const float fz = fmaf(q.A, q.dz, fmaf(q.B, q.uz, I.fz));
  I.fx = ok ? fx : I.fx;
  I.fy = ok ? fy : I.fy;
  I.fz = ok ? fz : I.fz;
}

__device__ __forceinline__ void force_pair(const FParams_t& P, ForceI& I, const float4 a, const float4 v) {
  uint chk = 0u;
  pair_add(I, pair_term<false>(P, I, a, v, chk));
}

__device__ __forceinline__ bool is_pair(const FParams_t& P, const ForceI& I, const float4 a) {
  const float dx = I.px - a.x, dy = I.py - a.y, dz = I.pz - a.z;
  const float dsq = fmaf(dz, dz, fmaf(dy, dy, dx * dx));
  return dsq < P.rd2 && dsq > 0.0f;
}

__device__ __forceinline__ void force_impl(const FParams_t& P, const Span S, int N, uint* fq) {
  const int t = threadIdx.x;
  const int i = S.p0 + S.blk * (int)blockDim.x + t;
  const uint* __restrict__ off = pbuf<const uint>(FAccel, AGRIDOFF);
  const uint* __restrict__ cnt = pbuf<const uint>(FAccel, AGRIDCNT);
  const uint* __restrict__ bits = pbuf<const uint>(FAccel, ANBRBITS);
  const float4* __restrict__ fr = pbuf<const float4>(FAccel, AFREC);
  const int srch = P.gridSrch;
  int gc = FX_GRID_UNDEF;
  if (i < S.p1) gc = pbuf<const int>(FPnts, FGCELL)[i];
  const bool act = gc != FX_GRID_UNDEF;
  const int base = stencil_base(P, gc);
  ForceI I;
  I.px = I.py = I.pz = I.vx = I.vy = I.vz = 0.0f;
  I.di = 1.0f;
  I.pi = 0.0f;
  I.fx = I.fy = I.fz = 0.0f;

  if (bits == nullptr || fr == nullptr) {
    // no density-stage records (a host without ANBRBITS/AFREC): test every
    // candidate and evaluate pairs in place
    if (act) {
      const fx_float3* __restrict__ pos = pbuf<const fx_float3>(FPnts, FPOS);
      const fx_float3* __restrict__ vev = pbuf<const fx_float3>(FPnts, FVEVAL);
      const float* __restrict__ rho = pbuf<const float>(FPnts, FPRESS);
      const fx_float3 p = pos[i], v = vev[i];
      I.px = p.x; I.py = p.y; I.pz = p.z;
      I.vx = v.x; I.vy = v.y; I.vz = v.z;
      I.di = rho[i];
      I.pi = (I.di - P.prest_dens) * P.pintstiff;
      for (int r = 0; r < srch * srch; r++) {
        int jb, je;
        row_range(P, base, r, off, cnt, jb, je);
        for (int j = jb; j < je; j++) {
          const fx_float3 q = pos[j], u = vev[j];
          const float4 a = make_float4(q.x, q.y, q.z, rho[j]);
          if (is_pair(P, I, a)) force_pair(P, I, a, make_float4(u.x, u.y, u.z, 0.0f));
        }
      }
      pbuf<fx_float3>(FPnts, FFORCE)[i] = fx_float3{I.fx, I.fy, I.fz};
    }
    return;
  }

  if (act) {
    const float4 a = fr[2 * (size_t)i], v = fr[2 * (size_t)i + 1];
    I.px = a.x; I.py = a.y; I.pz = a.z;
    I.vx = v.x; I.vy = v.y; I.vz = v.z;
    I.di = a.w;
    I.pi = (I.di - P.prest_dens) * P.pintstiff;
  }
  // a particle without recorded bits (too many candidates) tests its own
  const bool ovf = act && nbr_words(P, gc, off, cnt) > nbr_cap();
  if (ovf) {
    for (int r = 0; r < srch * srch; r++) {
      int jb, je;
      row_range(P, base, r, off, cnt, jb, je);
      for (int j = jb; j < je; j++) {
        const float4 a = fr[2 * (size_t)j];
        if (is_pair(P, I, a)) force_pair(P, I, a, fr[2 * (size_t)j + 1]);
      }
    }
  }
  const bool use = act && !ovf;
  const size_t NN = (size_t)N;
  const int fqn = FQ_SLOTS / (int)blockDim.x;  // ring entries per lane
  if (fqn < 16) {
    // blocks too large for a ring that holds a half-word per lane: evaluate
    // each lane's pairs in place
    int W = 0;
    for (int r = 0; r < srch * srch; r++) {
      int jb = 0, je = 0;
      if (use) row_range(P, base, r, off, cnt, jb, je);
      const int nw = (je - jb + 31) >> 5;
      for (int w = 0; w < nw; w++) {
        uint m = bits[(size_t)(W + w) * NN + i];
        while (m != 0u) {
          const uint j = (uint)(jb + (w << 5) + __builtin_ctz(m));
          m &= m - 1u;
          force_pair(P, I, fr[2 * (size_t)j], fr[2 * (size_t)j + 1]);
        }
      }
      W += nw;
    }
    if (act) pbuf<fx_float3>(FPnts, FFORCE)[i] = fx_float3{I.fx, I.fy, I.fz};
    return;
  }
  int head = 0, qn = 0;  // ring holds entries head .. head+qn-1 (mod fqn)
  int W = 0;
  // evaluates the ring's first f entries of every lane (fewer if it holds
  // fewer); a lane whose ring is empty evaluates record 0 and discards the
  // result.
  auto drain = [&](int f) {
#pragma unroll 2
    for (int e = 0; e < f; e++) {
      const bool ok = e < qn;
      const uint j = ok ? fq[head * (int)blockDim.x + t] : 0u;
      const float4 a = fr[2 * (size_t)j], v = fr[2 * (size_t)j + 1];
      ForceI J = I;
      force_pair(P, J, a, v);
      if (ok) {
        I.fx = J.fx;
        I.fy = J.fy;
        I.fz = J.fz;
        head = (head + 1 == fqn) ? 0 : head + 1;
      }
    }
    qn = max(qn - f, 0);
  };
  for (int r = 0; r < srch * srch; r++) {
    int jb = 0, je = 0;
    if (use) row_range(P, base, r, off, cnt, jb, je);
    const int nw = (je - jb + 31) >> 5;
    const int maxw = min(wave_max(nw), FX_NBR_WORDS);
    for (int w = 0; w < maxw; w++) {
      uint word = 0;
      if (w < nw) word = bits[(size_t)(W + w) * NN + i];
      for (int h = 0; h < 32; h += 16) {  // a word in two halves of 16 candidates
        uint m = (word >> h) & 0xffffu;
        const int pc = __popc(m);
        // make room: every lane must fit this half-word's pairs
        if (__any(qn + pc > fqn)) {
          const int need = wave_max(qn + pc - fqn);
          drain(min(max(need, wave_min(use ? qn : 0x7fffffff)), fqn));
        }
        int tail = head + qn;
        if (tail >= fqn) tail -= fqn;
        while (m != 0u) {
          const int b = __builtin_ctz(m);
          m &= m - 1u;
          fq[tail * (int)blockDim.x + t] = (uint)(jb + (w << 5) + h + b);
          tail = (tail + 1 == fqn) ? 0 : tail + 1;
          qn++;
        }
      }
    }
    W += nw;
  }
  drain(min(wave_max(qn), fqn));
  if (act) pbuf<fx_float3>(FPnts, FFORCE)[i] = fx_float3{I.fx, I.fy, I.fz};
}

#ifndef FW_AHEAD
#define FW_AHEAD 4  // bitmask words loaded ahead of their use
#endif

// Word-queue force.  Each lane reads its bitmask words as one stream (row
// r's words follow row r-1's) and queues every non-zero word whole, with the
// record index of its bit 0: two words in registers, up to K more in LDS.
// The wave then evaluates pairs in batches: a batch takes the same number of
// pairs from every lane (as many as the shortest queue holds, more only when
// a queue must make room), each lane's pairs in candidate order, FW_STEP
// pairs' terms evaluated at a time.  Queuing words instead of pairs costs one LDS
// write per word, and a deep queue of words keeps nearly every lane busy in
// the batches, so nearly every pair gather carries a pair.
#ifndef FW_STEP
#define FW_STEP 3  // pair terms evaluated per drain step
#endif
#ifndef FW_QBYTES
#define FW_QBYTES 16384  // LDS queue per block: (word, base) pairs, 4 words per lane at 512 threads
#endif

template <int R, int S>
__device__ __forceinline__ void force_walk_q(const FParams_t& P, ForceI& I, const uint* __restrict__ bits,
                                             size_t NN, int i, int nwords, int (&E_)[R], int (&G)[R], uint* Qw,
                                             uint* Qb, int K, const float4* srcA, const float4* srcV, bool use) {
  const int t = threadIdx.x, nt = blockDim.x;
  uint cur = 0u, nxt = 0u;  // current word (bits not yet taken) and the next one
  int curb = 0, nxtb = 0;   // their bases
  int qh = 0, qc = 0;       // LDS queue head and length
  int qn = 0;               // pairs held
  // the lane's next pair, in candidate order; false when it holds none
  auto take = [&](uint& j) -> bool {
    const bool ok = cur != 0u;
    j = ok ? (uint)(curb + __builtin_ctz(cur)) : 0u;
    cur &= cur - 1u;
    if (ok && cur == 0u) {
      cur = nxt;
      curb = nxtb;
      nxt = 0u;
      if (qc > 0) {
        nxt = Qw[qh * nt + t];
        nxtb = (int)Qb[qh * nt + t];
        qh = (qh + 1 == K) ? 0 : qh + 1;
        qc--;
      }
    }
    return ok;
  };
  // f pairs from every lane (a lane that runs out evaluates record 0 and
  // discards it), FW_STEP pair terms evaluated at a time and added in order
  auto drain = [&](int f) {
    int e = 0;
    for (; e + FW_STEP <= f; e += FW_STEP) {
      uint j[FW_STEP];
      bool ok[FW_STEP];
      PairTerm q[FW_STEP];
      uint chk = 0u;
#pragma unroll
      for (int u = 0; u < FW_STEP; u++) ok[u] = take(j[u]);
#pragma unroll
      for (int u = 0; u < FW_STEP; u++)
        q[u] = pair_term<false>(P, I, srcA[S * (size_t)j[u]], srcV[S * (size_t)j[u]], chk);
#pragma unroll
      for (int u = 0; u < FW_STEP; u++) pair_add_if(I, q[u], ok[u]);
    }
    for (; e < f; e++) {
      uint j, chk = 0u;
      const bool ok = take(j);
      pair_add_if(I, pair_term<false>(P, I, srcA[S * (size_t)j], srcV[S * (size_t)j], chk), ok);
    }
    qn = max(qn - f, 0);
  };
  const int maxf = wave_max(nwords);
  // The bitmask is read once, as a stream: non-temporal loads keep it from
  // displacing the neighbour records in L1 and L2 (force 3.81 -> 3.79 ms per
  // launch over 200 dam-break steps, 0.470 -> 0.451 ms at the 4M beach scene).
  // Non-temporal stores in the density stage measured slower (3.85 ms).
  uint nx4[FW_AHEAD];
#pragma unroll
  for (int k = 0; k < FW_AHEAD; k++) nx4[k] = k < nwords ? __builtin_nontemporal_load(&bits[(size_t)k * NN + i]) : 0u;
  for (int f0 = 0; f0 < maxf; f0 += FW_AHEAD) {
    uint cw[FW_AHEAD];
#pragma unroll
    for (int k = 0; k < FW_AHEAD; k++) {
      cw[k] = nx4[k];
      const int fn = f0 + FW_AHEAD + k;
      nx4[k] = fn < nwords ? __builtin_nontemporal_load(&bits[(size_t)fn * NN + i]) : 0u;
    }
#pragma unroll
    for (int k = 0; k < FW_AHEAD; k++) {
      const int f = f0 + k;
      if (f >= maxf) break;
      const uint word = cw[k];
      if (word != 0u) {
        while (f >= E_[0]) {  // move to the row holding word f
#pragma unroll
          for (int r = 0; r < R - 1; r++) {
            E_[r] = E_[r + 1];
            G[r] = G[r + 1];
          }
          E_[R - 1] = INT_MAX;
        }
      }
      const int held = (cur != 0u ? 1 : 0) + (nxt != 0u ? 1 : 0) + qc;
      const bool full = word != 0u && held == K + 2;
      if (__any(full)) {  // free a word slot: the full lanes finish their current word
        const int need = wave_max(full ? __popc(cur) : 0);
        drain(max(need, wave_min(use ? qn : 0x7fffffff)));
      }
      if (word != 0u) {
        const int base = G[0] + (f << 5);
        if (cur == 0u) {
          cur = word;
          curb = base;
        } else if (nxt == 0u) {
          nxt = word;
          nxtb = base;
        } else {
          int tl = qh + qc;
          if (tl >= K) tl -= K;
          Qw[tl * nt + t] = word;
          Qb[tl * nt + t] = (uint)base;
          qc++;
        }
        qn += __popc(word);
      }
    }
  }
  drain(wave_max(qn));
}

template <int SR>
__device__ __forceinline__ void force_q_impl(const FParams_t& P, const Span S, int N, uint* lq) {
  constexpr int R = SR * SR;
  const int t = threadIdx.x, nt = blockDim.x;
  const int i = S.p0 + S.blk * nt + t;
  const uint* __restrict__ off = pbuf<const uint>(FAccel, AGRIDOFF);
  const uint* __restrict__ cnt = pbuf<const uint>(FAccel, AGRIDCNT);
  const uint* __restrict__ bits = pbuf<const uint>(FAccel, ANBRBITS);
  const float4* __restrict__ fr = pbuf<const float4>(FAccel, AFREC);
  int gc = FX_GRID_UNDEF;
  if (i < S.p1) gc = pbuf<const int>(FPnts, FGCELL)[i];
  const bool act = gc != FX_GRID_UNDEF;
  const int shift = (P.gridRes.z + 1) * P.gridRes.x + 1;
  ForceI I;
  I.px = I.py = I.pz = I.vx = I.vy = I.vz = 0.0f;
  I.di = 1.0f;
  I.pi = 0.0f;
  I.fx = I.fy = I.fz = 0.0f;
  // the lane's row windows: row r covers words [W_r, W_{r+1}) of its bitmask;
  // E_[r] = W_{r+1}, and the record of word f, bit b is G[r] + 32 f + b
  int E_[R], G[R];
  int nwords = 0;
  if (act) {
#pragma unroll
    for (int r = 0; r < R; r++) {
      const int c0 = gc + P.gridAdj[r * SR] - shift;
      const int jb = (int)off[c0], je = (int)off[c0 + SR];
      G[r] = jb - (nwords << 5);
      nwords += (je - jb + 31) >> 5;
      E_[r] = nwords;
    }
    const float4 a = fr[2 * (size_t)i], v = fr[2 * (size_t)i + 1];
    I.px = a.x; I.py = a.y; I.pz = a.z;
    I.vx = v.x; I.vy = v.y; I.vz = v.z;
    I.di = a.w;
    I.pi = (I.di - P.prest_dens) * P.pintstiff;
  } else {
#pragma unroll
    for (int r = 0; r < R; r++) E_[r] = G[r] = 0;
  }
  const bool ovf = act && nwords > nbr_cap();
  if (ovf) {  // no recorded bits: test every candidate
    const int base = stencil_base(P, gc);
    for (int r = 0; r < R; r++) {
      int jb, je;
      row_range(P, base, r, off, cnt, jb, je);
      for (int j = jb; j < je; j++) {
        const float4 a = fr[2 * (size_t)j];
        if (is_pair(P, I, a)) force_pair(P, I, a, fr[2 * (size_t)j + 1]);
      }
    }
  }
  const bool use = act && !ovf;
  const int K = min(FW_QBYTES / (8 * nt), 16);
  force_walk_q<R, 2>(P, I, bits, (size_t)N, i, use ? nwords : 0, E_, G, lq, lq + K * nt, K, fr, fr + 1, use);
  if (act) pbuf<fx_float3>(FPnts, FFORCE)[i] = fx_float3{I.fx, I.fy, I.fz};
}

// Dispatch: the word queue needs the density stage's records and at least
// 4 LDS words per lane (blocks of up to 512 threads, the reference's launch
// geometry); otherwise the ring or candidate-testing pass.
__device__ __forceinline__ void force_q(const FParams_t& P, const Span S, int N, uint* lq) {
  if (FAccel.mbuf[ANBRBITS] == 0 || FAccel.mbuf[AFREC] == 0 || FW_QBYTES / (8 * (int)blockDim.x) < 4 ||
      P.gridSrch > 3) {
    force_impl(P, S, N, lq);
    return;
  }
  if (P.gridSrch == 3)
    force_q_impl<3>(P, S, N, lq);
  else
    force_q_impl<2>(P, S, N, lq);
}

extern "C" __global__ __launch_bounds__(1024) void computeForce(int pnum) {
  __shared__ uint lq[FW_QBYTES / 4];
  force_q(*cparams(&FParams), Span{0, pnum, 0, xcd_block()}, pnum, lq);
}

extern "C" __global__ __launch_bounds__(1024) void computeForceBatch(BatchArgs B, int ntotal) {
  __shared__ uint lq[FW_QBYTES / 4];
  const FParams_t* P;
  const Span S = batch_span(B, xcd_block(), P);
  force_q(*P, S, ntotal, lq);
}

// The persistent loop costs the kernel registers (101 VGPRs, 4 waves per
// SIMD); held at the one-block-per-entry kernel's 5 waves (96, no spills).
extern "C" __global__ __launch_bounds__(1024) __attribute__((amdgpu_waves_per_eu(5))) void computeForceBatchP(
    BatchArgs B, int ntotal) {
  __shared__ uint lq[FW_QBYTES / 4];
  batch_items(B, [&](int b) {
    const FParams_t* P;
    const Span S = batch_span(B, b, P);
    force_q(*P, S, ntotal, lq);
  });
}

// ------------------------------------------------------ the step's last pass
//
// When another step follows, the force launch also advances its particles and
// makes the next step's insert (and, in a recorded step of a rollout, writes
// the particles as they are before the advance to the tape): a particle's
// position and evaluation velocity are at hand as its pair record, its force
// need not be read back, and the passes' traffic lies beside other
// waves' pair arithmetic.  Neighbours are read from the records and the
// offsets only, which neither changes; the counts were cleared before
// (clear_counts).  What this pass writes is not read before the next launch and is
// stored non-temporally, so that it does not displace the records (4M
// particles on the beach, a step from step 20 751 -> 721 us, from step 80
// 1143 -> 1109).  Against passes of their own for the advance with the insert
// (which took 75 us of 1034 at the beach): 43.2 -> 39.9 us a step at 16,384
// particles, 110 -> 105 at 262,144, 214 -> 210 at 1,000,000, at the 4M beach
// 731 -> 721 and 1115 -> 1109.

// a tape slot, in the layout of adjTapeRecord: pos, vel, veval, force (12 B
// each), rho, the sort's permutation, cell (4 B each), then the cell offsets
struct TapeDst {
  char* dst;
  const uint* src;  // the sort's permutation
  int n;
  int cells;
};

// what follows the forces: nothing (0), the advance and the next insert (1),
// the tape before them (2); dt and scale of a batch are its scenes'
struct FxNext {
  int mode;
  float time, dt, ss;
  const float* clock;
  TapeDst tape;
};

__device__ __forceinline__ void tape_store(const TapeDst& T, int i, bool own) {
  const size_t N = (size_t)T.n;
  if (own) {
    const fx_float3 x = ld3(pbuf<const fx_float3>(FPnts, FPOS), (size_t)i);
    const fx_float3 v = ld3(pbuf<const fx_float3>(FPnts, FVEL), (size_t)i);
    const fx_float3 e = ld3(pbuf<const fx_float3>(FPnts, FVEVAL), (size_t)i);
    const fx_float3 f = ld3(pbuf<const fx_float3>(FPnts, FFORCE), (size_t)i);
    st3(reinterpret_cast<fx_float3*>(T.dst), (size_t)i, x.x, x.y, x.z);
    st3(reinterpret_cast<fx_float3*>(T.dst + 12 * N), (size_t)i, v.x, v.y, v.z);
    st3(reinterpret_cast<fx_float3*>(T.dst + 24 * N), (size_t)i, e.x, e.y, e.z);
    st3(reinterpret_cast<fx_float3*>(T.dst + 36 * N), (size_t)i, f.x, f.y, f.z);
    uint* w = reinterpret_cast<uint*>(T.dst + 48 * N);
    w[i] = __float_as_uint(pbuf<const float>(FPnts, FPRESS)[i]);
    w[N + i] = T.src[i];
    w[2 * N + i] = pbuf<const uint>(FPnts, FGCELL)[i];
  }
  const uint* __restrict__ off = pbuf<const uint>(FAccel, AGRIDOFF);
  uint* o = reinterpret_cast<uint*>(T.dst + 60 * N);
  for (int k = (int)(blockIdx.x * blockDim.x + threadIdx.x); k < T.cells; k += (int)(gridDim.x * blockDim.x)) o[k] = off[k];
}

template <bool Nt>
__device__ __forceinline__ fx_float3 advance_from(const FParams_t& P, int i, const fx_float3 pos, fx_float3 vel,
                                                  const fx_float3 ve, const fx_float3 f, float time, float dt,
                                                  float ss);
__device__ __forceinline__ fx_float3 park(int i);

// Every thread of the block calls it; own: the lane writes particle i, in
// cell gc, with the forces in I.  lds: 34 words of the block's LDS.
__device__ __forceinline__ void force_end(const FParams_t& P, const Span S, int i, bool own, int gc, const ForceI& I,
                                          const FxNext& X, float dt, float ss, uint* lds) {
  const bool act = own && gc != FX_GRID_UNDEF;
  // (stored in every step: a slot whose particle leaves the grid keeps its last force)
  if (act) {
    if (X.mode == 1)
      put3<true>(pbuf<fx_float3>(FPnts, FFORCE), (size_t)i, I.fx, I.fy, I.fz);
    else
      st3(pbuf<fx_float3>(FPnts, FFORCE), (size_t)i, I.fx, I.fy, I.fz);
  }
  if (X.mode == 0) return;
  if (X.mode == 2) tape_store(X.tape, i, own);
  fx_float3 x = fx_float3{0.0f, 0.0f, 0.0f};
  if (act) {
    x = advance_from<true>(P, i, fx_float3{I.px, I.py, I.pz}, ld3nt(pbuf<const fx_float3>(FPnts, FVEL), (size_t)i),
                           fx_float3{I.vx, I.vy, I.vz}, fx_float3{I.fx, I.fy, I.fz},
                           X.clock != nullptr ? X.clock[0] : X.time, dt, ss);
  } else if (own) {
    x = park(i);
  }
  lds_barrier();  // the waves' queues in the block's LDS are done with
  insert_at<true>(P, S, i, own, x, true, reinterpret_cast<uint(*)[17]>(lds));
}

// ----------------------------------------------------------- force by wave
//
// The library's own force stage (stencil rows of 2 or 3 cells): the word
// queue above with three costs taken out.
//
// Gathers.  A wave's 64 scattered 16-byte loads take 37 cycles of a CU's
// texture path whatever their width, 21 when neighbouring lanes read the two
// halves of one record (16 when four lanes share a 128-byte line; measured on
// records in L1).  So lanes 2k and 2k + 1 read both halves of the even lane's
// record together, then both halves of the odd lane's, and exchange what is
// the other's: seven v_cndmask with a DPP source a pair, written as asm (the
// compiler makes a move and a select of each).
//
// Queue.  All words but the current one lie in LDS, and the two that follow
// it are read a step ahead, so that a lane that finishes a word waits for
// nothing; the queue above read the next word when it was needed, inside a
// branch, up to three times a step.
//
// Terms.  Square root and reciprocal by near_sqrt and near_rcp (8
// instructions instead of 27), with one check for the FQ_STEP terms of a
// step; a step with an argument outside their range is evaluated again with
// the IEEE sequences.  The bits are the same.
//
// Force per launch, queue above / here (us, HIP events around the stage):
// the compressed 4M dam break from step 5 1950 / 1640, from step 60
// 4800 / 4110; the 4M beach from step 20 285 / 260, from step 90 765 / 687;
// at rest density 1,000,000 at step 40 88 / 77, at step 140 218 / 184,
// 262,144 at step 90 92 / 78, 65,536 at step 40 44 / 34.  FQ_STEP 2 / 3 / 4 /
// 5 gave 1708 / 1632 / 1640 / 1727, 4586 / 4287 / 4160 / 4255 and
// 290 / 267 / 261 / 284 us on the first three; 8 instead of 16 queued words
// 1857, 4830 and 284 (at FQ_STEP 3).  118 VGPRs, four waves a SIMD; held at
// 96 it spills (2250 us).  The texture path of the gathers (busy for 0.93 to
// 0.97 of the cycles) and VALU issue (about 52 instructions a pair and lane;
// 0.22 to 0.29 a cycle and SIMD, where FMAs alone reach 0.21 and two-operand
// instructions 0.40) bound it together.
#define FQ_STEP 4 // pairs a lane and step

template <int SR>
__device__ __forceinline__ void force_wave(const FParams_t& P, int i, int gc, int N, const uint* __restrict__ bits,
                                           int cap, uint* lds, ForceI& I) {
  constexpr int R = SR * SR;
  const int lane = (int)(threadIdx.x & 63u);
  const bool odd = (lane & 1) != 0;
  uint* q = lds + (threadIdx.x >> 6) * (2 * FX_WALK_K * 64) + lane;
  const uint* __restrict__ off = pbuf<const uint>(FAccel, AGRIDOFF);
  const float4* __restrict__ fr = pbuf<const float4>(FAccel, AFREC);
  const float4* __restrict__ half = fr + (odd ? 1 : 0);  // the half of a record this lane reads
  const bool act = gc != FX_GRID_UNDEF;
  if (__ballot(act) == 0ull) return;
  const int shift = (P.gridRes.z + 1) * P.gridRes.x + 1;
  // row r: candidates from jb[r], words [E_[r - 1], E_[r]) of the bitmask
  int jb[R], E_[R];
#pragma unroll
  for (int r = 0; r < R; r++) jb[r] = E_[r] = 0;
  if (act) {
#pragma unroll
    for (int r = 0; r < R; r++) {
      const int c0 = gc + P.gridAdj[r * SR] - shift;
      jb[r] = (int)off[c0];
      E_[r] = (int)off[c0 + SR];
    }
    const float4 a = fr[2 * (size_t)i], v = fr[2 * (size_t)i + 1];
    I.px = a.x; I.py = a.y; I.pz = a.z;
    I.vx = v.x; I.vy = v.y; I.vz = v.z;
    I.di = a.w;
    I.pi = (I.di - P.prest_dens) * P.pintstiff;
  }
  int nwords = 0, longest = 0;
#pragma unroll
  for (int r = 0; r < R; r++) {
    const int len = E_[r] - jb[r];
    longest = max(longest, len);
    nwords += (len + 31) >> 5;
    E_[r] = nwords;
  }
  if (act && nwords > cap) {  // no recorded bits: test every candidate
    const int base = stencil_base(P, gc);
    for (int r = 0; r < R; r++) {
      int b, e;
      row_range(P, base, r, off, off, b, e);  // from the offsets alone: the counts may be cleared
      for (int j = b; j < e; j++) {
        const float4 a = fr[2 * (size_t)j];
        if (is_pair(P, I, a)) force_pair(P, I, a, fr[2 * (size_t)j + 1]);
      }
    }
    nwords = 0;
#pragma unroll
    for (int r = 0; r < R; r++) E_[r] = 0;
  }
  word_walk<R, 2, FQ_STEP>(bits, (size_t)N, i, nwords, longest, jb, E_, q, [&](const uint (&j)[FQ_STEP], const bool (&ok)[FQ_STEP]) __attribute__((always_inline)) {
    float4 e[FQ_STEP], o[FQ_STEP];  // this lane's half of the even lane's record, and of the odd lane's
#pragma unroll
    for (int u = 0; u < FQ_STEP; u++) {
      const uint jx = lane_other(j[u]);
      e[u] = half[odd ? jx : j[u]];
      o[u] = half[odd ? j[u] : jx];
    }
    PairTerm t[FQ_STEP];
    float4 a[FQ_STEP];
    uint chk = 0u;
#pragma unroll
    for (int u = 0; u < FQ_STEP; u++) {
      swap_halves(e[u], o[u], a[u]);
      t[u] = pair_term<true>(P, I, a[u], o[u], chk);
    }
    if (__any(chk >= FX_NEAR_SPAN)) {
#pragma unroll
      for (int u = 0; u < FQ_STEP; u++) t[u] = pair_term<false>(P, I, a[u], o[u], chk);
    }
    bool every = true;
#pragma unroll
    for (int u = 0; u < FQ_STEP; u++) every = every && ok[u];
    if (__all(every)) {
#pragma unroll
      for (int u = 0; u < FQ_STEP; u++) pair_add(I, t[u]);
    } else {
#pragma unroll
      for (int u = 0; u < FQ_STEP; u++) pair_add_if(I, t[u], ok[u]);
    }
  });
}

extern __shared__ uint force_lds[];  // FX_FORCE_LDS(threads) bytes

__device__ __forceinline__ ForceI no_force() {
  ForceI I;
  I.px = I.py = I.pz = I.vx = I.vy = I.vz = 0.0f;
  I.di = 1.0f;
  I.pi = 0.0f;
  I.fx = I.fy = I.fz = 0.0f;
  return I;
}

__device__ __forceinline__ void force_wave_any(const FParams_t& P, const Span S, int N, const uint* bits, int cap,
                                               const FxNext& X, float dt, float ss) {
  const int i = S.p0 + S.blk * (int)blockDim.x + (int)threadIdx.x;
  const int gc = i < S.p1 ? pbuf<const int>(FPnts, FGCELL)[i] : FX_GRID_UNDEF;
  ForceI I = no_force();
  if (P.gridSrch == 3)
    force_wave<3>(P, i, gc, N, bits, cap, force_lds, I);
  else
    force_wave<2>(P, i, gc, N, bits, cap, force_lds, I);
  force_end(P, S, i, i < S.p1, gc, I, X, dt, ss, force_lds);
}

// Bounds of 1024 threads, twice what is launched, keep the compiler's schedule
// at four waves a SIMD: 280 instead of 260 us on the beach with 512.
extern "C" __global__ __launch_bounds__(1024) void computeForceWave(int pnum, const uint* bits, int cap, FxNext X) {
  force_wave_any(*cparams(&FParams), Span{0, pnum, 0, xcd_block()}, pnum, bits, cap, X, X.dt, X.ss);
}

extern "C" __global__ __launch_bounds__(1024) void computeForceWaveBatch(BatchArgs B, int ntotal, const uint* bits,
                                                                                int cap, FxNext X) {
  const FParams_t* P;
  const Span S = batch_span(B, xcd_block(), P);
  force_wave_any(*P, S, ntotal, bits, cap, X, P->dt, P->sim_scale);
}

// Four lanes to a particle, for launches of few waves: those wait for the
// chain of their busiest lane (a step's gathers, then its terms, some 20
// times over), and a quarter of the pairs a lane shortens it.  The wave turns
// the words of its 16 particles into a list of neighbours each, in candidate
// order; a particle's lanes evaluate four entries at a time and add the
// terms in order through DPP broadcasts, so the sums are the same bits.  Per
// stage, one lane / four (us, HIP events around it): 16,384 compressed
// 22.0 / 14.3; at rest density 16,384 21.6 / 14.2, 65,537 from step 10
// 22.8 / 19.1 and from step 80 24.3 / 20.2, 100,000 23.3 / 25.3, 131,072
// 23.7 / 28.9.  1 / 2 / 3 / 4 entries a lane and step gave 15.5 / 14.2 /
// 14.3 / 14.5 at 16,384 and 19.3 / 19.1 / 19.1 / 20.1 at 65,537.
#define FL_CAP 128  // list entries of a particle: the pairs of four words
#define FL_STEP 2   // entries a lane and step

// I + the terms of the particle's first nv lanes, in lane order
__device__ __forceinline__ void add_lanes(ForceI& I, const PairTerm& q, int nv) {
  auto one = [&](auto kk) __attribute__((always_inline)) {
    constexpr int K = decltype(kk)::value;
    if (K < nv) {  // the same for the four lanes
      const float A = lane_bcast<4, K>(q.A), B = lane_bcast<4, K>(q.B);
      I.fx = fmaf(A, lane_bcast<4, K>(q.dx), fmaf(B, lane_bcast<4, K>(q.ux), I.fx));
      I.fy = fmaf(A, lane_bcast<4, K>(q.dy), fmaf(B, lane_bcast<4, K>(q.uy), I.fy));
      I.fz = fmaf(A, lane_bcast<4, K>(q.dz), fmaf(B, lane_bcast<4, K>(q.uz), I.fz));
    }
  };
  one(std::integral_constant<int, 0>());
  one(std::integral_constant<int, 1>());
  one(std::integral_constant<int, 2>());
  one(std::integral_constant<int, 3>());
}

template <int SR>
__device__ __forceinline__ void force_lists(const FParams_t& P, int i, int gc, bool in, int N,
                                            const uint* __restrict__ bits, int cap, uint* lds, ForceI& I) {
  constexpr int G = 4, R = SR * SR;
  const int lane = (int)(threadIdx.x & 63u), sub = lane & (G - 1);
  // the particle's list; strides of 4 mod 32 words keep the lists of a wave in different banks
  uint* list = lds + ((threadIdx.x >> 6) * (64 / G) + lane / G) * (FL_CAP + G);
  const uint* __restrict__ off = pbuf<const uint>(FAccel, AGRIDOFF);
  const float4* __restrict__ fr = pbuf<const float4>(FAccel, AFREC);
  // The lane's first three words, beside the cell and before it is known how
  // many the particle has (the buffer holds cap words of every particle):
  // 19.2 -> 18.8 us at 65,537 particles.
  uint w0 = 0u, w1 = 0u, w2 = 0u;
  if (in) {
    const size_t NN = (size_t)N;
    if (sub < cap) w0 = __builtin_nontemporal_load(&bits[(size_t)sub * NN + i]);
    if (sub + G < cap) w1 = __builtin_nontemporal_load(&bits[(size_t)(sub + G) * NN + i]);
    if (sub + 2 * G < cap) w2 = __builtin_nontemporal_load(&bits[(size_t)(sub + 2 * G) * NN + i]);
  }
  const bool act = gc != FX_GRID_UNDEF;
  if (__ballot(act) == 0ull) return;
  const int shift = (P.gridRes.z + 1) * P.gridRes.x + 1;
  // words [E_[r - 1], E_[r]) of the bitmask are row r's; bit 0 of word f is candidate B_[r] + 32 f
  int E_[R], B_[R];
#pragma unroll
  for (int r = 0; r < R; r++) E_[r] = B_[r] = 0;
  int nwords = 0;
  if (act) {
#pragma unroll
    for (int r = 0; r < R; r++) {
      const int c0 = gc + P.gridAdj[r * SR] - shift;
      B_[r] = (int)off[c0];
      E_[r] = (int)off[c0 + SR];
    }
    const float4 a = fr[2 * (size_t)i], v = fr[2 * (size_t)i + 1];
    I.px = a.x; I.py = a.y; I.pz = a.z;
    I.vx = v.x; I.vy = v.y; I.vz = v.z;
    I.di = a.w;
    I.pi = (I.di - P.prest_dens) * P.pintstiff;
  }
#pragma unroll
  for (int r = 0; r < R; r++) {
    const int nw = (E_[r] - B_[r] + 31) >> 5;
    B_[r] -= nwords << 5;
    nwords += nw;
    E_[r] = nwords;
  }
  if (act && nwords > cap) {  // no recorded bits: test every candidate
    const int base = stencil_base(P, gc);
    for (int r = 0; r < R; r++) {
      int b, e;
      row_range(P, base, r, off, off, b, e);
      for (int j = b; j < e; j++) {
        const float4 a = fr[2 * (size_t)j];
        if (is_pair(P, I, a)) force_pair(P, I, a, fr[2 * (size_t)j + 1]);
      }
    }
    nwords = 0;
  }
  const size_t NN = (size_t)N;
  int head = 0, qn = 0;  // the list holds entries head .. head + qn - 1 (mod FL_CAP)
  // G * U entries of the list, the last of them repeated beyond nv
  auto take = [&](auto uu, int nv) __attribute__((always_inline)) {
    constexpr int U = decltype(uu)::value;
    float4 a[U], v[U];
#pragma unroll
    for (int u = 0; u < U; u++) {
      const size_t j = 2 * (size_t)list[(head + min(u * G + sub, nv - 1)) & (FL_CAP - 1)];
      a[u] = fr[j];
      v[u] = fr[j + 1];
    }
    PairTerm q[U];
    uint chk = 0u;
#pragma unroll
    for (int u = 0; u < U; u++) q[u] = pair_term<true>(P, I, a[u], v[u], chk);
    if (__any(chk >= FX_NEAR_SPAN)) {
#pragma unroll
      for (int u = 0; u < U; u++) q[u] = pair_term<false>(P, I, a[u], v[u], chk);
    }
#pragma unroll
    for (int u = 0; u < U; u++) add_lanes(I, q[u], nv - u * G);
    head += nv;
    qn -= nv;
  };
  // down to fewer than G entries a list, and those too if `all`
  auto drain = [&](bool all) __attribute__((always_inline)) {
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront", "local");  // other lanes' list entries
    while (qn >= G * FL_STEP) take(std::integral_constant<int, FL_STEP>(), G * FL_STEP);
    while (qn >= G || (all && qn > 0)) take(std::integral_constant<int, 1>(), min(qn, G));
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront", "local");
  };
  const int maxf = wave_max(nwords);
  for (int f0 = 0; f0 < maxf; f0 += G) {  // a word a lane
    const int f = f0 + sub;
    uint m = f < nwords ? w0 : 0u;
    w0 = w1;
    w1 = w2;
    w2 = f + 3 * G < nwords ? __builtin_nontemporal_load(&bits[(size_t)(f + 3 * G) * NN + i]) : 0u;
    int base = B_[0];
#pragma unroll
    for (int r = 1; r < R; r++) base = f >= E_[r - 1] ? B_[r] : base;
    base += f << 5;
    const int pc = __popc(m);
    // pairs in the words of the lanes up to this one, and of all four
    const int p1 = (int)__builtin_amdgcn_update_dpp(0, pc, 0x90, 0xf, 0xf, true);  // quad_perm 0,0,1,2
    int pre = pc + (sub >= 1 ? p1 : 0);
    const int p2 = (int)__builtin_amdgcn_update_dpp(0, pre, 0x40, 0xf, 0xf, true);  // quad_perm 0,0,0,1
    pre += sub >= 2 ? p2 : 0;
    const int tot = (int)__builtin_amdgcn_update_dpp(0, pre, 0xFF, 0xf, 0xf, true);  // quad_perm 3,3,3,3
    if (__any(qn + tot > FL_CAP)) drain(false);
    if (__any(qn + tot > FL_CAP)) drain(true);  // fewer than G held and four full words coming
    int tail = head + qn + pre - pc;
    while (m != 0u) {
      list[tail & (FL_CAP - 1)] = (uint)(base + __builtin_ctz(m));
      m &= m - 1u;
      tail++;
    }
    qn += tot;
  }
  drain(true);
}

__device__ __forceinline__ void force_lists_any(const FParams_t& P, const Span S, int N, const uint* bits, int cap,
                                                const FxNext& X, float dt, float ss) {
  const int i = S.p0 + (S.blk * (int)blockDim.x + (int)threadIdx.x) / 4;
  const int gc = i < S.p1 ? pbuf<const int>(FPnts, FGCELL)[i] : FX_GRID_UNDEF;
  ForceI I = no_force();
  if (P.gridSrch == 3)
    force_lists<3>(P, i, gc, i < S.p1, N, bits, cap, force_lds, I);
  else
    force_lists<2>(P, i, gc, i < S.p1, N, bits, cap, force_lds, I);
  force_end(P, S, i, i < S.p1 && (threadIdx.x & 3u) == 0u, gc, I, X, dt, ss, force_lds);
}

extern "C" __global__ __launch_bounds__(FX_FORCE4_THREADS) void computeForceWave4(int pnum, const uint* bits, int cap,
                                                                                 FxNext X) {
  force_lists_any(*cparams(&FParams), Span{0, pnum, 0, xcd_block()}, pnum, bits, cap, X, X.dt, X.ss);
}

extern "C" __global__ __launch_bounds__(FX_FORCE4_THREADS) void computeForceWaveBatch4(BatchArgs B, int ntotal,
                                                                                      const uint* bits, int cap,
                                                                                      FxNext X) {
  const FParams_t* P;
  const Span S = batch_span(B, xcd_block(), P);
  force_lists_any(*P, S, ntotal, bits, cap, X, P->dt, P->sim_scale);
}

// ------------------------------------------------------ neighbour statistics

// The largest number of bitmask words any in-range particle's stencil needs,
// on a state whose counts and offsets are current (after insert and scan; the
// particles need not be sorted): out[0] = max.  Sizes the reverse mode's tape.
__device__ __forceinline__ void max_words_impl(const FParams_t& P, const Span S, uint* out) {
  const int i = S.p0 + S.blk * (int)blockDim.x + (int)threadIdx.x;
  if (i >= S.p1) return;
  const int gc = pbuf<const int>(FPnts, FGCELL)[i];
  if (gc == FX_GRID_UNDEF) return;
  const int w = nbr_words(P, gc, pbuf<const uint>(FAccel, AGRIDOFF), pbuf<const uint>(FAccel, AGRIDCNT));
  atomicMax(out, (uint)w);
}

extern "C" __global__ void fxMaxWords(uint* out, int pnum) {
  max_words_impl(*cparams(&FParams), Span{0, pnum, 0, (int)blockIdx.x}, out);
}

extern "C" __global__ void fxMaxWordsBatch(BatchArgs B, uint* out) {
  const FParams_t* P;
  const Span S = batch_span(B, blockIdx.x, P);
  max_words_impl(*P, S, out);
}

// Sums over all in-range particles of the stencil candidates (members of the
// stencil cells, self included) and of the in-radius pairs (0 < d2 < rd2),
// on the cell-sorted set: out[0] += C, out[1] += P.  The measurement behind
// the flop model of the density and force stages; the role of the
// reference's neighbour-count validation (fluids4.0/fluid_system.cpp:959-1011).
__device__ __forceinline__ void count_pairs_impl(const FParams_t& P, const Span S, unsigned long long* out) {
  const int i = S.p0 + S.blk * (int)blockDim.x + (int)threadIdx.x;
  unsigned long long nc = 0, np = 0;
  if (i < S.p1) {
    const int gc = pbuf<const int>(FPnts, FGCELL)[i];
    if (gc != FX_GRID_UNDEF) {
      const fx_float3* __restrict__ pos = pbuf<const fx_float3>(FPnts, FPOS);
      const uint* __restrict__ off = pbuf<const uint>(FAccel, AGRIDOFF);
      const uint* __restrict__ cnt = pbuf<const uint>(FAccel, AGRIDCNT);
      const fx_float3 p = pos[i];
      const int base = stencil_base(P, gc);
      for (int r = 0; r < P.gridSrch * P.gridSrch; r++) {
        int jb, je;
        row_range(P, base, r, off, cnt, jb, je);
        nc += (unsigned long long)(je - jb);
        for (int j = jb; j < je; j++) {
          const fx_float3 q = pos[j];
          const float dx = p.x - q.x, dy = p.y - q.y, dz = p.z - q.z;
          const float dsq = fmaf(dz, dz, fmaf(dy, dy, dx * dx));
          np += (dsq < P.rd2 && dsq > 0.0f) ? 1u : 0u;
        }
      }
    }
  }
  // wave64 reduction, one atomic per wave
  for (int o = 32; o > 0; o >>= 1) {
    nc += __shfl_xor(nc, o, 64);
    np += __shfl_xor(np, o, 64);
  }
  if ((threadIdx.x & 63) == 0 && (nc | np) != 0) {
    atomicAdd(&out[0], nc);
    atomicAdd(&out[1], np);
  }
}

extern "C" __global__ void fxCountPairs(unsigned long long* out, int pnum) {
  count_pairs_impl(*cparams(&FParams), Span{0, pnum, 0, (int)blockIdx.x}, out);
}

extern "C" __global__ void fxCountPairsBatch(BatchArgs B, unsigned long long* out) {
  const FParams_t* P;
  const Span S = batch_span(B, blockIdx.x, P);
  count_pairs_impl(*P, S, out);
}

// ------------------------------------------------------ volume sampling

// Gaussian splat of the particles onto a brick of res.x * res.y * res.z
// voxels spanning [bmin, bmax] (sampleParticles,
// fluids4.0/fluid_kernels.cu:259-300), a consumer of the cell table: voxel
// (x, y, z) sits at bmin + (x/res.x, y/res.y, z/res.z) * (bmax - bmin) and
// sums gausskern * exp(-r^2 / h2), h2 = 2 r2 / 8, over the particles of its
// 27 stencil cells with 0 < d^2 < rd2 (r in simulation units), in the
// stencil's cell order; the result, times `scalar`, goes to
// brick[(z * res.y + y) * res.x + x].  Voxels whose cell is outside
// [1, gridRes - gridSrch] get 0 at that same index (the reference writes
// those at (y * res.z + z) * res.x + x, a transposed index).  Positions are
// the current set's; the cell table is the one of the last sort.
//
// A wave takes a cube of 4 x 4 x 4 voxels (they share cells, and 16-byte runs
// of the brick); a stencil row is one run of particles (its cells are
// consecutive), and the bounds of all rows of 2 or 3 cells are loaded at once.
// The exponential is a power of two: its exponent d^2 * k, with
// k = -d2 / h2 * log2(e) in two floats khi + klo from the host, and the
// exponent's low part added to first order; no root, division or range check,
// and a smaller error than expf(-(r * r) / h2) of a rounded r.  160 x 80 x 80
// voxels, 131,072 particles: 96 us with expf, a root and a division a pair and
// voxels in planes of 8 x 8, 53 us so.  The candidates that a voxel walks
// while its wave's longest row lasts bound it, with the gathers' latency.
#define SV_EDGE 4  // voxels of a wave along each axis
#define SV_STEP 2  // particles loaded at a time: 1 / 2 / 3 / 4 gave 55 / 53 / 53 / 53 us
template <int SR>
__device__ __forceinline__ float sample_voxel(const FParams_t& P, float px, float py, float pz, int gs, int numPnts,
                                              float khi, float klo) {
  const fx_float3* __restrict__ pos = pbuf<const fx_float3>(FPnts, FPOS);
  const uint* __restrict__ off = pbuf<const uint>(FAccel, AGRIDOFF);
  constexpr int R = SR > 0 ? SR * SR : 1;
  const float rd2 = P.rd2;
  float v = 0.0f;
  auto row = [&](int jb, int je) {
    for (int j = jb; j < je; j += SV_STEP) {
      fx_float3 q[SV_STEP];
#pragma unroll
      for (int u = 0; u < SV_STEP; u++) q[u] = ld3(pos, (size_t)min(j + u, je - 1));
#pragma unroll
      for (int u = 0; u < SV_STEP; u++) {
        const float dx = px - q[u].x, dy = py - q[u].y, dz = pz - q[u].z;
        const float dsq = dx * dx + dy * dy + dz * dz;
        const float t = dsq * khi, l = fmaf(dsq, klo, fmaf(dsq, khi, -t));
        const float e = __builtin_amdgcn_exp2f(t);
        const float w = v + fmaf(e, l * 0.693147180559945f, e);
        v = dsq < rd2 && dsq > 0.0f && (u == 0 || j + u < je) ? w : v;
      }
    }
  };
  if (SR > 0) {
    int jb[R], je[R];
#pragma unroll
    for (int r = 0; r < R; r++) {
      const int c0 = gs + P.gridAdj[r * SR];
      jb[r] = (int)off[c0];
      je[r] = min((int)off[c0 + SR], numPnts);
    }
#pragma unroll
    for (int r = 0; r < R; r++) row(jb[r], je[r]);
  } else {
    const int srch = P.gridSrch;
    for (int r = 0; r < srch * srch; r++) {
      const int c0 = gs + P.gridAdj[r * srch];
      row((int)off[c0], min((int)off[c0 + srch], numPnts));
    }
  }
  return v;
}

__device__ __forceinline__ void sample_brick(int x, int y, int z, float* brick, const fx_int3 res, const fx_float3 bmin,
                                             const fx_float3 bmax, int numPnts, float scalar, float khi, float klo) {
  const FParams_t& P = *cparams(&FParams);
  if (x >= res.x || y >= res.y || z >= res.z) return;
  const size_t out = ((size_t)z * res.y + y) * res.x + x;
  const float px = bmin.x + ((float)x / (float)res.x) * (bmax.x - bmin.x);
  const float py = bmin.y + ((float)y / (float)res.y) * (bmax.y - bmin.y);
  const float pz = bmin.z + ((float)z / (float)res.z) * (bmax.z - bmin.z);
  const int gx = (int)((px - P.gridMin.x) * P.gridDelta.x);
  const int gy = (int)((py - P.gridMin.y) * P.gridDelta.y);
  const int gz = (int)((pz - P.gridMin.z) * P.gridDelta.z);
  if (gx < 1 || gx > P.gridRes.x - P.gridSrch || gy < 1 || gy > P.gridRes.y - P.gridSrch || gz < 1 ||
      gz > P.gridRes.z - P.gridSrch) {
    brick[out] = 0.0f;
    return;
  }
  const int nadj = (P.gridRes.z + 1) * P.gridRes.x + 1;
  const int gs = (gy * P.gridRes.z + gz) * P.gridRes.x + gx - nadj;
  const float v = P.gridSrch == 3   ? sample_voxel<3>(P, px, py, pz, gs, numPnts, khi, klo)
                  : P.gridSrch == 2 ? sample_voxel<2>(P, px, py, pz, gs, numPnts, khi, klo)
                                    : sample_voxel<0>(P, px, py, pz, gs, numPnts, khi, klo);
  brick[out] = v * P.gausskern * scalar;
}

// libfluidsx's launch: blocks of 256 threads over 8 x 8 x 4 voxels, four waves
extern "C" __global__ __launch_bounds__(256) void fxSampleBrick(float* brick, fx_int3 res, fx_float3 bmin,
                                                                fx_float3 bmax, int numPnts, float scalar, float khi,
                                                                float klo) {
  const int t = (int)threadIdx.x, w = t >> 6;
  const int x = (int)blockIdx.x * 2 * SV_EDGE + (w & 1) * SV_EDGE + t % SV_EDGE;
  const int y = (int)blockIdx.y * 2 * SV_EDGE + (w >> 1) * SV_EDGE + t / SV_EDGE % SV_EDGE;
  const int z = (int)blockIdx.z * SV_EDGE + t / (SV_EDGE * SV_EDGE) % SV_EDGE;
  sample_brick(x, y, z, brick, res, bmin, bmax, numPnts, scalar, khi, klo);
}

// The reference's kernel name and arguments (fluids4.0/fluid_kernels.cu:259),
// one voxel a thread of blocks of any shape; the same values.
extern "C" __global__ void sampleParticles(float* brick, fx_int3 res, fx_float3 bmin, fx_float3 bmax, int numPnts,
                                           float scalar) {
  const FParams_t& P = *cparams(&FParams);
  const float h2 = 2.0f * P.r2 / 8.0f;
  const double k = -(double)P.d2 / (double)h2 * 1.4426950408889634;
  const float khi = (float)k, klo = (float)(k - (double)khi);
  sample_brick((int)(blockIdx.x * blockDim.x + threadIdx.x), (int)(blockIdx.y * blockDim.y + threadIdx.y),
               (int)(blockIdx.z * blockDim.z + threadIdx.z), brick, res, bmin, bmax, numPnts, scalar, khi, klo);
}

// ------------------------------------------------------------------- emit

// emitParticles (fluids4.0/fluid_kernels.cu:231-257): each of `emit` threads
// respawns one particle at a point of the box (-170,10,-20)..(-190,60,20)
// quantized to 1/256 per axis by three bytes of a 32-bit value v, with
// velocity (5,-2,0) and zero veval and force.  The reference draws v from a
// per-particle XORWOW state and respawns particle v & (numPnts-1), so two
// threads can pick the same particle and the result depends on their order.
// Here v is a counter-based SplitMix64 of (frame, thread index) and the
// particles are a frame-seeded bijection of the thread index,
// j = (A i + b) mod numPnts with A prime (2654435761): min(emit, numPnts)
// distinct particles, whatever the thread order.
__device__ __forceinline__ unsigned long long fx_splitmix64(unsigned long long x) {
  x += 0x9E3779B97F4A7C15ull;
  x = (x ^ (x >> 30)) * 0xBF58476D1CE4E5B9ull;
  x = (x ^ (x >> 27)) * 0x94D049BB133111EBull;
  return x ^ (x >> 31);
}

extern "C" __global__ void emitParticles(float frame, int emit, int numPnts) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= emit || i >= numPnts) return;
  const unsigned long long h = fx_splitmix64((unsigned long long)__float_as_uint(frame));
  const uint v = (uint)(fx_splitmix64(h ^ fx_splitmix64((unsigned long long)i)) >> 32);
  const unsigned long long n = (unsigned long long)numPnts;
  const uint j = (uint)((2654435761ull * (unsigned long long)i + h % n) % n);
  const fx_float3 bmin = {-170.0f, 10.0f, -20.0f}, bmax = {-190.0f, 60.0f, 20.0f};
  const float ux = (float)(v & 0xFFu) / 256.0f;
  const float uy = (float)((v >> 8) & 0xFFu) / 256.0f;
  const float uz = (float)((v >> 16) & 0xFFu) / 256.0f;
  fx_float3 p;
  p.x = bmin.x + ux * (bmax.x - bmin.x);
  p.y = bmin.y + uy * (bmax.y - bmin.y);
  p.z = bmin.z + uz * (bmax.z - bmin.z);
  pbuf<fx_float3>(FPnts, FPOS)[j] = p;
  pbuf<fx_float3>(FPnts, FVEVAL)[j] = fx_float3{0.0f, 0.0f, 0.0f};
  pbuf<fx_float3>(FPnts, FVEL)[j] = fx_float3{5.0f, -2.0f, 0.0f};
  pbuf<fx_float3>(FPnts, FFORCE)[j] = fx_float3{0.0f, 0.0f, 0.0f};
}

// ----------------------------------------------------------------- advance

// Integrator (particles.cu:237-322): penalty walls on bound_min/bound_max
// (Y-min with slope and friction, Y-max with friction, X-min moving wall whose
// stiffness term is scaled by 'wall', X-max, Z-min, Z-max), gravity, the
// acceleration limit, the velocity limit applied to the old velocity, and the
// leapfrog update; returns the new position.
template <bool Nt>
__device__ __forceinline__ fx_float3 advance_from(const FParams_t& P, int i, const fx_float3 pos, fx_float3 vel,
                                                  const fx_float3 ve, const fx_float3 f, float time, float dt,
                                                  float ss) {
  fx_float3* __restrict__ posb = pbuf<fx_float3>(FPnts, FPOS);
  fx_float3* __restrict__ velb = pbuf<fx_float3>(FPnts, FVEL);
  fx_float3* __restrict__ vevb = pbuf<fx_float3>(FPnts, FVEVAL);
  const float m = P.pmass;
  float ax = f.x * m, ay = f.y * m, az = f.z * m;
  const float rad = P.pradius, stiff = P.bound_stiff, damp = P.bound_damp;
  const float slope = P.bound_slope, fric = P.bound_friction;
  const fx_float3 bmin = P.bound_min, bmax = P.bound_max;
  float diff, adj, nx, ny, nz;

  // Y-min, sloped floor with friction
  diff = rad - (pos.y - (bmin.y + (pos.x - bmin.x) * slope)) * ss;
  if (diff > FX_EPSILON) {
    nx = -slope;
    ny = 1.0f - slope;
    nz = 0.0f;
    adj = stiff * diff - damp * (nx * ve.x + ny * ve.y + nz * ve.z);
    nx *= adj; ny *= adj; nz *= adj;
    ax += nx - ve.x * fric;
    ay += ny - ve.y * fric;
    az += nz - ve.z * fric;
  }
  // Y-max with friction
  diff = rad - (bmax.y - pos.y) * ss;
  if (diff > FX_EPSILON) {
    nx = 0.0f; ny = -1.0f; nz = 0.0f;
    adj = stiff * diff - damp * (nx * ve.x + ny * ve.y + nz * ve.z);
    nx *= adj; ny *= adj; nz *= adj;
    ax += nx - ve.x * fric;
    ay += ny - ve.y * fric;
    az += nz - ve.z * fric;
  }
  // X-min, moving wall; its stiffness term is scaled by 'wall'
  const float sarg = time * P.bound_wall_freq + pos.z / 400.0f;
  // in double, as the reference (its 0.5 are double literals) and the oracle:
  // an FP32 restatement would round (s + 1) force / 2 once where the double
  // path may round twice
  const float wall = (float)(((double)fx_sinf(sarg) * 0.5 + 0.5) * (double)P.bound_wall_force);
  diff = rad - (pos.x - (bmin.x + wall)) * ss;
  if (diff > FX_EPSILON) {
    nx = 1.0f; ny = 0.0f; nz = 0.0f;
    adj = wall * stiff * diff - damp * (nx * ve.x + ny * ve.y + nz * ve.z);
    ax += nx * adj; ay += ny * adj; az += nz * adj;
  }
  // X-max
  diff = rad - (bmax.x - pos.x) * ss;
  if (diff > FX_EPSILON) {
    nx = -1.0f; ny = 0.0f; nz = 0.0f;
    adj = stiff * diff - damp * (nx * ve.x + ny * ve.y + nz * ve.z);
    ax += nx * adj; ay += ny * adj; az += nz * adj;
  }
  // Z-min
  diff = rad - (pos.z - bmin.z) * ss;
  if (diff > FX_EPSILON) {
    nx = 0.0f; ny = 0.0f; nz = 1.0f;
    adj = stiff * diff - damp * (nx * ve.x + ny * ve.y + nz * ve.z);
    ax += nx * adj; ay += ny * adj; az += nz * adj;
  }
  // Z-max
  diff = rad - (bmax.z - pos.z) * ss;
  if (diff > FX_EPSILON) {
    nx = 0.0f; ny = 0.0f; nz = -1.0f;
    adj = stiff * diff - damp * (nx * ve.x + ny * ve.y + nz * ve.z);
    ax += nx * adj; ay += ny * adj; az += nz * adj;
  }
  // gravity
  ax += P.gravity.x;
  ay += P.gravity.y;
  az += P.gravity.z;
  // acceleration limit
  float speed = ax * ax + ay * ay + az * az;
  if (speed > P.AL2) {
    const float s = P.AL / sqrtf(speed);
    ax *= s; ay *= s; az *= s;
  }
  // velocity limit, applied to the old velocity
  speed = vel.x * vel.x + vel.y * vel.y + vel.z * vel.z;
  if (speed > P.VL2) {
    const float s = P.VL / sqrtf(speed);
    vel.x *= s; vel.y *= s; vel.z *= s;
  }
  // leapfrog
  const float vnx = ax * dt + vel.x, vny = ay * dt + vel.y, vnz = az * dt + vel.z;
  put3<Nt>(vevb, (size_t)i, (vel.x + vnx) * 0.5f, (vel.y + vny) * 0.5f, (vel.z + vnz) * 0.5f);
  put3<Nt>(velb, (size_t)i, vnx, vny, vnz);
  const float dts = dt / ss;
  const float x = pos.x + vnx * dts, y = pos.y + vny * dts, z = pos.z + vnz * dts;
  put3<Nt>(posb, (size_t)i, x, y, z);
  return fx_float3{x, y, z};
}

// GRID_UNDEF particles are parked at (-1000)^3 with zero velocity.
__device__ __forceinline__ fx_float3 park(int i) {
  pbuf<fx_float3>(FPnts, FPOS)[i] = fx_float3{-1000.0f, -1000.0f, -1000.0f};
  pbuf<fx_float3>(FPnts, FVEL)[i] = fx_float3{0.0f, 0.0f, 0.0f};
  return fx_float3{-1000.0f, -1000.0f, -1000.0f};
}

__device__ __forceinline__ void advance_one(const FParams_t& P, int i, float time, float dt, float ss) {
  if (pbuf<const int>(FPnts, FGCELL)[i] == FX_GRID_UNDEF) {
    park(i);
    return;
  }
  advance_from<false>(P, i, pbuf<const fx_float3>(FPnts, FPOS)[i], pbuf<const fx_float3>(FPnts, FVEL)[i],
               pbuf<const fx_float3>(FPnts, FVEVAL)[i], pbuf<const fx_float3>(FPnts, FFORCE)[i], time, dt, ss);
}

extern "C" __global__ void advanceParticles(float time, float dt, float ss, int numPnts) {
  const int ppt = ppt_of(5);
  if (ppt == 1) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < numPnts) advance_one(*cparams(&FParams), i, time, dt, ss);
    return;
  }
  for (int k = 0; k < ppt; k++) {
    const int i = (blockIdx.x * ppt + k) * blockDim.x + threadIdx.x;
    if (i < numPnts) advance_one(*cparams(&FParams), i, time, dt, ss);
  }
}

// Same integrator with the simulation time read from device memory, for
// captured step graphs whose launches cannot carry a per-step time argument.
// The set exchange (exchange_tables) moves that clock on by dt each step (the
// host's AdvanceTime, particles.cpp:396-400).
extern "C" __global__ void advanceParticlesClock(const float* clock, float dt, float ss, int numPnts) {
  const int ppt = ppt_of(5);
  if (ppt == 1) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < numPnts) advance_one(*cparams(&FParams), i, clock[0], dt, ss);
    return;
  }
  for (int k = 0; k < ppt; k++) {
    const int i = (blockIdx.x * ppt + k) * blockDim.x + threadIdx.x;
    if (i < numPnts) advance_one(*cparams(&FParams), i, clock[0], dt, ss);
  }
}

// The set exchange as a launch of its own (64 threads).
extern "C" __global__ void fxPublishTables(FxExchange E) { exchange_tables(E); }

// Batch integrator: the time comes from clock[0] when clock is given, else
// from the argument; dt and the scale from each scene's parameters.
__device__ __forceinline__ void advance_entry(const BatchArgs& B, int b, const float* clock, float time) {
  const int ppt = ppt_of(5);
  const FParams_t* P;
  const Span S = batch_span(B, b, P);
  for (int k = 0; k < ppt; k++) {
    const int i = S.p0 + (S.blk * ppt + k) * (int)blockDim.x + (int)threadIdx.x;
    if (i < S.p1) advance_one(*P, i, clock != nullptr ? clock[0] : time, P->dt, P->sim_scale);
  }
}

extern "C" __global__ void advanceParticlesBatch(BatchArgs B, const float* clock, float time) {
  advance_entry(B, blockIdx.x, clock, time);
}

extern "C" __global__ void advanceParticlesBatchP(BatchArgs B, const float* clock, float time) {
  batch_items(B, [&](int b) { advance_entry(B, b, clock, time); });
}

// ------------------------------------------- the ranked sort of other hosts

extern "C" __global__ void countingSortFullRanked(int pnum) {
  const int ppt = ppt_of(2);
  const Span S{0, pnum, 0, xcd_block()};
  if (ppt == 1) {
    sort_full_impl(*cparams(&FParams), S);
    return;
  }
  for (int k = 0; k < ppt; k++) sort_full_impl(*cparams(&FParams), sub_span(S, ppt, k));
}
