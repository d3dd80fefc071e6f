/* fx_walk.hpp -- a wave walks the recorded neighbours of its 64 particles.
 *
 * The density stage leaves one bit per stencil candidate of a particle, row r
 * of the stencil in a word-aligned run.  word_walk gives each lane its
 * particle's set bits in candidate order, the same number from every lane at
 * a time, so that the pair arithmetic of the caller runs with nearly all
 * lanes busy and no candidate is tested twice.  The forward force and both
 * kernels of its adjoint use it.
 */
#ifndef FX_WALK_HPP
#define FX_WALK_HPP

#include <climits>

// Wave-wide max / min with the same DPP pattern; lane 63 ends up with the
// reduction of all 64 lanes and is read back as a scalar.
template <bool kMax>
__device__ __forceinline__ int wave_reduce(int v) {
  const int id = kMax ? INT_MIN : INT_MAX;
  int t;
#define FX_RED_STEP(ctrl, rmask)                                    \
  t = __builtin_amdgcn_update_dpp(id, v, ctrl, rmask, 0xf, false); \
  v = kMax ? max(v, t) : min(v, t);
  FX_RED_STEP(0x111, 0xf)  // row_shr:1
  FX_RED_STEP(0x112, 0xf)  // row_shr:2
  FX_RED_STEP(0x114, 0xf)  // row_shr:4
  FX_RED_STEP(0x118, 0xf)  // row_shr:8
  FX_RED_STEP(0x142, 0xa)  // row_bcast:15
  FX_RED_STEP(0x143, 0xc)  // row_bcast:31
#undef FX_RED_STEP
  return __builtin_amdgcn_readlane(v, 63);
}
__device__ __forceinline__ int wave_max(int v) { return wave_reduce<true>(v); }
__device__ __forceinline__ int wave_min(int v) { return wave_reduce<false>(v); }

// The value of the neighbouring lane (2k and 2k + 1 exchange).
__device__ __forceinline__ uint lane_other(uint v) {
  return __builtin_amdgcn_update_dpp(0u, v, 0xB1, 0xf, 0xf, true);  // quad_perm 1,0,3,2
}

// Lanes 2k and 2k + 1 have read both halves of the even lane's record (e, each
// lane one half) and of the odd lane's (o); a becomes the lane's own first
// half and o its own second half (three words of it).
__device__ __forceinline__ void swap_halves(const float4& e, float4& o, float4& a) {
  // a, the (pos, rho) half: an even lane's e, an odd lane takes the even
  // lane's o.  o becomes the (veval, 0) half: an odd lane's own, an even
  // lane takes the odd lane's e.  Every lane of the wave runs this; a DPP
  // source needs two cycles after a VALU write of it.
  __asm__("s_nop 1\n\ts_mov_b64 vcc, %8\n\t"
          "v_cndmask_b32_dpp %0, %4, %9, vcc quad_perm:[1,0,3,2] row_mask:0xf bank_mask:0xf\n\t"
          "v_cndmask_b32_dpp %1, %5, %10, vcc quad_perm:[1,0,3,2] row_mask:0xf bank_mask:0xf\n\t"
          "v_cndmask_b32_dpp %2, %6, %11, vcc quad_perm:[1,0,3,2] row_mask:0xf bank_mask:0xf\n\t"
          "v_cndmask_b32_dpp %3, %7, %12, vcc quad_perm:[1,0,3,2] row_mask:0xf bank_mask:0xf"
          : "=&v"(a.x), "=&v"(a.y), "=&v"(a.z), "=&v"(a.w)
          : "v"(o.x), "v"(o.y), "v"(o.z), "v"(o.w), "s"(0x5555555555555555ull), "v"(e.x),
            "v"(e.y), "v"(e.z), "v"(e.w)
          : "vcc");
  __asm__("s_nop 1\n\ts_mov_b64 vcc, %6\n\t"
          "v_cndmask_b32_dpp %0, %3, %0, vcc quad_perm:[1,0,3,2] row_mask:0xf bank_mask:0xf\n\t"
          "v_cndmask_b32_dpp %1, %4, %1, vcc quad_perm:[1,0,3,2] row_mask:0xf bank_mask:0xf\n\t"
          "v_cndmask_b32_dpp %2, %5, %2, vcc quad_perm:[1,0,3,2] row_mask:0xf bank_mask:0xf"
          : "+v"(o.x), "+v"(o.y), "+v"(o.z)
          : "v"(e.x), "v"(e.y), "v"(e.z), "s"(0xAAAAAAAAAAAAAAAAull)
          : "vcc");
}

#define FX_WALK_K 16  // queued words a lane: 8 KB of LDS a wave; a power of two

// Row r's candidates begin at jb[r] and take words [E_[r - 1], E_[r]) of the
// lane's nwords (word f at bits[f * NN + i]); longest is the longest row, in
// candidates.  q: the lane's place in the wave's 8 KB.  eval(j, ok) takes
// STEP pairs of every lane: j[u] is MUL times the candidate, 0 where the lane
// has none left (ok[u] false).  All 64 lanes call it.
template <int R, uint MUL, int STEP, class Eval>
__device__ __forceinline__ void word_walk(const uint* __restrict__ bits, size_t NN, int i, int nwords, int longest,
                                          const int (&jb)[R], const int (&E_)[R], uint* q, const Eval& eval) {
  constexpr int MASK = FX_WALK_K * 64 - 1, AHEAD = 4;  // bitmask words loaded ahead of their use
  static_assert(R <= FX_WALK_K, "a word of every row fits the queue");
  uint* qw = q;                   // words, 64 apart
  uint* qb = q + FX_WALK_K * 64;  // and where they begin
  // the current word and what its bit 0 stands for, in records; the
  // queue's first two (0 where it holds fewer)
  uint cur = 0u, curb = 0u, n1 = 0u, n1b = 0u, n2 = 0u, n2b = 0u;
  int head = 0, cnt = 0;  // of the queue, n1 and n2 included
  int qn = 0;             // pairs held
  auto ahead = [&]() __attribute__((always_inline)) {
    const int h2 = (head + 64) & MASK;
    n1 = qw[head];
    n1b = qb[head];
    n2 = qw[h2];
    n2b = qb[h2];
    n1 = cnt > 0 ? n1 : 0u;
    n2 = cnt > 1 ? n2 : 0u;
  };
  // STEP pairs from every lane (a lane that has none left evaluates record
  // 0 and discards it), each lane's in candidate order
  auto step = [&]() __attribute__((always_inline)) {
    uint j[STEP];
    bool ok[STEP];
    const int have = min(cnt, 2);
#pragma unroll
    for (int u = 0; u < STEP; u++) {
      ok[u] = cur != 0u;
      j[u] = ok[u] ? curb + MUL * (uint)__builtin_ctz(cur) : 0u;
      const uint rest = cur & (cur - 1u);
      const bool next = rest == 0u;
      cur = next ? n1 : rest;
      curb = next ? n1b : curb;
      n1 = next ? n2 : n1;
      n1b = next ? n2b : n1b;
      n2 = next ? 0u : n2;
      qn -= ok[u] ? 1 : 0;
    }
    const int used = have - (n1 != 0u ? 1 : 0) - (n2 != 0u ? 1 : 0);
    cnt -= used;
    head = (head + 64 * used) & MASK;
    ahead();
    eval(j, ok);
  };
  // A pass reads the bitmask once, as a stream: non-temporal loads.
  if (wave_max(longest) <= 32) {
    // a word a row: the queue holds them all
    uint w[R];
#pragma unroll
    for (int r = 0; r < R; r++) {
      const int f = r == 0 ? 0 : E_[r - 1];
      w[r] = f < E_[r] ? __builtin_nontemporal_load(&bits[(size_t)f * NN + i]) : 0u;
    }
#pragma unroll
    for (int r = 0; r < R; r++) {  // a zero word is written over by the next
      qw[64 * cnt] = w[r];
      qb[64 * cnt] = MUL * (uint)jb[r];
      cnt += w[r] != 0u ? 1 : 0;
      qn += __popc(w[r]);
    }
  } else {
    const int maxf = wave_max(nwords);
    uint nx[AHEAD];
#pragma unroll
    for (int k = 0; k < AHEAD; k++) nx[k] = k < nwords ? __builtin_nontemporal_load(&bits[(size_t)k * NN + i]) : 0u;
    for (int f0 = 0; f0 < maxf; f0 += AHEAD) {
      uint cw[AHEAD];
#pragma unroll
      for (int k = 0; k < AHEAD; k++) {
        cw[k] = nx[k];
        const int fn = f0 + AHEAD + k;
        nx[k] = fn < nwords ? __builtin_nontemporal_load(&bits[(size_t)fn * NN + i]) : 0u;
      }
#pragma unroll
      for (int k = 0; k < AHEAD; k++) {
        const int f = f0 + k;
        if (f >= maxf) break;
        const uint word = cw[k];
        int base = jb[0], first = 0;  // of the row that holds word f
#pragma unroll
        for (int r = 1; r < R; r++) {
          const int b = jb[r], e = E_[r - 1];
          base = f >= e ? b : base;
          first = f >= e ? e : first;
        }
        const bool full = word != 0u && cnt == FX_WALK_K;
        if (__any(full)) {
          // free a slot: the full lanes finish their current word, every lane
          // gives as many pairs as the shortest queue holds
          ahead();
          int f1 = max(wave_max(full ? __popc(cur) + 1 : 0), wave_min(nwords > 0 ? qn : INT_MAX));
          do {
            step();
            f1 -= STEP;
          } while (f1 > 0 || __any(word != 0u && cnt == FX_WALK_K));
        }
        if (word != 0u) {
          const int t = (head + 64 * cnt) & MASK;
          qw[t] = word;
          qb[t] = MUL * (uint)(base + ((f - first) << 5));
          cnt++;
          qn += __popc(word);
        }
      }
    }
  }
  ahead();
  while (__any(qn > 0)) step();
}

#endif
