// KV k-means clustering and centroid-scored token selection for gfx950 (MI355X).
//
// Replaces the reference's Triton kernels in cache_hub/kmeans.py:
//   _triton_assign_kernel :7-79, _triton_update_kernel :82-124, _triton_k_means_train :127-196,
//   _triton_reverse_index_kernel :199-262, _triton_index_add_kernel :265-329.
// The reference scatters every token into its cluster sum with fp32 atomics (16.8 M atomics per head and
// iteration at 131072 x 128).  Here the assignment is a dense bf16 MFMA contraction with an arg-max
// epilogue in registers, tokens are then grouped by cluster tile by tile and every cluster is summed by one
// workgroup in fp64, which is exact for bf16 data and therefore independent of order -- and of how the sums were
// arrived at: a run of iterations may keep them in the workspace and apply only the tokens that changed cluster
// (sq_kmeans_train_stateful).  A counting sort in ascending token order yields the reverse index.
#include <algorithm>

#include "common.hpp"

namespace sq {
namespace {

constexpr int kD = 128;
constexpr int kCB = 64;            // centroids per LDS stage
constexpr int kTileTok = 256;      // tokens per workgroup in assign / sort kernels
constexpr int kMaxC = 8192;
constexpr int kBigTok = 2;         // tokens per thread of the grouping kernel
constexpr int kBigTile = 1024 * kBigTok;   // and per workgroup

// ------------------------------------------------------------------------------------------ fill
__global__ void fill_i32_kernel(int32_t* p, int64_t n, int32_t v) {
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x) p[i] = v;
}

// ---------------------------------------------------------------------------------------- assign
// What the NEAR form of the assignment keeps from step to step beside the sums (below)
struct NearState {
  int32_t* order;      // [G,N] the tokens cluster by cluster, as they were when the sums began to be carried
  int32_t* cursor;     // [G,C] places handed out while `order` is formed
  uint16_t* used;      // [G,C,128] the centroids c' the last assignment was made with; of the tokens x a cluster got there:
  float* used_low;     // [G,C] the lowest score <x, c'>
  float* used_far;     // [G,C] the largest distance from the line along c' (not a number: unknown)
  uint32_t* low;       // [G,C] the same, collected by the assignment under way: score and squared distance, as bits
  uint32_t* far2;      // [G,C]
  float* norm2;        // [G,C] |c|^2 of the present centroids
  uint32_t* mask;      // [G,C,C/32] bit j of row a: centroid j can win a token of cluster a
  unsigned long long* pairs;   // pairs of a token and a centroid the masks leave to be looked at, by every kPairSample-th block of clusters
  unsigned long long limit;    // more than these: everything is walked, from then on (an eighth of all pairs of such blocks)
  unsigned long long* excess;  // centroids walked by every kWalkSample-th workgroup of the first such assignment, kWalkShare times, less all; above 0 (signed): the same
  int32_t* dense;      // 1: one of the two has happened; 0: what is walked has not been counted yet
  int32_t* odd;        // [G] not 0: a centroid that is no finite number
  int32_t G;
};

struct AssignArgs {
  const uint16_t* data;  // [G,N,128] bf16
  const uint16_t* cent;  // [G,C,128] bf16
  int32_t* idx;          // [G,N]
  int64_t d_sg, d_sn, c_sg, c_sc, i_sg;
  int32_t N, C;
  double* keep_sum;      // TRACK: [G,C,128] the clusters' exact sums, carried from the previous step
  int32_t* keep_cnt;     // TRACK: [G,C] and their sizes
  NearState near;        // NEAR
};

__device__ __forceinline__ int wave_inclusive_scan(int v, int lane) {
#pragma unroll
  for (int d = 1; d < 64; d <<= 1) {
    const int o = __shfl_up(v, d);
    if (lane >= d) v += o;
  }
  return v;
}

__device__ __forceinline__ float dot8_bf16(const uint4& x, const uint4& y, float acc) {
  typedef __attribute__((ext_vector_type(2))) __bf16 bf16x2_t;
  const uint32_t a[4] = {x.x, x.y, x.z, x.w}, b[4] = {y.x, y.y, y.z, y.w};
#pragma unroll
  for (int e = 0; e < 4; ++e) acc = __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(bf16x2_t, a[e]), __builtin_bit_cast(bf16x2_t, b[e]), acc, false);
  return acc;
}
// over the 16 lanes of a row
__device__ __forceinline__ float sum16(float v) {
#pragma unroll
  for (int d = 1; d < 16; d <<= 1) v += __shfl_xor(v, d);
  return v;
}

constexpr int kNearMaxC = 2048;
constexpr int kPairSample = 8, kWalkSample = 4, kWalkShare = 5;
constexpr uint32_t kInfBits = 0x7f800000u, kNanBits = 0x7fc00000u;
// Squared lengths the bounds need of a token and of a centroid: 32-bit products of two of them are still good to 1e-7.  Below, they
// know nothing, and everything is walked.
constexpr float kFaint = 1e-18f;

// Squared distance of a token x from the line along a centroid c, xx = |x|^2 and on_line = <x, c>^2 / |c|^2.  The fp32 sums are within
// 3e-5 of the terms, 1e-3 of them covers that.  Not a number: unknown.
__device__ __forceinline__ float far_squared(float xx, float on_line) {
  const float d2 = xx - on_line + 1e-3f * (xx + on_line);
  return xx >= kFaint && d2 >= 0.f ? d2 : __uint_as_float(kNanBits);
}

constexpr int kAssignWaves = 4;   // x 64 tokens; two workgroups per CU put two waves on every SIMD

// Workgroup = 256 tokens of one group, 64 per wave (two 32-token operand sets in registers): every centroid fragment
// read from LDS feeds two MFMAs, which halves the LDS traffic per MFMA -- with 32 tokens per wave the fragment reads
// of the four SIMDs add up to the LDS's whole 128 bytes per cycle.  Centroids stream through LDS in blocks of 64
// (global_load_lds, unpadded rows, 16-byte chunks XOR-swizzled by row so that the MFMA operand reads are conflict
// free), double buffered with one barrier per block; the arg-max over one half block's scores runs underneath the
// MFMAs of the next half block (see `phase` below).
// TRACK: the sums that are carried across iterations.  After the first few Lloyd iterations hardly any token changes its
// cluster (configuration 4: 1 % in the fourth iteration, 0.1 % in the tenth), yet a full re-sum reads every row again.
// The sums are exact (fp64 of bf16 values), so they can be carried: `idx` holds the previous iteration's assignment on
// entry, and a token whose cluster changes is subtracted from its old cluster's sum and added to its new one's, in any
// order, by fp64 atomics that round nothing -- the result is the sum a full re-sum would give, bit for bit.  The
// workgroup lists its movers in LDS and applies them itself at the end (one channel per thread, the first 128 threads
// adding, the others subtracting); kmeans_update_kernel then turns sums and sizes into centroids.
// PARTS: launches that leave CUs idle.  A workgroup's length is its chain of centroid blocks, whatever the number of
// tokens (4096 tokens x 1024 centroids: 16 workgroups, 16 us).  With PARTS = 2 or 4 a workgroup takes 256 / PARTS tokens
// and its waves share the centroids: wave w walks part w % PARTS of the blocks, each part streaming through buffers of its
// own, and the parts' (score, index) pairs meet in LDS at the end.  A score is the same chain of MFMAs in any part and the
// lowest index wins ties inside a part and across them, so the assignment is the same to the bit.
// NEAR: centroids that cannot win are left out, by bounds that hold for every token of a cluster (the triangle inequality, as in
// C. Elkan, "Using the triangle inequality to accelerate k-means", 2003); the assignment is the same to the bit.  The last
// assignment left for every cluster a, with c' the centroid it was made with, its tokens' lowest score s = <x, c'> and their largest
// distance R from the line along c'.  For all of them <x, c_j - c_a> <= s / |c'|^2 <c', c_j - c_a> + R |c_j - c_a| where the first product
// is negative, and that takes products of centroids only (kmeans_bounds_kernel).  A centroid for which it is clearly negative cannot win.
// Tokens are taken in `order`, so a workgroup's 256 belong to a few clusters, and it walks the list of the centroids that can
// win any of them.  Whatever is not a finite number, or smaller than kFaint, has everything walked.
// What it takes is a chain of dependent loads, some 9 us a workgroup, four rounds of them: ids, rows and old clusters, masks, the block of
// centroids.  4 x 131072 tokens around 512 centres, 1024 centroids: 117 - 130 -> 46 to 59 us a step, by the keys, beside 9 us for the bounds, and of a
// run of ten steps, seven of which have bounds, 1410 -> 1102 us.  Three workgroups per CU (168 registers) spill: 35 us a workgroup.
template <bool TRACK, int PARTS, bool NEAR = false>
__global__ __launch_bounds__(kAssignWaves * 64, 1) void kmeans_assign_kernel(AssignArgs a) {
  static_assert(PARTS == 1 || PARTS == 2 || PARTS == kAssignWaves, "waves per part");
  static_assert(!NEAR || (TRACK && PARTS == 1), "the assignment before this one is needed");
  __shared__ __attribute__((aligned(16))) char smem[PARTS * 2 * kCB * 256];
  __shared__ int32_t s_chg_n;
  __shared__ uint2 s_chg[TRACK ? kTileTok / PARTS : 1];   // (token, old cluster << 16 | new cluster)
  __shared__ float s_best[PARTS > 1 ? kAssignWaves * 64 : 1];
  __shared__ int32_t s_bidx[PARTS > 1 ? kAssignWaves * 64 : 1];
  __shared__ uint32_t s_mask[NEAR ? kNearMaxC / 32 : 1];
  __shared__ uint16_t s_list[NEAR ? kNearMaxC : 1];   // the centroids to walk, ascending
  __shared__ uint32_t s_low[NEAR ? kNearMaxC : 1], s_far2[NEAR ? kNearMaxC : 1];   // by place in the list
  __shared__ float s_norm2[NEAR ? kNearMaxC : 1];
  __shared__ int32_t s_all;
  typedef __attribute__((address_space(3))) void* lds_ptr_t;
  // NEAR: the tiles of all groups in turn, so that the large clusters in front of every group's `order` come first
  const int g_id = NEAR ? (int)(blockIdx.x % a.near.G) : (int)blockIdx.y, tile = NEAR ? (int)(blockIdx.x / a.near.G) : (int)blockIdx.x;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int c32 = lane & 31, g = lane >> 5;
  const int part = wave % PARTS, sub = wave / PARTS;   // share of the centroids, 64 tokens of the tile
  const int tok0 = tile * (kTileTok / PARTS) + sub * 64;

  // token fragments (B operand of S^T = Cent . Data^T): lane (column = token 32 tb + c32, k-group g)
  const uint16_t* db = a.data + (int64_t)g_id * a.d_sg;
  uint4 tf[2][8];
  const int form = NEAR ? *a.near.dense : 0;
  const bool dense = NEAR && (form == 1 || *a.near.pairs > a.near.limit);
  int tok[2];
#pragma unroll
  for (int tb = 0; tb < 2; ++tb) {
    tok[tb] = min(tok0 + 32 * tb + c32, a.N - 1);
    if constexpr (NEAR) {
      const int n = a.near.order[(int64_t)g_id * a.N + tok[tb]];   // (asked for either way: not behind the answer to `dense`)
      if (!dense) tok[tb] = min(max(n, 0), a.N - 1);
    }
  }
  int old_idx[2] = {-1, -1};
  if constexpr (TRACK) {
    // NEAR wants them first of all, the others at the very end
#pragma unroll
    for (int tb = 0; tb < 2; ++tb)
      if (tok0 + 32 * tb + c32 < a.N) old_idx[tb] = a.idx[(int64_t)g_id * a.i_sg + tok[tb]];
  }
#pragma unroll
  for (int tb = 0; tb < 2; ++tb) {
    const int n = tok[tb];
    const uint16_t* rp = db + (int64_t)n * a.d_sn + 8 * g;
#pragma unroll
    for (int kk = 0; kk < 8; ++kk) tf[tb][kk] = *(const uint4*)(rp + 16 * kk);
  }
  if constexpr (TRACK) {
    if (tid == 0) s_chg_n = 0;   // (the block loop below passes at least one barrier before anyone adds to it)
  }
  const uint16_t* cb = a.cent + (int64_t)g_id * a.c_sg;
  // per-lane source of the wave's 1 KB copies of a block (4 centroid rows each, four copies per wave and part), as a byte
  // offset from the block's first row (the swizzle repeats every four copies); rows past C are clamped to the last
  // centroid, which only a block that runs past C has to do
  constexpr int kCopies = 4 * PARTS;
  int64_t src_off[4];
#pragma unroll
  for (int c = 0; c < 4; ++c) {
    const int row = 4 * (sub * kCopies + c) + (lane >> 4);
    src_off[c] = ((int64_t)row * a.c_sc + 8 * ((lane & 15) ^ (row & 15))) * 2;
  }
  int n_list = 0;        // NEAR: length of s_list
  bool whole = !NEAR;    // all centroids, in order
  auto stage = [&](int chunk, int st) {
    char* buf = smem + (2 * part + st) * (kCB * 256);
    if (NEAR && !whole) {   // places behind the list's end: copies of its last centroid
      int crow[4];
#pragma unroll
      for (int c = 0; c < 4; ++c) crow[c] = s_list[min(chunk * kCB + 4 * (sub * 4 + c) + (lane >> 4), n_list - 1)];
#pragma unroll
      for (int c = 0; c < 4; ++c) {
        const int row = 4 * (sub * 4 + c) + (lane >> 4);
        __builtin_amdgcn_global_load_lds((const void*)(cb + (int64_t)crow[c] * a.c_sc + 8 * ((lane & 15) ^ (row & 15))),
                                         (lds_ptr_t)(buf + (sub * 4 + c) * 1024), 16, 0, 0);
      }
      return;
    }
    const char* blk = (const char*)cb + (int64_t)chunk * kCB * a.c_sc * 2;
    if ((chunk + 1) * kCB <= a.C) {
#pragma unroll
      for (int c = 0; c < kCopies; ++c)
        __builtin_amdgcn_global_load_lds((const void*)(blk + src_off[c & 3] + (int64_t)(c >> 2) * 32 * a.c_sc),
                                         (lds_ptr_t)(buf + (sub * kCopies + c) * 1024), 16, 0, 0);
    } else {
#pragma unroll
      for (int c = 0; c < kCopies; ++c) {
        const int q = sub * kCopies + c;
        const int row = 4 * q + (lane >> 4);
        const int ch = (lane & 15) ^ (row & 15);
        const int crow = min(chunk * kCB + row, a.C - 1);
        __builtin_amdgcn_global_load_lds((const void*)(cb + (int64_t)crow * a.c_sc + 8 * ch), (lds_ptr_t)(buf + q * 1024), 16, 0, 0);
      }
    }
  };
  // Fragment number n = 8 half + kk of a block: centroid row 32 half + c32, 16-byte chunk (2 kk + g) ^ (row & 15).  The
  // reads go through lds_read128 / lds_wait (explicit lgkmcnt counts): left to the compiler, every wait was a full
  // lgkmcnt(0), i.e. also for the fragments requested a moment ago.
  const int ksw = c32 & 15;
  const uint32_t smem_addr = (uint32_t)(uintptr_t)(lds_ptr_t)smem + part * (2 * kCB * 256);
  uint32_t fa[8];
#pragma unroll
  for (int kk = 0; kk < 8; ++kk) fa[kk] = smem_addr + c32 * 256 + (((2 * kk + g) ^ ksw) << 4);
  auto frag = [&](uint32_t boff, auto NUM) {
    constexpr int n = decltype(NUM)::value;
    return lds_read128<(n >> 3) * 8192>(fa[n & 7] + boff);
  };
  // Running arg-max in ascending centroid order with strict '>' = lowest index on ties (kmeans.py:62-65), four scores
  // at a time: the group's maximum (v_max3 + v_max) is compared with the running best; a group that wins leaves its
  // id and its first three scores behind, from which the position inside the group follows at the end (the first score
  // equal to the best; if none of the three, the fourth).  Eight vector instructions per four scores instead of
  // twelve.  Rows past C (C % 64 == 32) are clamped copies of the last centroid; they come after it in this order and
  // can never beat it strictly.
  float best[2] = {-INFINITY, -INFINITY};
  float keep0[2] = {0.f, 0.f}, keep1[2] = {0.f, 0.f}, keep2[2] = {0.f, 0.f};
  int bgrp[2] = {0, 0}, bhalf[2] = {0, 0};
  // S[tb][h]: scores of token set tb against centroid half h (32 centroids) of the current block.  A block is
  // computed in two phases of 16 MFMAs, half 0 then half 1, each as two accumulator chains (tb = 0, 1) over the eight
  // 16-wide slices of the dimension.  Underneath the MFMAs of one phase runs the arg-max over the results of the
  // previous phase, as one hand-ordered instruction stream: an MFMA occupies the matrix pipe for 32 cycles, half a
  // group's arg-max (four vector instructions) issues behind it.  The accumulators are not double-buffered; with
  // the MFMAs in their VGPR form (build flag) the arg-max reads them without copies out of the accumulation registers.
  f32x16_t S[2][2];
#pragma unroll
  for (int tb = 0; tb < 2; ++tb)
#pragma unroll
    for (int i = 0; i < 16; ++i) S[tb][1][i] = -INFINITY;   // "previous phase" of the very first one
  // One group of four scores against the running best, as one instruction block in the short encodings with the
  // condition in VCC (the compiler's form of the same selects is a masked block of moves behind s_and_saveexec):
  // VCC = not (m > best); a group that wins leaves its id and its first three scores behind.
  auto group_step = [&](const f32x16_t& P, int tb, auto Q) {
    constexpr int q = decltype(Q)::value;
    float m;
    float &b = best[tb], &k0 = keep0[tb], &k1 = keep1[tb], &k2 = keep2[tb];
    int& grp = bgrp[tb];
    asm volatile(
        "v_max3_f32 %[m], %[p0], %[p1], %[p2]\n\t"
        "v_max_f32_e32 %[m], %[m], %[p3]\n\t"
        "v_cmp_le_f32_e32 vcc, %[m], %[best]\n\t"
        "v_cndmask_b32_e32 %[k0], %[p0], %[k0], vcc\n\t"
        "v_cndmask_b32_e32 %[k1], %[p1], %[k1], vcc\n\t"
        "v_cndmask_b32_e32 %[k2], %[p2], %[k2], vcc\n\t"
        "v_cndmask_b32_e32 %[grp], %[qq], %[grp], vcc\n\t"
        "v_max_f32_e32 %[best], %[best], %[m]"
        : [m] "=&v"(m), [best] "+v"(b), [k0] "+v"(k0), [k1] "+v"(k1), [k2] "+v"(k2), [grp] "+v"(grp)
        : [p0] "v"(P[4 * q]), [p1] "v"(P[4 * q + 1]), [p2] "v"(P[4 * q + 2]), [p3] "v"(P[4 * q + 3]), [qq] "n"(q)
        : "vcc");
  };
  // The 16 centroid fragments of a block (half h, slice kk -> number 8 h + kk) are requested kFragAhead steps before
  // the MFMA pair that uses them: an LDS read takes longer than one pair of MFMAs when eight waves read at once.
  constexpr int kFragAhead = 3;
  auto phase = [&](auto H, uint32_t boff, int half_id, u32x4_t (&fr)[16]) {
    constexpr int h = decltype(H)::value;   // centroid half computed now; the arg-max runs over half 1 - h
    const float before0 = best[0], before1 = best[1];
    static_for<0, 8>([&](auto KK) {
      constexpr int kk = decltype(KK)::value;
      constexpr int cur = 8 * h + kk, nxt = cur + kFragAhead;
      if constexpr (nxt < 16) fr[nxt] = frag(boff, std::integral_constant<int, nxt>{});
      lds_wait<(15 - cur < kFragAhead ? 15 - cur : kFragAhead)>(fr[cur]);
      const bf16x8_t af = __builtin_bit_cast(bf16x8_t, fr[cur]);
      static_for<0, 2>([&](auto TB) {
        constexpr int tb = decltype(TB)::value;
        const bf16x8_t t = __builtin_bit_cast(bf16x8_t, tf[tb][kk]);
        if constexpr (kk == 0) {
          const f32x16_t zero = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
          S[tb][h] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(af, t, zero, 0, 0, 0);
        } else {
          S[tb][h] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(af, t, S[tb][h], 0, 0, 0);
        }
        __builtin_amdgcn_sched_barrier(0);
        // group kk of the previous phase's 8 groups (token set kk >> 2, scores 4 (kk & 3) .. + 3), behind the first
        // MFMA of the pair
        constexpr int ctb = kk >> 2, q = kk & 3;
        if constexpr (tb == 0) group_step(S[ctb][1 - h], ctb, std::integral_constant<int, q>{});
        __builtin_amdgcn_sched_barrier(0);
      });
    });
    // the scores just examined belong to the half before this one
    bhalf[0] = (best[0] > before0) ? half_id - 1 : bhalf[0];
    bhalf[1] = (best[1] > before1) ? half_id - 1 : bhalf[1];
  };
  const int nchunks = (a.C + kCB - 1) / kCB;
  // this part's blocks c0 .. c1 - 1; every part passes the barrier of every step, also one whose blocks have run out
  const int steps = (nchunks + PARTS - 1) / PARTS;
  const int c0 = PARTS > 1 ? min(part * steps, nchunks) : 0;
  const int c1 = PARTS > 1 ? min(c0 + steps, nchunks) : nchunks;
  auto walk = [&](int c0, int c1, int steps) __attribute__((always_inline)) {
    if (PARTS == 1 || c0 < c1) stage(c0, 0);
    for (int step = 0; step < steps; ++step) {
      const int chunk = c0 + step;
      __builtin_amdgcn_s_waitcnt(0);
      // block `chunk` has landed for every wave, and every wave has finished reading block chunk - 1, whose buffer the
      // next block may now overwrite; it has this block's 32 MFMAs per wave to arrive
      __syncthreads();
      __builtin_amdgcn_sched_barrier(0);
      if (PARTS > 1 && chunk >= c1) continue;   // wave-uniform
      if (chunk + 1 < c1) stage(chunk + 1, (step + 1) & 1);
      const uint32_t boff = (step & 1) * (kCB * 256);
      u32x4_t fr[16];
      static_for<0, kFragAhead>([&](auto I) { fr[decltype(I)::value] = frag(boff, I); });
      __builtin_amdgcn_sched_barrier(0);
      phase(std::integral_constant<int, 0>{}, boff, 2 * chunk, fr);
      phase(std::integral_constant<int, 1>{}, boff, 2 * chunk + 1, fr);
    }
    {   // the last half block
      const float before0 = best[0], before1 = best[1];
      static_for<0, 2>([&](auto TB) {
        static_for<0, 4>([&](auto Q) { group_step(S[decltype(TB)::value][1], decltype(TB)::value, Q); });
      });
      bhalf[0] = (best[0] > before0) ? 2 * c1 - 1 : bhalf[0];
      bhalf[1] = (best[1] > before1) ? 2 * c1 - 1 : bhalf[1];
    }
  };
  float bv2[2];
  int bidx2[2];
  auto result = [&]() __attribute__((always_inline)) {   // best score and its place, the same in a token's two lanes
#pragma unroll
    for (int tb = 0; tb < 2; ++tb) {
      const int in_group = (keep0[tb] == best[tb]) ? 0 : (keep1[tb] == best[tb]) ? 1 : (keep2[tb] == best[tb]) ? 2 : 3;
      int bidx = bhalf[tb] * 32 + 4 * g + 8 * bgrp[tb] + in_group;
      float bv = best[tb];
      const float ob = __shfl_xor(bv, 32);
      const int oi = __shfl_xor(bidx, 32);
      if (ob > bv || (ob == bv && oi < bidx)) {
        bv = ob;
        bidx = oi;
      }
      bv2[tb] = bv;
      bidx2[tb] = bidx;
      if constexpr (PARTS > 1) {
        if (g == 0) {
          s_best[wave * 64 + 32 * tb + c32] = bv;
          s_bidx[wave * 64 + 32 * tb + c32] = bidx;
        }
      }
    }
  };
  if constexpr (!NEAR) {
    walk(c0, c1, steps);
    result();
  } else {
    const int words = a.C / 32;
    float xx[2] = {0.f, 0.f};
    bool all = dense;
    if (!dense) {
      if (tid < words) s_mask[tid] = 0u;
      if (tid == 0) s_all = a.near.odd[g_id];
      // the masks of the wave's clusters: lane l looks at token l of its 64, a lane whose neighbour's token is in the same cluster adds
      // nothing; four rows in flight
      const int mine = g ? old_idx[1] : old_idx[0];
      const bool valid = tok0 + lane < a.N, known = valid && (uint32_t)mine < (uint32_t)a.C;
      const int before = __shfl_up(mine, 1);
      unsigned long long heads = __ballot(known && (lane == 0 || mine != before));
      const uint32_t* rows = a.near.mask + (int64_t)g_id * a.C * words;
      auto four = [&](uint32_t (&r)[4]) __attribute__((always_inline)) {
#pragma unroll
        for (int u = 0; u < 4; ++u) {
          const int at = heads != 0 ? __ffsll(heads) - 1 : -1;
          const int c = at >= 0 ? __builtin_amdgcn_readlane(mine, at) : -1;
          r[u] = at >= 0 && lane < words ? rows[(int64_t)c * words + lane] : 0u;
          heads &= heads - 1;
        }
      };
      uint32_t r[4];
      four(r);
      // |x|^2 of this lane's tokens: half of the channels here, the others in the lane 32 away
#pragma unroll
      for (int tb = 0; tb < 2; ++tb) {
        float t = 0.f;
#pragma unroll
        for (int kk = 0; kk < 8; ++kk) t = dot8_bf16(tf[tb][kk], tf[tb][kk], t);
        xx[tb] = t + __shfl_xor(t, 32);
      }
      const bool stray = !(xx[0] < INFINITY && xx[1] < INFINITY) || valid != known;
      uint32_t bits = r[0] | r[1] | r[2] | r[3];
      while (heads != 0) {
        four(r);
        bits |= r[0] | r[1] | r[2] | r[3];
      }
      __syncthreads();
      if (lane < words && bits != 0) atomicOr(&s_mask[lane], bits);
      if (stray) s_all = 1;
      __syncthreads();
      all = s_all != 0;
    }
    if (!all) {   // every wave counts, each writes its share of the list
      uint32_t m = lane < words ? s_mask[lane] : 0u;
      const int n = __popc(m), inc = wave_inclusive_scan(n, lane);
      n_list = __builtin_amdgcn_readlane(inc, 63);
      if ((lane & (kAssignWaves - 1)) == wave)
        for (int at = inc - n; m != 0; m &= m - 1) s_list[at++] = (uint16_t)(32 * lane + __ffs(m) - 1);
    }
    if (n_list == 0) {   // (a cluster's own centroid is never left out, so only where `all`)
      n_list = a.C;
      whole = true;
    }
    auto centroid_at = [&](int at) { return whole ? at : (int)s_list[at]; };
    if (!dense)
      for (int i = tid; i < n_list; i += kAssignWaves * 64) {
        s_low[i] = kInfBits;
        s_far2[i] = 0u;
      }
    __syncthreads();
    if (!dense)   // (before the walk, which waits for memory anyway)
      for (int i = tid; i < n_list; i += kAssignWaves * 64) s_norm2[i] = a.near.norm2[(int64_t)g_id * a.C + centroid_at(i)];
    const int blocks = (n_list + kCB - 1) / kCB;
    walk(0, blocks, blocks);
    result();
    int place[2];
#pragma unroll
    for (int tb = 0; tb < 2; ++tb) {
      place[tb] = min(bidx2[tb], n_list - 1);
      bidx2[tb] = centroid_at(place[tb]);
    }
    if (!dense) {
#pragma unroll
      for (int tb = 0; tb < 2; ++tb) {
        const float d2 = far_squared(xx[tb], bv2[tb] * bv2[tb] / s_norm2[place[tb]]);   // (written before the walk's barriers)
        if (g == 0 && tok0 + 32 * tb + c32 < a.N) {
          atomicMin(&s_low[place[tb]], bv2[tb] > 0.f ? __float_as_uint(bv2[tb]) : 0u);
          atomicMax(&s_far2[place[tb]], __float_as_uint(d2));   // (not a number: above everything)
        }
      }
      __syncthreads();
      for (int i = tid; i < n_list; i += kAssignWaves * 64)
        if (s_low[i] != kInfBits) {
          atomicMin(a.near.low + (int64_t)g_id * a.C + centroid_at(i), s_low[i]);
          atomicMax(a.near.far2 + (int64_t)g_id * a.C + centroid_at(i), s_far2[i]);
        }
      // (a run's first carried step has the longest lists; counted in each, in front of the walk, it was 0.3 - 2 us of a step)
      if (form == 0 && tid == kAssignWaves * 64 - 1 && (tile + g_id) % kWalkSample == 0)
        atomicAdd(a.near.excess, (unsigned long long)((long long)kWalkShare * n_list - a.C));
    }
  }
  if constexpr (PARTS > 1) {
    __syncthreads();
#pragma unroll
    for (int tb = 0; tb < 2; ++tb)
#pragma unroll
      for (int p = 1; p < PARTS; ++p) {
        const float ob = s_best[(sub * PARTS + p) * 64 + 32 * tb + c32];
        const int oi = s_bidx[(sub * PARTS + p) * 64 + 32 * tb + c32];
        if (ob > bv2[tb]) {   // a tie stays with the lower part, whose indices are lower; so does a token without a score above -inf (NaN)
          bv2[tb] = ob;
          bidx2[tb] = oi;
        }
      }
  }
  const bool writes = g == 0 && part == 0;
#pragma unroll
  for (int tb = 0; tb < 2; ++tb) {
    const int bidx = bidx2[tb];
    const int n = tok[tb];
    const bool valid = tok0 + 32 * tb + c32 < a.N;
    // cluster sizes come out of the counting sort that follows (per-tile histograms), not out of global atomics
    if (writes && valid && (!NEAR || old_idx[tb] != bidx)) a.idx[(int64_t)g_id * a.i_sg + n] = bidx;
    if constexpr (TRACK) {
      const bool changed = writes && valid && old_idx[tb] != bidx;
      const unsigned long long m = __ballot(changed);
      if (m != 0) {   // wave-uniform
        int base = 0;
        if (lane == 0) base = atomicAdd(&s_chg_n, __popcll(m));
        base = __shfl(base, 0);
        if (changed) {
          const int pos = base + __popcll(m & ((1ull << lane) - 1ull));
          s_chg[pos] = make_uint2((uint32_t)n, ((uint32_t)old_idx[tb] << 16) | (uint32_t)bidx);
        }
      }
    }
  }
  if constexpr (TRACK) {
    __syncthreads();
    const int n_chg = s_chg_n;
    if (n_chg == 0) return;
    const int ch = tid & (kD - 1);
    const bool adds = tid < kD;
    const uint16_t* drow = db + ch;
    double* sg = a.keep_sum + (int64_t)g_id * a.C * kD + ch;
    int32_t* cg = a.keep_cnt + (int64_t)g_id * a.C;
    // NEAR: the movers of a cluster are in few workgroups, 100 and more in one, and mostly go the same way: eight rows in flight, and
    // what goes to one cluster is added up first (exactly, as everything here)
    constexpr int kMove = NEAR ? 8 : 1;
    double sum = 0;
    int to = a.C, count = 0;
    auto hand_over = [&]() {
      if (to < a.C) {   // (an old assignment that is no cluster: nothing to take it out of)
        unsafeAtomicAdd(sg + (int64_t)to * kD, adds ? sum : -sum);
        if (ch == 0) atomicAdd(cg + to, adds ? count : -count);
      }
    };
    for (int i0 = 0; i0 < n_chg; i0 += kMove) {
      uint2 e[kMove];
      uint16_t x16[kMove];
#pragma unroll
      for (int u = 0; u < kMove; ++u) e[u] = s_chg[min(i0 + u, n_chg - 1)];
#pragma unroll
      for (int u = 0; u < kMove; ++u) x16[u] = drow[(int64_t)e[u].x * a.d_sn];
#pragma unroll
      for (int u = 0; u < kMove; ++u) {
        const int c = adds ? (int)(e[u].y & 0xffffu) : (int)(e[u].y >> 16);
        if (i0 + u >= n_chg) continue;
        if (!NEAR || c != to) {
          hand_over();
          sum = 0;
          count = 0;
          to = c;
        }
        sum += (double)bf16_bits_to_f32(x16[u]);
        ++count;
      }
    }
    hand_over();
  }
}

// Which centroids can win a token of which cluster (NEAR).  With data whose clusters overlap nothing can be left out, and the gather
// and the lists only cost: where more than an eighth of all (token, centroid) pairs remain, everything is walked in the tokens' own
// order, from that step on.  A cluster's mask does not say what a workgroup walks, which is all that any of its clusters wants: where clusters
// are small, 256 tokens of many clusters have long lists out of short masks.  So what is walked is counted too, in the first carried step,
// and more than a fifth ends it the same way (ten steps of 16 x 16384 tokens, 1024 centroids around 512 centres of width 0.5: 1.28 times
// the run without bounds -> 1.10, and of 64 x 4096, width 0.3: 1.97 -> 1.16, both with the trial's and the bounds' savings below; a
// third, a fifth and an eighth are alike within 1 % at 4 x 131072 and 4 x 70000).
// A wave takes 32 clusters a (columns) against 32 centroids j (rows), so that a lane has one cluster.
struct BoundsArgs {
  const uint16_t* cent;   // [G,C,128] bf16
  NearState near;
  const int32_t* cnt;     // [G,C]
  int64_t c_sg, c_sc;
  int32_t C;
  int32_t every;          // blocks of clusters: every so many-th
};

constexpr int kBoundsWaves = 8;
__global__ __launch_bounds__(kBoundsWaves * 64) void kmeans_bounds_kernel(BoundsArgs a) {
  // rows of 256 bytes, chunk c of row r in slot c ^ (r & 15): centroids a, used centroids a, a block of centroids j per wave
  // (80 KB and not a byte more: two workgroups on a CU, 9.1 us instead of 11.7; what is wanted in addition goes where a wave's block was)
  __shared__ __attribute__((aligned(16))) char smem[(2 + kBoundsWaves) * 32 * 256];
  typedef __attribute__((address_space(3))) void* lds_ptr_t;
  const int g_id = blockIdx.z;
  const int lane = threadIdx.x & 63, c32 = lane & 31, g = lane >> 5;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int block = blockIdx.x * a.every, cl = 32 * block + c32, words = a.C / 32, jb = kBoundsWaves * blockIdx.y + wave;
  const uint16_t* cb = a.cent + (int64_t)g_id * a.c_sg;
  const uint16_t* ub = a.near.used + (int64_t)g_id * a.C * kD;
  auto copy = [&](const uint16_t* base, int64_t stride, int row0, int part, int q) {   // rows 4 q .. 4 q + 3 of a block of 32
    const int r = 4 * q + (lane >> 4);
    __builtin_amdgcn_global_load_lds((const void*)(base + (int64_t)min(row0 + r, a.C - 1) * stride + 8 * ((lane & 15) ^ (r & 15))),
                                     (lds_ptr_t)(smem + part * 8192 + q * 1024), 16, 0, 0);
  };
  if (*a.near.dense == 1) return;   // (asked before the rows are fetched: 16 groups of 1024 centroids 8.5 -> 4.6 us, 64 groups 29 -> 5)
  copy(cb, a.c_sc, 32 * block, 0, wave);
  copy(ub, kD, 32 * block, 1, wave);
#pragma unroll
  for (int q = 0; q < 8; ++q) copy(cb, a.c_sc, 32 * jb, 2 + wave, q);
  const int64_t gc = (int64_t)g_id * a.C;
  const float far = a.near.used_far[gc + cl], low = a.near.used_low[gc + cl];
  const int size = a.cnt[gc + cl];
  __builtin_amdgcn_s_waitcnt(0);
  __syncthreads();
  auto frag = [&](int part, int kk) { return *(const uint4*)(smem + part * 8192 + c32 * 256 + (((2 * kk + g) ^ (c32 & 15)) << 4)); };
  float cc = 0.f, uu = 0.f, uc = 0.f, jj = 0.f;
  f32x16_t vu = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f}, vc = vu;
#pragma unroll
  for (int kk = 0; kk < 8; ++kk) {
    const uint4 fc = frag(0, kk), fu = frag(1, kk), fj = frag(2 + wave, kk);
    vu = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8_t, fj), __builtin_bit_cast(bf16x8_t, fu), vu, 0, 0, 0);
    vc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8_t, fj), __builtin_bit_cast(bf16x8_t, fc), vc, 0, 0, 0);
    cc = dot8_bf16(fc, fc, cc);
    uu = dot8_bf16(fu, fu, uu);
    uc = dot8_bf16(fu, fc, uc);
    jj = dot8_bf16(fj, fj, jj);
  }
  cc += __shfl_xor(cc, 32);
  uu += __shfl_xor(uu, 32);
  uc += __shfl_xor(uc, 32);
  jj += __shfl_xor(jj, 32);
  float* const norm2 = (float*)(smem + (2 + wave) * 8192);   // (the wave has read its block, and reads these alone)
  if (g == 0) norm2[c32] = jj;
  if (jb == 0 && g == 0) {
    a.near.norm2[gc + cl] = cc;
    if (!(cc < INFINITY)) a.near.odd[g_id] = 1;
  }
  // Left out where scale <c', c_a - c_j> - slack > R |c_j - c_a|, without the root of the right side.  |x| <= 32 R by the margin in
  // R, so the slack covers the errors of two scores (2e-5 |x| times the centroids' lengths) and of the products here.  Of a faint
  // centroid nothing is known: scale is no number then, and nothing left out; a lead whose square is hardly above the smallest 32-bit numbers is none.
  const float scale = fminf(uu, cc) >= kFaint ? low / uu : __uint_as_float(kNanBits), far2 = far * far, len_c = __builtin_amdgcn_sqrtf(cc);
  uint32_t bits = 0;
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    const float4 n4 = *(const float4*)&norm2[8 * q + 4 * g];
    const float n[4] = {n4.x, n4.y, n4.z, n4.w};
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const int i = 4 * q + e;
      const float dist2 = n[e] + cc - 2.f * vc[i] + 1e-3f * (n[e] + cc);
      const float lead = scale * (uc - vu[i]) - 4e-3f * far * (len_c + __builtin_amdgcn_sqrtf(n[e]));
      if (!(lead > 1e-18f && lead * lead > far2 * dist2)) bits |= 1u << (8 * q + 4 * g + e);
    }
  }
  bits |= (uint32_t)__shfl_xor((int)bits, 32);
  if (jb >= words) bits = 0;   // (a wave without a block of its own: the last rows over again)
  if (g == 0) {
    if (jb < words) a.near.mask[(gc + cl) * words + jb] = bits;
    ((int32_t*)norm2)[32 + c32] = __popc(bits);
  }
  if (block % kPairSample != 0) return;   // (one word to add to, for all of them 5 us)
  __syncthreads();
  if (threadIdx.x < 64) {   // (lane: cluster c32 again)
    unsigned long long sum = 0;
    if (g == 0)
      for (int w = 0; w < kBoundsWaves; ++w) sum += ((const int32_t*)(smem + (2 + w) * 8192))[32 + c32];
    sum *= (unsigned long long)size;
#pragma unroll
    for (int d = 1; d < 32; d <<= 1) sum += __shfl_xor(sum, d);
    if (lane == 0) atomicAdd(a.near.pairs, sum);
  }
}

// The tokens of a group cluster by cluster, for the NEAR form: places from the clusters' sizes, then every tile of kOrderTile tokens
// reserves its share of a cluster's range.  The order inside a cluster is whatever comes out; no result depends on it.
struct OrderArgs {
  const int32_t* idx;   // [G,N]
  const int32_t* cnt;   // [G,C]
  NearState near;
  int64_t i_sg;
  int32_t N, C;
};

// Clusters come in falling order of size (32 steps of a quarter of the mean): those that hold several groups of the data, whose tokens
// everything has to be walked for, are the large ones, and as the last workgroups they would run alone.
__global__ __launch_bounds__(1024) void order_start_kernel(OrderArgs a) {
  constexpr int kSteps = 32;
  __shared__ int32_t total[kSteps];
  const int g = blockIdx.x, t = threadIdx.x;
  if (g == 0) {
    if (t == 0) {
      *a.near.pairs = 0;
      *a.near.excess = 0;
      *a.near.dense = 0;
    }
    for (int i = t; i < a.near.G; i += 1024) a.near.odd[i] = 0;
  }
  if (t < kSteps) total[t] = 0;
  __syncthreads();
  int at[kNearMaxC / 1024], step[kNearMaxC / 1024];
#pragma unroll
  for (int u = 0; u < kNearMaxC / 1024; ++u) {
    const int i = 1024 * u + t;
    if (i >= a.C) continue;
    const int n = a.cnt[(int64_t)g * a.C + i];
    step[u] = kSteps - 1 - (int)min((int64_t)n * 4 * a.C / a.N, (int64_t)(kSteps - 1));
    at[u] = atomicAdd(&total[step[u]], n);
  }
  __syncthreads();
#pragma unroll
  for (int u = 0; u < kNearMaxC / 1024; ++u) {
    const int i = 1024 * u + t;
    if (i >= a.C) continue;
    for (int w = 0; w < step[u]; ++w) at[u] += total[w];
    a.near.cursor[(int64_t)g * a.C + i] = at[u];
    a.near.low[(int64_t)g * a.C + i] = kInfBits;
    a.near.far2[(int64_t)g * a.C + i] = 0u;
  }
}

constexpr int kOrderTile = 4096;

__global__ __launch_bounds__(1024) void order_fill_kernel(OrderArgs a) {
  __shared__ int32_t hist[kNearMaxC];
  const int g = blockIdx.y, t = threadIdx.x;
  if (*a.near.pairs > a.near.limit) {
    if (g == 0 && blockIdx.x == 0 && t == 0) *a.near.dense = 1;
    return;
  }
  for (int i = t; i < a.C; i += 1024) hist[i] = 0;
  __syncthreads();
  int c[kOrderTile / 1024], rank[kOrderTile / 1024];
#pragma unroll
  for (int u = 0; u < kOrderTile / 1024; ++u) {
    const int n = blockIdx.x * kOrderTile + u * 1024 + t;
    c[u] = n < a.N ? a.idx[(int64_t)g * a.i_sg + n] : -1;
    if (c[u] >= a.C) c[u] = -1;
    rank[u] = c[u] >= 0 ? atomicAdd(&hist[c[u]], 1) : 0;
  }
  __syncthreads();
  for (int i = t; i < a.C; i += 1024)
    if (hist[i] > 0) hist[i] = atomicAdd(a.near.cursor + (int64_t)g * a.C + i, hist[i]);
  __syncthreads();
#pragma unroll
  for (int u = 0; u < kOrderTile / 1024; ++u) {
    if (c[u] < 0) continue;
    const int at = hist[c[u]] + rank[u];
    if (at < a.N) a.near.order[(int64_t)g * a.N + at] = blockIdx.x * kOrderTile + u * 1024 + t;
  }
}

// What the bounds want to know of a cluster's tokens, before an assignment has collected it: against the centroid the sums have just
// given (the one the tokens were assigned by can still be far from their mean: 121 us for the step to come, 62 us from here).
// SAMPLE: a trial with the clusters whose pairs are counted (every kPairSample-th block of 32), and of each a token from each of up to 16
// tiles, out of the grouping of the sums.  Their distances are at most the cluster's, so where the bounds leave too much in by these
// they do by all, and the order and the pass over all rows can be spared (this pass and its bounds, 8 x 33000 tokens, 1024 centroids:
// 28 us with all clusters, 12 us with these).  Otherwise all tokens, bound by the rows it gathers: 30 us for 134 MB.  Not for clusters of
// 8 times the mean size and more, which would hold up the launch.
struct ReachArgs {
  const uint16_t* data;   // [G,N,128] bf16
  const uint16_t* cent;   // [G,C,128] bf16
  const int32_t* cnt;     // [G,C]
  NearState near;
  const int32_t* tile_order;   // SAMPLE: SumArgs' order and start
  const int32_t* tile_start;
  int64_t d_sg, d_sn, c_sg, c_sc;
  int32_t N, C, nT;
};

template <bool SAMPLE>
__global__ __launch_bounds__(256) void near_reach_kernel(ReachArgs a) {
  constexpr int kRows = SAMPLE ? 1 : 4;   // in flight per thread
  __shared__ float s_low[16], s_far2[16];
  const int c = SAMPLE ? (int)(blockIdx.x / 32 * kPairSample * 32 + blockIdx.x % 32) : (int)blockIdx.x;
  const int g = blockIdx.y, o = threadIdx.x & 15, r = threadIdx.x >> 4;
  const int64_t gc = (int64_t)g * a.C + c;
  int m = a.cnt[gc];
  if (!SAMPLE) {
    if (g == 0 && c == 0 && threadIdx.x == 0) *a.near.pairs = 0;
    if (*a.near.dense == 1) return;
  }
  const uint4 cen = *(const uint4*)(a.cent + (int64_t)g * a.c_sg + (int64_t)c * a.c_sc + 8 * o);
  if (threadIdx.x < 16) *(uint4*)(a.near.used + gc * kD + 8 * o) = cen;
  if (!SAMPLE && (int64_t)m * a.C >= 8 * (int64_t)a.N) {
    if (threadIdx.x == 0) a.near.used_far[gc] = __uint_as_float(kNanBits);
    return;
  }
  const int32_t* ids;
  if constexpr (SAMPLE) {   // thread's row: the first token of the cluster in tile r
    const int32_t* st = a.tile_start + ((int64_t)g * a.nT + min(r, a.nT - 1)) * (a.C + 1) + c;
    ids = a.tile_order + (int64_t)g * a.N + (int64_t)min(r, a.nT - 1) * kBigTile + st[0];
    m = r < a.nT && st[1] > st[0] ? r + 1 : 0;   // one round of the loop below, or none
  } else {
    ids = a.near.order + (int64_t)g * a.N + a.near.cursor[gc] - m;   // the cursor has moved to the end of the range
  }
  const uint16_t* db = a.data + (int64_t)g * a.d_sg + 8 * o;
  const float inv_n = 1.f / sum16(dot8_bf16(cen, cen, 0.f));
  float low = INFINITY, far2 = 0.f;
  for (int i0 = r; i0 < m; i0 += 16 * kRows) {
    uint4 x[kRows];
#pragma unroll
    for (int u = 0; u < kRows; ++u) x[u] = *(const uint4*)(db + (int64_t)ids[SAMPLE ? 0 : min(i0 + 16 * u, m - 1)] * a.d_sn);
#pragma unroll
    for (int u = 0; u < kRows; ++u) {
      const float score = sum16(dot8_bf16(x[u], cen, 0.f)), xx = sum16(dot8_bf16(x[u], x[u], 0.f)), d2 = far_squared(xx, score * score * inv_n);
      low = fminf(low, score);
      far2 = far2 != far2 || far2 >= d2 ? far2 : d2;   // keeps what is not a number
    }
  }
  if (o == 0) {
    s_low[r] = low;
    s_far2[r] = far2;
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    for (int i = 1; i < 16; ++i) {
      low = fminf(low, s_low[i]);
      far2 = far2 != far2 || far2 >= s_far2[i] ? far2 : s_far2[i];
    }
    a.near.used_low[gc] = fmaxf(low, 0.f);
    a.near.used_far[gc] = sqrtf(far2);
  }
}

// ------------------------------------------------------------------------- counting sort by cluster
struct SortArgs {
  const int32_t* idx;     // [G,N]
  int32_t* tile_hist;     // [G,nT,C]  in: per-tile histogram, after scan: exclusive prefix over tiles
  int32_t* total;         // [G,C]     cluster sizes (written by the scan)
  int32_t* dst;           // clusters [G,C,M]
  int64_t i_sg, dst_sg, dst_sc;
  int32_t N, C, nT, M;
};

__global__ __launch_bounds__(kTileTok) void sort_hist_kernel(SortArgs a) {
  extern __shared__ int32_t hist[];
  const int tile = blockIdx.x, g = blockIdx.y;
  for (int c = threadIdx.x; c < a.C; c += blockDim.x) hist[c] = 0;
  __syncthreads();
  const int n = tile * kTileTok + threadIdx.x;
  if (n < a.N) {
    const int c = a.idx[(int64_t)g * a.i_sg + n];
    if (c >= 0 && c < a.C) atomicAdd(&hist[c], 1);
  }
  __syncthreads();
  int32_t* out = a.tile_hist + ((int64_t)g * a.nT + tile) * a.C;
  for (int c = threadIdx.x; c < a.C; c += blockDim.x) out[c] = hist[c];
}

// Exclusive prefix over tiles of every cluster's per-tile count.  Workgroup = 32 clusters x 32 tile segments:
// each thread sums its segment, the 32 segment sums are scanned through LDS, then each thread rewrites its segment.
constexpr int kScanSegs = 32;
__global__ __launch_bounds__(32 * kScanSegs) void sort_scan_tiles_kernel(SortArgs a) {
  __shared__ int32_t seg_sum[kScanSegs][32];
  const int cl = threadIdx.x & 31, seg = threadIdx.x >> 5;
  const int c = blockIdx.x * 32 + cl, g = blockIdx.y;
  const int per = (a.nT + kScanSegs - 1) / kScanSegs;
  const int tb = seg * per, te = min(tb + per, a.nT);
  int32_t* h = a.tile_hist + (int64_t)g * a.nT * a.C + c;
  int sum = 0;
  if (c < a.C)
    for (int t = tb; t < te; ++t) sum += h[(int64_t)t * a.C];
  seg_sum[seg][cl] = sum;
  __syncthreads();
  int run = 0, total = 0;
#pragma unroll
  for (int q = 0; q < kScanSegs; ++q) {
    const int v = seg_sum[q][cl];
    if (q < seg) run += v;
    total += v;
  }
  if (c >= a.C) return;
  for (int t = tb; t < te; ++t) {
    const int v = h[(int64_t)t * a.C];
    h[(int64_t)t * a.C] = run;
    run += v;
  }
  if (seg == 0) a.total[(int64_t)g * a.C + c] = total;
}

__global__ __launch_bounds__(kTileTok) void sort_scatter_kernel(SortArgs a) {
  __shared__ int32_t cl[kTileTok];
  const int tile = blockIdx.x, g = blockIdx.y, t = threadIdx.x;
  const int n = tile * kTileTok + t;
  const int c = (n < a.N) ? a.idx[(int64_t)g * a.i_sg + n] : -1;
  cl[t] = c;
  __syncthreads();
  if (c < 0 || c >= a.C) return;
  int rank = 0;
  for (int u = 0; u < t; ++u) rank += (cl[u] == c);   // tokens of a tile keep their ascending order
  const int base = a.tile_hist[((int64_t)g * a.nT + tile) * a.C + c] + rank;
  if (base < a.M) a.dst[(int64_t)g * a.dst_sg + (int64_t)c * a.dst_sc + base] = n;
}

// Grouping without a global order, for the callers that only sum the rows of a cluster afterwards (centroid update,
// index_add): those sums are exact, so neither the order of the addends nor where a cluster's tokens lie matters.  A
// workgroup sorts its own tile of kBigTile tokens by cluster and nothing else: LDS histogram (the atomic's return value is
// the token's rank inside its (tile, cluster) range), exclusive prefix over the clusters, token ids written to
// order[tile * kBigTile + start[c] + rank].  start[tile][0..C] goes to memory; the sum kernel of cluster c walks the
// tiles and picks up order[tile][start[c] .. start[c + 1]) from each.  One launch, no pass that depends on all tiles.
//
// Clusters are summed by one workgroup each, so a cluster that has swallowed a large part of the tokens (the second
// Lloyd iteration from evenly spaced seeds does that: 50 000 of 131 072 tokens in one cluster, 0.5 ms in one workgroup)
// would hold up the whole step.  Tiles all have the same number of tokens, so the tile's workgroup takes that work: a
// (tile, cluster) range of kHeavy tokens or more is summed right here, in fp64, into rec[tile][start / kHeavy][128]
// (ranges that long cannot share a block of kHeavy positions, so the slot is unique), and the cluster's workgroup adds
// the records instead of the rows.
constexpr int kHeavy = 64;                      // tokens of one cluster in one tile from which the tile sums them itself
constexpr int kSlots = kBigTile / kHeavy;

struct GroupArgs {
  const int32_t* idx;     // [G,N]
  const uint16_t* src;    // [G,N,128] bf16 rows that will be summed
  int32_t* start;         // [G,nT,C+1]
  int32_t* order;         // [G,N]
  double* rec;            // [G,nT,kSlots,128]
  int64_t i_sg, s_sg, s_sn;
  int32_t N, C, nT;
};

__device__ __forceinline__ void add_row_bf16(double (&acc)[8], const uint4& raw) {
  const uint32_t w[4] = {raw.x, raw.y, raw.z, raw.w};
#pragma unroll
  for (int e = 0; e < 8; ++e) {
    const uint32_t bits = (e & 1) ? (w[e >> 1] >> 16) : (w[e >> 1] & 0xffffu);
    acc[e] += (double)bf16_bits_to_f32(bits);
  }
}

constexpr int kMaxItems = 2 * kSlots;   // pieces of at most kHeavy rows: sum over ranges of ceil(m / kHeavy) <= kBigTile / kHeavy + ranges

__global__ __launch_bounds__(1024) void tile_group_kernel(GroupArgs a) {
  extern __shared__ double racc[];       // [kSlots][128] sums of the long ranges; then C counters / start positions; then the sorted ids
  __shared__ int32_t wsum[16];
  __shared__ int32_t item[kMaxItems][3]; // (first position, rows, slot) of a piece of a long range
  __shared__ int32_t used[kSlots];
  __shared__ int32_t n_items;
  int32_t* hist = (int32_t*)(racc + kSlots * kD);
  int32_t* ids = hist + a.C;
  const int tile = blockIdx.x, g = blockIdx.y, t = threadIdx.x, lane = t & 63, wave = t >> 6;
  int c[kBigTok], rank[kBigTok];
#pragma unroll
  for (int u = 0; u < kBigTok; ++u) {
    const int n = tile * kBigTile + u * 1024 + t;
    c[u] = (n < a.N) ? a.idx[(int64_t)g * a.i_sg + n] : -1;
    if (c[u] >= a.C) c[u] = -1;
  }
  for (int i = t; i < a.C; i += 1024) hist[i] = 0;
  for (int i = t; i < kSlots * kD; i += 1024) racc[i] = 0;
  if (t < kSlots) used[t] = 0;
  if (t == 0) n_items = 0;
  __syncthreads();
#pragma unroll
  for (int u = 0; u < kBigTok; ++u) rank[u] = (c[u] >= 0) ? atomicAdd(&hist[c[u]], 1) : 0;
  __syncthreads();
  int32_t* out = a.start + ((int64_t)g * a.nT + tile) * (a.C + 1);
  int carry = 0;
  for (int c0 = 0; c0 < a.C; c0 += 1024) {
    const int i = c0 + t;
    const int v = (i < a.C) ? hist[i] : 0;
    const int inc = wave_inclusive_scan(v, lane);
    if (lane == 63) wsum[wave] = inc;
    __syncthreads();
    int wbase = 0, all = 0;
#pragma unroll
    for (int w = 0; w < 16; ++w) {
      const int x = wsum[w];
      if (w < wave) wbase += x;
      all += x;
    }
    const int ex = carry + wbase + inc - v;
    if (i < a.C) {
      hist[i] = ex;
      out[i] = ex;
      if (v >= kHeavy) {
        const int pieces = (v + kHeavy - 1) / kHeavy, sl = ex / kHeavy;
        const int first = atomicAdd(&n_items, pieces);
        used[sl] = 1;
        for (int k = 0; k < pieces; ++k) {
          item[first + k][0] = ex + k * kHeavy;
          item[first + k][1] = min(kHeavy, v - k * kHeavy);
          item[first + k][2] = sl;
        }
      }
    }
    carry += all;
    __syncthreads();
  }
  if (t == 0) out[a.C] = carry;
  int32_t* ord = a.order + (int64_t)g * a.N + (int64_t)tile * kBigTile;
#pragma unroll
  for (int u = 0; u < kBigTok; ++u)
    if (c[u] >= 0) {
      const int pos = hist[c[u]] + rank[u], n = tile * kBigTile + u * 1024 + t;
      ord[pos] = n;
      ids[pos] = n;
    }
  __syncthreads();
  const int ni = n_items;
  if (ni == 0) return;
  // a piece per wave: four rows at a time (16 lanes of 16 bytes each), all of a lane's rows requested before the first is used
  const int o = lane & 15, rg = lane >> 4;
  const uint16_t* sb = a.src + (int64_t)g * a.s_sg + 8 * o;
  for (int it = wave; it < ni; it += 16) {
    const int p0 = item[it][0], m = item[it][1], sl = item[it][2];
    uint4 raw[kHeavy / 4];
#pragma unroll
    for (int u = 0; u < kHeavy / 4; ++u) {
      const int i = rg + 4 * u;
      raw[u] = make_uint4(0, 0, 0, 0);
      if (i < m) raw[u] = *(const uint4*)(sb + (int64_t)ids[p0 + i] * a.s_sn);
    }
    double acc[8] = {0, 0, 0, 0, 0, 0, 0, 0};
#pragma unroll
    for (int u = 0; u < kHeavy / 4; ++u) add_row_bf16(acc, raw[u]);
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      acc[e] += __shfl_xor(acc[e], 16);
      acc[e] += __shfl_xor(acc[e], 32);
    }
    if (lane < 16) {
#pragma unroll
      for (int e = 0; e < 8; ++e) atomicAdd(&racc[sl * kD + 8 * o + e], acc[e]);   // exact sums: the order does not matter
    }
  }
  __syncthreads();
  double* rec = a.rec + ((int64_t)g * a.nT + tile) * kSlots * kD;
  for (int i = t; i < kSlots * kD; i += 1024)
    if (used[i / kD]) rec[i] = racc[i];
}

// ------------------------------------------------------------------------- per-cluster sum + update
struct SumArgs {
  const uint16_t* src;    // [G,N,128] bf16 rows to sum (keys for the update, values for index_add)
  const int32_t* order;   // [G,N] token ids, every tile of kBigTile tokens grouped by cluster
  const int32_t* start;   // [G,nT,C+1] where a cluster's range begins inside its tile
  const double* rec;      // [G,nT,kSlots,128] sums of the ranges of kHeavy tokens or more
  uint16_t* dst;          // [G,C,128] bf16: centroids (update) or value sums (index_add)
  int32_t* cnt;           // [G,C] cluster sizes, or null
  int64_t s_sg, s_sn, d_sg, d_sc;
  int32_t N, C, nT, mode; // mode 0: plain sum cast to bf16; 1: mean; 2: mean + L2 normalise (1,2: only where cnt > 0)
  double* keep_sum;       // [G,C,128] or null: the exact sums, left for the iterations that only apply changes
  int32_t* keep_cnt;      // [G,C] or null
};

// From a cluster's exact sum (channel t of thread t < 128) and size to its stored row: sum rounded once to fp32, mean
// (kmeans.py:121), optional L2 normalisation with the squared norm summed in fp64 in a fixed tree (:122-123), bf16
// store only where the cluster has tokens (:120, 124).  Shared by the full re-sum and by the update from kept sums, so
// the two give the same bits.  All threads of the workgroup call it (it has barriers); ss_red: 128 doubles of LDS.
__device__ __forceinline__ void finish_cluster(double s, int cnt, int mode, double* ss_red, int t, uint16_t* dst_row, int32_t* cnt_out) {
  float x = 0.f;
  if (t < kD) {
    x = (float)s;                                   // exact sum rounded once to fp32
    if (mode >= 1) x = x / (float)cnt;
    ss_red[t] = (double)x * (double)x;
  }
  __syncthreads();
  if (mode == 2) {
    for (int d = kD / 2; d > 0; d >>= 1) {
      if (t < d) ss_red[t] += ss_red[t + d];
      __syncthreads();
    }
    if (t < kD) x = x / sqrtf((float)ss_red[0]);
  }
  if (t < kD && (mode == 0 || cnt > 0)) dst_row[t] = (uint16_t)f32_to_bf16_bits(x);
  if (cnt_out && t == 0) *cnt_out = cnt;
}

constexpr int kSumRows = 4;   // rows in flight per thread (8: slower, 2: the same)
constexpr int kListCap = 2048;   // token ids staged in LDS at a time

__global__ __launch_bounds__(256) void cluster_sum_kernel(SumArgs a) {
  __shared__ double red[4][kD];
  __shared__ double ss_red[kD];
  __shared__ int32_t list[kListCap];
  __shared__ int32_t wsum[4], wbig[4];
  __shared__ int32_t slot[64];
  const int c = blockIdx.x, g = blockIdx.y, t = threadIdx.x, lane = t & 63, wave = t >> 6;
  const int o = t & 15, r = t >> 4;
  const int32_t* st = a.start + (int64_t)g * a.nT * (a.C + 1) + c;
  const int32_t* ord = a.order + (int64_t)g * a.N;
  const uint16_t* sb = a.src + (int64_t)g * a.s_sg + 8 * o;
  double acc[8] = {0, 0, 0, 0, 0, 0, 0, 0};
  double extra = 0;   // channel t of the ranges the tiles have summed already
  int cnt = 0;
  for (int tb = 0; tb < a.nT; tb += 64) {   // 64 tiles at a time, four threads per tile
    const int tile = tb + (t >> 2), q = t & 3;
    int s0 = 0, mine = 0, big = 0;
    if (tile < a.nT) {
      s0 = st[(int64_t)tile * (a.C + 1)];
      mine = st[(int64_t)tile * (a.C + 1) + 1] - s0;
    }
    if (mine >= kHeavy) {
      big = mine;
      mine = 0;
    }
    if (q == 0) slot[t >> 2] = big ? s0 / kHeavy : -1;
    const int inc = wave_inclusive_scan(q == 0 ? mine : 0, lane);
    const int binc = wave_inclusive_scan(q == 0 ? big : 0, lane);
    if (lane == 63) {
      wsum[wave] = inc;
      wbig[wave] = binc;
    }
    __syncthreads();
    int base = __shfl(inc, lane & ~3) - mine, all = 0, all_big = 0;   // where this tile's ids go in the list
#pragma unroll
    for (int w = 0; w < 4; ++w) {
      const int x = wsum[w];
      if (w < wave) base += x;
      all += x;
      all_big += wbig[w];
    }
    if (all_big > 0 && t < kD) {
      const int nt = min(64, a.nT - tb);
      for (int j = 0; j < nt; ++j)
        if (slot[j] >= 0) extra += a.rec[(((int64_t)g * a.nT + tb + j) * kSlots + slot[j]) * kD + t];
    }
    cnt += all_big;
    const int32_t* mo = ord + (int64_t)tile * kBigTile + s0;
    for (int w0 = 0; w0 < all; w0 += kListCap) {   // the ids of these tiles' tokens, kListCap at a time
      const int jb = max(0, w0 - base), je = min(mine, w0 + kListCap - base);
      for (int j = jb + q; j < je; j += 4) list[base + j - w0] = mo[j];
      __syncthreads();
      const int m = min(all - w0, kListCap);
      for (int i0 = r; i0 < m; i0 += 16 * kSumRows) {  // kSumRows rows in flight per thread
        uint4 raw[kSumRows];
#pragma unroll
        for (int u = 0; u < kSumRows; ++u) {
          const int i = i0 + 16 * u;
          raw[u] = make_uint4(0, 0, 0, 0);
          if (i < m) raw[u] = *(const uint4*)(sb + (int64_t)list[i] * a.s_sn);
        }
#pragma unroll
        for (int u = 0; u < kSumRows; ++u) add_row_bf16(acc, raw[u]);
      }
      __syncthreads();
    }
    cnt += all;
    __syncthreads();
  }
#pragma unroll
  for (int e = 0; e < 8; ++e) {   // the wave's four rows, then the four waves through LDS
    acc[e] += __shfl_xor(acc[e], 16);
    acc[e] += __shfl_xor(acc[e], 32);
  }
  if (lane < 16) {
#pragma unroll
    for (int e = 0; e < 8; ++e) red[wave][8 * o + e] = acc[e];
  }
  __syncthreads();
  double s = 0;
  if (t < kD) {
    s = extra;
#pragma unroll
    for (int rr = 0; rr < 4; ++rr) s += red[rr][t];
    if (a.keep_sum) a.keep_sum[((int64_t)g * a.C + c) * kD + t] = s;
  }
  if (a.keep_cnt && t == 0) a.keep_cnt[(int64_t)g * a.C + c] = cnt;
  finish_cluster(s, cnt, a.mode, ss_red, t, a.dst + (int64_t)g * a.d_sg + (int64_t)c * a.d_sc, a.cnt ? a.cnt + (int64_t)g * a.C + c : nullptr);
}

// ------------------------------------------------------------------------- centroids from the carried sums
struct UpdateArgs {
  const double* sum;      // [G,C,128]
  const int32_t* cnt;     // [G,C]
  uint16_t* dst;          // centroids [G,C,128] bf16
  int32_t* cnt_out;       // [G,C]
  int64_t d_sg, d_sc;
  int32_t C, mode;
  NearState near;         // order null: not kept
};

__global__ __launch_bounds__(kD) void kmeans_update_kernel(UpdateArgs a) {
  __shared__ double ss_red[kD];
  const int c = blockIdx.x, g = blockIdx.y, t = threadIdx.x;
  const double s = a.sum[((int64_t)g * a.C + c) * kD + t];
  const int cnt = a.cnt[(int64_t)g * a.C + c];
  const int64_t gc = (int64_t)g * a.C + c;
  uint16_t* row = a.dst + (int64_t)g * a.d_sg + (int64_t)c * a.d_sc;
  if (a.near.order && *a.near.dense != 1) {
    if (gc == 0 && t == 0) {
      *a.near.dense = *a.near.pairs > a.near.limit || (long long)*a.near.excess > 0 ? 1 : 2;
      *a.near.pairs = 0;
      *a.near.excess = 0;
    }
    a.near.used[gc * kD + t] = row[t];
    if (t == 0) {
      a.near.used_low[gc] = __uint_as_float(a.near.low[gc]);
      a.near.used_far[gc] = sqrtf(__uint_as_float(a.near.far2[gc]));
      a.near.low[gc] = kInfBits;
      a.near.far2[gc] = 0u;
    }
  }
  finish_cluster(s, cnt, a.mode, ss_red, t, row, a.cnt_out + gc);
}

// ---------------------------------------------------------------------------------- top-k selection
struct TopkArgs {
  const uint16_t* query;   // [B,Hq,128] bf16
  const uint16_t* cent;    // [G,C,128] bf16
  const int32_t* clusters; // [G,C,M]
  const int32_t* size;     // [G,C]
  int32_t* out;            // [G,k], rows out_sg apart
  int64_t out_sg;
  float* score;            // workspace [G,C]
  int32_t* start;          // workspace [G,C] start position of each cluster in rank order (two-kernel path)
  unsigned long long* scored;   // workspace [G,C] score and tag of the shared score phase (one-launch path; the memory of `score` and `start`)
  uint32_t tag;
  int32_t share;           // waves (64 clusters each) per workgroup of the shared score phase
  int64_t q_sb, q_sh, c_sg, c_sc, cl_sg, cl_sc;
  int32_t C, M, k, Hkv, group;
};

// Cluster score = max over the kv head's q heads of <q_h, centroid>: one thread per centroid, the centroid row in
// registers (sixteen 16-byte loads), the group's queries in LDS as fp32; every dot product is one fp32 FMA chain over
// d = 0..127 in order.
__global__ __launch_bounds__(256) void topk_score_kernel(TopkArgs a) {
  __shared__ float qs[16][kD];
  const int g = blockIdx.y, b = g / a.Hkv, kvh = g % a.Hkv;
  const int nh = a.group < 16 ? a.group : 16;
  for (int i = threadIdx.x; i < nh * kD; i += blockDim.x) {
    const int h = i / kD, d = i % kD;
    qs[h][d] = bf16_bits_to_f32(a.query[(int64_t)b * a.q_sb + (int64_t)(kvh * a.group + h) * a.q_sh + d]);
  }
  __syncthreads();
  const int c = blockIdx.x * blockDim.x + threadIdx.x;
  if (c >= a.C) return;
  const uint16_t* cp = a.cent + (int64_t)g * a.c_sg + (int64_t)c * a.c_sc;
  float best = -INFINITY;
  if (a.group <= 16) {
    float cf[kD];
#pragma unroll
    for (int j = 0; j < kD / 8; ++j) {
      const uint4 w = *(const uint4*)(cp + 8 * j);
      const uint32_t ww[4] = {w.x, w.y, w.z, w.w};
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        cf[8 * j + 2 * e] = bf16_bits_to_f32(ww[e] & 0xffffu);
        cf[8 * j + 2 * e + 1] = bf16_bits_to_f32(ww[e] >> 16);
      }
    }
    for (int h = 0; h < nh; ++h) {
      float sacc = 0.f;
#pragma unroll
      for (int d = 0; d < kD; ++d) sacc += qs[h][d] * cf[d];
      best = fmaxf(best, sacc);
    }
  } else {   // more than 16 q heads per kv head: straight from memory
    for (int h = 0; h < a.group; ++h) {
      const uint16_t* qp = a.query + (int64_t)b * a.q_sb + (int64_t)(kvh * a.group + h) * a.q_sh;
      float sacc = 0.f;
      for (int d = 0; d < kD; ++d) sacc += bf16_bits_to_f32(qp[d]) * bf16_bits_to_f32(cp[d]);
      best = fmaxf(best, sacc);
    }
  }
  a.score[(int64_t)g * a.C + c] = best;
}

// Order the clusters by (score descending, index ascending), prefix-sum their sizes in that order and emit the first k
// token ids: one workgroup per group, everything in LDS.  The order comes from a bitonic sort of 64-bit keys
// (score mapped to an unsigned integer of the same order in the high word, ~index in the low word; a counting rank
// with C compares per cluster took 50 us at C = 1024).  Each output position finds its cluster by a binary search
// over the prefix; positions past the total number of tokens get -1.
__global__ __launch_bounds__(1024) void topk_emit_kernel(TopkArgs a) {
  extern __shared__ int32_t sh[];          // [P] 64-bit keys (P = C rounded up to a power of two), then [C + 1] prefix
  int P = 1;
  while (P < a.C) P <<= 1;
  unsigned long long* key = (unsigned long long*)sh;
  int32_t* pre = sh + 2 * P;
  __shared__ int32_t part[1024];
  const int g = blockIdx.x, t = threadIdx.x;
  const int32_t* size = a.size + (int64_t)g * a.C;
  for (int c = t; c < P; c += blockDim.x) {
    unsigned long long kk = 0;             // padding sorts behind every cluster
    if (c < a.C) {
      const uint32_t bits = __float_as_uint(a.score[(int64_t)g * a.C + c] + 0.0f);    // -0.0 counts as +0.0
      const uint32_t ord = (bits & 0x80000000u) ? ~bits : (bits | 0x80000000u);
      kk = ((unsigned long long)ord << 32) | (0xffffffffu - (uint32_t)c);
    }
    key[c] = kk;
  }
  __syncthreads();
  for (int len = 2; len <= P; len <<= 1)
    for (int d = len >> 1; d > 0; d >>= 1) {
      for (int i = t; i < P / 2; i += blockDim.x) {
        const int lo = ((i & ~(d - 1)) << 1) | (i & (d - 1)), hi = lo | d;
        const bool descending = (lo & len) == 0;
        const unsigned long long x = key[lo], y = key[hi];
        if ((x < y) == descending) {
          key[lo] = y;
          key[hi] = x;
        }
      }
      __syncthreads();
    }
  auto by_rank = [&](int r) { return (int)(0xffffffffu - (uint32_t)key[r]); };
  // exclusive prefix of the (clamped) sizes in rank order: per-thread runs of `per` ranks, a scan over the 1024 run sums
  const int per = (a.C + 1023) / 1024;
  int run = 0;
  for (int i = 0; i < per; ++i) {
    const int r = t * per + i;
    if (r < a.C) run += min(size[by_rank(r)], a.M);
  }
  part[t] = run;
  __syncthreads();
  for (int d = 1; d < 1024; d <<= 1) {   // Hillis-Steele inclusive scan
    const int v = (t >= d) ? part[t - d] : 0;
    __syncthreads();
    part[t] += v;
    __syncthreads();
  }
  int acc = part[t] - run;
  for (int i = 0; i < per; ++i) {
    const int r = t * per + i;
    if (r < a.C) {
      pre[r] = acc;
      acc += min(size[by_rank(r)], a.M);
    }
  }
  if (t == 1023) pre[a.C] = part[1023];
  __syncthreads();
  const int total = pre[a.C];
  int32_t* out = a.out + (int64_t)g * a.out_sg;
  for (int p = t; p < a.k; p += blockDim.x) {
    int32_t id = -1;
    if (p < total) {
      int lo = 0, hi = a.C;               // the rank r with pre[r] <= p < pre[r + 1]
      while (hi - lo > 1) {
        const int mid = (lo + hi) >> 1;
        if (pre[mid] <= p) lo = mid;
        else hi = mid;
      }
      id = a.clusters[(int64_t)g * a.cl_sg + (int64_t)by_rank(lo) * a.cl_sc + (p - pre[lo])];
    }
    out[p] = id;
  }
}


// ---- the same selection in one launch, without ordering all clusters (at most 1024 clusters and 16 q heads per kv head;
// other shapes take the two kernels above).  One workgroup of 1024 threads per group, one cluster per thread:
//   1. scores of all clusters on the matrix cores (fp32 accumulation of exact bf16 products), maximum over the q heads;
//   2. the clusters that can take part are found from one histogram in LDS: 512 equal bins between the largest and the
//      smallest score, weighted by cluster size, read from the top bin down by one wave until k tokens are covered.  The
//      bin of a score is a monotone function of it, so all clusters above the pivot bin together hold fewer than k
//      tokens and those in it complete them: every cluster at or above the pivot bin is a candidate;
//   3. only the candidates (a few dozen of 1024 for k = 4096) are ordered by (score descending, index ascending): rank and
//      number of tokens ahead by comparing all pairs while there are at most 256 of them, the bitonic network otherwise;
//   4. every output position finds its cluster by binary search.
// Bound by latency: a chain of dependent steps of one workgroup, each run once, so that fetching its instructions counts as
// much as running them.  4 x 1024 clusters, k = 4096, in us (clock reads in the kernel; in brackets: one workgroup in four scores
// with a masked maximum per head column, hand-over by fences and an arrival counter, two rounds of 256 bins over the key
// bits, ranks and prefix in separate passes): scores 2.9 (4.0), hand-over 0.8 (3.1), pivot 1.2 (1.9), order 1.0 (1.5), ids
// 1.9 (2.0); the kernel 8.8 (14.1).
constexpr int kSelCount = 256;   // candidates ranked by counting; more go through the bitonic network
constexpr int kSelBins = 512;

// inclusive sum over the lanes of a wave
__device__ __forceinline__ int wave_scan_add(int v) {
  v += __builtin_amdgcn_update_dpp(0, v, 0x111, 0xf, 0xf, false);   // row_shr 1, 2, 4, 8: within 16 lanes
  v += __builtin_amdgcn_update_dpp(0, v, 0x112, 0xf, 0xf, false);
  v += __builtin_amdgcn_update_dpp(0, v, 0x114, 0xf, 0xf, false);
  v += __builtin_amdgcn_update_dpp(0, v, 0x118, 0xf, 0xf, false);
  v += __builtin_amdgcn_update_dpp(0, v, 0x142, 0xa, 0xf, false);   // row_bcast 15: into rows 1 and 3
  v += __builtin_amdgcn_update_dpp(0, v, 0x143, 0xc, 0xf, false);   // row_bcast 31: into rows 2 and 3
  return v;
}

// maximum over the 16 lanes of a row by rotations within the row (DPP row_ror 1, 2, 4, 8): no LDS traffic
__device__ __forceinline__ float row_max16(float v) {
  v = fmaxf(v, __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x121, 0xf, 0xf, false)));
  v = fmaxf(v, __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x122, 0xf, 0xf, false)));
  v = fmaxf(v, __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x124, 0xf, 0xf, false)));
  return fmaxf(v, __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x128, 0xf, 0xf, false)));
}

// maximum over the four rows of 16 lanes: lanes 16, 32 and 48 away
__device__ __forceinline__ float max_of_rows(float v) {
  const auto x = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  v = fmaxf(__uint_as_float(x[0]), __uint_as_float(x[1]));
  const auto y = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  return fmaxf(__uint_as_float(y[0]), __uint_as_float(y[1]));
}

// One CU draws about 36 GB/s from memory: a head's whole centroid matrix (256 KB at 1024 clusters) took one workgroup 7 us.
// So workgroups of a (sequence, kv head) score a share of its clusters each, into the workspace, and whoever then finds all
// scores there carries on with steps 2 - 4.  Nobody waits for anybody.
//
// A score travels in one 64-bit word with the call's tag (`call_tag` in common.hpp), so finding the words of the call is
// having its scores: no counter, and no state from before the call that would have to be cleared.
//   1. the words are stored as device-scope atomics, which write through the storing XCD's L2, and every wave waits for its
//      own to be acknowledged (s_waitcnt vmcnt(0));
//   2. behind the workgroup barrier every thread loads one word with a device-scope load, which neither the CU's vector
//      cache nor its XCD's L2 answers from a line of its own.  The workgroup that passes its barrier last finds all words.
//      So may one just before it: both then write the same ids;
//   3. who has written the ids clears the words, so that a replay of the call from a graph, whose tag is the same, does not
//      take them for its own.  Nobody needs them any more: all parts have stored theirs, and a part that finds some cleared
//      leaves the ids to whoever cleared them.
// Waves (of 64 clusters) per workgroup: two, while that makes no more workgroups than there are CUs; beyond it the second
// workgroup on a CU and the ids written by several of them cost more than the shorter score phase saves.  us for 1024 clusters,
// k = 4096, shares of 2 / 4 / 16 waves: 4 heads 8.8 / 9.8 / 14.5, 32 heads 9.1 / 9.9 / 14.5, 64 heads 11.7 / 10.2 / 14.6,
// 128 heads 18.1 / 14.7 / 15.2, 256 heads 28.8 / 23.5 / 17.8; for 512 clusters 4 heads 7.8 / 8.7 / 11.1, 64 heads 8.4 / 9.1 / 11.3.
inline int topk_share(int64_t G, int waves) {
  int share = 2;
  while (share < 16 && G * ((waves + share - 1) / share) > 256) share *= 2;
  return share;
}

__global__ __launch_bounds__(1024) void topk_select_kernel(TopkArgs a) {
  __shared__ float sc[1024];
  __shared__ __align__(16) unsigned long long ckey[1024];
  __shared__ __align__(16) int32_t hw[kSelBins];
  __shared__ __align__(16) int32_t csize[1024];
  __shared__ int32_t pre[1025], rank_cluster[1024], misc[4];
  __shared__ float s_ext[2][16];
  const int g = blockIdx.x, t = threadIdx.x, lane = t & 63;
  const int parts = gridDim.y, part = blockIdx.y;
  const int b = g / a.Hkv, kvh = g % a.Hkv;
  const int nh = a.group;
  const bool have = t < a.C;
  unsigned long long* const word = a.scored + (int64_t)g * a.C;
  int sz = have ? a.size[(int64_t)g * a.C + t] : 0;   // requested ahead of the score phase
  // ---- 1. scores on the matrix cores: wave w takes clusters 64 w .. 64 w + 63 in four blocks of 16; per block
  // S[head, cluster] = queries . centroids^T on v_mfma_f32_16x16x32_bf16.  Lane (r = lane % 16, q = lane / 16) feeds query
  // head r (the group's last one again in the places of rows it does not have, which leaves the maximum what it is),
  // columns 32 kk + 8 q .. + 7, as the A operand and the same columns of centroid r as the B operand, and receives
  // S[head 4 q + i][cluster r], i < 4: the maximum over the heads is three in the lane and two exchanges.
  if ((t >> 6) < a.share) {
    const int wave = part * a.share + (t >> 6), r = lane & 15, q4 = lane >> 4;
    typedef __attribute__((ext_vector_type(4))) float f32x4;
    uint4 qf[4], cf[4][4];
    const uint16_t* qp = a.query + (int64_t)b * a.q_sb + (int64_t)(kvh * a.group + min(r, nh - 1)) * a.q_sh + 8 * q4;
#pragma unroll
    for (int kk = 0; kk < 4; ++kk) qf[kk] = *(const uint4*)(qp + 32 * kk);
    // all 20 loads are on their way before the first is used: one trip to memory instead of one per block
#pragma unroll
    for (int blk = 0; blk < 4; ++blk) {
      const int row = min(64 * wave + 16 * blk + r, a.C - 1);
      const uint16_t* cp = a.cent + (int64_t)g * a.c_sg + (int64_t)row * a.c_sc + 8 * q4;
#pragma unroll
      for (int kk = 0; kk < 4; ++kk) cf[blk][kk] = *(const uint4*)(cp + 32 * kk);
    }
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int blk = 0; blk < 4; ++blk) {
      const int c = 64 * wave + 16 * blk + r;
      f32x4 acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int kk = 0; kk < 4; ++kk)
        acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, qf[kk]), __builtin_bit_cast(bf16x8_t, cf[blk][kk]), acc, 0, 0, 0);
      // from -inf, so that a score that is NaN for every head ranks as in the two-kernel route and not by the sign of the NaN
      const float v = max_of_rows(fmaxf(fmaxf(fmaxf(acc[0], acc[1]), fmaxf(acc[2], acc[3])), -INFINITY));
      if (q4 == 0) {
        if (parts == 1) sc[c] = v;
        else if (c < a.C) __hip_atomic_store(word + c, ((unsigned long long)a.tag << 32) | __float_as_uint(v), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      }
    }
  }
  if (t < kSelBins) hw[t] = 0;
  if (t < 2) misc[t] = 0;
  ckey[t] = 0;
  float s = 0.f;
  if (parts > 1) {
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");   // step 1: this wave's scores have arrived
    __syncthreads();
    const unsigned long long w = have ? __hip_atomic_load(word + t, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) : 0;
    if (have && (uint32_t)(w >> 32) != a.tag) misc[1] = 1;
    __syncthreads();
    if (misc[1] != 0) return;    // uniform: somebody else finishes the job
    s = __uint_as_float((uint32_t)w);
  } else {
    __syncthreads();
    if (have) s = sc[t];
  }
  sz = min(sz, a.M);
  s += 0.0f;    // -0.0 counts as +0.0
  const uint32_t bits = __float_as_uint(s);
  const uint32_t key32 = (bits & 0x80000000u) ? ~bits : (bits | 0x80000000u);   // ordered like the scores
  // ---- 2. histogram between the extremes of the scores (of clusters that hold tokens), weighted by size
  {
    const bool in = sz > 0;
    const float hi = max_of_rows(row_max16(in ? s : -INFINITY)), lo = max_of_rows(row_max16(in ? -s : -INFINITY));
    if (lane == 0) {
      s_ext[0][t >> 6] = hi;
      s_ext[1][t >> 6] = lo;
    }
  }
  __syncthreads();
  const float top = row_max16(s_ext[0][lane & 15]), bottom = -row_max16(s_ext[1][lane & 15]);
  // Equal steps of the score.  Where the range is not a positive finite number (equal scores, infinities, nothing to
  // select) every cluster is in bin 0, i.e. a candidate.
  const float range = top - bottom;
  int bin = 0;
  if (range > 0.f && range < INFINITY) {
    const float x = (top - s) * ((float)(kSelBins - 1) / range);   // a range too small for the quotient: infinite or NaN, bin 0 or the last
    bin = (int)fminf(x, (float)(kSelBins - 1));
  }
  if (sz > 0) atomicAdd(&hw[bin], sz);
  __syncthreads();
  if (t < 64) {
    constexpr int per = kSelBins / 64;
    int w[per], sum = 0;
#pragma unroll
    for (int i = 0; i < per; ++i) {
      w[i] = hw[per * lane + i];
      sum += w[i];
    }
    const int inc = wave_scan_add(sum);
    const unsigned long long m = __ballot(inc >= a.k);
    int pivot = kSelBins - 1;             // fewer than k tokens in all: everything
    if (m != 0) {
      const int lp = __ffsll((long long)m) - 1;
      int cum = inc - sum, at = per * lane;
#pragma unroll
      for (int i = 0; i < per; ++i) {
        cum += w[i];
        at += cum < a.k ? 1 : 0;
      }
      pivot = __builtin_amdgcn_readlane(at, lp);
    }
    if (t == 0) misc[2] = pivot;
  }
  __syncthreads();
  // ---- 3. candidates and their order
  if (sz > 0 && bin <= misc[2]) {
    const int pos = atomicAdd(&misc[0], 1);
    ckey[pos] = ((unsigned long long)key32 << 32) | (0xffffffffu - (uint32_t)t);
    csize[pos] = sz;
  }
  __syncthreads();
  const int m = misc[0];
  if (m <= kSelCount) {
    if (t < m) {
      const unsigned long long mine = ckey[t];
      int rank = 0, ahead = 0;
      // four candidates a round, read whether they count or not (places behind the last hold key 0, which never does)
      for (int j = 0; j < m; j += 4) {
        unsigned long long k4[4];
        int z4[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          k4[i] = ckey[j + i];
          z4[i] = csize[j + i];
        }
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const bool before = k4[i] > mine;
          rank += before ? 1 : 0;
          ahead += before ? z4[i] : 0;
        }
      }
      rank_cluster[rank] = (int)(0xffffffffu - (uint32_t)mine);
      pre[rank] = ahead;
      if (rank == m - 1) pre[m] = ahead + csize[t];
    }
    if (m == 0 && t == 0) pre[0] = 0;
  } else {
    int P = 1;
    while (P < m) P <<= 1;
    // (the places behind the last candidate hold key 0, which sorts behind every candidate)
    for (int len = 2; len <= P; len <<= 1)
      for (int d = len >> 1; d > 0; d >>= 1) {
        if (t < P / 2) {
          const int lo = ((t & ~(d - 1)) << 1) | (t & (d - 1)), hi = lo | d;
          const bool descending = (lo & len) == 0;
          const unsigned long long x = ckey[lo], y = ckey[hi];
          if ((x < y) == descending) {
            ckey[lo] = y;
            ckey[hi] = x;
          }
        }
        __syncthreads();
      }
    if (t < m) {
      const int c = (int)(0xffffffffu - (uint32_t)ckey[t]);
      rank_cluster[t] = c;
      csize[t] = min(a.size[(int64_t)g * a.C + c], a.M);
    }
    __syncthreads();
    // exclusive prefix of the sizes in rank order (one wave)
    if (t < 64) {
      const int per = (m + 63) / 64;
      int run = 0;
      for (int i = 0; i < per; ++i) {
        const int r = lane * per + i;
        if (r < m) run += csize[r];
      }
      const int inc = wave_scan_add(run);
      int acc = inc - run;
      for (int i = 0; i < per; ++i) {
        const int r = lane * per + i;
        if (r < m) {
          pre[r] = acc;
          acc += csize[r];
        }
      }
      if (lane == 63) pre[m] = inc;
    }
  }
  __syncthreads();
  // ---- 4. the token ids
  const int total = pre[m];
  int32_t* out = a.out + (int64_t)g * a.out_sg;
  constexpr int U = 4;   // positions per thread and round: their table reads are independent and overlap
  for (int p0 = t; p0 < a.k; p0 += U * 1024) {
    int64_t off[U];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int p = p0 + u * 1024;
      off[u] = -1;
      if (p < a.k && p < total) {
        int lo = 0, hi = m;               // the rank r with pre[r] <= p < pre[r + 1]
        while (hi - lo > 1) {
          const int mid = (lo + hi) >> 1;
          if (pre[mid] <= p) lo = mid;
          else hi = mid;
        }
        off[u] = (int64_t)g * a.cl_sg + (int64_t)rank_cluster[lo] * a.cl_sc + (p - pre[lo]);
      }
    }
    int32_t id[U];
#pragma unroll
    for (int u = 0; u < U; ++u) id[u] = off[u] >= 0 ? a.clusters[off[u]] : -1;
#pragma unroll
    for (int u = 0; u < U; ++u)
      if (p0 + u * 1024 < a.k) out[p0 + u * 1024] = id[u];
  }
  if (parts > 1 && have) __hip_atomic_store(word + t, 0ull, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

struct WsLayout {
  size_t off_bytes, hist_bytes, order_bytes, score_bytes, start_bytes, total_bytes, rec_bytes;
  size_t sum_bytes, cnt_bytes;   // the sums and sizes carried from step to step (sq_kmeans_train_stateful)
  size_t near_order_bytes = 0, used_bytes = 0, mask_bytes = 0, table_bytes = 0, ctl_bytes = 0;   // NearState, where that form runs
  int nT, C;
  size_t rec_offset() const { return off_bytes + hist_bytes + order_bytes + score_bytes + start_bytes + total_bytes; }
  size_t sum_offset() const { return rec_offset() + rec_bytes; }
  size_t cnt_offset() const { return sum_offset() + sum_bytes; }
  size_t near_offset() const { return cnt_offset() + cnt_bytes; }
  size_t all() const { return near_offset() + near_order_bytes + used_bytes + mask_bytes + 6 * table_bytes + ctl_bytes; }
  NearState near(char* ws, int64_t G, int64_t N) const {
    NearState n = {};
    if (near_order_bytes == 0) return n;
    char* p = ws + near_offset();
    auto take = [&](size_t bytes) { char* q = p; p += bytes; return q; };
    n.order = (int32_t*)take(near_order_bytes);
    n.used = (uint16_t*)take(used_bytes);
    n.mask = (uint32_t*)take(mask_bytes);
    n.cursor = (int32_t*)take(table_bytes);
    n.used_low = (float*)take(table_bytes);
    n.used_far = (float*)take(table_bytes);
    n.low = (uint32_t*)take(table_bytes);
    n.far2 = (uint32_t*)take(table_bytes);
    n.norm2 = (float*)take(table_bytes);
    n.pairs = (unsigned long long*)take(ctl_bytes);
    n.excess = n.pairs + 1;
    n.dense = (int32_t*)(n.pairs + 2);
    n.odd = n.dense + 2;
    const unsigned long long blocks = C / 32, looked_at = (blocks + kPairSample - 1) / kPairSample;
    n.limit = (unsigned long long)G * N * C / 8 * looked_at / blocks;
    n.G = (int)G;
    return n;
  }
};

WsLayout ws_layout(int64_t G, int64_t N, int64_t C, bool bounded = false) {
  WsLayout w;
  auto up = [](size_t x) { return (x + 255) / 256 * 256; };
  w.nT = (int)((N + kTileTok - 1) / kTileTok);
  w.C = (int)C;
  w.off_bytes = up((size_t)G * (C + 1) * 4);
  w.hist_bytes = up((size_t)G * w.nT * (C + 1) * 4);   // per-tile histograms of the ordered sort, or range starts of the grouping
  w.order_bytes = up((size_t)G * N * 4);
  w.score_bytes = up((size_t)G * C * 4);
  w.start_bytes = up((size_t)G * C * 4);
  w.total_bytes = up((size_t)G * C * 4);
  w.rec_bytes = up((size_t)G * ((N + kBigTile - 1) / kBigTile) * kSlots * kD * 8);
  w.sum_bytes = up((size_t)G * C * kD * 8);
  w.cnt_bytes = up((size_t)G * C * 4);
  if (bounded) {
    w.near_order_bytes = up((size_t)G * N * 4);
    w.used_bytes = up((size_t)G * C * kD * 2);
    w.mask_bytes = up((size_t)G * C * (C / 32) * 4);
    w.table_bytes = up((size_t)G * C * 4);
    w.ctl_bytes = up((size_t)(6 + G) * 4);
  }
  return w;
}

int check_ws(const DLTensor* ws, size_t need, int dev, const char* who) {
  SQ_REQUIRE(ws && on_gpu(ws) && ws->device.device_id == dev, SQ_EWORKSPACE, "%s: workspace missing or not on the device", who);
  SQ_REQUIRE((size_t)numel_of(ws) * (ws->dtype.bits / 8) >= need && is_compact(ws), SQ_EWORKSPACE,
             "%s: workspace too small: need %zu bytes", who, need);
  SQ_REQUIRE(((uintptr_t)data_of(ws) & 255) == 0, SQ_EWORKSPACE, "%s: workspace not 256-byte aligned", who);
  return SQ_OK;
}

int check_current_device(int dev, const char* who) {
  int cur = -1;
  SQ_HIP(hipGetDevice(&cur));
  SQ_REQUIRE(cur == dev, SQ_EDEVICE, "%s: tensors live on device %d but the current device is %d", who, dev, cur);
  return SQ_OK;
}

// tokens of every cluster in ascending order into clusters[G,C,M] (reverse index), sizes into total_out
int run_sort(const DLTensor* idx, char* wsp, const WsLayout& w, int32_t* dst, int64_t dst_sg, int64_t dst_sc, int M,
             int32_t* total_out, int C, hipStream_t st) {
  const int64_t G = idx->shape[0], N = idx->shape[1];
  SortArgs s;
  s.idx = (const int32_t*)data_of(idx);
  s.tile_hist = (int32_t*)(wsp + w.off_bytes);
  s.total = total_out;
  s.dst = dst;
  s.i_sg = stride_of(idx, 0);
  s.dst_sg = dst_sg;
  s.dst_sc = dst_sc;
  s.N = (int)N;
  s.C = C;
  s.nT = w.nT;
  s.M = M;
  hipLaunchKernelGGL(sort_hist_kernel, dim3(w.nT, (unsigned)G), dim3(kTileTok), (size_t)C * 4, st, s);
  hipLaunchKernelGGL(sort_scan_tiles_kernel, dim3((C + 31) / 32, (unsigned)G), dim3(32 * kScanSegs), 0, st, s);
  hipLaunchKernelGGL(sort_scatter_kernel, dim3(w.nT, (unsigned)G), dim3(kTileTok), 0, st, s);
  SQ_HIP(hipGetLastError());
  return SQ_OK;
}

// every tile of kBigTile tokens grouped by cluster into `order`, the ranges' starts into the histogram region
int run_group(const DLTensor* idx, const DLTensor* src, char* wsp, const WsLayout& w, hipStream_t st) {
  const int64_t G = idx->shape[0], N = idx->shape[1];
  GroupArgs s;
  s.idx = (const int32_t*)data_of(idx);
  s.src = (const uint16_t*)data_of(src);
  s.start = (int32_t*)(wsp + w.off_bytes);
  s.order = (int32_t*)(wsp + w.off_bytes + w.hist_bytes);
  s.rec = (double*)(wsp + w.rec_offset());
  s.i_sg = stride_of(idx, 0);
  s.s_sg = stride_of(src, 0);
  s.s_sn = stride_of(src, 1);
  s.N = (int)N;
  s.C = w.C;
  s.nT = (int)((N + kBigTile - 1) / kBigTile);
  const size_t lds = (size_t)kSlots * kD * 8 + ((size_t)w.C + kBigTile) * 4;
  static bool raised[64] = {};
  int dev = 0;
  SQ_HIP(hipGetDevice(&dev));
  if (dev >= 0 && dev < 64 && !raised[dev]) {   // up to 72 KB for 8192 clusters, above the default limit
    SQ_HIP(hipFuncSetAttribute((const void*)tile_group_kernel, hipFuncAttributeMaxDynamicSharedMemorySize, (int)((size_t)kSlots * kD * 8 + ((size_t)kMaxC + kBigTile) * 4)));
    raised[dev] = true;
  }
  hipLaunchKernelGGL(tile_group_kernel, dim3(s.nT, (unsigned)G), dim3(1024), lds, st, s);
  SQ_HIP(hipGetLastError());
  return SQ_OK;
}

// sums of `src` rows per cluster after run_group
int run_cluster_sum(const DLTensor* src, char* wsp, const WsLayout& w, DLTensor* dst, int32_t* cnt, int mode, hipStream_t st, bool keep = false) {
  const int64_t G = src->shape[0], N = src->shape[1];
  SumArgs s;
  s.src = (const uint16_t*)data_of(src);
  s.start = (const int32_t*)(wsp + w.off_bytes);
  s.order = (const int32_t*)(wsp + w.off_bytes + w.hist_bytes);
  s.rec = (const double*)(wsp + w.rec_offset());
  s.dst = (uint16_t*)data_of(dst);
  s.cnt = cnt;
  s.s_sg = stride_of(src, 0);
  s.s_sn = stride_of(src, 1);
  s.d_sg = stride_of(dst, 0);
  s.d_sc = stride_of(dst, 1);
  s.N = (int)N;
  s.C = w.C;
  s.nT = (int)((N + kBigTile - 1) / kBigTile);
  s.mode = mode;
  s.keep_sum = keep ? (double*)(wsp + w.sum_offset()) : nullptr;
  s.keep_cnt = keep ? (int32_t*)(wsp + w.cnt_offset()) : nullptr;
  hipLaunchKernelGGL(cluster_sum_kernel, dim3((unsigned)w.C, (unsigned)G), dim3(256), 0, st, s);
  SQ_HIP(hipGetLastError());
  return SQ_OK;
}

int check_gnd(const DLTensor* t, const char* name, int dev) {
  int rc = check_tensor(t, name, 3, dev);
  if (rc) return rc;
  SQ_REQUIRE(dtype_of(t) == DType::BF16, SQ_EDTYPE, "%s must be bf16", name);
  SQ_REQUIRE(t->shape[2] == kD, SQ_EUNSUPPORTED, "%s: last dimension must be 128, got %lld", name, (long long)t->shape[2]);
  SQ_REQUIRE(stride_of(t, 0) % 8 == 0 && stride_of(t, 1) % 8 == 0, SQ_ESHAPE, "%s: strides must be multiples of 8 elements", name);
  return SQ_OK;
}

int check_i32(const DLTensor* t, const char* name, int ndim, int dev) {
  SQ_REQUIRE(t != nullptr, SQ_EINVAL, "%s is null", name);
  SQ_REQUIRE(on_gpu(t) && t->device.device_id == dev, SQ_EDEVICE, "%s is not on the same ROCm device", name);
  SQ_REQUIRE(dtype_of(t) == DType::I32 && t->ndim == ndim && is_compact(t), SQ_ESHAPE, "%s must be a compact int32 tensor of rank %d", name, ndim);
  return SQ_OK;
}

}  // namespace
}  // namespace sq

using namespace sq;

extern "C" size_t sq_kmeans_workspace_bytes(int64_t groups, int64_t num_tokens, int64_t num_centroids, int64_t dim) {
  (void)dim;
  if (groups <= 0 || num_tokens <= 0 || num_centroids <= 0) return 0;
  return ws_layout(groups, num_tokens, num_centroids).all();
}

namespace {
// Four parts while the launch's 64-token workgroups fit the CUs one each, two while its 128-token ones do: the waves that
// share the centroids then run on CUs that would idle.  Beyond that a split workgroup only takes another's CU (an unsplit
// launch with one workgroup per CU holds its 16 KB blocks twice, a launch of four parts its CU's whole LDS).
// segment_k_means, ten steps, 1024 centroids: 4096 tokens 335 -> 267 us, 16384 tokens 342 -> 277, 20000 (two parts) 350 -> 292.
// Unsplit all the same
//  * up to 128 tokens with up to three blocks of centroids, where the chain is short and the shares' meeting is not (64 tokens x 96
//    centroids: 6.7 us a step, 7.9 with four parts; 256 centroids 8.0 / 8.0, 512: 10.8 / 9.1);
//  * from 32 groups on, where every group has centroids of its own and a full chip reads them all at once, a launch over half
//    the CUs, unless its chain is long: 32 groups x 500 tokens, 256 workgroups of four parts against 64 whole ones, 256
//    centroids 12.1 us whole, 14.1 split, 1024: 27.4 / 26.2; 1000 tokens in two parts 320 centroids 14.3 / 15.7.
int assign_parts(int64_t G, int64_t N, int64_t C) {
  constexpr int64_t kCUs = 256;
  const int64_t blocks = (C + kCB - 1) / kCB;
  if (!(blocks > 3 || (blocks > 1 && N > 128))) return 1;
  if (G * ((N + 63) / 64) <= (G < 32 || blocks >= 16 ? kCUs : kCUs / 2)) return 4;
  return G * ((N + 127) / 128) <= (G < 32 || blocks >= 8 ? kCUs : kCUs / 2) ? 2 : 1;
}

template <bool TRACK>
void launch_assign(const AssignArgs& a, int64_t G, hipStream_t st) {
  const int64_t N = a.N;
  auto grid = [&](int tokens) { return dim3((unsigned)((N + tokens - 1) / tokens), (unsigned)G); };
  const dim3 block(kAssignWaves * 64);
  const int parts = assign_parts(G, N, a.C);
  if (parts == 4)
    hipLaunchKernelGGL((kmeans_assign_kernel<TRACK, 4>), grid(kTileTok / 4), block, 0, st, a);
  else if (parts == 2)
    hipLaunchKernelGGL((kmeans_assign_kernel<TRACK, 2>), grid(kTileTok / 2), block, 0, st, a);
  else
    hipLaunchKernelGGL((kmeans_assign_kernel<TRACK, 1>), grid(kTileTok), block, 0, st, a);
}

int kmeans_train_impl(const DLTensor* data, DLTensor* centroids, DLTensor* idx, DLTensor* cnt, DLTensor* workspace,
                      int32_t normalize, int32_t state, void* stream, const char* who, bool bounded = false) {
  SQ_REQUIRE(data && centroids && idx && cnt, SQ_EINVAL, "%s: data, centroids, idx and cnt must be non-null", who);
  SQ_REQUIRE(state >= SQ_KMEANS_STATELESS && state <= SQ_KMEANS_APPLY_CHANGES, SQ_EINVAL, "%s: state %d not supported", who, (int)state);
  const int dev = data->device.device_id;
  int rc;
  if ((rc = check_gnd(data, "data", dev)) || (rc = check_gnd(centroids, "centroids", dev)) || (rc = check_i32(idx, "idx", 2, dev)) ||
      (rc = check_i32(cnt, "cnt", 2, dev)))
    return rc;
  const int64_t G = data->shape[0], N = data->shape[1], C = centroids->shape[1];
  SQ_REQUIRE(G > 0 && N > 0 && C > 0, SQ_ESHAPE, "%s: empty tensor", who);
  SQ_REQUIRE(centroids->shape[0] == G && idx->shape[0] == G && idx->shape[1] == N && cnt->shape[0] == G && cnt->shape[1] == C,
             SQ_ESHAPE, "%s: shapes of data/centroids/idx/cnt disagree", who);
  SQ_REQUIRE(C % 32 == 0, SQ_ESHAPE, "num_centroids %% 32 != 0 (num_centroids = %lld)", (long long)C);
  SQ_REQUIRE(C <= kMaxC, SQ_EUNSUPPORTED, "%s: more than %d centroids", who, kMaxC);
  SQ_REQUIRE(N < (1ll << 31) - 65536, SQ_EUNSUPPORTED, "%s: too many tokens", who);
  SQ_REQUIRE(!bounded || C <= kNearMaxC, SQ_EUNSUPPORTED, "%s: more than %d centroids", who, kNearMaxC);
  const bool near = bounded && assign_parts(G, N, C) == 1;
  const WsLayout w = ws_layout(G, N, C, bounded);
  if ((rc = check_ws(workspace, w.all(), dev, who)) || (rc = check_current_device(dev, who))) return rc;
  hipStream_t st = (hipStream_t)stream;
  char* wsp = data_of(workspace);

  AssignArgs a;
  a.data = (const uint16_t*)data_of(data);
  a.cent = (const uint16_t*)data_of(centroids);
  a.idx = (int32_t*)data_of(idx);
  a.d_sg = stride_of(data, 0);
  a.d_sn = stride_of(data, 1);
  a.c_sg = stride_of(centroids, 0);
  a.c_sc = stride_of(centroids, 1);
  a.i_sg = stride_of(idx, 0);
  a.N = (int)N;
  a.C = (int)C;
  a.keep_sum = (double*)(wsp + w.sum_offset());
  a.keep_cnt = (int32_t*)(wsp + w.cnt_offset());
  const int mode = normalize ? 2 : 1;
  a.near = near ? w.near(wsp, G, N) : NearState{};
  const unsigned blocks = (unsigned)C / 32, looked_at = (blocks + kPairSample - 1) / kPairSample;
  auto launch_bounds = [&](bool trial) {
    BoundsArgs ba;
    ba.cent = a.cent;
    ba.near = a.near;
    ba.cnt = a.keep_cnt;
    ba.c_sg = a.c_sg;
    ba.c_sc = a.c_sc;
    ba.C = (int)C;
    ba.every = trial ? kPairSample : 1;
    hipLaunchKernelGGL(kmeans_bounds_kernel, dim3(trial ? looked_at : blocks, (blocks + kBoundsWaves - 1) / kBoundsWaves, (unsigned)G), dim3(kBoundsWaves * 64), 0, st, ba);
  };
  if (state == SQ_KMEANS_APPLY_CHANGES) {
    if (near) {
      const unsigned tiles = (unsigned)((N + kTileTok - 1) / kTileTok);
      launch_bounds(false);
      hipLaunchKernelGGL((kmeans_assign_kernel<true, 1, true>), dim3(tiles * (unsigned)G), dim3(kAssignWaves * 64), 0, st, a);
    } else {
      launch_assign<true>(a, G, st);
    }
    UpdateArgs u;
    u.sum = a.keep_sum;
    u.cnt = a.keep_cnt;
    u.dst = (uint16_t*)data_of(centroids);
    u.cnt_out = (int32_t*)data_of(cnt);
    u.d_sg = stride_of(centroids, 0);
    u.d_sc = stride_of(centroids, 1);
    u.C = (int)C;
    u.mode = mode;
    u.near = a.near;
    hipLaunchKernelGGL(kmeans_update_kernel, dim3((unsigned)C, (unsigned)G), dim3(kD), 0, st, u);
    SQ_HIP(hipGetLastError());
    return SQ_OK;
  }
  launch_assign<false>(a, G, st);
  SQ_HIP(hipGetLastError());
  if ((rc = run_group(idx, data, wsp, w, st))) return rc;
  if ((rc = run_cluster_sum(data, wsp, w, centroids, (int32_t*)data_of(cnt), mode, st, state == SQ_KMEANS_KEEP_SUMS))) return rc;   // cnt = cluster sizes
  if (state == SQ_KMEANS_KEEP_SUMS && near) {
    OrderArgs o;
    o.idx = a.idx;
    o.cnt = a.keep_cnt;
    o.near = a.near;
    o.i_sg = a.i_sg;
    o.N = (int)N;
    o.C = (int)C;
    hipLaunchKernelGGL(order_start_kernel, dim3((unsigned)G), dim3(1024), 0, st, o);
    ReachArgs ra;
    ra.data = a.data;
    ra.cent = a.cent;
    ra.cnt = a.keep_cnt;
    ra.near = a.near;
    ra.d_sg = a.d_sg;
    ra.d_sn = a.d_sn;
    ra.c_sg = a.c_sg;
    ra.c_sc = a.c_sc;
    ra.N = (int)N;
    ra.C = (int)C;
    ra.nT = (int)((N + kBigTile - 1) / kBigTile);
    ra.tile_start = (const int32_t*)(wsp + w.off_bytes);
    ra.tile_order = (const int32_t*)(wsp + w.off_bytes + w.hist_bytes);
    hipLaunchKernelGGL((near_reach_kernel<true>), dim3(looked_at * 32, (unsigned)G), dim3(256), 0, st, ra);
    launch_bounds(true);
    hipLaunchKernelGGL(order_fill_kernel, dim3((unsigned)((N + kOrderTile - 1) / kOrderTile), (unsigned)G), dim3(1024), 0, st, o);
    hipLaunchKernelGGL((near_reach_kernel<false>), dim3((unsigned)C, (unsigned)G), dim3(256), 0, st, ra);
    SQ_HIP(hipGetLastError());
  }
  return SQ_OK;
}
}  // namespace

extern "C" int sq_kmeans_train(const DLTensor* data, DLTensor* centroids, DLTensor* idx, DLTensor* cnt, DLTensor* workspace,
                               int32_t normalize, void* stream) {
  return kmeans_train_impl(data, centroids, idx, cnt, workspace, normalize, SQ_KMEANS_STATELESS, stream, "sq_kmeans_train");
}

extern "C" int sq_kmeans_train_stateful(const DLTensor* data, DLTensor* centroids, DLTensor* idx, DLTensor* cnt, DLTensor* workspace,
                                        int32_t normalize, int32_t state, void* stream) {
  return kmeans_train_impl(data, centroids, idx, cnt, workspace, normalize, state, stream, "sq_kmeans_train_stateful");
}

extern "C" size_t sq_kmeans_workspace_bytes_bounded(int64_t groups, int64_t num_tokens, int64_t num_centroids, int64_t dim) {
  (void)dim;
  if (groups <= 0 || num_tokens <= 0 || num_centroids <= 0) return 0;
  return ws_layout(groups, num_tokens, num_centroids, true).all();
}

extern "C" int sq_kmeans_train_bounded(const DLTensor* data, DLTensor* centroids, DLTensor* idx, DLTensor* cnt, DLTensor* workspace,
                                       int32_t normalize, int32_t state, void* stream) {
  return kmeans_train_impl(data, centroids, idx, cnt, workspace, normalize, state, stream, "sq_kmeans_train_bounded", true);
}

extern "C" int sq_reverse_index(const DLTensor* idx, DLTensor* clusters, DLTensor* cluster_size, DLTensor* workspace, void* stream) {
  SQ_REQUIRE(idx && clusters && cluster_size, SQ_EINVAL, "sq_reverse_index: idx, clusters and cluster_size must be non-null");
  const int dev = idx->device.device_id;
  int rc;
  if ((rc = check_i32(idx, "idx", 2, dev)) || (rc = check_i32(clusters, "clusters", 3, dev)) ||
      (rc = check_i32(cluster_size, "cluster_size", 2, dev)))
    return rc;
  const int64_t G = idx->shape[0], N = idx->shape[1], C = clusters->shape[1], M = clusters->shape[2];
  SQ_REQUIRE(G > 0 && N > 0 && C > 0 && M > 0, SQ_ESHAPE, "sq_reverse_index: empty tensor");
  SQ_REQUIRE(clusters->shape[0] == G && cluster_size->shape[0] == G && cluster_size->shape[1] == C, SQ_ESHAPE,
             "sq_reverse_index: shapes of idx/clusters/cluster_size disagree");
  SQ_REQUIRE(C <= kMaxC, SQ_EUNSUPPORTED, "sq_reverse_index: more than %d centroids", kMaxC);
  const WsLayout w = ws_layout(G, N, C);
  if ((rc = check_ws(workspace, w.all(), dev, "sq_reverse_index")) || (rc = check_current_device(dev, "sq_reverse_index"))) return rc;
  hipStream_t st = (hipStream_t)stream;
  hipLaunchKernelGGL(fill_i32_kernel, dim3(256), dim3(256), 0, st, (int32_t*)data_of(clusters), G * C * M, 0);
  return run_sort(idx, data_of(workspace), w, (int32_t*)data_of(clusters), C * M, M, (int)M,
                  (int32_t*)data_of(cluster_size), (int)C, st);
}

extern "C" int sq_index_add(const DLTensor* value, const DLTensor* idx, DLTensor* out, DLTensor* workspace, void* stream) {
  SQ_REQUIRE(value && idx && out, SQ_EINVAL, "sq_index_add: value, idx and out must be non-null");
  const int dev = value->device.device_id;
  int rc;
  if ((rc = check_gnd(value, "value", dev)) || (rc = check_gnd(out, "out", dev)) || (rc = check_i32(idx, "idx", 2, dev))) return rc;
  const int64_t G = value->shape[0], N = value->shape[1], C = out->shape[1];
  SQ_REQUIRE(G > 0 && N > 0 && C > 0, SQ_ESHAPE, "sq_index_add: empty tensor");
  SQ_REQUIRE(out->shape[0] == G && idx->shape[0] == G && idx->shape[1] == N, SQ_ESHAPE, "sq_index_add: shapes disagree");
  SQ_REQUIRE(C <= kMaxC, SQ_EUNSUPPORTED, "sq_index_add: more than %d centroids", kMaxC);
  const WsLayout w = ws_layout(G, N, C);
  if ((rc = check_ws(workspace, w.all(), dev, "sq_index_add")) || (rc = check_current_device(dev, "sq_index_add"))) return rc;
  hipStream_t st = (hipStream_t)stream;
  char* wsp = data_of(workspace);
  if ((rc = run_group(idx, value, wsp, w, st))) return rc;
  return run_cluster_sum(value, wsp, w, out, nullptr, 0, st);
}

extern "C" int sq_topk_select(const DLTensor* query, const DLTensor* centroids, const DLTensor* clusters,
                              const DLTensor* cluster_size, DLTensor* out, DLTensor* workspace, int32_t num_kv_groups,
                              void* stream) {
  SQ_REQUIRE(query && centroids && clusters && cluster_size && out, SQ_EINVAL, "sq_topk_select: null tensor argument");
  const int dev = query->device.device_id;
  int rc;
  if ((rc = check_gnd(query, "query", dev)) || (rc = check_gnd(centroids, "centroids", dev)) ||
      (rc = check_i32(clusters, "clusters", 3, dev)) || (rc = check_i32(cluster_size, "cluster_size", 2, dev)))
    return rc;
  // out may be the leading columns of a wider int32 matrix (a decode list that continues with other tokens)
  SQ_REQUIRE(on_gpu(out) && out->device.device_id == dev, SQ_EDEVICE, "out is not on the same ROCm device");
  SQ_REQUIRE(dtype_of(out) == DType::I32 && out->ndim == 2 && stride_of(out, 1) == 1 && stride_of(out, 0) >= out->shape[1], SQ_ESHAPE,
             "out must be int32 [G, k] with contiguous rows");
  const int64_t B = query->shape[0], Hq = query->shape[1], G = centroids->shape[0], C = centroids->shape[1];
  const int64_t M = clusters->shape[2], k = out->shape[1];
  SQ_REQUIRE(num_kv_groups > 0 && Hq % num_kv_groups == 0, SQ_EINVAL, "sq_topk_select: num_kv_groups %d does not divide Hq", num_kv_groups);
  const int64_t Hkv = Hq / num_kv_groups;
  SQ_REQUIRE(G == B * Hkv, SQ_ESHAPE, "sq_topk_select: centroids has %lld groups, expected B*Hkv = %lld", (long long)G, (long long)(B * Hkv));
  SQ_REQUIRE(clusters->shape[0] == G && clusters->shape[1] == C && cluster_size->shape[0] == G && cluster_size->shape[1] == C &&
                 out->shape[0] == G && k > 0 && M > 0,
             SQ_ESHAPE, "sq_topk_select: shapes disagree");
  SQ_REQUIRE(C <= kMaxC, SQ_EUNSUPPORTED, "sq_topk_select: more than %d centroids", kMaxC);
  const WsLayout w = ws_layout(G, 1, C);
  if ((rc = check_ws(workspace, w.all(), dev, "sq_topk_select")) || (rc = check_current_device(dev, "sq_topk_select"))) return rc;
  hipStream_t st = (hipStream_t)stream;
  char* wsp = data_of(workspace);
  TopkArgs a;
  a.query = (const uint16_t*)data_of(query);
  a.cent = (const uint16_t*)data_of(centroids);
  a.clusters = (const int32_t*)data_of(clusters);
  a.size = (const int32_t*)data_of(cluster_size);
  a.out = (int32_t*)data_of(out);
  a.out_sg = stride_of(out, 0);
  a.score = (float*)(wsp + w.off_bytes + w.hist_bytes + w.order_bytes);
  a.start = (int32_t*)(wsp + w.off_bytes + w.hist_bytes + w.order_bytes + w.score_bytes);
  a.scored = (unsigned long long*)a.score;   // `start` follows `score`
  a.tag = 0;
  a.q_sb = stride_of(query, 0);
  a.q_sh = stride_of(query, 1);
  a.c_sg = stride_of(centroids, 0);
  a.c_sc = stride_of(centroids, 1);
  a.cl_sg = C * M;
  a.cl_sc = M;
  a.C = (int)C;
  a.M = (int)M;
  a.k = (int)k;
  a.Hkv = (int)Hkv;
  a.group = num_kv_groups;
  if (C <= 1024 && num_kv_groups <= 16) {   // one launch, only the clusters that can fill k are ordered
    const int waves = (int)((C + 63) / 64);
    a.share = topk_share(G, waves);
    const unsigned parts = (unsigned)((waves + a.share - 1) / a.share);
    if (parts > 1) a.tag = call_tag();
    hipLaunchKernelGGL(topk_select_kernel, dim3((unsigned)G, parts), dim3(1024), 0, st, a);
    SQ_HIP(hipGetLastError());
    return SQ_OK;
  }
  hipLaunchKernelGGL(topk_score_kernel, dim3((unsigned)((C + 255) / 256), (unsigned)G), dim3(256), 0, st, a);
  int P = 1;
  while (P < C) P <<= 1;
  const size_t emit_lds = (size_t)(2 * P + C + 1) * 4;
  if (emit_lds > 48 * 1024)   // beyond the default limit of dynamic LDS (C > 4096)
    SQ_HIP(hipFuncSetAttribute((const void*)topk_emit_kernel, hipFuncAttributeMaxDynamicSharedMemorySize, (int)emit_lds));
  hipLaunchKernelGGL(topk_emit_kernel, dim3((unsigned)G), dim3(1024), emit_lds, st, a);
  SQ_HIP(hipGetLastError());
  return SQ_OK;
}
