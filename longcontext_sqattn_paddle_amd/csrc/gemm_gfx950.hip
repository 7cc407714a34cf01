// out = x . weight^T (+ bias) for the projections of a prompt: x [M, K], weight [N, K] as a Linear layer stores it.
//
// The prompt's products (model_hub/qwen.py:302-326) have few rows and, three of the four, few output features: 512 x 3584 outputs
// are 28 tiles of 256 x 256 for 256 CUs.  The tensor library leaves most of the chip idle there (down_proj of 512 rows 196 us, of 64
// rows 91 us, where the weight streams from memory in 21).  Here the sum over K is split over workgroups until they fill the
// chip; a second kernel adds the parts and the bias.
//
// Workgroup = 8 waves, a BM x BN tile of the output.  Per step of 64 elements of K the tiles of x and weight go to LDS with
// global_load_lds into a ring of NB buffers, requested NB - 1 steps ahead, one barrier per step; 128-byte rows, 16-byte chunk c of row r in
// slot c ^ ((r >> 1) & 7), so that the 16 rows a quarter-wave reads at one chunk index fall into 16 different bank
// groups.  MFMA 32x32x16, x rows as the A and weight rows as the B operand: a lane holds one output feature and 16 rows of a 32 x 32 block.
#include <algorithm>

#include "common.hpp"

namespace sq {
namespace {

constexpr int kBK = 64;            // elements of K per step
constexpr int kRowBytes = kBK * 2;
constexpr int kThreads = 512;

struct GemmArgs {
  const char* x;
  const char* w;
  const void* bias;
  void* out;
  float* part;          // [splits, M, N] fp32, or null: the tile is the result
  int64_t x_row, w_row, o_row;   // bytes, bytes, elements
  int32_t M, N, steps, splits, tiles_m, tiles_n;
};

template <bool BF16>
__device__ __forceinline__ f32x16_t mfma32(const u32x4_t& a, const u32x4_t& b, f32x16_t c) {
  if constexpr (BF16) return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8_t, a), __builtin_bit_cast(bf16x8_t, b), c, 0, 0, 0);
  else return __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(f16x8_t, a), __builtin_bit_cast(f16x8_t, b), c, 0, 0, 0);
}
template <bool BF16>
__device__ __forceinline__ uint32_t to_bits16(float v) {
  if constexpr (BF16) return f32_to_bf16_bits(v);
  else return (uint32_t)__builtin_bit_cast(uint16_t, (_Float16)v);
}
template <bool BF16>
__device__ __forceinline__ float from_bits16(uint32_t b) {
  if constexpr (BF16) return bf16_bits_to_f32(b);
  else return (float)__builtin_bit_cast(_Float16, (uint16_t)b);
}

template <bool BF16, int BM, int BN, int WM, int WN, int NB>
__global__ __launch_bounds__(kThreads) void gemm_kernel(GemmArgs a) {
  static_assert(WM * WN == 8 && BM % (32 * WM) == 0 && BN % (32 * WN) == 0, "eight waves of whole 32 x 32 blocks");
  constexpr int MA = BM / WM / 32, MB = BN / WN / 32;
  constexpr int PER = (BM + BN) / 64;          // copies of 1 KB (8 rows) per wave and step
  constexpr int kBuf = (BM + BN) * kRowBytes;
  extern __shared__ __attribute__((aligned(16))) char smem[];
  typedef __attribute__((address_space(3))) void* lds_ptr_t;
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  // blockIdx -> (part of K, tile): the row tiles of one (weight tile, part) on one XCD, next to each other, so that the weight is
  // fetched once; with the part as the fastest index an XCD also stays with few parts of x
  const int r8 = blockIdx.x >> 3, group = r8 / a.tiles_m * 8 + (blockIdx.x & 7);
  if (group >= a.tiles_n * a.splits) return;
  const int m0 = r8 % a.tiles_m * BM, split = group % a.splits, n0 = group / a.splits * BN;
  const int s0 = (int)((int64_t)a.steps * split / a.splits), n_steps = (int)((int64_t)a.steps * (split + 1) / a.splits) - s0;

  // this wave's copies: 1 KB number PER wave + c of the tile of x (BM / 8 of them), then of weight; rows past the end are copies of the last
  uint32_t off[PER];
#pragma unroll
  for (int c = 0; c < PER; ++c) {
    const int q = PER * wave + c;
    const bool is_x = q < BM / 8;
    const int r = 8 * (is_x ? q : q - BM / 8) + (lane >> 3);
    const uint32_t chunk = (uint32_t)((lane & 7) ^ ((r >> 1) & 7)) * 16u;
    off[c] = is_x ? (uint32_t)min(m0 + r, a.M - 1) * (uint32_t)a.x_row + chunk : (uint32_t)min(n0 + r, a.N - 1) * (uint32_t)a.w_row + chunk;
  }
  auto copy = [&](int s, int buf, int c) __attribute__((always_inline)) {
    const int q = PER * wave + c;
    const char* base = (q < BM / 8 ? a.x : a.w) + (int64_t)(s0 + s) * kRowBytes;
    uint32_t o = off[c];
    asm volatile("" : "+v"(o));   // a 32-bit per-lane offset next to the uniform 64-bit base
    __builtin_amdgcn_global_load_lds((const void*)(base + o), (lds_ptr_t)(smem + buf * kBuf + q * 1024), 16, 0, 0);
  };
  auto stage = [&](int s, int buf) __attribute__((always_inline)) { static_for<0, PER>([&](auto C) { copy(s, buf, decltype(C)::value); }); };
  const int c32 = lane & 31, g = lane >> 5, wm = wave / WN, wn = wave % WN;
  const uint32_t smem_addr = (uint32_t)(uintptr_t)(lds_ptr_t)smem;
  uint32_t xa[4], wa[4];   // k-step j of 16: the lane's chunk 2 j + g
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const uint32_t slot = (uint32_t)(((2 * j + g) ^ ((c32 >> 1) & 7)) << 4);
    xa[j] = smem_addr + (wm * (BM / WM) + c32) * kRowBytes + slot;
    wa[j] = smem_addr + (BM + wn * (BN / WN) + c32) * kRowBytes + slot;
  }
  f32x16_t acc[MA][MB];
#pragma unroll
  for (int i = 0; i < MA; ++i)
#pragma unroll
    for (int j = 0; j < MB; ++j)
#pragma unroll
      for (int e = 0; e < 16; ++e) acc[i][j][e] = 0.f;

  constexpr int kReads = MA + MB, kMfmas = MA * MB;
  u32x4_t fx[2][MA], fw[2][MB];
  int buf = 0;
  auto read = [&](auto J, auto R) __attribute__((always_inline)) {
    constexpr int j = decltype(J)::value, r = decltype(R)::value;
    if constexpr (r < MA) fx[j & 1][r] = lds_read128<r * 32 * kRowBytes>(xa[j] + (uint32_t)(buf * kBuf));
    else fw[j & 1][r - MA] = lds_read128<(r - MA) * 32 * kRowBytes>(wa[j] + (uint32_t)(buf * kBuf));
  };
  auto arrived = [&](auto J, auto Behind) __attribute__((always_inline)) {   // with Behind reads requested after them
    constexpr int j = decltype(J)::value, n = decltype(Behind)::value;
    static_for<0, MA>([&](auto I) { lds_wait<n>(fx[j & 1][decltype(I)::value]); });
    static_for<0, MB>([&](auto I) { lds_wait<n>(fw[j & 1][decltype(I)::value]); });
  };
  using std::integral_constant;
  using zero = integral_constant<int, 0>;
  if constexpr (kMfmas > 2) {
    // The barrier stands in front of a step's last k-step: the next step's copies have landed there (everybody's, once it is passed), so that
    // its first fragments are read between this step's last MFMAs; and this step's buffer, read out by then, is refilled.  The matrix pipe
    // does not stand for the reads between two steps: a step of the 256 x 128 tile 0.74 us, in the order below 0.82.
    constexpr auto reads_before = [](int i) { return 2 * i >= kMfmas ? kReads : 2 * i * kReads / kMfmas; };   // with the first half of the MFMAs
    auto multiply = [&](auto J, auto Copies, int s, int refill) __attribute__((always_inline)) {
      constexpr int j = decltype(J)::value, next = (j + 1) & 3;
      static_for<0, kMfmas>([&](auto I) {
        constexpr int i = decltype(I)::value, p = i / MB, q = i % MB;
        static_for<reads_before(i), reads_before(i + 1)>([&](auto R) { read(integral_constant<int, next>{}, R); });
        if constexpr (decltype(Copies)::value) static_for<i * PER / kMfmas, (i + 1) * PER / kMfmas>([&](auto C) { copy(s + NB, refill, decltype(C)::value); });
        acc[p][q] = mfma32<BF16>(fx[j & 1][p], fw[j & 1][q], acc[p][q]);
        __builtin_amdgcn_sched_barrier(0);   // left alone, the scheduler moves MFMAs behind the next k-step's waits
      });
      arrived(integral_constant<int, next>{}, zero{});
    };
    auto step = [&](int s, auto Copies) __attribute__((always_inline)) {
      static_for<0, 3>([&](auto J) { multiply(J, std::false_type{}, 0, 0); });
      const int refill = buf;
      if (decltype(Copies)::value || s + 1 < n_steps) {
        // copies of the NB - 2 steps behind the next one may still be on their way
        if (decltype(Copies)::value || n_steps - 1 - s >= NB - 1) asm volatile("s_waitcnt vmcnt(%0)" ::"n"((NB - 2) * PER) : "memory");
        else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        asm volatile("s_barrier" ::: "memory");
        buf = buf == NB - 1 ? 0 : buf + 1;
      }
      multiply(integral_constant<int, 3>{}, Copies, s, refill);   // the last step reads its own buffer once more, for nobody
    };
#pragma unroll
    for (int s = 0; s < NB; ++s)
      if (s < n_steps) stage(s, s);
    if (n_steps >= NB) asm volatile("s_waitcnt vmcnt(%0)" ::"n"((NB - 1) * PER) : "memory");
    else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    asm volatile("s_barrier" ::: "memory");
    static_for<0, kReads>([&](auto R) { read(zero{}, R); });
    arrived(zero{}, zero{});
    int s = 0;
    for (; s + NB < n_steps; ++s) step(s, std::true_type{});
    for (; s < n_steps; ++s) step(s, std::false_type{});
  } else {
    // One or two MFMAs a k-step: memory bounds these tiles.  The order above is no faster here and its deeper queue of copies costs launches
    // of few steps 2 to 4 us (4096 x 4096 of 200 rows 22.7 against 25.9, 1024 x 8192 of 512 rows 22.7 against 29.5).
#pragma unroll
    for (int s = 0; s < NB - 1; ++s)
      if (s < n_steps) stage(s, s);
    for (int s = 0; s < n_steps; ++s) {
      // the copies of this step have landed: at most those of the NB - 2 steps behind it are still on their way
      if (n_steps - 1 - s >= NB - 2) asm volatile("s_waitcnt vmcnt(%0)" ::"n"((NB - 2) * PER) : "memory");
      else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
      asm volatile("s_barrier" ::: "memory");   // ... everybody's; and everybody is done with the buffer that is refilled now
      if (s + NB - 1 < n_steps) stage(s + NB - 1, buf == 0 ? NB - 1 : buf - 1);
      static_for<0, kReads>([&](auto R) { read(zero{}, R); });
      static_for<0, 4>([&](auto J) {
        constexpr int j = decltype(J)::value;
        if constexpr (j < 3) static_for<0, kReads>([&](auto R) { read(integral_constant<int, j + 1>{}, R); });
        arrived(J, integral_constant<int, (j < 3 ? kReads : 0)>{});
#pragma unroll
        for (int p = 0; p < MA; ++p)
#pragma unroll
          for (int q = 0; q < MB; ++q) acc[p][q] = mfma32<BF16>(fx[j & 1][p], fw[j & 1][q], acc[p][q]);
      });
      buf = buf == NB - 1 ? 0 : buf + 1;
    }
  }
#pragma unroll
  for (int q = 0; q < MB; ++q) {
    const int n = n0 + wn * (BN / WN) + 32 * q + c32;
    if (n >= a.N) continue;
    const float bias = a.bias && !a.part ? from_bits16<BF16>(((const uint16_t*)a.bias)[n]) : 0.f;
#pragma unroll
    for (int p = 0; p < MA; ++p)
#pragma unroll
      for (int e = 0; e < 16; ++e) {
        const int m = m0 + wm * (BM / WM) + 32 * p + 8 * (e >> 2) + 4 * g + (e & 3);
        if (m >= a.M) continue;
        if (a.part) a.part[((int64_t)split * a.M + m) * a.N + n] = acc[p][q][e];
        else ((uint16_t*)a.out)[(int64_t)m * a.o_row + n] = (uint16_t)to_bits16<BF16>(acc[p][q][e] + bias);
      }
  }
}

// The parts added in order, plus the bias, rounded once: four neighbouring features per thread
template <bool BF16>
__global__ __launch_bounds__(256) void gemm_add_kernel(GemmArgs a) {
  const int quads = a.N / 4;
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (i >= (int64_t)a.M * quads) return;
  const int m = (int)(i / quads), n = (int)(i % quads) * 4;
  const float* p = a.part + (int64_t)m * a.N + n;
  const int64_t stride = (int64_t)a.M * a.N;
  float4 s = make_float4(0.f, 0.f, 0.f, 0.f);
#pragma unroll 4
  for (int k = 0; k < a.splits; ++k) {
    const float4 v = *(const float4*)(p + k * stride);
    s.x += v.x;
    s.y += v.y;
    s.z += v.z;
    s.w += v.w;
  }
  if (a.bias) {
    const uint2 b = *(const uint2*)((const uint16_t*)a.bias + n);
    s.x += from_bits16<BF16>(b.x & 0xffffu);
    s.y += from_bits16<BF16>(b.x >> 16);
    s.z += from_bits16<BF16>(b.y & 0xffffu);
    s.w += from_bits16<BF16>(b.y >> 16);
  }
  *(uint2*)((uint16_t*)a.out + (int64_t)m * a.o_row + n) =
      make_uint2(to_bits16<BF16>(s.x) | (to_bits16<BF16>(s.y) << 16), to_bits16<BF16>(s.z) | (to_bits16<BF16>(s.w) << 16));
}

struct GemmPlan {
  int bm = 0, splits = 0;
  float us = 0.f;
};

// Tile and number of parts by an estimate of the time; constants fitted (us) over 11 shapes of 64 to 1024 rows.  The 256-row tile is charged
// the 0.82 us a step it took before its fragments were read across the barrier (0.74): with 0.74 another tile is chosen for 235 of
// 7114 shapes, which then take 2.5 % longer in the mean (152 of them longer).  3584 features, K = 18944,
// tile / parts: 64 rows 64 / 1 133, 64 / 4 45, 64 / 8 31, 64 / 16 (two rounds) 37; 512 rows 256 / 1 225, 256 / 4 80 (now 78), 256 / 8 97, 128 / 2 93,
// 64 / 1 130.
GemmPlan plan_gemm(int64_t M, int64_t N, int64_t K) {
  constexpr int kCUs = 256, kBN = 128;
  const int steps = (int)(K / kBK);
  GemmPlan best;
  best.us = 1e9f;
  for (int bm : {64, 128, 256}) {
    if (bm > 64 && M <= bm / 2) continue;
    const float step = bm == 64 ? 0.42f : (bm == 128 ? 0.56f : 0.82f);   // on a nearly idle chip; 17 % more on a full one
    const int64_t tiles_m = (M + bm - 1) / bm, tiles_n = (N + kBN - 1) / kBN;
    for (int s = 1; s == 1 || (s <= 32 && steps / s >= 4); ++s) {
      const int64_t rounds = ((tiles_n * s + 7) / 8 * tiles_m + kCUs / 8 - 1) / (kCUs / 8);   // of the fullest XCD
      const float fill = (float)(tiles_m * tiles_n * s) / (float)(rounds * kCUs);
      float us = rounds * (((steps + s - 1) / s) * step * (1.f + 0.17f * fill) + 6.f);
      if (s > 1) us += 3.f + (float)s * M * N * 8e-6f / 4.f;   // the parts written and read again
      if (us < best.us) best = GemmPlan{bm, s, us};
    }
  }
  return best;
}

}  // namespace
}  // namespace sq

using namespace sq;

// Where the split product is mostly the faster one: the BLAS library's time goes by its own tile and split choices for the exact
// sizes, so no rule on sizes meets every one.  7865 shapes measured (N 64 to 8192, K 64 to 20352 in steps of 64, 5 to 2048 rows; weights
// cold where they are large), library / here in us:
//  * up to 256 rows and 8192 features the library's tiles fill less than a quarter of the chip: 4608 x 3584 of 64 rows 19.5 / 14.9,
//    256 rows 35.6 / 22.8; 3584 x 3584 of 128 rows 22.5 / 16.0; 2048 x 8192 of 5 rows 19.2 / 13.4.  More features fill it: 14336 x 4096
//    of 64 rows 29.6 / 34.1.  Small products are about as long on either side (K below 2048: 0.85 to 1.2), but a call of the library's
//    takes 14 us on the host, one of these 5 to 7;
//  * not few rows of a weight of 64 MB and more whose rows are multiples of 8 KB, which fall on few memory channels here: 8192 x 8192 of 16
//    rows 31.1 / 43.6, of 64 rows 34.3 / 43.5; 4096 x 16384 of 24 rows 33.8 / 45.7 (58 shapes: 0.87 in the mean);
//  * not 161 to 255 rows that leave half a 32-row block empty, of 6144 features and more at K of 2048 to 4096: 6144 x 4096 of
//    200 rows 26.5 / 30.2, 8192 x 3584 of 176 rows 24.5 / 29.5 (54 shapes: 0.95; the whole blocks: 36 shapes, 1.20);
//  * beyond 256 rows where K is at least twice N: 3584 x 18944 of 512 rows 197 / 78, 1024 rows 190 / 135; 4096 x 14336 of 512
//    rows 94.9 / 70.4; 1024 x 8192 of 1024 rows 34.2 / 29.3.  Not 4608 x 3584 (512 rows 32.5 / 36.2) or 4096 x 4096 (30.8 / 30.6).
//    Beyond 640 rows the output itself fills much of the chip where K is short: 1024 x 4096 of 1024 rows 17.8 / 21.8 (37 shapes: 0.85),
//    3584 x 8192 of 777 rows 54.3 / 63.5 (19 shapes: 0.99);
//  * beyond 1024 rows only where K is five times N: 3584 x 18944 of 2048 rows 361 / 254, but 2048 x 8192 of 1500 56.0 / 66.2.
// Of the 7697 shapes taken 46 are more than 2 % slower as calls, by up to 16 % (3072 x 16384 of 2048 rows 180 / 210); in the mean 1.28 times
// faster on the GPU, 1.8 times as calls.
extern "C" int32_t sq_linear_preferred(int64_t M, int64_t N, int64_t K) {
  if (M <= 0 || N <= 0 || K < kBK || K % kBK || N % 4) return 0;
  if (M <= 256) {
    if (N > 8192) return 0;
    if (K % 4096 == 0 && N * K >= 1 << 25 && M <= (N > 6144 || K >= 4 * N ? 64 : 16)) return 0;
    return !(M > 160 && M % 32 && N >= 6144 && K >= 2048 && K <= 4096);
  }
  if (M <= 1024) return K >= 2 * N && !(M > 640 && ((N >= 1024 && K <= 4096) || (N >= 3072 && K <= 8192)));
  return M <= 2048 && K >= 5 * N;
}

extern "C" size_t sq_linear_workspace_bytes(int64_t M, int64_t N, int64_t K) {
  if (M <= 0 || N <= 0 || K < kBK || K % kBK) return 0;
  const GemmPlan p = plan_gemm(M, N, K);
  return p.splits > 1 ? (size_t)p.splits * M * N * sizeof(float) : 0;
}

extern "C" int sq_linear(const DLTensor* x, const DLTensor* weight, const DLTensor* bias, DLTensor* out, DLTensor* workspace, void* stream) {
  SQ_REQUIRE(x && weight && out, SQ_EINVAL, "sq_linear: x, weight and out must be non-null");
  const int dev = x->device.device_id;
  int rc;
  if ((rc = check_tensor(x, "x", 2, dev)) || (rc = check_tensor(weight, "weight", 2, dev)) || (rc = check_tensor(out, "out", 2, dev))) return rc;
  const DType dt = dtype_of(x);
  SQ_REQUIRE((dt == DType::BF16 || dt == DType::F16) && dtype_of(weight) == dt && dtype_of(out) == dt, SQ_EDTYPE, "sq_linear: x, weight and out must all be bf16 or all fp16");
  const int64_t M = x->shape[0], K = x->shape[1], N = weight->shape[0];
  SQ_REQUIRE(M > 0 && N > 0 && weight->shape[1] == K && out->shape[0] == M && out->shape[1] == N, SQ_ESHAPE, "sq_linear: shapes disagree");
  SQ_REQUIRE(K >= kBK && K % kBK == 0 && N % 4 == 0, SQ_EUNSUPPORTED, "sq_linear: K must be a multiple of 64 and N of 4 (got %lld, %lld)", (long long)K, (long long)N);
  const int64_t xs = stride_of(x, 0), ws = stride_of(weight, 0), os = stride_of(out, 0);
  SQ_REQUIRE(xs >= K && ws >= K && os >= N && xs % 8 == 0 && ws % 8 == 0 && os % 4 == 0, SQ_ESHAPE, "sq_linear: rows must not overlap and must start on 16-byte (out: 8-byte) boundaries");
  // a tile's rows are reached by 32-bit offsets from the operand's start
  SQ_REQUIRE((M - 1) * xs + K < (1ll << 31) && (N - 1) * ws + K < (1ll << 31) && M < (1 << 30) && N < (1 << 30), SQ_EUNSUPPORTED, "sq_linear: operands of 4 GiB and more are not supported");
  if (bias) {
    if ((rc = check_tensor(bias, "bias", 1, dev))) return rc;
    SQ_REQUIRE(dtype_of(bias) == dt && bias->shape[0] == N && stride_of(bias, 0) == 1, SQ_ESHAPE, "sq_linear: bias must be a contiguous [%lld] of x's dtype", (long long)N);
  }
  const GemmPlan plan = plan_gemm(M, N, K);
  GemmArgs a = {};
  a.x = data_of(x);
  a.w = data_of(weight);
  a.bias = bias ? data_of(bias) : nullptr;
  a.out = data_of(out);
  a.x_row = xs * 2;
  a.w_row = ws * 2;
  a.o_row = os;
  a.M = (int)M;
  a.N = (int)N;
  a.steps = (int)(K / kBK);
  a.splits = plan.splits;
  a.tiles_m = (int)((M + plan.bm - 1) / plan.bm);
  a.tiles_n = (int)((N + 127) / 128);
  if (plan.splits > 1) {
    const size_t need = (size_t)plan.splits * M * N * sizeof(float);
    SQ_REQUIRE(workspace && on_gpu(workspace) && workspace->device.device_id == dev && is_compact(workspace) &&
                   (size_t)numel_of(workspace) * (workspace->dtype.bits / 8) >= need && ((uintptr_t)data_of(workspace) & 15) == 0,
               SQ_EWORKSPACE, "sq_linear: needs a compact, 16-byte aligned workspace of %zu bytes on the tensors' device", need);
    a.part = (float*)data_of(workspace);
  }
  int cur = -1;
  SQ_HIP(hipGetDevice(&cur));
  SQ_REQUIRE(cur == dev, SQ_EDEVICE, "sq_linear: tensors live on device %d but the current device is %d", dev, cur);
  hipStream_t st = (hipStream_t)stream;
  const unsigned blocks = (unsigned)(((int64_t)a.tiles_n * a.splits + 7) / 8 * 8 * a.tiles_m);
#define SQ_GEMM(BF, BM, WM, WN, NB)                                                                                                \
  do {                                                                                                                             \
    constexpr int smem = NB * (BM + 128) * kRowBytes;                                                                              \
    SQ_HIP(hipFuncSetAttribute((const void*)gemm_kernel<BF, BM, 128, WM, WN, NB>, hipFuncAttributeMaxDynamicSharedMemorySize, smem)); \
    hipLaunchKernelGGL((gemm_kernel<BF, BM, 128, WM, WN, NB>), dim3(blocks), dim3(kThreads), smem, st, a);                         \
  } while (0)
#define SQ_GEMMS(BF)                                  \
  do {                                                \
    if (plan.bm == 64) SQ_GEMM(BF, 64, 2, 4, 5);      \
    else if (plan.bm == 128) SQ_GEMM(BF, 128, 2, 4, 4); \
    else SQ_GEMM(BF, 256, 4, 2, 3);                   \
  } while (0)
  if (dt == DType::BF16) SQ_GEMMS(true);
  else SQ_GEMMS(false);
#undef SQ_GEMMS
#undef SQ_GEMM
  SQ_HIP(hipGetLastError());
  if (plan.splits > 1) {
    const unsigned n = (unsigned)((M * (N / 4) + 255) / 256);
    if (dt == DType::BF16) hipLaunchKernelGGL((gemm_add_kernel<true>), dim3(n), dim3(256), 0, st, a);
    else hipLaunchKernelGGL((gemm_add_kernel<false>), dim3(n), dim3(256), 0, st, a);
    SQ_HIP(hipGetLastError());
  }
  return SQ_OK;
}
