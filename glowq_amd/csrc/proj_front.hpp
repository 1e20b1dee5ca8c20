// r[m, j] = fp16(sum_k x[m, k] R[j, k]) by workgroups in front of the grid of a group launch that needs r at its end (gemm.hip,
// skinny_tiled.hip): a tile of 32 kA token rows by 32 kA rows of R per workgroup, both operands by direct-to-LDS loads in stages of 128
// columns of K, kStages of them in a ring (swizzled like the activations of gemm_tiled_kernel: slot c' of row q holds the row's 16-byte
// piece c' ^ (q % 16)).  kA = 1: the waves deal a stage's eight k-steps among themselves; kA = 2: two by two waves own 32 x 32 each (and eight
// waves deal the k-steps in halves).  The waves' sums meet in LDS once, in wave order, and r goes out with stores that pass the caches
// of this part of the chip, acknowledged before the tile's word goes up.
// Long K is cut over `slices` workgroups of a tile: all but the first leave their fp32 sums in the workspace and raise words of their own,
// and the first adds them in slice order (bounded: without them it walks all of K by itself).
// What bounds such a workgroup is a memory round trip a stage: the compiler waits for all loads to LDS in front of a barrier (the release of
// __syncthreads covers LDS writes, which it takes them for), so a stage is in flight only while the one before it is multiplied,
// however many the ring holds.  It has most of the group launch's time for it.  A launch of its own for r takes two dependent launches from some twenty rows on (tiles with K cut over
// workgroups, their sum).
// K % 128 == 0, rank % 8 == 0, 16-byte aligned x, R and r, x and R below 4 GiB.
#pragma once

#include "common.hpp"
#include "handover.hpp"

namespace glowq {

// What the kernels hand to their workgroups in front: workgroup p takes slice p % slices of tile p / slices, the tiles of a row block next to
// each other; word p of `pub` is its word, that of a tile's first slice the tile's.  Behind `count` of them, up to `front`, come workgroups that
// only hold a place until r is there (see plan_front in gemm.hip).
struct FrontArgs {
  const half_t* x;
  const half_t* R;
  half_t* r_out;
  unsigned long long* pub;
  float* partials;  // [workgroup][1024 kA kA], with slices > 1
  int M, K, rank;
  int front, count, a, slices;  // workgroups in front, those of them with work, kA, slices of K
  unsigned spin;  // looks at a word before a reader does without; kNeverRaised: a test in which no word goes up
  int any_cost;   // a test in which every launch that can computes r itself
};
constexpr unsigned kNeverRaised = 0xFFFFFFFFu;

// Whether the words [p0, p1) step `step` of this launch are all up, looked at by every lane of a wave at most `spin` + 1 times.
__device__ __forceinline__ bool wait_words(const unsigned long long* pub, int p0, int p1, int step, unsigned long long tag, unsigned spin) {
  const int lane = (int)threadIdx.x & 63;
  bool all = false;
  for (unsigned looks = 0; !all && looks <= spin && spin != kNeverRaised; ++looks) {
    bool up = true;
    for (int p = p0 + lane * step; p < p1; p += 64 * step)
      up = up && (__hip_atomic_load(pub + p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) & kTagMask) == tag;
    all = __builtin_amdgcn_ballot_w64(!up) == 0;
    if (!all) __builtin_amdgcn_s_sleep(2);
  }
  return all;
}

template <int kWaves, int kA>
struct ProjFront {
  static_assert((kWaves == 4 || kWaves == 8) && (kA == 1 || kA == 2), "four or eight waves, tiles of 32 or 64");
  static constexpr int kRow = 256;  // bytes of a staged row
  // (five stages of the small tiles: 80 KB of LDS leave two workgroups on a compute unit where there were three, and with the wait above the further
  // ones were never in flight: no faster)
  static constexpr int kStages = kA == 1 ? 3 : 2;
  static constexpr int kStageBytes = 64 * kA * kRow;
  static constexpr int kLds = kStages * kStageBytes;
  static constexpr int kLoads = 16 * kA / kWaves;  // of a wave per stage, a kilobyte (four rows) each
  static_assert(kWaves * 4096 <= kLds, "the waves' sums");

  // stages [st0, st1) of the tile at (m0, j0): the waves' sums in `smem` ([wave][register][lane] floats)
  static __device__ __forceinline__ void accumulate(const FrontArgs& f, int m0, int j0, int st0, int st1, unsigned char* smem) {
    const int tid = (int)threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int ln = lane & 31, lh = lane >> 5, K = f.K;
    const auto rsrc = [](const void* p, size_t bytes) {
      return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(p), 0, (int)(uint32_t)bytes, 0x00020000);
    };
    const __amdgpu_buffer_rsrc_t rs_x = rsrc(f.x, (size_t)f.M * K * 2), rs_r = rsrc(f.R, (size_t)f.rank * K * 2);  // rows past the end: zeros
    const int sub = 4 * (wave & 3) + (lane >> 4);  // row of this lane's pieces within a block of sixteen
    const uint32_t lane_off = (uint32_t)sub * (uint32_t)K * 2u + (uint32_t)((lane & 15) ^ sub) * 16u;
    auto request = [&](int st) __attribute__((always_inline)) {
      typedef __attribute__((address_space(3))) void* lds_ptr_t;
      unsigned char* dst = smem + (size_t)((st - st0) % kStages) * kStageBytes;
#pragma unroll
      for (int i = 0; i < kLoads; ++i) {
        const int q = (wave >> 2) + (kWaves / 4) * i;  // block of sixteen rows: 2 kA of x, then 2 kA of R
        const bool of_x = (kWaves / 4) * i < 2 * kA;
        const uint32_t row = (uint32_t)(of_x ? m0 + 16 * q : j0 + 16 * (q - 2 * kA));
        // (past the end: an offset past the end of the descriptor, so that the count of loads in flight holds to the last stage)
        const uint32_t off = st < st1 ? row * (uint32_t)K * 2u + (uint32_t)st * 256u : 0xFFFF0000u;
        __builtin_amdgcn_raw_ptr_buffer_load_lds(of_x ? rs_x : rs_r, (lds_ptr_t)(dst + (16 * q + 4 * (wave & 3)) * kRow), 16, (int)lane_off, (int)off, 0, 0);
      }
    };
    f16v acc;
#pragma unroll
    for (int i = 0; i < 16; ++i) acc[i] = 0.f;
    const int wr = kA == 1 ? 0 : ((wave >> 1) & 1) * 32, wc = kA == 1 ? 0 : (wave & 1) * 32;
    constexpr int kSteps = kA == 1 ? 8 / kWaves : 32 / kWaves;  // k-steps of a wave per stage
    const int t0 = kA == 1 ? wave * kSteps : (wave >> 2) * kSteps;
#pragma unroll
    for (int i = 0; i < kStages - 1; ++i) request(st0 + i);
    for (int st = st0; st < st1; ++st) {
      constexpr int n = (kStages - 2) * kLoads;
      __builtin_amdgcn_s_waitcnt((n & 15) | 0x0F70 | ((n >> 4) << 14));  // this wave's part of stage st has landed ...
      __syncthreads();                                                   // ... and everybody's; everybody is done with stage st - 1
      request(st + kStages - 1);
      const unsigned char* base = smem + (size_t)((st - st0) % kStages) * kStageBytes;
#pragma unroll
      for (int t = 0; t < kSteps; ++t) {
        const int slot = ((2 * (t0 + t) + lh) ^ (ln & 15)) << 4;
        const h8 af = *reinterpret_cast<const h8*>(base + (wr + ln) * kRow + slot);
        const h8 bf = *reinterpret_cast<const h8*>(base + (32 * kA + wc + ln) * kRow + slot);
        acc = __builtin_amdgcn_mfma_f32_32x32x16_f16(af, bf, acc, 0, 0, 0);
      }
    }
    __builtin_amdgcn_s_waitcnt(0x0F70);  // nothing may land in the stages any more
    __syncthreads();
    float* red = reinterpret_cast<float*>(smem);  // [wave][register][lane]
#pragma unroll
    for (int i = 0; i < 16; ++i) red[(wave * 16 + i) * 64 + lane] = acc[i];
    __syncthreads();
  }
  // the sums of the tile's entries (row, col .. col + 3), e = row * 8 kA + col / 4
  static __device__ __forceinline__ f4 sums_of(int e, const unsigned char* smem) {
    const float* red = reinterpret_cast<const float*>(smem);
    const int row = e / (8 * kA), col = (e % (8 * kA)) * 4;
    const int at = ((((row & 31) >> 3) * 4 + (row & 3)) * 64 + ((row >> 2) & 1) * 32 + (col & 31));
    const int first = kA == 1 ? 0 : (row >> 5) * 2 + (col >> 5);
    constexpr int kParts = kA == 1 ? kWaves : kWaves / 4, kStride = kA == 1 ? 1 : 4;
    f4 v = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int p = 0; p < kParts; ++p) v += *reinterpret_cast<const f4*>(red + (first + p * kStride) * 1024 + at);
    return v;
  }

  // workgroup p in front, by its first 64 kWaves threads (the others must be gone: the barriers count the waves that arrive)
  static __device__ __forceinline__ void run(const FrontArgs& f, int p, unsigned long long tag, unsigned char* smem) {
    const int tid = (int)threadIdx.x;
    const int tile = p / f.slices, slice = p - tile * f.slices;
    const int cols = (f.rank + 32 * kA - 1) / (32 * kA);
    const int m0 = tile / cols * (32 * kA), j0 = tile % cols * (32 * kA);
    const int stages = f.K >> 7, per = (stages + f.slices - 1) / f.slices;
    constexpr int kQuads = 256 * kA * kA, kThreads = 64 * kWaves;
    accumulate(f, m0, j0, min(slice * per, stages), min((slice + 1) * per, stages), smem);
    if (slice > 0) {
      float* out = f.partials + (size_t)p * (4 * kQuads);
      for (int e = tid; e < kQuads; e += kThreads) {
        const f4 v = sums_of(e, smem);
#pragma unroll
        for (int h = 0; h < 2; ++h)
          __hip_atomic_store(reinterpret_cast<unsigned long long*>(out + 4 * e) + h, __builtin_bit_cast(unsigned long long, float2{v[2 * h], v[2 * h + 1]}),
                             __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      }
    } else {
      bool have = f.slices == 1 || wait_words(f.pub, p + 1, p + f.slices, 1, tag, f.spin);
      if (f.slices > 1) have = __syncthreads_and(have) != 0;  // one answer for the workgroup
      if (!have) {
        __syncthreads();
        accumulate(f, m0, j0, 0, stages, smem);
      }
      for (int e = tid; e < kQuads; e += kThreads) {
        f4 v = sums_of(e, smem);
        if (have)
          for (int z = 1; z < f.slices; ++z) {
            const unsigned long long* in = reinterpret_cast<const unsigned long long*>(f.partials + (size_t)(p + z) * (4 * kQuads) + 4 * e);
            const float2 lo = __builtin_bit_cast(float2, __hip_atomic_load(in, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT));
            const float2 hi = __builtin_bit_cast(float2, __hip_atomic_load(in + 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT));
            v += f4{lo.x, lo.y, hi.x, hi.y};
          }
        const int m = m0 + e / (8 * kA), j = j0 + e % (8 * kA) * 4;
        if (m < f.M && j < f.rank) {
          const h4 o = {(half_t)v[0], (half_t)v[1], (half_t)v[2], (half_t)v[3]};
          __hip_atomic_store(reinterpret_cast<unsigned long long*>(f.r_out + (size_t)m * f.rank + j), __builtin_bit_cast(unsigned long long, o),
                             __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
      }
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // the stores are acknowledged: they are where every reader looks
    __syncthreads();
    if (tid == 0 && f.spin != kNeverRaised) __hip_atomic_store(f.pub + p, tag, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  }
};

// Workgroup p < f.front of a launch.
template <int kWaves>
__device__ __forceinline__ void run_front(const FrontArgs& f, int p, unsigned long long tag, unsigned char* smem) {
  if (p >= f.count) {
    if (threadIdx.x < 64) wait_words(f.pub, (p - f.count) % (f.count / f.slices) * f.slices, (p - f.count) % (f.count / f.slices) * f.slices + 1, 1, tag, f.spin);
  } else if (f.a == 2) {
    ProjFront<kWaves, 2>::run(f, p, tag, smem);
  } else {
    ProjFront<kWaves, 1>::run(f, p, tag, smem);
  }
}
constexpr size_t front_lds(const FrontArgs& f) { return (size_t)(f.a == 2 ? 2 : 3) * 64 * f.a * 256; }

}  // namespace glowq
