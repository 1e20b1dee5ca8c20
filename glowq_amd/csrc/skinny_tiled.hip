// Matrix-core kernel for a handful of token rows (5..32, from 2 on the longest streams) on members that bring the tiled copy of their weights
// (tiled.hpp): the weights are streamed once, every 16-byte load of a wave is one contiguous kilobyte and lands in
// the lanes' registers as the B operand of v_mfma_f32_32x32x16_f16 -- no pass through LDS, no per-lane scale and
// zero-point gather (both ride in the stream).
//
// Arithmetic: that of the reference's GEMV (src/cuda_w4a16/csrc/gemv_w4a16.cu:96-112, which the reference uses up to 128
// token rows): the weight (code - zero) * scale is never rounded to fp16.  The codes go to the matrix cores as they are
// -- a nibble masked in place is the fp16 subnormal code * 2^-24 (or code * 2^-20; the activations of those columns
// are staged divided by 16) -- the eight instructions of a 128-column half leave sum code * x per (token row, output
// row), a ninth adds -zero * sum x (the per-row sums of the activations come as one more A fragment), and the scale
// is applied to that sum in fp32: y += scale * 2^24 * sum.  Five vector instructions per code word instead of the
// thirteen a dequantisation to fp16 takes: the vector ALUs, not memory, bound the dequantising form.
// (The division by 16 is exact for |x| >= 2^-10; below, x / 16 is a subnormal and x is rounded to a multiple of 2^-20,
// an absolute error of 2^-21 and less.  The row sums are carried as two halves, good to 2^-22 of their value.)
// Up to 16 token rows the products are tiles of 16 by 16 (v_mfma_f32_16x16x32_f16: half the matrix time and half the LDS reads of 32 rows
// that are half empty): v_permlane16_swap trades rows of sixteen lanes between two neighbouring words, after which each holds sixteen
// columns over the k values of both, and one more product per fragment, against ones, leaves the row sums in fp32 (no sums in the
// producers, whose vector instructions a step had to wait for).  All eight fragments of a step are asked for at its head.  Launch
// without a correction, 16 rows, us: 2 x 14336 x 4096 18.4 -> 15.3 (4.0 TB/s), 2 x 17408 x 5120 26.4 -> 23.2, 17408 x 5120 19.7 -> 15.4,
// 5120 x 17408 20.0 -> 16.3.
// kCanon: the narrow tiles on the canonical buffers, for groups without a tiled copy: a lane takes 16 bytes (four words) of the row that is its
// column, and word j of all lanes is an operand by itself -- the k values of a product may come in any order that the activations share, which
// are read from where those words' columns are staged, in the order the masks leave the codes.  A load instruction covers half a cache line of
// sixteen rows, so the two halves are asked for together and without the non-temporal hint (18944 x 3584, 16 rows: 13.4, with it 14.2; asked
// for half a step apart 15.9); scales and zero-points come for four super-blocks at a time (with two gathers a super-block 15.2).
// From 9 rows on (kWhole) the activations stay whole, as in the rounding kernel of skinny.hip that has these rows otherwise: the masks of two neighbouring
// words make one operand of the low nibbles and one of the high ones, with sums of their own (error of the output at |x| around 1e-4, against
// x / 16 in fp16: 2.1e-4 / 2.0e-3; same matrix and vector instructions: 14336 x 4096 at 16 rows 12.8 us / 12.6, 1024 x 5120 9.2 / 9.5, 4096 x 14336
// 19.5 / 19.7, 2 x 14336 x 4096 15.9 / 15.2, with r inside 19.9 / 18.2.  As code - zero, nine vector instructions a word instead of five: 13.4, 9.6, 20.2), and sums that are not finite are taken again
// with code - zero, which gives an infinite activation's products their signs.  At 8 rows two sums cost 2 to 5 % more, and the
// raw-code form of skinny.hip divides by 16 as well.
// Launch without a correction, 8 and 16 rows, us, against the kernels of skinny.hip: 14336 x 4096 15.7, 16.9 -> 11.6, 12.5, 18944 x 3584
// 17.9, 20.8 -> 12.5, 13.4, 1024 x 5120 8.9, 9.8 -> 8.2, 8.4, 4096 x 14336 15.3, 17.5 -> 14.8, 15.3, 8192 x 2048 6.3, 6.9 -> 5.3, 6.3.
//
// A workgroup owns 32 cw output columns of one member (a row block of 32 per consumer wave) and all token rows.  Its
// waves come in K groups that walk contiguous parts of the K range in step and meet in LDS at the end; a K group is
// `cw` consumer waves (four as a rule; more where that brings the column tiles down to one per compute unit) and kPW
// producer waves.
//   * Consumers keep kD sets of weight registers in rotation: the set of super-block v is refilled with super-block
//     v + kD as soon as its words have been masked, so up to kD - 1 super-blocks of a wave are in flight while it
//     computes.  They wait for nothing but their weights.
//   * Producers load the activations of the super-blocks ahead (token rows x 512 bytes; four sets of registers in rotation -- with one,
//     every step took an L2 round trip under load: 3 to 17 % of the launches) in memory order (the tiled copy
//     holds the nibbles of a word in the order the masks deliver them: no permutation), divide the pairs at positions
//     2, 3 and 6, 7 of every octet by 16, from 17 rows on sum every row's two
//     128-column halves in fp32, and leave all of it in the LDS stage the consumers do not read (528-byte rows:
//     conflict-free 16-byte reads).  One barrier per super-block.  A wave's loads return in order: a consumer that
//     fetched activations as well would have to drain its weight requests with every step.
// The correction is a K-extension behind the weights: in the last rotation the sets are refilled with the blocks of
// the tiled left factor (fp16, already in B-operand order), r follows the last super-block through the stages, and
// acc += alpha * (r . L^T) from an accumulator of its own.
// kProj: the launch computes r = x R^T itself.  Workgroups in front of the grid (roles dealt as in handover.hpp) produce
// blocks of four token rows by four rows of R in the arithmetic of shared_proj_block_kernel and write them to r_out with
// stores that pass the caches private to a part of the chip (two blocks at a time where the workgroup has eight waves
// and more), each raises its flag when its stores are acknowledged, and the first of them turns the flags into one ready
// word.  The producer waves of the other workgroups look for that word when
// they are about to send r through the stages -- during the last super-block, so the producers in front have the whole
// weight stream to get there -- and read r with loads that pass those caches; one that does not see the word within its
// bound computes the pieces of r it would have loaded, so every wave ends whatever becomes of the workgroups in front.
// Few column tiles (o_proj, down_proj): K is also cut into gridDim.y slices, each workgroup leaves its fp32 tile in the
// caller's workspace and skinny_tiled_reduce_kernel adds the slices in order.  Calls of 33 to 64 rows run in this arithmetic on
// gemm_tiled_kernel (gemm.hip).
#include <algorithm>
#include <atomic>
#include <cstdlib>

#include <type_traits>

#include "common.hpp"
#include "dequant.hpp"
#include "handover.hpp"
#include "proj_block.hpp"
#include "tiled.hpp"

namespace glowq {

struct TileMember {
  const unsigned char* wt;  // tiled weights (tiled.hpp)
  const unsigned char* lt;  // tiled left factor or nullptr
  const half_t* bias;
  half_t* y;
  int N, ldy;
  int col0;                 // first column of the member in a row of the partial buffer (members padded to 128)
  // kCanon: wt is the packed weight itself, lt the left factor [N, rank]
  const half_t* scales;
  const int32_t* qzeros;
  int ldw, lds, ldz;
};

struct TileArgs {
  const half_t* r;  // [M, rank] or nullptr
  TileMember mem[GLOWQ_MAX_MEMBERS];
  int blk_end[GLOWQ_MAX_MEMBERS];
  int n_members;
  int M, K, rank;
  float alpha;
  int slices;       // gridDim.y
  float* partials;  // [slice][M][ldp] fp32 when slices > 1
  int ldp;
  int tiles;        // column tiles of the whole group: the grid's x extent
  int cw;           // consumer waves per K group: a tile is 32 cw columns
  // kProj (the launch computes r itself; `r` then points at r_out)
  const half_t* R;          // [rank, K]
  half_t* r_out;            // [M, rank]
  unsigned long long* pub;  // [0]: the ready word; [kTiledFlags + p]: the flag of producer p
  unsigned spin;            // polls of the ready word before a producer wave computes its pieces of r itself
  int producers;            // workgroups in front that produce r
  int teams;                // blocks of r a producer works on at a time: teams of four waves (1 or 2)
};
constexpr int kTiledFlags = 512;  // the producers' flags lie 4096 bytes behind the ready word
constexpr int kTiledMaxProducers = 512;
constexpr size_t kTiledHandoverBytes = (size_t)(kTiledFlags + kTiledMaxProducers) * 8;
// blocks of r a producer in front may have to compute (gate|up of a 14B layer, rank 256, 35 producers: 3.7 blocks each at
// eight rows 26.8 us against 30.9 with the projection launch, 5.5 at twelve 27.4 against 31.3, 7.3 at sixteen 30.5 to 31.5
// against 31.5)
constexpr int kTiledProjBlocks = 6;

namespace {

// The code of column k of a word (nibble k in the canonical buffers) moves to nibble (0,4,1,5,2,6,3,7)[k]: the four
// masks of the kernels then deliver the eight codes in column order.
__device__ __forceinline__ uint32_t mask_order_word(uint32_t w) {
  uint32_t o = 0;
#pragma unroll
  for (int k = 0; k < 8; ++k) o |= ((w >> (4 * k)) & 0xFu) << (4 * ((k >> 1) + 4 * (k & 1)));
  return o;
}

// total over a row of 16 lanes, in every lane of it
__device__ __forceinline__ float row16_total_t(float v) {
  int t;
  t = __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), 0x121, 0xF, 0xF, true);  // row_ror:1
  v += __builtin_bit_cast(float, t);
  t = __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), 0x122, 0xF, 0xF, true);  // row_ror:2
  v += __builtin_bit_cast(float, t);
  t = __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), 0x124, 0xF, 0xF, true);  // row_ror:4
  v += __builtin_bit_cast(float, t);
  t = __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), 0x128, 0xF, 0xF, true);  // row_ror:8
  v += __builtin_bit_cast(float, t);
  return v;
}

constexpr int kRowBytes = 528;  // 512 bytes of a token row's super-block + 16: rows 8 apart share no bank
constexpr int kD = 4;           // weight register sets in rotation
#ifndef GLOWQ_TILED_AUX
#define GLOWQ_TILED_AUX 2
#endif
constexpr int kStreamAux = GLOWQ_TILED_AUX;  // cache policy of the weight loads: non-temporal, every byte is used once

}  // namespace

// kRows: token rows a K group stages (8, 16 or 32).  kWk: K groups per workgroup.  kPW: producer waves per K group.
// The leading scalar arguments arrive in registers with the wave (kernel-argument preload): what a workgroup of the
// first member needs to request its first weights and activations, without a round trip to the argument buffer.
// Consumer waves a K group may have and the workgroup size that goes with it: 768 threads at most.
constexpr int tiled_max_cw(int wk, int pw) { return wk > 1 ? 4 : 12 - pw; }
constexpr int tiled_max_threads(int wk, int pw) { return (tiled_max_cw(wk, pw) + pw) * 64 * wk; }

template <int kRows, int kWk, int kPW, bool kProj = false, bool kCanon = false>
__global__ __launch_bounds__(tiled_max_threads(kWk, kPW))
void skinny_tiled_kernel(const half_t* __restrict__ x, const int M, const int K, const int slices,
                         const unsigned char* __restrict__ wt0, const int blk_end0, const int N0, const int cw, const TileArgs g) {
  extern __shared__ __attribute__((aligned(16))) unsigned char smem_all[];
  static_assert(kRows <= 32, "one 32-row tile per consumer wave");
  constexpr int kPQ = (kRows + 2 * kPW - 1) / (2 * kPW);  // 16-byte pieces of a super-block of x per producer thread
  static_assert(kPQ * 2 * kPW == kRows, "whole passes");
  constexpr bool kNarrow = kRows <= 16;          // tiles of 16 token rows by 16 columns
  static_assert(kNarrow || !kCanon, "the canonical buffers are read by the narrow tiles");
  constexpr bool kWhole = kCanon && kRows > 8;   // activations are not divided by 16
  constexpr int kSigBytes = kNarrow ? 0 : kRows * 16;  // per 128-column half: a 16-byte fragment of sums per token row
  constexpr int kStage = kRows * kRowBytes + 2 * kSigBytes;
  const int group_threads = (cw + kPW) * 64;  // the consumer waves, then the producer waves
  const int gk = kWk > 1 ? __builtin_amdgcn_readfirstlane((int)threadIdx.x >= group_threads ? 1 : 0) : 0;
  static_assert(kWk <= 2, "gk is a comparison");
  const int tig = (int)threadIdx.x - gk * group_threads;  // thread within the K group
  const int lane = tig & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tig >> 6);
  const bool producer = wave >= cw;
  const int ln = lane & 31, lh = lane >> 5;
  unsigned char* smem = smem_all + gk * 2 * kStage;

  int tile = (int)blockIdx.x;
  unsigned long long tag = 0;
  if constexpr (kProj) {
    tag = launch_tag();
    const int front = g.producers;
    const int role = front_role(tile, front);
    if (role >= 0) {
      if (role >= front || blockIdx.y != 0) return;
      {
        // teams of four waves, each with a block of its own at a time
        const int teams = g.teams;
        if ((int)threadIdx.x >= 256 * teams) return;  // (the body's barriers count the waves that arrive)
        const int team = (int)threadIdx.x >> 8, ttid = (int)threadIdx.x & 255;
        float* part = reinterpret_cast<float*>(smem_all) + team * (4 * 16 + 16);
        const int jblocks = (g.rank + 3) >> 2;
        float* vals = part + 4 * 16;
        const int nblocks = jblocks * ((M + 3) >> 2);
        // blocks of four token rows by four rows of R, dealt round robin to the producers.  (Blocks of eight token rows,
        // half as many: 21.5 against 20.1 us at 12 rows on gate|up of an 8B layer, 32.0 against 27.5 on a 14B layer's;
        // three 16-byte pieces of every row in flight per thread instead of two, a row of 5120 columns in one round trip:
        // no difference.)
        for (int b0 = role * teams; b0 < nblocks; b0 += g.producers * teams) {
          const int b = b0 + team;
          const bool active = b < nblocks;
          const int bj = b % jblocks, bm = b / jblocks;
          proj_block_body<4, 4>(x, g.R, M, K, g.rank, 4 * bj, 4 * bm, part,
                                [&](int m, int j, float v) { vals[(m - 4 * bm) * 4 + (j - 4 * bj)] = v; }, ttid, active);
          __syncthreads();
          // pairs of neighbouring entries of a token row go out as one 32-bit store (ranks are multiples of 8)
          if (active && ttid < 8) {
            const int mi = ttid >> 1, pp = ttid & 1;
            const int m = 4 * bm + mi, j = 4 * bj + 2 * pp;
            if (m < M && j < g.rank) {
              const h2 v = {(half_t)vals[mi * 4 + 2 * pp], (half_t)vals[mi * 4 + 2 * pp + 1]};
              __hip_atomic_store(reinterpret_cast<uint32_t*>(g.r_out + (size_t)m * g.rank + j), __builtin_bit_cast(uint32_t, v),
                                 __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            }
          }
          __syncthreads();  // (part and vals are free for the next block)
        }
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // the stores are acknowledged: r is where every reader looks
        __syncthreads();
        if (threadIdx.x == 0 && g.spin != 0xFFFFFFFFu)  // (that value: a test in which the flags never go up)
          __hip_atomic_store(g.pub + kTiledFlags + role, tag, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      }
      // the first producer is also the collector: one wave, lane l takes flags l, l + 64, ...
      if (role != 0 || threadIdx.x >= 64) return;
      bool all = false;
      for (unsigned spins = 0; !all && spins <= g.spin && g.spin != 0xFFFFFFFFu; ++spins) {
        bool mine = true;
        for (int p = (int)threadIdx.x; p < g.producers; p += 64)
          mine = mine && (__hip_atomic_load(g.pub + kTiledFlags + p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) & kTagMask) == tag;
        all = __builtin_amdgcn_ballot_w64(!mine) == 0;
        if (!all) __builtin_amdgcn_s_sleep(2);
      }
      if (all && threadIdx.x == 0) __hip_atomic_store(g.pub, tag, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      return;
    }
    if (tile >= g.tiles) return;  // (a front larger than the grid behind it leaves places between its workgroups empty)
  }
  const int SB = K >> 8;
  // The workgroup's super-blocks (slice blockIdx.y of K) are dealt to its K groups in contiguous parts of `pg`; every
  // group runs the same number of steps, a whole number of rotations of the register sets.  Steps past the end of a
  // group's part read past the end of its descriptor, which returns zeros (zero codes at scale zero), and in the last
  // rotation they are skipped.
  const int per = (SB + slices - 1) / slices;
  const int s0 = min((int)blockIdx.y * per, SB), s1 = min(s0 + per, SB);
  const int pg = (s1 - s0 + kWk - 1) / kWk;
  const int sb0 = min(s0 + gk * pg, s1), sb1 = min(sb0 + pg, s1);
  const int rounds = max(1, (pg + kD - 1) / kD);
  const int steps = rounds * kD;
  const bool wg_corr = g.r != nullptr && blockIdx.y == 0;  // the first slice of a group that has an r: uniform
  const int LBall = (g.rank + 63) >> 6;                     // correction blocks of 64 rank columns

  const auto rsrc = [](const void* p, size_t bytes) {
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(p), 0, (int)(uint32_t)bytes, 0x00020000);
  };

  if (producer) {
    // ---- producer waves: the activations of step v + 1 go from registers to the stage the consumers do not read,
    // the loads of step v + 2 go out, barrier.  After the last super-block the first 256 columns of r follow through
    // the stages, then the later passes of a rank above 256.
    const int pt = tig - cw * 64;              // 0 .. 64 kPW - 1
    const int prow = pt >> 5, pcol = pt & 31;  // piece q of this thread: token row 2 kPW q + prow, 16-byte piece pcol
    const __amdgpu_buffer_rsrc_t rs_x = rsrc(x, (size_t)M * K * 2);
    const __amdgpu_buffer_rsrc_t rs_r = rsrc(g.r != nullptr ? (const void*)g.r : (const void*)x, g.r != nullptr ? (size_t)M * g.rank * 2 : 0);
    // kXD sets of activation registers in rotation: a piece has kXD - 1 steps to arrive
    constexpr int kXD = kNarrow || kPQ <= 4 ? 4 : 2;
    static_assert(kD % kXD == 0, "the sets rotate with the steps of a round");
    u32x4 avs[kXD][kPQ];
    auto load_a = [&](u32x4 (&av)[kPQ], bool is_r, int idx) __attribute__((always_inline)) {
      const __amdgpu_buffer_rsrc_t rs = is_r ? rs_r : rs_x;
      const uint32_t ld = (uint32_t)(is_r ? g.rank : K);
#pragma unroll
      for (int q = 0; q < kPQ; ++q) {
        const uint32_t row = (uint32_t)min(2 * kPW * q + prow, M - 1);
        uint32_t off = (row * ld + (uint32_t)pcol * 8u) * 2u;
        if (is_r && idx * 256 + pcol * 8 >= g.rank) off = 0x80000000u;  // zeros past the rank (not the next row, which may not be finite)
        av[q] = __builtin_amdgcn_raw_buffer_load_b128(rs, (int)off, idx * 512, 0);
      }
    };
    auto store_a = [&](const u32x4 (&av)[kPQ], int stage, bool is_r) __attribute__((always_inline)) {
      unsigned char* dst = smem + stage * kStage + prow * kRowBytes + pcol * 16;
      unsigned char* sig = smem + stage * kStage + kRows * kRowBytes + (pcol >> 4) * kSigBytes + prow * 16;
      const h2 ones = {(half_t)1.f, (half_t)1.f};
      const h2 sixteenth = {(half_t)0.0625f, (half_t)0.0625f};
#pragma unroll
      for (int q = 0; q < kPQ; ++q) {
        if constexpr (kWhole) {
          // the pairs of columns that a mask leaves in the low bits of a byte, (0, 4) and (2, 6), of two neighbouring words, then those it leaves
          // in the high bits, (1, 5) and (3, 7): a piece of the stage holds one kind; r as it is
          const u32x4 v = av[q];
          unsigned char* piece = dst + 2 * kPW * q * kRowBytes;
          if (is_r) {
            *reinterpret_cast<u32x4*>(piece) = v;
          } else {
            piece -= 8 * (pcol & 1);
            *reinterpret_cast<u32x2*>(piece) = u32x2{__builtin_amdgcn_perm(v.z, v.x, 0x05040100u), __builtin_amdgcn_perm(v.w, v.y, 0x05040100u)};
            *reinterpret_cast<u32x2*>(piece + 16) = u32x2{__builtin_amdgcn_perm(v.z, v.x, 0x07060302u), __builtin_amdgcn_perm(v.w, v.y, 0x07060302u)};
          }
          continue;
        }
        if constexpr (kCanon) {
          // columns in the order the masks deliver the codes of a canonical word: (0, 4), (1, 5) / 16, (2, 6), (3, 7) / 16; r as it is
          const u32x4 v = av[q];
          u32x4 o = {__builtin_amdgcn_perm(v.z, v.x, 0x05040100u), __builtin_amdgcn_perm(v.z, v.x, 0x07060302u),
                     __builtin_amdgcn_perm(v.w, v.y, 0x05040100u), __builtin_amdgcn_perm(v.w, v.y, 0x07060302u)};
          o.y = __builtin_bit_cast(uint32_t, bitcast_u32<h2>(o.y) * sixteenth);
          o.w = __builtin_bit_cast(uint32_t, bitcast_u32<h2>(o.w) * sixteenth);
          *reinterpret_cast<u32x4*>(dst + 2 * kPW * q * kRowBytes) = is_r ? v : o;
          continue;
        }
        if constexpr (kNarrow) {
          u32x4 o = av[q];
          o.y = __builtin_bit_cast(uint32_t, bitcast_u32<h2>(o.y) * sixteenth);
          o.w = __builtin_bit_cast(uint32_t, bitcast_u32<h2>(o.w) * sixteenth);
          *reinterpret_cast<u32x4*>(dst + 2 * kPW * q * kRowBytes) = o;
          continue;
        }
        // the sixteen lanes pcol / 16 hold the 128 columns of one half of the token row: their sum, in fp32
        const h8 v = __builtin_bit_cast(h8, av[q]);
        float sum = __builtin_amdgcn_fdot2(h2{v[0], v[1]}, ones, 0.f, false);
        sum = __builtin_amdgcn_fdot2(h2{v[2], v[3]}, ones, sum, false);
        sum = __builtin_amdgcn_fdot2(h2{v[4], v[5]}, ones, sum, false);
        sum = __builtin_amdgcn_fdot2(h2{v[6], v[7]}, ones, sum, false);
        sum = row16_total_t(sum);
        u32x4 o = av[q];
        o.y = __builtin_bit_cast(uint32_t, bitcast_u32<h2>(o.y) * sixteenth);
        o.w = __builtin_bit_cast(uint32_t, bitcast_u32<h2>(o.w) * sixteenth);
        *reinterpret_cast<u32x4*>(dst + 2 * kPW * q * kRowBytes) = o;
        if ((pcol & 15) == 0) {
          // sum * 2^-8 as two halves (the zero-point fragment carries -zero * 2^-16)
          const float sc = sum * 0.00390625f;
          const half_t hi = (half_t)sc;
          const half_t lo = (half_t)(sc - (float)hi);
          const uint32_t pr = (uint32_t)__builtin_bit_cast(uint16_t, hi) | ((uint32_t)__builtin_bit_cast(uint16_t, lo) << 16);
          *reinterpret_cast<u32x4*>(sig + 2 * kPW * q * 16) = u32x4{pr, pr, pr, pr};
        }
      }
    };
    // kProj: the first 256 columns of r from r_out once the ready word is up (loads that pass the caches the producers'
    // stores passed); without the word within the bound, the thread computes the eight entries of each of its pieces
    // `polls`: how often the wave looks before it gives up (one look where it may come back later).  True: the loads
    // are out.
    auto ask_r_handed = [&](u32x4 (&av)[kPQ], unsigned polls) __attribute__((always_inline)) -> bool {
      int seen = 0;
      if (lane == 0) {
        for (unsigned spins = 0; !seen && spins < polls && g.spin != 0xFFFFFFFFu; ++spins) {
          seen = (__hip_atomic_load(g.pub, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) & kTagMask) == tag;
          if (!seen && spins + 1 < polls) __builtin_amdgcn_s_sleep(2);
        }
      }
      seen = __builtin_amdgcn_readfirstlane(seen);
      if (seen) {
#pragma unroll
        for (int q = 0; q < kPQ; ++q) {
          const uint32_t row = (uint32_t)min(2 * kPW * q + prow, M - 1);
          uint32_t off = (row * (uint32_t)g.rank + (uint32_t)pcol * 8u) * 2u;
          if (pcol * 8 >= g.rank) off = 0x80000000u;
          av[q] = __builtin_amdgcn_raw_buffer_load_b128(rs_r, (int)off, 0, 16);
        }
      }
      return seen != 0;
    };
    auto load_r_handed = [&](u32x4 (&av)[kPQ]) __attribute__((always_inline)) {
      if (ask_r_handed(av, g.spin == 0xFFFFFFFFu ? 0u : g.spin + 1u)) return;
      for (int q = 0; q < kPQ; ++q) {
        const int row = min(2 * kPW * q + prow, M - 1);
        h8 own;
        for (int e = 0; e < 8; ++e) {
          const int j = pcol * 8 + e;
          float a = 0.f;
          if (j < g.rank) {
            const half_t* Rrow = g.R + (size_t)j * K;
            const half_t* xrow = x + (size_t)row * K;
            for (int kk = 0; kk < K; ++kk) a = __builtin_fmaf((float)Rrow[kk], (float)xrow[kk], a);
          }
          own[e] = (half_t)a;
        }
        av[q] = __builtin_bit_cast(u32x4, own);
      }
    };
    // what follows the last super-block through the stages (step `steps`) is r
    const auto fetch = [&](u32x4 (&av)[kPQ], int j) __attribute__((always_inline)) {
      const bool is_r = j >= steps;
      if constexpr (kProj) {
        if (!is_r) load_a(av, false, min(sb0 + j, SB - 1));
      } else {
        load_a(av, is_r, is_r ? 0 : min(sb0 + j, SB - 1));  // (past r: once more, never stored)
      }
    };
#pragma unroll
    for (int j = 0; j < kXD; ++j) fetch(avs[j], j);
    store_a(avs[0], 0, false);
    fetch(avs[0], kXD);
    __syncthreads();
    bool have_r = false;
    const auto produce = [&](int i, auto set_const) __attribute__((always_inline)) {  // step i: set (i + 1) % kXD
      constexpr int set = decltype(set_const)::value;
      if constexpr (kProj) {
        // r that was not there a step earlier is waited for during the last super-block, for the stage that super-block
        // does not read
        if (set == 0 && i + 1 == steps && wg_corr && gk == 0 && !have_r) load_r_handed(avs[0]);
      }
      store_a(avs[set], (i + 1) & 1, i + 1 >= steps);  // step i + 1's activations (or r after the last step)
      fetch(avs[set], i + 1 + kXD);
      if constexpr (kProj) {
        // one look a step before: as a rule the workgroups in front are long done
        if (i + 2 == steps && wg_corr && gk == 0) have_r = ask_r_handed(avs[0], 1u);
      }
      __syncthreads();
    };
    using std::integral_constant;
    for (int i = 0; i < steps; i += kD) {
      produce(i, integral_constant<int, 1 % kXD>{});
      produce(i + 1, integral_constant<int, 2 % kXD>{});
      produce(i + 2, integral_constant<int, 3 % kXD>{});
      produce(i + 3, integral_constant<int, 4 % kXD>{});
    }
    if (wg_corr) {
      for (int pass = 1; pass * kD < LBall; ++pass) {
        __syncthreads();
        load_a(avs[0], true, pass);
        store_a(avs[0], 0, true);
        __syncthreads();
      }
    }
    if constexpr (kWk > 1) {
      __syncthreads();
      __syncthreads();
    }
    return;
  }

  // ---- consumer waves -----------------------------------------------------------------------------------------------
  // the member: the first one from the leading arguments, the others from the argument buffer
  const unsigned char* wt = wt0;
  int mem_N = N0, blk_base = 0, mi = 0;
  if (tile >= blk_end0) {
#pragma unroll
    for (int i = 1; i < GLOWQ_MAX_MEMBERS; ++i)
      if (i < g.n_members && tile >= g.blk_end[i - 1]) {
        wt = g.mem[i].wt;
        mem_N = g.mem[i].N;
        blk_base = g.blk_end[i - 1];
        mi = i;
      }
  }
  const int rb = (tile - blk_base) * cw + wave;  // this wave's row block of the member
  const bool live = rb < ((mem_N + 31) >> 5);   // a wave past the member's rows still meets the barriers
  // chunk (rb, sb) lies at (sb * RB + rb) * kChunk: the descriptor starts at the wave's chunk of super-block 0 and ends
  // behind its chunk of the group's last super-block
  const int chunk_stride = ((mem_N + 31) >> 5) * tiled::kChunk;
  const int ldw = kCanon ? g.mem[mi].ldw : 0, lds = kCanon ? g.mem[mi].lds : 0, ldz = kCanon ? g.mem[mi].ldz : 0;
  const int crows = live ? min(32, mem_N - rb * 32) : 0;  // kCanon: rows of the block that exist
  const size_t crow0 = (size_t)(live ? rb : 0) * 32;
  // kCanon: the last row may be the end of its buffer whatever the stride (a member cut from a wider one), and requests run past K
  const auto span = [&](size_t ld, int used) { return crows > 0 ? (size_t)(crows - 1) * ld + used : 0; };
  const __amdgpu_buffer_rsrc_t rs_w = kCanon ? rsrc(wt + crow0 * ldw * 4, span(ldw, K / 8) * 4)
                                             : rsrc(wt + (size_t)(live ? rb : 0) * tiled::kChunk, live && sb1 > 0 ? (size_t)(sb1 - 1) * chunk_stride + tiled::kChunk : 0);
  const int b_off = lane * 16;

  struct BSet {
    u32x4 w[4];  // kCanon: [2 half + c], columns 16 c + lane % 16, k words 4 (lane / 16) .. + 3 of the half
    u32x2 side;  // the lane's column: (scale | -zero * 2^-16) of the two halves (kCanon: from `turn`)
  };
  BSet bs[kD];
  const __amdgpu_buffer_rsrc_t rs_s = rsrc(kCanon ? (const void*)(g.mem[mi].scales + crow0 * lds) : (const void*)wt, kCanon ? span(lds, 2 * SB) * 2 : 0);
  const __amdgpu_buffer_rsrc_t rs_z = rsrc(kCanon ? (const void*)(g.mem[mi].qzeros + crow0 * ldz) : (const void*)wt, kCanon ? span(ldz, (2 * SB + 7) / 8) * 4 : 0);
  const int c_row = lane & 15;
  int w_at[2], s_at[2], z_at[2];
#pragma unroll
  for (int c = 0; c < 2; ++c) {
    w_at[c] = (16 * c + c_row) * ldw * 4 + (lane >> 4) * 16;
    s_at[c] = (16 * c + c_row) * lds * 2;
    z_at[c] = (16 * c + c_row) * ldz * 4;
  }
  // kCanon: scales and zero-points of the super-blocks of a rotation in columns c = 0, 1 (a gather over sixteen rows, hence four
  // super-blocks at a time), asked for a rotation ahead.  The four pairs of scales start early enough to lie in the row.
  struct Side {
    u32x4 s[2];
    uint32_t z0[2], z1[2];
  };
  Side ahead = {}, now = {};
  const auto request_side = [&](int sbq) __attribute__((always_inline)) {
    const int at = min(sbq, SB - kD) * 4, word = min(sbq, SB - 1) >> 2, last = (SB - 1) >> 2;
#pragma unroll
    for (int c = 0; c < 2; ++c) {
      ahead.s[c] = __builtin_amdgcn_raw_buffer_load_b128(rs_s, s_at[c], at, 0);
      ahead.z0[c] = __builtin_amdgcn_raw_buffer_load_b32(rs_z, z_at[c], word * 4, 0);
      ahead.z1[c] = __builtin_amdgcn_raw_buffer_load_b32(rs_z, z_at[c], min(word + 1, last) * 4, 0);
    }
  };
  const auto turn = [&](int sbq, bool more) __attribute__((always_inline)) {
    const int skip = min(sbq, SB - 1) - min(sbq, SB - kD);
#pragma unroll
    for (int c = 0; c < 2; ++c) {
      u32x4 v = ahead.s[c];
      if (skip & 1) v = u32x4{v.y, v.z, v.w, v.w};
      if (skip & 2) v = u32x4{v.z, v.w, v.w, v.w};
      now.s[c] = v;
      now.z0[c] = __builtin_amdgcn_alignbit(ahead.z1[c], ahead.z0[c], 8 * (sbq & 3));
    }
    if (more) request_side(sbq + kD);
  };
  auto request = [&](BSet& b, int sbq) __attribute__((always_inline)) {
    if constexpr (kCanon) {
#pragma unroll
      for (int j = 0; j < 4; ++j) b.w[2 * (j & 1) + (j >> 1)] = __builtin_amdgcn_raw_buffer_load_b128(rs_w, w_at[j >> 1], sbq * 128 + (j & 1) * 64, 0);
      return;
    }
#pragma unroll
    for (int j = 0; j < 4; ++j) b.w[j] = __builtin_amdgcn_raw_buffer_load_b128(rs_w, b_off + j * 1024, sbq * chunk_stride, kStreamAux);
    b.side = __builtin_bit_cast(u32x2, __builtin_amdgcn_raw_buffer_load_b64(rs_w, ln * 8, sbq * chunk_stride + tiled::kCodeBytes, kStreamAux));
  };
  // two super-blocks up front, the other two once the first activations are staged: with all four at once the whole
  // chip asks for half a long matrix before any wave can begin
  if constexpr (kCanon) request_side(sb0);
  request(bs[0], sb0);
  request(bs[1], sb0 + 1);

  // a member without a left factor (GlowQ-S) reads zeros for its correction blocks
  const TileMember mem = g.mem[mi];
  const bool has_l = wg_corr && gk == 0 && mem.lt != nullptr && live;
  const __amdgpu_buffer_rsrc_t rs_l = kCanon ? rsrc(has_l ? mem.lt + crow0 * g.rank * 2 : wt, has_l ? (size_t)crows * g.rank * 2 : 0) : rsrc(has_l ? mem.lt + (size_t)rb * LBall * tiled::kLChunk : wt, has_l ? (size_t)LBall * tiled::kLChunk : 0);

  // block q (64 columns of the rank) of the left factor into a set
  const auto request_left = [&](BSet& b, int q) __attribute__((always_inline)) {
#pragma unroll
    for (int t = 0; t < 4; ++t) {
      if constexpr (kCanon) {  // w[2 t + c]: columns 32 t + 8 (lane / 16) .. + 7 of the block
        const int col = q * 64 + (t >> 1) * 32 + (lane >> 4) * 8;
        const int at = ((16 * (t & 1) + c_row) * g.rank + col) * 2;
        b.w[t] = __builtin_amdgcn_raw_buffer_load_b128(rs_l, col < g.rank ? at : (int)0x80000000u, 0, 0);
      } else {
        b.w[t] = __builtin_amdgcn_raw_buffer_load_b128(rs_l, b_off + t * 1024, q * tiled::kLChunk, 0);
      }
    }
  };
  // Up to 16 token rows: tiles of 16 rows by 16 columns, two to a row block (acc[c][i]: row 4 (lane / 16) + i, column 16 c + lane % 16).
  // Rows of sixteen lanes of two neighbouring words change places, and each of the two then holds the codes of sixteen columns over
  // the 32 k values of both.
  f4 nacc[2] = {};
  const auto spread = [](uint32_t a, uint32_t b, uint32_t& lo, uint32_t& hi) __attribute__((always_inline)) {
    const auto v = __builtin_amdgcn_permlane16_swap(a, b, false, false);
    lo = v[0];
    hi = v[1];
  };
  const int nrow_off = (lane & (kRows - 1) & 15) * kRowBytes;
  const int nq = lane >> 4;  // k octet of the lane: word nq % 2 of a pair, lane half nq / 2
  f16v acc;
#pragma unroll
  for (int i = 0; i < 16; ++i) acc[i] = 0.f;
  const uint32_t half0 = lh == 0 ? 0xFFFFFFFFu : 0u;  // the zero-point fragment lives in the first lane half
  const int arow_off = ln * kRowBytes + 128 * lh;  // 32-row tiles
  const int sig_off = kRows * kRowBytes + ln * 16;

  // One super-block: the codes of the register set `b` against the staged rows, half by half.
  // kRefill: each register of the set is refilled with super-block sb_next as soon as its words have been masked.
  auto compute = [&](auto d_const, int sb_next, BSet& b, auto refill_const) __attribute__((always_inline)) {
    constexpr int d = decltype(d_const)::value, stage = d & 1;
    constexpr bool kRefill = decltype(refill_const)::value;
    const unsigned char* st = smem + stage * kStage;
    const u32x2 side = b.side;
    if constexpr (kNarrow) {
      uint32_t sw[2][2];  // [half][c]
      if constexpr (kCanon) {
        sw[0][0] = now.s[0][d], sw[0][1] = now.s[1][d], sw[1][0] = sw[0][0] >> 16, sw[1][1] = sw[0][1] >> 16;
      } else {
        spread(side.x, side.x, sw[0][0], sw[0][1]);
        spread(side.y, side.y, sw[1][0], sw[1][1]);
      }
      // the pairs a mask leaves at code * 2^-20 are staged divided by 16 (but kWhole)
      const h2 one = {(half_t)1.f, (half_t)1.f}, sixteen = {(half_t)16.f, (half_t)16.f};
      const uint32_t o1 = __builtin_bit_cast(uint32_t, one), o16 = __builtin_bit_cast(uint32_t, sixteen);
      const h8 ones = __builtin_bit_cast(h8, u32x4{o1, kWhole ? o1 : o16, o1, kWhole ? o1 : o16});
      // all fragments of the step are asked for at once: one LDS round trip for it instead of eight
      const unsigned char* xs = st + nrow_off + (kCanon ? 64 * nq : 128 * (nq >> 1) + 16 * (nq & 1));
      h8 af[8];
#pragma unroll
      for (int t = 0; t < 8; ++t) af[t] = *reinterpret_cast<const h8*>(xs + 256 * (t >> 2) + (kCanon ? 16 : 32) * (t & 3));
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int gh = 0; gh < 2; ++gh) {
        f4 pg[2] = {}, sx = {};
        if constexpr (kWhole) {
          // codes * 2^-24 and codes * 2^-20 into sums of their own, so that the activations stay whole
#pragma unroll
          for (int c = 0; c < 2; ++c) {
            f4 pl = {}, ph = {};
#pragma unroll
            for (int j = 0; j < 4; j += 2) {
              const uint32_t wa = b.w[2 * gh + c][j], wb = b.w[2 * gh + c][j + 1], ha = wa >> 8, hb = wb >> 8;
              const h8 lo = __builtin_bit_cast(h8, u32x4{wa & 0x000F000Fu, ha & 0x000F000Fu, wb & 0x000F000Fu, hb & 0x000F000Fu});
              const h8 hi = __builtin_bit_cast(h8, u32x4{wa & 0x00F000F0u, ha & 0x00F000F0u, wb & 0x00F000F0u, hb & 0x00F000F0u});
              pl = __builtin_amdgcn_mfma_f32_16x16x32_f16(af[4 * gh + j], lo, pl, 0, 0, 0);
              ph = __builtin_amdgcn_mfma_f32_16x16x32_f16(af[4 * gh + j + 1], hi, ph, 0, 0, 0);
              if (c == 0) {
                sx = __builtin_amdgcn_mfma_f32_16x16x32_f16(af[4 * gh + j], ones, sx, 0, 0, 0);
                sx = __builtin_amdgcn_mfma_f32_16x16x32_f16(af[4 * gh + j + 1], ones, sx, 0, 0, 0);
              }
            }
            __builtin_amdgcn_sched_barrier(0);
            const float sf = (float)__builtin_bit_cast(half_t, (uint16_t)(sw[gh][c] & 0xFFFFu)) * 0x1p24f;
            const float nz = (float)((now.z0[c] >> (8 * d + 4 * gh)) & 15u) * -0x1p-24f;
#pragma unroll
            for (int i = 0; i < 4; ++i) nacc[c][i] = __builtin_fmaf(sf, __builtin_fmaf(nz, sx[i], __builtin_fmaf(0.0625f, ph[i], pl[i])), nacc[c][i]);
          }
          if constexpr (kRefill)
            if (gh == 1) request(b, sb_next);  // (both halves of a cache line together)
          continue;
        }
        if constexpr (kCanon) {
#pragma unroll
          for (int j = 0; j < 4; ++j) {
#pragma unroll
            for (int c = 0; c < 2; ++c) {
              const uint32_t wd = b.w[2 * gh + c][j], hi = wd >> 8;
              const h8 bf = __builtin_bit_cast(h8, u32x4{wd & 0x000F000Fu, wd & 0x00F000F0u, hi & 0x000F000Fu, hi & 0x00F000F0u});
              pg[c] = __builtin_amdgcn_mfma_f32_16x16x32_f16(af[4 * gh + j], bf, pg[c], 0, 0, 0);
            }
            sx = __builtin_amdgcn_mfma_f32_16x16x32_f16(af[4 * gh + j], ones, sx, 0, 0, 0);
          }
          if constexpr (kRefill)
            if (gh == 1) request(b, sb_next);  // (both halves of a cache line together)
        }
#pragma unroll
        for (int p = 0; p < (kCanon ? 0 : 2); ++p) {
          const u32x4 raw = b.w[2 * gh + p];
#pragma unroll
          for (int i = 0; i < 4; i += 2) {
            const h8 a = af[4 * gh + 2 * p + (i >> 1)];
            uint32_t w[2];
            spread(raw[i], raw[i + 1], w[0], w[1]);
#pragma unroll
            for (int c = 0; c < 2; ++c) {
              const uint32_t hi = w[c] >> 8;
              const h8 bf = __builtin_bit_cast(h8, u32x4{w[c] & 0x000F000Fu, w[c] & 0x00F000F0u, hi & 0x000F000Fu, hi & 0x00F000F0u});
              pg[c] = __builtin_amdgcn_mfma_f32_16x16x32_f16(a, bf, pg[c], 0, 0, 0);
            }
            sx = __builtin_amdgcn_mfma_f32_16x16x32_f16(a, ones, sx, 0, 0, 0);
          }
          if constexpr (kRefill) b.w[2 * gh + p] = __builtin_amdgcn_raw_buffer_load_b128(rs_w, b_off + (2 * gh + p) * 1024, sb_next * chunk_stride, kStreamAux);
        }
#pragma unroll
        for (int c = 0; c < 2; ++c) {
          const float sf = (float)__builtin_bit_cast(half_t, (uint16_t)(sw[gh][c] & 0xFFFFu)) * 0x1p24f;
          const float nz = kCanon ? (float)((now.z0[c] >> (8 * d + 4 * gh)) & 15u) * -0x1p-24f
                                  : (float)__builtin_bit_cast(half_t, (uint16_t)(sw[gh][c] >> 16)) * 0x1p-8f;  // -zero * 2^-24
#pragma unroll
          for (int i = 0; i < 4; ++i) nacc[c][i] = __builtin_fmaf(sf, __builtin_fmaf(nz, sx[i], pg[c][i]), nacc[c][i]);
        }
      }
      if constexpr (kRefill && !kCanon)
        b.side = __builtin_bit_cast(u32x2, __builtin_amdgcn_raw_buffer_load_b64(rs_w, ln * 8, sb_next * chunk_stride + tiled::kCodeBytes, kStreamAux));
      return;
    }
#pragma unroll
    for (int gh = 0; gh < 2; ++gh) {
      f16v pg;
#pragma unroll
      for (int p = 0; p < 2; ++p) {
        const u32x4 raw = b.w[2 * gh + p];
        if constexpr (kRefill) b.w[2 * gh + p] = __builtin_amdgcn_raw_buffer_load_b128(rs_w, b_off + (2 * gh + p) * 1024, sb_next * chunk_stride, kStreamAux);
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const uint32_t wd = raw[i], hi = wd >> 8;
          const h8 bf = __builtin_bit_cast(h8, u32x4{wd & 0x000F000Fu, wd & 0x00F000F0u, hi & 0x000F000Fu, hi & 0x00F000F0u});
          const h8 af = *reinterpret_cast<const h8*>(st + arow_off + 256 * gh + 64 * p + 16 * i);
          if (p == 0 && i == 0) {
            const f16v zero = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
            pg = __builtin_amdgcn_mfma_f32_32x32x16_f16(af, bf, zero, 0, 0, 0);
          } else {
            pg = __builtin_amdgcn_mfma_f32_32x32x16_f16(af, bf, pg, 0, 0, 0);
          }
        }
      }
      // the zero-point: k values 0 and 1 of the first lane half carry -zero * 2^-16 against the row's sum * 2^-8 (hi, lo)
      const uint32_t sw = side[gh];
      const h8 bz = __builtin_bit_cast(h8, u32x4{__builtin_amdgcn_perm(sw, sw, 0x03020302u) & half0, 0u, 0u, 0u});
      const float sf = (float)__builtin_bit_cast(half_t, (uint16_t)(sw & 0xFFFFu)) * 0x1p24f;
      const h8 az = *reinterpret_cast<const h8*>(st + sig_off + gh * kSigBytes);
      pg = __builtin_amdgcn_mfma_f32_32x32x16_f16(az, bz, pg, 0, 0, 0);
#pragma unroll
      for (int i = 0; i < 16; ++i) acc[i] = __builtin_fmaf(sf, pg[i], acc[i]);
    }
    if constexpr (kRefill)
      b.side = __builtin_bit_cast(u32x2, __builtin_amdgcn_raw_buffer_load_b64(rs_w, ln * 8, sb_next * chunk_stride + tiled::kCodeBytes, kStreamAux));
  };

  __syncthreads();
  request(bs[2], sb0 + 2);
  request(bs[3], sb0 + 3);

  // step d of a rotation at super-block sb: compute on stage d % 2; barrier.  Last rotation: a step past the group's
  // part is skipped, and the sets are refilled with the blocks of the tiled left factor (set q: block q; past the rank
  // they lie past the end of the descriptor).
  auto step = [&](int sb, auto d_const, auto last_const) __attribute__((always_inline)) {
    constexpr int d = decltype(d_const)::value;
    constexpr bool kLast = decltype(last_const)::value;
    if constexpr (kLast) {
      if (sb < sb1) compute(d_const, 0, bs[d], std::false_type{});
      request_left(bs[d], d);
    } else {
      compute(d_const, sb + kD, bs[d], std::true_type{});
    }
    __syncthreads();
  };
  using std::integral_constant;
  int sb = sb0;
  for (int rd = 0; rd < rounds - 1; ++rd, sb += kD) {
    if constexpr (kCanon) turn(sb, true);
    step(sb, integral_constant<int, 0>{}, std::false_type{});
    step(sb + 1, integral_constant<int, 1>{}, std::false_type{});
    step(sb + 2, integral_constant<int, 2>{}, std::false_type{});
    step(sb + 3, integral_constant<int, 3>{}, std::false_type{});
  }
  if constexpr (kCanon) turn(sb, false);
  step(sb, integral_constant<int, 0>{}, std::true_type{});
  step(sb + 1, integral_constant<int, 1>{}, std::true_type{});
  step(sb + 2, integral_constant<int, 2>{}, std::true_type{});
  step(sb + 3, integral_constant<int, 3>{}, std::true_type{});

  // kWhole, a sum that is not finite: an infinite activation makes infinities of both signs of sum code * x and -zero * sum x, and no number of
  // their sum.  The wave walks its part of K again with code - zero as the operand, whose products have the signs they should have
  // (words and activations straight from memory: such a call has worse things than this walk to wait for).
  if constexpr (kWhole) {
    float size = 0.f;
#pragma unroll
    for (int i = 0; i < 8; ++i) size += __builtin_fabsf(nacc[i >> 2][i & 3]);
    if (live && __builtin_amdgcn_ballot_w64(!(size < __builtin_inff())) != 0) {
      const half_t* xr = x + (size_t)min(lane & 15, M - 1) * K + 32 * nq;
      nacc[0] = nacc[1] = f4{};
#pragma unroll 1
      for (int again = sb0; again < sb1; ++again) {
        BSet b;
        request(b, again);
#pragma unroll 1
        for (int gh = 0; gh < 2; ++gh) {
          const int grp = 2 * again + gh;
#pragma unroll
          for (int c = 0; c < 2; ++c) {
            const size_t row = crow0 + min(16 * c + c_row, crows - 1);
            const uint32_t z = nibble((uint32_t)g.mem[mi].qzeros[row * ldz + (grp >> 3)], grp & 7);
            const h2 zb_lo = bitcast_u32<h2>(z * 0x00010001u + 0xE400E400u), zb_hi = bitcast_u32<h2>(z * 0x00100010u + 0xD400D400u);
            f4 sum = {};
#pragma unroll
            for (int j = 0; j < 4; ++j) {
              const u32x4 v = *reinterpret_cast<const u32x4*>(xr + again * 256 + gh * 128 + 8 * j);
              const u32x4 o = {__builtin_amdgcn_perm(v.z, v.x, 0x05040100u), __builtin_amdgcn_perm(v.z, v.x, 0x07060302u),
                               __builtin_amdgcn_perm(v.w, v.y, 0x05040100u), __builtin_amdgcn_perm(v.w, v.y, 0x07060302u)};
              const uint32_t wd = gh == 0 ? b.w[c][j] : b.w[2 + c][j];
              sum = __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(h8, o), dequant_word<false>(wd, zb_lo, zb_hi, h2{}), sum, 0, 0, 0);
            }
            const float sc = (float)g.mem[mi].scales[row * lds + grp];
#pragma unroll
            for (int i = 0; i < 4; ++i) nacc[c][i] = __builtin_fmaf(sc, sum[i], nacc[c][i]);
          }
        }
      }
    }
  }

  // ---- the correction: set q holds block q of the tiled left factor (B fragments of its four k-steps as they are),
  // stage 0 the first 256 columns of r.  Ranks above 256 take further passes, each with its loads in the open.  K groups
  // other than the first hold zeros in their sets.
  if (wg_corr) {
    f16v acc2;
    f4 nacc2[2] = {};
#pragma unroll
    for (int i = 0; i < 16; ++i) acc2[i] = 0.f;
    for (int pass = 0; pass * kD < LBall; ++pass) {
      if (pass > 0) {
        __syncthreads();  // the fragment reads of the pass before are done
#pragma unroll
        for (int q = 0; q < kD; ++q) request_left(bs[q], pass * kD + q);
        __syncthreads();
      }
      if constexpr (kNarrow) {
        const unsigned char* ar = smem + nrow_off + (kCanon ? 16 * nq : 64 * (nq >> 1) + 16 * (nq & 1));
#pragma unroll
        for (int q = 0; q < kD; ++q)
#pragma unroll
          for (int t = 0; t < 4; t += 2) {
            const h8 af = *reinterpret_cast<const h8*>(ar + 128 * q + (kCanon ? 32 : 16) * t);
            u32x4 bw[2] = {bs[q].w[t], bs[q].w[t + 1]};
#pragma unroll
            for (int e = 0; e < (kCanon ? 0 : 4); ++e) {
              uint32_t lo, hi;
              spread(bs[q].w[t][e], bs[q].w[t + 1][e], lo, hi);
              bw[0][e] = lo;
              bw[1][e] = hi;
            }
#pragma unroll
            for (int c = 0; c < 2; ++c) nacc2[c] = __builtin_amdgcn_mfma_f32_16x16x32_f16(af, __builtin_bit_cast(h8, bw[c]), nacc2[c], 0, 0, 0);
          }
        continue;
      }
      const unsigned char* ar = smem + ln * kRowBytes + 64 * lh;
#pragma unroll
      for (int q = 0; q < kD; ++q)
#pragma unroll
        for (int t = 0; t < 4; ++t) {
          const h8 af = *reinterpret_cast<const h8*>(ar + 128 * q + 16 * t);
          acc2 = __builtin_amdgcn_mfma_f32_32x32x16_f16(af, __builtin_bit_cast(h8, bs[q].w[t]), acc2, 0, 0, 0);
        }
    }
#pragma unroll
    for (int i = 0; i < 16; ++i) acc[i] = __builtin_fmaf(g.alpha, acc2[i], acc[i]);
#pragma unroll
    for (int c = 0; c < 2; ++c) nacc[c] += g.alpha * nacc2[c];
  }
  constexpr int kAccs = kNarrow ? 8 : 16;
  float out[kAccs];
#pragma unroll
  for (int i = 0; i < kAccs; ++i) out[i] = kNarrow ? nacc[(i >> 2) & 1][i & 3] : acc[i];

  // ---- the K groups' accumulators meet in LDS: groups 1.. leave theirs, group 0 adds them in order ---------------
  if constexpr (kWk > 1) {
    __syncthreads();  // every group is done with its stages
    float* red = reinterpret_cast<float*>(smem_all);
    if (gk > 0) {
#pragma unroll
      for (int i = 0; i < kAccs; ++i) red[(((gk - 1) * cw + wave) * kAccs + i) * 64 + lane] = out[i];
    }
    __syncthreads();
    if (gk > 0) return;
#pragma unroll
    for (int o = 1; o < kWk; ++o)
#pragma unroll
      for (int i = 0; i < kAccs; ++i) out[i] += red[(((o - 1) * cw + wave) * kAccs + i) * 64 + lane];
  }

  // ---- epilogue: entry i of a lane is token row 8 (i / 4) + 4 lh + i % 4, column ln of the wave's row block; of the narrow tiles row
  // 4 nq + i % 4, column 16 (i / 4) + lane % 16
  if (!live) return;
  const auto row_of = [&](int i) { return kNarrow ? 4 * nq + (i & 3) : 8 * (i >> 2) + 4 * lh + (i & 3); };
  const auto col_of = [&](int i) { return rb * 32 + (kNarrow ? 16 * (i >> 2) + (lane & 15) : ln); };
  if (slices > 1) {
    float* prow = g.partials + ((size_t)blockIdx.y * M) * g.ldp + mem.col0;
#pragma unroll
    for (int i = 0; i < kAccs; ++i)
      if (row_of(i) < M) prow[(size_t)row_of(i) * g.ldp + col_of(i)] = out[i];
    return;
  }
  constexpr int kPer = kNarrow ? 4 : 16;  // entries of a column
#pragma unroll
  for (int i0 = 0; i0 < kAccs; i0 += kPer) {
    const int n = col_of(i0);
    if (n >= mem.N) continue;
    const float bias = mem.bias ? (float)mem.bias[n] : 0.f;
#pragma unroll
    for (int i = i0; i < i0 + kPer; ++i)
      if (row_of(i) < M) mem.y[(size_t)row_of(i) * mem.ldy + n] = (half_t)(out[i] + bias);
  }
}

// y = fp16(sum over the K slices, in slice order, + bias).  One thread per (token row, four columns of the padded row).
__global__ __launch_bounds__(256) void skinny_tiled_reduce_kernel(const TileArgs g) {
  const int c4 = (int)(blockIdx.x * blockDim.x + threadIdx.x) * 4;
  const int m = (int)blockIdx.y;
  if (c4 >= g.ldp) return;
  f4 sum = {0.f, 0.f, 0.f, 0.f};
  for (int s = 0; s < g.slices; ++s) sum += *reinterpret_cast<const f4*>(g.partials + ((size_t)s * g.M + m) * g.ldp + c4);
  TileMember mem = g.mem[0];
  for (int i = 1; i < g.n_members; ++i)
    if (c4 >= g.mem[i].col0) mem = g.mem[i];
  const int n0 = c4 - mem.col0;
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    const int n = n0 + e;
    if (n < mem.N) mem.y[(size_t)m * mem.ldy + n] = (half_t)(sum[e] + (mem.bias ? (float)mem.bias[n] : 0.f));
  }
}

// ---- packing (conversion time) ------------------------------------------------------------------------------
// One thread per (row block, super-block, lane): its four 16-byte pieces; lanes 0..31 also write their column's side pair.
__global__ __launch_bounds__(256) void pack_tiled_weights_kernel(const int32_t* __restrict__ qweight, const half_t* __restrict__ scales,
                                                                 const int32_t* __restrict__ qzeros, unsigned char* __restrict__ out,
                                                                 int N, int K, int group_size, int ldw, int lds, int ldz) {
  const int SB = K >> 8;
  const long total = (long)((N + 31) >> 5) * SB * 64;
  for (long idx = (long)blockIdx.x * blockDim.x + threadIdx.x; idx < total; idx += (long)gridDim.x * blockDim.x) {
    const int l = (int)(idx & 63);
    const long chunk = idx >> 6;  // = sb * RB + rb
    const int RB = (N + 31) >> 5;
    const int rb = (int)(chunk % RB), sb = (int)(chunk / RB);
    const int row = rb * 32 + (l & 31), h = l >> 5;
    unsigned char* dst = out + (size_t)chunk * tiled::kChunk;
    const bool in = row < N;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      u32x4 v = {0u, 0u, 0u, 0u};
      if (in) {
        const int32_t* src = qweight + (size_t)row * ldw + sb * 32 + 16 * (j >> 1) + 8 * h + 4 * (j & 1);
        v = u32x4{mask_order_word((uint32_t)src[0]), mask_order_word((uint32_t)src[1]), mask_order_word((uint32_t)src[2]),
                  mask_order_word((uint32_t)src[3])};
      }
      *reinterpret_cast<u32x4*>(dst + 1024 * j + 16 * l) = v;
    }
    if (h == 0) {
      u32x2 side = {0u, 0u};
      if (in) {
#pragma unroll
        for (int gh = 0; gh < 2; ++gh) {
          const int grp = (sb * 256 + gh * 128) / group_size;
          const uint32_t z = nibble((uint32_t)qzeros[(size_t)row * ldz + (grp >> 3)], grp & 7);
          const half_t nz = (half_t)(-(float)z * 0x1p-16f);  // a multiple of 2^-24: exact
          side[gh] = (uint32_t)__builtin_bit_cast(uint16_t, scales[(size_t)row * lds + grp]) | ((uint32_t)__builtin_bit_cast(uint16_t, nz) << 16);
        }
      }
      *reinterpret_cast<u32x2*>(dst + tiled::kCodeBytes + 8 * (l & 31)) = side;
    }
  }
}

// One thread per (row block, rank block, lane, k-step): 8 consecutive halves of a row of L, those at positions 2, 3, 6, 7
// times 16.
__global__ __launch_bounds__(256) void pack_tiled_left_kernel(const half_t* __restrict__ L, unsigned char* __restrict__ out, int N,
                                                              int rank) {
  const int LB = (rank + 63) >> 6;
  const long total = (long)((N + 31) >> 5) * LB * 256;
  for (long idx = (long)blockIdx.x * blockDim.x + threadIdx.x; idx < total; idx += (long)gridDim.x * blockDim.x) {
    const int l = (int)(idx & 63), t = (int)((idx >> 6) & 3);
    const long chunk = idx >> 8;
    const int jb = (int)(chunk % LB), rb = (int)(chunk / LB);
    const int row = rb * 32 + (l & 31), k0 = jb * 64 + (l >> 5) * 32 + t * 8;
    h8 v;
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      const half_t val = (row < N && k0 + e < rank) ? L[(size_t)row * rank + k0 + e] : (half_t)0.f;
      v[e] = (e & 2) ? val * (half_t)16.f : val;  // the pairs the activations carry divided by 16
    }
    *reinterpret_cast<h8*>(out + (size_t)chunk * tiled::kLChunk + 1024 * t + 16 * l) = v;
  }
}

// ---- host side ----------------------------------------------------------------------------------------------
hipError_t launch_pack_tiled(const int32_t* qweight, const half_t* scales, const int32_t* qzeros, void* out, int N, int K,
                             int group_size, int ldw, int lds, int ldz, int num_cus, hipStream_t stream) {
  const long total = (long)((N + 31) >> 5) * (K >> 8) * 64;
  long blocks = (total + 255) / 256;
  if (blocks > (long)num_cus * 32) blocks = (long)num_cus * 32;
  if (blocks < 1) blocks = 1;
  hipLaunchKernelGGL(pack_tiled_weights_kernel, dim3((unsigned)blocks), dim3(256), 0, stream, qweight, scales, qzeros,
                     static_cast<unsigned char*>(out), N, K, group_size, ldw, lds, ldz);
  return hipGetLastError();
}

hipError_t launch_pack_tiled_left(const half_t* L, void* out, int N, int rank, int num_cus, hipStream_t stream) {
  const long total = (long)((N + 31) >> 5) * ((rank + 63) >> 6) * 256;
  long blocks = (total + 255) / 256;
  if (blocks > (long)num_cus * 32) blocks = (long)num_cus * 32;
  if (blocks < 1) blocks = 1;
  hipLaunchKernelGGL(pack_tiled_left_kernel, dim3((unsigned)blocks), dim3(256), 0, stream, L, static_cast<unsigned char*>(out), N, rank);
  return hipGetLastError();
}

// Every member brings its tiled weights (and its tiled left factor where it has one), K and the groups fit the layout,
// the rank is a multiple of 8 and at most 64 token rows.
bool skinny_tiled_supported(const GroupDev& g) {
  if (g.M < 1 || g.M > 64 || !tiled::applies(g.K, g.group_size)) return false;
  const half_t* r = g.r != nullptr ? g.r : (g.R != nullptr ? g.r_out : nullptr);
  if (r != nullptr && ((g.rank & 7) != 0 || g.rank < 8 || (reinterpret_cast<uintptr_t>(r) & 15u) != 0)) return false;
  if ((reinterpret_cast<uintptr_t>(g.x) & 15u) != 0) return false;
  if ((size_t)g.M * g.K * 2 >= (1ull << 32)) return false;
  for (int i = 0; i < g.n_members; ++i) {
    const MemberDev& m = g.mem[i];
    if (m.tiled == nullptr || (reinterpret_cast<uintptr_t>(m.tiled) & 15u) != 0) return false;
    if (tiled::weight_bytes(m.N, g.K) >= (1ull << 32)) return false;  // 32-bit offsets into the stream
    if (m.L != nullptr && r != nullptr && (m.tiled_L == nullptr || m.tiled_rank != g.rank || (reinterpret_cast<uintptr_t>(m.tiled_L) & 15u) != 0))
      return false;
  }
  return true;
}

// The narrow tiles on the canonical buffers: 5 to 16 token rows, K in four and more whole super-blocks, groups of 128 columns, and what the loads need of
// pointers and strides (codes and left factor 16 bytes, scales and zero-points four).
bool skinny_words_supported(const GroupDev& g) {
  if (g.M < 5 || g.M > 16 || (g.K & 255) != 0 || g.K < 1024 || g.group_size != 128) return false;
  const half_t* r = g.r != nullptr ? g.r : (g.R != nullptr ? g.r_out : nullptr);
  if (r != nullptr && ((g.rank & 7) != 0 || g.rank < 8 || (reinterpret_cast<uintptr_t>(r) & 15u) != 0)) return false;
  if ((reinterpret_cast<uintptr_t>(g.x) & 15u) != 0 || (size_t)g.M * g.K * 2 >= (1ull << 31)) return false;
  for (int i = 0; i < g.n_members; ++i) {
    const MemberDev& m = g.mem[i];
    if ((reinterpret_cast<uintptr_t>(m.qweight) & 15u) != 0 || (m.ldw & 3) != 0 || m.ldw < g.K / 8 || (size_t)m.ldw * 128 >= (1ull << 31)) return false;
    if ((reinterpret_cast<uintptr_t>(m.scales) & 3u) != 0 || (m.lds & 1) != 0 || (reinterpret_cast<uintptr_t>(m.qzeros) & 3u) != 0) return false;
    if ((size_t)m.lds * 64 >= (1ull << 31) || (size_t)m.ldz * 128 >= (1ull << 31)) return false;
    if (m.L != nullptr && r != nullptr && (reinterpret_cast<uintptr_t>(m.L) & 15u) != 0) return false;
  }
  return true;
}

// How the launch cuts K and staffs a K group: `wk` K groups inside a workgroup (their sums meet in LDS), `slices`
// workgroups per tile (their sums meet in the workspace), `pw` producer waves per K group, `cw` consumer waves (a tile is 32 cw columns).
// Workgroups stay at 768 threads and below (a 1024-thread workgroup gets 128 registers per lane and the chip runs such workgroups in
// two rounds).
struct TiledPlan {
  int wk, slices, pw, cw;
  bool front;  // the launch computes r itself
};
static int tiled_tiles(const GroupDev& g, int cw) {
  int t = 0;
  for (int i = 0; i < g.n_members; ++i) t += ((g.mem[i].N + 31) / 32 + cw - 1) / cw;
  return t;
}
static int proj_blocks(int M, int rank) { return ((rank + 3) / 4) * ((M + 3) / 4); }  // of four token rows by four rows of R
// Up to 16 rows: the cheapest cut by what the launches were seen to take (us): 4.2 and the longer, a fifth of the shorter, of the steps of a
// K group (whole rotations, 0.34 each and 0.04 per consumer wave; of two K groups 0.49 or 0.72; a compute unit draws a super-block of a row
// block in 0.11) and the bytes of the group at 4.9 TB/s; 3.3 for slices and the launch that adds them.  r ahead of the launch is 2.3 and its
// products, inside it 1.0 where the workgroups in front, on the compute units the tiles leave free, are done in time: 4.0 and 0.53 per
// thousand columns of K for each of the blocks a team of four waves computes (q|k|v of a 14B layer at twelve rows, six blocks each on 32
// compute units, 22.5 against 14.3 on wider tiles).  Tiles on a quarter of the chip and less are cut in K rather than given a front.
// Predicted / measured at 16 rows without a correction: 5120 x 5120 10.6 / 9.6, 17408 x 5120 15.5 / 15.4, 2 x 17408 x 5120 24.7 / 23.2,
// 5120 x 17408 18.2 / 16.7, 4096 x 14336 14.6 / 14.0.
// (One K group at a wave per SIMD leaves vector and matrix instructions to alternate; two of them pay where the tiles are a row block or
// two wide: 4096 x 4096 7.9 against 10.2, but 2 x 14336 x 4096 at four 16.9 against 15.5.)
static TiledPlan narrow_plan(const GroupDev& g, int num_cus, size_t ws_bytes, bool fused, bool canon) {
  const int SB = g.K >> 8;
  const bool corrected = g.r != nullptr || g.R != nullptr;
  double rows = 0;
  for (int i = 0; i < g.n_members; ++i) rows += (g.mem[i].N + 31) / 32 * 32;
  const double stream_us = rows * (g.K * 0.53125 + (corrected ? 2. * g.rank : 0.)) / 4.9e6;
  TiledPlan best{1, 1, 1, 1, false};
  double best_us = 1e30;
  bool one_round = false;
  for (int cw = 1; cw <= 8; ++cw) {
    const int tiles = tiled_tiles(g, cw);
    if (cw < 8 && tiles > num_cus) continue;
    if (one_round && SB < 8) break;  // (a launch this short: nothing to gain from wider tiles)
    one_round = true;
    const double rounds = (double)((tiles + num_cus - 1) / num_cus);
    const size_t per_slice = (size_t)g.M * tiles * cw * 32 * sizeof(float);
    for (int wk = 1; wk <= (cw <= 2 && SB >= 4 ? 2 : 1); ++wk) {
      long top = cw <= 4 ? std::min<long>(num_cus / std::max(tiles, 1), SB / (4 * wk)) : 1;
      top = std::min<long>(top, (long)(ws_bytes / per_slice));
      for (int s = 1, last = 0; s == 1 || s <= top; ++s) {
        const int per = (SB + s - 1) / s, slices = (SB + per - 1) / per;
        if (slices == last) continue;
        last = slices;
        const int steps = ((per + wk - 1) / wk + kD - 1) / kD * kD;
        const double step_us = rounds * steps * std::max(wk == 1 ? 0.34 + 0.04 * cw : (cw == 1 ? 0.49 : 0.72), cw * wk * 0.11);
        double us = 4.2 + std::max(step_us, stream_us) + 0.2 * std::min(step_us, stream_us) + (slices > 1 ? 3.3 : 0.);
        const int pw = (fused || canon) && g.M > 8 ? 2 : 1;  // (one wave with all pieces of 16 rows and more to do runs out of registers)
        bool front = false;
        if (g.R != nullptr) {
          const int threads = (cw + pw) * 64 * wk, free_cus = (num_cus - tiles) & ~3;  // (the front is padded to a multiple of four: handover.hpp)
          const int blocks = proj_blocks(g.M, g.rank), teams = blocks > free_cus && threads >= 512 ? 2 : 1;
          front = fused && slices == 1 && threads >= 256 && tiles * 4 > num_cus && free_cus > 0 && (free_cus * kTiledProjBlocks >= blocks || g.pub_mute);
          if (front) us = 1.0 + std::max(us, 4.0 + 0.53e-3 * g.K * ((blocks + free_cus * teams - 1) / (free_cus * teams)));
          else us += 2.3 + 0.065e-6 * g.M * (double)g.K * g.rank;
        }
        if (us < best_us) best_us = us, best = TiledPlan{wk, slices, pw, cw, front};
      }
    }
  }
  return best;
}
static TiledPlan tiled_plan(const GroupDev& g, int num_cus, size_t ws_bytes, bool fused, bool canon) {
  if (g.M <= 16) return narrow_plan(g, num_cus, ws_bytes, fused, canon);
  const int SB = g.K >> 8;
  // one K group of four consumer and four producer waves (two of two producers, 8B shapes at 32 rows, us: gate|up 26.4 against 26.3,
  // down_proj 27.1 against 25.5)
  TiledPlan p{1, 1, 4, 4, false};
  // a few tiles more than compute units would run as two rounds, the second nearly empty: wider tiles where they bring the count
  // down to one round
  if (tiled_tiles(g, 4) > num_cus) {
    for (int cw = 5; cw <= 8; ++cw)
      if (tiled_tiles(g, cw) <= num_cus) {
        p.cw = cw;
        break;
      }
  }
  // slices where the tiles alone leave most of the chip empty
  const int tiles = tiled_tiles(g, p.cw);
  const size_t per_slice = (size_t)g.M * tiles * p.cw * 32 * sizeof(float);
  long s = tiles * 2 <= num_cus ? num_cus / std::max(tiles, 1) : 1;
  s = std::max(1L, std::min(s, std::min((long)SB / 4, per_slice > 0 ? (long)(ws_bytes / per_slice) : 1L)));
  const int per = (SB + (int)s - 1) / (int)s;  // slices of equal depth: no more of them than leave none empty
  p.slices = (SB + per - 1) / per;
  return p;
}

// The most workspace tiled_plan and narrow_plan ask for: they cut K only where tiles x slices stay within num_cus workgroups, and into slices only
// tiles of up to four consumer waves (128 columns): one 128-column fp32 tile per token row for each of them.
size_t tiled_split_workspace_bytes(int M, int num_cus) { return M > 4 ? (size_t)num_cus * (size_t)M * 128 * sizeof(float) : 0; }

template <int kRows, int kWk, int kPW, bool kProj = false, bool kCanon = false>
static hipError_t launch_tiled_t(TileArgs& a, const half_t* x, int num_cus, hipStream_t stream) {
  auto kern = skinny_tiled_kernel<kRows, kWk, kPW, kProj, kCanon>;
  size_t lds = (size_t)kWk * 2 * (kRows * kRowBytes + (kRows <= 16 ? 0 : 2 * kRows * 16));
  const size_t red = (size_t)(kWk - 1) * a.cw * (kRows <= 16 ? 8 : 16) * 64 * sizeof(float);
  if (lds < red) lds = red;
  static LdsLimit lds_limit;
  if (hipError_t e = ensure_dynamic_lds(reinterpret_cast<const void*>(kern), lds, lds_limit); e != hipSuccess) return e;
  if (a.cw < 1 || a.cw > tiled_max_cw(kWk, kPW)) return hipErrorInvalidValue;
  const int threads = (a.cw + kPW) * 64 * kWk;
  int grid_x = a.tiles;
  if constexpr (kProj) {
    // The workgroups in front take places the launch leaves free on the chip, so that every workgroup starts at once and
    // none with a column tile waits behind a producer.  The readers ask for r during their last super-block, so a
    // producer has most of the launch for its blocks: up to kTiledProjBlocks of them.
    static std::atomic<long> asked_for{-1};
    static std::atomic<int> resident{0};
    const long shape = (long)lds * 4096 + threads;
    int per_cu = 0;
    if (asked_for.load(std::memory_order_acquire) == shape) {
      per_cu = resident.load(std::memory_order_relaxed);
    } else {
      if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, reinterpret_cast<const void*>(kern), threads, lds) != hipSuccess) per_cu = 0;
      resident.store(per_cu, std::memory_order_relaxed);
      asked_for.store(shape, std::memory_order_release);
    }
    // (one workgroup per compute unit, whatever the occupancy allows: two that share a compute unit share its LDS
    // bandwidth and matrix cores, and the launch gets longer -- gate|up of a 14B layer at eight rows with 131 producers
    // beside 218 tiles 42 us against 30.5)
    const long capacity = per_cu >= 1 ? num_cus : 0;
    long want = (capacity - (long)a.tiles) & ~3L;  // (the front is padded to a multiple of four: handover.hpp)
    const int nblocks = proj_blocks(a.M, a.rank);
    if (want > nblocks) want = nblocks;
    if (want > kTiledMaxProducers) want = kTiledMaxProducers;
    if (threads < 256 || want < 1 || ((long)kTiledProjBlocks * want < nblocks && a.spin != 0xFFFFFFFFu)) return hipErrorNotReady;
    a.producers = (int)want;
    a.teams = (nblocks > want && threads >= 512) ? 2 : 1;  // two blocks at a time where the workgroup has the waves
    grid_x = front_grid(a.tiles, a.producers);
  }
  hipLaunchKernelGGL(kern, dim3(grid_x, a.slices), dim3(threads), lds, stream, x, a.M, a.K, a.slices, a.mem[0].wt,
                     a.blk_end[0], a.mem[0].N, a.cw, a);
  note_launch(grid_x, a.slices, threads, kProj ? "%s<%d,%d,%d,1> with %d consumer waves" : "%s<%d,%d,%d> with %d consumer waves",
              kCanon ? "skinny_words_kernel" : "skinny_tiled_kernel", kRows, kWk, kPW, a.cw);
  if (hipError_t e = hipGetLastError(); e != hipSuccess || a.slices == 1) return e;
  hipLaunchKernelGGL(skinny_tiled_reduce_kernel, dim3((a.ldp / 4 + 255) / 256, a.M), dim3(256), 0, stream, a);
  return hipGetLastError();
}

template <bool kCanon>
static hipError_t launch_narrow(TileArgs& a, const half_t* x, const TiledPlan& plan, bool proj, int num_cus, hipStream_t stream) {
  const int key = (a.M <= 8 ? 8 : 16) * 100 + plan.wk * 10 + plan.pw;
  if (proj) {
    if (!plan.front) return hipErrorNotReady;
    switch (key) {
      case 821: return launch_tiled_t<8, 2, 1, true, kCanon>(a, x, num_cus, stream);
      case 811: return launch_tiled_t<8, 1, 1, true, kCanon>(a, x, num_cus, stream);
      case 1622: return launch_tiled_t<16, 2, 2, true, kCanon>(a, x, num_cus, stream);
      case 1612: return launch_tiled_t<16, 1, 2, true, kCanon>(a, x, num_cus, stream);
    }
    return hipErrorInvalidValue;
  }
  switch (key) {
    case 821: return launch_tiled_t<8, 2, 1, false, kCanon>(a, x, num_cus, stream);
    case 811: return launch_tiled_t<8, 1, 1, false, kCanon>(a, x, num_cus, stream);
    case 1620 + (kCanon ? 2 : 1): return launch_tiled_t<16, 2, kCanon ? 2 : 1, false, kCanon>(a, x, num_cus, stream);
    case 1610 + (kCanon ? 2 : 1): return launch_tiled_t<16, 1, kCanon ? 2 : 1, false, kCanon>(a, x, num_cus, stream);
  }
  return hipErrorInvalidValue;
}

// `canon`: the narrow tiles on the canonical buffers (skinny_words_supported)
hipError_t launch_skinny_tiled(GroupDev& g, int num_cus, hipStream_t stream, bool canon) {
  TileArgs a;
  a.r = g.r;
  // the launch computes r itself (run_group set g.pub to the head of the workspace): up to 16 token rows and rank 256 (r
  // goes through the stages in one pass), K whole, nothing else in the workspace (no slices)
  const bool proj = g.pub != nullptr;
  a.R = g.R;
  a.r_out = g.r_out;
  a.pub = g.pub;
  a.spin = g.pub_mute ? 0xFFFFFFFFu : g.pub_spin;
  a.producers = 0;
  a.teams = 1;
  if (proj) {
    if (g.M > 16 || g.rank > 256 || (g.rank & 7) != 0 || (g.K & 7) != 0 || g.R == nullptr || g.r_out == nullptr || g.ws_bytes < kTiledHandoverBytes)
      return hipErrorNotReady;
    a.r = g.r_out;
  }
  a.n_members = g.n_members;
  a.M = g.M;
  a.K = g.K;
  a.rank = g.rank;
  a.alpha = g.alpha;
  const bool ws_ok = g.ws != nullptr && (reinterpret_cast<uintptr_t>(g.ws) & 15u) == 0;
  a.partials = ws_ok ? static_cast<float*>(g.ws) : nullptr;
  const TiledPlan plan = tiled_plan(g, num_cus, ws_ok ? g.ws_bytes : 0, proj, canon);
  a.slices = plan.slices;
  a.cw = plan.cw;
  int tiles = 0, col = 0;
  for (int i = 0; i < g.n_members; ++i) {
    const MemberDev& m = g.mem[i];
    TileMember& t = a.mem[i];
    t.wt = canon ? reinterpret_cast<const unsigned char*>(m.qweight) : static_cast<const unsigned char*>(m.tiled);
    t.lt = (m.L != nullptr && (g.r != nullptr || proj)) ? (canon ? reinterpret_cast<const unsigned char*>(m.L) : static_cast<const unsigned char*>(m.tiled_L)) : nullptr;
    t.scales = m.scales;
    t.qzeros = m.qzeros;
    t.ldw = m.ldw;
    t.lds = m.lds;
    t.ldz = m.ldz;
    t.bias = m.bias;
    t.y = m.y;
    t.N = m.N;
    t.ldy = m.ldy;
    t.col0 = col;
    const int mt = ((m.N + 31) / 32 + plan.cw - 1) / plan.cw;
    tiles += mt;
    col += mt * plan.cw * 32;
    a.blk_end[i] = tiles;
  }
  a.tiles = tiles;
  a.ldp = col;
  if (g.M <= 16) return canon ? launch_narrow<true>(a, g.x, plan, proj, num_cus, stream) : launch_narrow<false>(a, g.x, plan, proj, num_cus, stream);
  return launch_tiled_t<32, 1, 4>(a, g.x, num_cus, stream);
}

}  // namespace glowq
