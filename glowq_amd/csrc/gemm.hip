// Prefill GEMM for gfx950: y[M,N] = x[M,K] . deq(W)[N,K]^T (+ alpha * r[M,rank] . L[N,rank]^T) on fp16 MFMA
// with fp32 accumulation.
//
// A workgroup of 4 waves owns a BM x BN output tile (BM = 32*kMT rows, BN = 128*kNT columns); the waves
// split the columns, each holding kMT x kNT accumulator tiles of 32x32 (v_mfma_f32_32x32x16_f16).
//   * Activations go global -> registers -> LDS (double-buffered, rows padded to 144 bytes so that the
//     16-byte fragment reads of 32 consecutive rows fall into distinct banks) and are read back as MFMA
//     A fragments by all four waves.
//   * Weights never touch LDS or HBM as fp16: the B operand of the 32x32x16 MFMA wants, per lane, 8
//     consecutive k of one output column -- exactly one int32 word of 8 int4 codes.  A lane loads 16 bytes
//     (4 words = the 4 MFMA k-steps of a 64-deep block) and dequantises them in registers to
//     fp16((code - zero) * scale): the codes are masked into the mantissa of 1024.0 / 64.0, the offset
//     and zero-point are removed by one exact packed subtraction, and one packed multiply rounds once,
//     which is bit-identical to the reference's dequantisation.  Every weight is dequantised exactly once.
//   * The masks deliver the codes of a word in the order (0,4,1,5,2,6,3,7); the activations are permuted
//     the same way on their way into LDS, so no instruction is spent on reordering weights.
//   * The rank-r correction is a K-extension that runs first: acc = r . L^T on the same pipeline with an
//     fp16 B operand, acc *= alpha, then the quantised K loop accumulates on top.
#include <cstdlib>

#include <algorithm>
#include <type_traits>

#include "common.hpp"
#include "dequant.hpp"
#include "handover.hpp"
#include "proj_front.hpp"
#include "tiled.hpp"

namespace glowq {

constexpr int kBK = 64;              // k depth of one pipeline step
constexpr int kARow = kBK + 8;       // padded LDS row, in halves (144 bytes)

struct GemmArgs {
  const half_t* x;        // [M, K]
  const half_t* r;        // [M, rank] or nullptr
  const int32_t* qweight; // [N, ldw] (quantised B) or nullptr
  const half_t* scales;
  const int32_t* qzeros;
  const half_t* bmat;     // [N, ldb] fp16 B operand: L for the correction, or the whole B of a plain GEMM
  const half_t* bias;
  half_t* y;              // [M, ldy] (fp32 in the kernels with YT = float)
  const unsigned char* wt;  // the member's tiled weights (tiled.hpp) or nullptr
  const unsigned char* lt;  // its tiled left factor or nullptr
  int M, N, K, group_size, rank;
  int ldw, lds, ldz, ldb, ldy;
  float alpha;
};

// The result is rounded to fp16 in either form; fp32 outputs hold that value widened, which a caller that wants them would
// otherwise do in a launch and two passes of its own (Qwen2.5-7B layer at 333 rows: 34 us of 326).  The form is a template argument of
// the kernels on the tiled copy: a branch on it around every store costs 5 to 8 % of a launch, one per column far more (the
// accumulators leave the registers).
__device__ __forceinline__ void store_y(half_t* y, float v) { *y = (half_t)v; }
__device__ __forceinline__ void store_y(float* y, float v) { *y = (float)(half_t)v; }

// One launch covers every member of a group: workgroup b serves member i for blk_end[i-1] <= b < blk_end[i].
struct GemmGroup {
  GemmArgs m[GLOWQ_MAX_MEMBERS];
  int blk_end[GLOWQ_MAX_MEMBERS];
  int n;
  // split K (super-block form only): gridDim.y slices of whole super-blocks; every workgroup leaves its fp32 tile in
  // `partials` ([slice][tile][BM * BN] in accumulator-register order) and gemm_reduce_kernel adds them in slice order
  int slices;
  float* partials;
  // tail split (super-block form, slices == 1): workgroups [0, full) are whole tiles; behind them every tail tile comes
  // as tail_slices workgroups, slice t % tail_slices of tile full + t / tail_slices for t = blockIdx.x - full, which
  // leave partials ([slice][tail tile][BM * BN]) for gemm_reduce_kernel.  The last, partly filled round of workgroups
  // of a launch then costs its share of a round instead of a whole one.  tail_slices <= 1: off.
  int full, tail_slices;
  // the launch computes r itself (kProj of gemm_tiled_kernel, proj_front.hpp): `front.front` workgroups in front of the grid
  FrontArgs front;
};
// A launch that computes r itself keeps at the head of the workspace the words of its workgroups in front and the sums of their slices of
// r (4 KB each, 32 x 32 tiles); no more workgroups than this do work there.
constexpr int kMaxFront = 512;
constexpr size_t kGemmWordBytes = (size_t)kMaxFront * 8;
constexpr size_t kGemmHandoverBytes = kGemmWordBytes + (size_t)kMaxFront * 4096;

__device__ __forceinline__ h8 permute_for_nibble_order(const h8& v) {
  h8 p;
  p[0] = v[0]; p[1] = v[4]; p[2] = v[1]; p[3] = v[5];
  p[4] = v[2]; p[5] = v[6]; p[6] = v[3]; p[7] = v[7];
  return p;
}

// kQuant: B is the int4 weight (with the optional correction phase in front); otherwise B is plain fp16.
// kSuper (quantised B, K % 256 == 0, group sizes of 128 and up): the K loop walks 256-column super-blocks in which lane
// (column c, half h) owns the 64 contiguous bytes of codes [256 sb + 128 h, +128) of its weight row -- one quantisation
// group, one scale and zero-point per super-block -- and the weights reach the B operand through a wave-private LDS tile
// that is filled in memory order (8 lanes per 128-byte row segment).  Fragment loads straight from memory, one 16-byte
// request per lane and cache line, make every request pull a whole line out of L2.
template <int kMT, int kNT, bool kQuant, bool kSuper = false>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu((kMT * kNT >= 16 ? 1 : 2), (kMT * kNT >= 16 ? 1 : 8))))
void gemm_mfma_kernel(const GemmGroup gg, const int m_blocks) {
  // member of this workgroup, picked with scalar selects from fixed kernel-argument offsets
  // which tile and which slice of its K range this workgroup serves
  int wg = (int)blockIdx.x, slice = (int)blockIdx.y, nslices = gg.slices, part_tile = (int)blockIdx.x, part_tiles = (int)gridDim.x;
  if (kQuant && kSuper && gg.tail_slices > 1) {
    nslices = 1;
    if (wg >= gg.full) {
      const int t = wg - gg.full;
      part_tile = t / gg.tail_slices;
      slice = t - part_tile * gg.tail_slices;
      wg = gg.full + part_tile;
      nslices = gg.tail_slices;
      part_tiles = ((int)gridDim.x - gg.full) / gg.tail_slices;
    }
  }
  GemmArgs a = gg.m[0];
  int blk_base = 0;
#define GLOWQ_PICK(i)                                         \
  if (gg.n > i && wg >= gg.blk_end[i - 1]) {                 \
    a = gg.m[i];                                              \
    blk_base = gg.blk_end[i - 1];                             \
  }
  GLOWQ_PICK(1)
  GLOWQ_PICK(2)
  GLOWQ_PICK(3)
#undef GLOWQ_PICK
  extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
  constexpr int BM = 32 * kMT;
  constexpr int BN = 128 * kNT;
  half_t* lds_a = reinterpret_cast<half_t*>(smem);  // [2][BM][kARow]

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = tid >> 6;
  const int blk = wg - blk_base;
  const int bm = blk % m_blocks;  // row blocks vary fastest: neighbouring workgroups share weight columns
  const int bn = blk / m_blocks;
  const int m0 = bm * BM;
  const int ln = lane & 31;  // column inside a 32-wide tile (B operand, accumulator) / row inside a tile (A operand)
  const int lh = lane >> 5;  // which half of the k range of an MFMA step this lane feeds

  int ncol[kNT];  // weight row (= output column) this lane feeds, clamped for loads
#pragma unroll
  for (int tn = 0; tn < kNT; ++tn) ncol[tn] = min(bn * BN + wave * (32 * kNT) + tn * 32 + ln, a.N - 1);

  f16v acc[kMT][kNT];
#pragma unroll
  for (int tm = 0; tm < kMT; ++tm)
#pragma unroll
    for (int tn = 0; tn < kNT; ++tn)
#pragma unroll
      for (int i = 0; i < 16; ++i) acc[tm][tn][i] = 0.f;

  // ---- activation tile: global -> registers -> LDS ------------------------------------------------
  // BM rows x 8 octets (16 bytes); thread t takes octets t, t+256, ...: 8 consecutive threads read the
  // 128 contiguous bytes of one row.
  struct ARegs {
    u32x4 v[kMT];
  };
  ARegs areg, areg1;
  auto load_a_to = [&](ARegs& dst, const half_t* src, int ld, int kb) {
#pragma unroll
    for (int i = 0; i < kMT; ++i) {
      const int q = tid + 256 * i;
      const int row = min(m0 + (q >> 3), a.M - 1);
      dst.v[i] = *reinterpret_cast<const u32x4*>(src + (size_t)row * ld + kb + (q & 7) * 8);
    }
  };
  auto store_a_from = [&](const ARegs& srcr, int stage, bool permute) {
#pragma unroll
    for (int i = 0; i < kMT; ++i) {
      const int q = tid + 256 * i;
      half_t* dst = lds_a + ((size_t)stage * BM + (q >> 3)) * kARow + (q & 7) * 8;
      const h8 v = __builtin_bit_cast(h8, srcr.v[i]);
      *reinterpret_cast<h8*>(dst) = permute ? permute_for_nibble_order(v) : v;
    }
  };
  auto store_a = [&](int stage, bool permute) { store_a_from(areg, stage, permute); };
  // A fragment of MFMA step t for row tile tm: octet (4*lh + t) of row tm*32 + ln
  auto read_a = [&](int stage, int tm, int t) {
    const half_t* src = lds_a + ((size_t)stage * BM + tm * 32 + ln) * kARow + (4 * lh + t) * 8;
    return *reinterpret_cast<const h8*>(src);
  };
  auto mma_step = [&](int stage, const h8 (&bfrag)[kNT][4]) {
    constexpr int kChunk = kMT < 4 ? kMT : 4;  // row tiles whose A fragments are live at once
#pragma unroll
    for (int t = 0; t < 4; ++t) {
#pragma unroll
      for (int c = 0; c < kMT; c += kChunk) {
        h8 af[kChunk];
#pragma unroll
        for (int i = 0; i < kChunk; ++i) af[i] = read_a(stage, c + i, t);
#pragma unroll
        for (int tn = 0; tn < kNT; ++tn)
#pragma unroll
          for (int i = 0; i < kChunk; ++i)
            acc[c + i][tn] = __builtin_amdgcn_mfma_f32_32x32x16_f16(af[i], bfrag[tn][t], acc[c + i][tn], 0, 0, 0);
      }
    }
  };

  int stage = 0;

  // ---- phase 1: the correction as a K-extension, acc = r . L^T, fp16 B operand ----------------------
  if (kQuant && a.r != nullptr && slice == 0) {
    // ranks are multiples of 8: in a partial last block the octets of r past the rank count as zero and L is read
    // from the row's last octet (finite values)
    const int steps = (a.rank + kBK - 1) / kBK;
    auto load_r = [&](int kb) {
#pragma unroll
      for (int i = 0; i < kMT; ++i) {
        const int q = tid + 256 * i;
        const int row = min(m0 + (q >> 3), a.M - 1);
        const int k = kb + (q & 7) * 8;
        const u32x4 v = *reinterpret_cast<const u32x4*>(a.r + (size_t)row * a.rank + min(k, a.rank - 8));
        areg.v[i] = k < a.rank ? v : u32x4{0u, 0u, 0u, 0u};
      }
    };
    load_r(0);
    store_a(stage, false);
    __syncthreads();
    for (int ks = 0; ks < steps; ++ks) {
      h8 bfrag[kNT][4];
      if constexpr (kSuper) {
        // the wave's 32 kNT rows of L, 128 bytes of this block each, in memory order (8 lanes per row) through its LDS
        // tile, as the weights of the main loop: fragment loads straight from memory cost a line per lane
        unsigned char* ltile = smem + (size_t)2 * BM * kARow * sizeof(half_t) + (size_t)wave * (32 * kNT) * 144;
        u32x4 lreg[kNT * 4];
#pragma unroll
        for (int q = 0; q < kNT * 4; ++q)
          lreg[q] = *reinterpret_cast<const u32x4*>(a.bmat + (size_t)min(bn * BN + wave * (32 * kNT) + q * 8 + (lane >> 3), a.N - 1) * a.ldb +
                                                    min(ks * kBK + (lane & 7) * 8, a.rank - 8));
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");  // fragment reads of the previous block are done
        __builtin_amdgcn_wave_barrier();
#pragma unroll
        for (int q = 0; q < kNT * 4; ++q)
          *reinterpret_cast<u32x4*>(ltile + (q * 8 + (lane >> 3)) * 144 + (lane & 7) * 16) = lreg[q];
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
#pragma unroll
        for (int tn = 0; tn < kNT; ++tn)
#pragma unroll
          for (int t = 0; t < 4; ++t)
            bfrag[tn][t] = *reinterpret_cast<const h8*>(ltile + (tn * 32 + ln) * 144 + lh * 64 + t * 16);
      } else {
#pragma unroll
        for (int tn = 0; tn < kNT; ++tn)
#pragma unroll
          for (int t = 0; t < 4; ++t)
            bfrag[tn][t] = *reinterpret_cast<const h8*>(a.bmat + (size_t)ncol[tn] * a.ldb + min(ks * kBK + 32 * lh + 8 * t, a.rank - 8));
      }
      if (ks + 1 < steps) load_r((ks + 1) * kBK);
      mma_step(stage, bfrag);
      if (ks + 1 < steps) store_a(stage ^ 1, false);
      __syncthreads();
      stage ^= 1;
    }
    if (a.alpha != 1.0f) {
#pragma unroll
      for (int tm = 0; tm < kMT; ++tm)
#pragma unroll
        for (int tn = 0; tn < kNT; ++tn)
#pragma unroll
          for (int i = 0; i < 16; ++i) acc[tm][tn][i] *= a.alpha;
    }
  }

  // ---- phase 2: the main K loop ---------------------------------------------------------------------
  const int steps = a.K / kBK;
  const int gs_shift = __builtin_ctz(a.group_size);  // group sizes on this route are powers of two
  if constexpr (kQuant && kSuper) {
    // Sub-step ks = 4 sb + j covers columns {256 sb + 128 h + 32 j + [0, 32) : h = 0, 1}; the activation stage keeps
    // its [BM][64] shape with octets 0-3 = half 0 and octets 4-7 = half 1, so the fragment reads do not change.
    constexpr int kSeg = 144;  // bytes per row segment in the weight tile: 128 + 16, conflict-free fragment reads
    unsigned char* btile = smem + (size_t)2 * BM * kARow * sizeof(half_t) + (size_t)wave * (32 * kNT) * kSeg;
    // Every load of the loop is a buffer load: a uniform descriptor and a uniform byte offset that advances per step
    // (scalar registers) plus a 32-bit byte offset that a lane computes once.  With 64-bit addresses per lane and load
    // the address pairs alone spill the register file of the large tiles, and every reload of a spilled pair waits
    // for all loads in flight.  (The host keeps tensors whose byte extent does not fit 32 bits off this route.)
    const auto rsrc = [](const void* p, size_t bytes) {
      return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(p), 0, (int)(uint32_t)bytes, 0x00020000);
    };
    const __amdgpu_buffer_rsrc_t rs_x = rsrc(a.x, (size_t)a.M * a.K * 2);
    const __amdgpu_buffer_rsrc_t rs_w = rsrc(a.qweight, ((size_t)(a.N - 1) * a.ldw + (a.K >> 3)) * 4);
    const __amdgpu_buffer_rsrc_t rs_s = rsrc(a.scales, ((size_t)(a.N - 1) * a.lds + (a.K >> gs_shift)) * 2);
    const __amdgpu_buffer_rsrc_t rs_z = rsrc(a.qzeros, ((size_t)(a.N - 1) * a.ldz + (((a.K >> gs_shift) + 7) >> 3)) * 4);
    uint32_t a_off[kMT], b_off[kNT * 4], s_off[kNT], z_off[kNT];
#pragma unroll
    for (int i = 0; i < kMT; ++i) {
      const int q = tid + 256 * i;
      const int oct = q & 7;
      a_off[i] = ((uint32_t)min(m0 + (q >> 3), a.M - 1) * (uint32_t)a.K + (oct >> 2) * 128 + (oct & 3) * 8) * 2u;
    }
#pragma unroll
    for (int q = 0; q < kNT * 4; ++q)
      b_off[q] = ((uint32_t)min(bn * BN + wave * (32 * kNT) + q * 8 + (lane >> 3), a.N - 1) * (uint32_t)a.ldw + (lane & 7) * 4) * 4u;
#pragma unroll
    for (int tn = 0; tn < kNT; ++tn) {
      s_off[tn] = (uint32_t)ncol[tn] * (uint32_t)a.lds * 2u;
      z_off[tn] = (uint32_t)ncol[tn] * (uint32_t)a.ldz * 4u;
    }
    auto load_a_sub = [&](ARegs& dst, int ks) {
      const int kc = min(ks, steps - 1);
      const int step_off = ((kc >> 2) * 256 + (kc & 3) * 32) * 2;
#pragma unroll
      for (int i = 0; i < kMT; ++i) dst.v[i] = __builtin_amdgcn_raw_buffer_load_b128(rs_x, (int)a_off[i], step_off, 0);
    };
    struct BLoad {
      u32x4 w[kNT * 4];  // a super-block of the wave's 32 kNT weight rows in load order: row 8 q + lane / 8, piece lane % 8
      uint32_t s[kNT], z[kNT];
    };
    uint32_t cur_s[kNT], cur_z[kNT];
    auto issue_b = [&](int sb, BLoad& bl) {
      const int sbc = min(sb, (steps >> 2) - 1);
      const uint32_t grp = (uint32_t)((sbc * 256 + lh * 128) >> gs_shift);
#pragma unroll
      for (int q = 0; q < kNT * 4; ++q) bl.w[q] = __builtin_amdgcn_raw_buffer_load_b128(rs_w, (int)b_off[q], sbc * 128, 0);
#pragma unroll
      for (int tn = 0; tn < kNT; ++tn) {
        bl.s[tn] = (uint32_t)(unsigned short)__builtin_amdgcn_raw_buffer_load_b16(rs_s, (int)(s_off[tn] + grp * 2u), 0, 0);
        bl.z[tn] = (uint32_t)__builtin_amdgcn_raw_buffer_load_b32(rs_z, (int)(z_off[tn] + (grp >> 3) * 4u), 0, 0);
      }
    };
    auto stage_b = [&](const BLoad& bl) {
      __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");  // fragment reads of the previous super-block are done
      __builtin_amdgcn_wave_barrier();
#pragma unroll
      for (int q = 0; q < kNT * 4; ++q)
        *reinterpret_cast<u32x4*>(btile + (q * 8 + (lane >> 3)) * kSeg + (lane & 7) * 16) = bl.w[q];
#pragma unroll
      for (int tn = 0; tn < kNT; ++tn) {
        cur_s[tn] = bl.s[tn];
        cur_z[tn] = bl.z[tn];
      }
      __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
      __builtin_amdgcn_wave_barrier();
      __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    };
    BLoad bl;
    // j is a compile-time constant at every call site (the loop below is unrolled by four)
    auto step = [&](int ks, int j, ARegs& a_fill, const ARegs& a_store) {
      const int sb = ks >> 2;
      if (j == 0) stage_b(bl);
      const int grp = (sb * 256 + lh * 128) >> gs_shift;
      u32x4 raw[kNT];
      h2 zb_lo[kNT], zb_hi[kNT], s2[kNT];
#pragma unroll
      for (int tn = 0; tn < kNT; ++tn) {
        const half_t z = (half_t)(float)nibble(cur_z[tn], grp & 7);
        const half_t zl = (half_t)(-1024.0f) - z, zh = (half_t)(-64.0f) - z;
        zb_lo[tn] = h2{zl, zl};
        zb_hi[tn] = h2{zh, zh};
        s2[tn] = bitcast_u32<h2>(cur_s[tn] | (cur_s[tn] << 16));
        raw[tn] = *reinterpret_cast<const u32x4*>(btile + (tn * 32 + ln) * kSeg + lh * 64 + j * 16);
      }
      load_a_sub(a_fill, ks + 2);
      if (j == 0) issue_b(sb + 1, bl);  // behind the activation loads: waiting for those leaves the weights in flight
      // one code word per MFMA step is dequantised right before its MFMAs: 8 fragment registers live instead of 32
      constexpr int kChunk = kMT < 4 ? kMT : 4;
#pragma unroll
      for (int t = 0; t < 4; ++t) {
        h8 bf[kNT];
#pragma unroll
        for (int tn = 0; tn < kNT; ++tn) bf[tn] = dequant_word(raw[tn][t], zb_lo[tn], zb_hi[tn], s2[tn]);
#pragma unroll
        for (int c = 0; c < kMT; c += kChunk) {
          h8 af[kChunk];
#pragma unroll
          for (int i = 0; i < kChunk; ++i) af[i] = read_a(stage, c + i, t);
#pragma unroll
          for (int tn = 0; tn < kNT; ++tn)
#pragma unroll
            for (int i = 0; i < kChunk; ++i)
              acc[c + i][tn] = __builtin_amdgcn_mfma_f32_32x32x16_f16(af[i], bf[tn], acc[c + i][tn], 0, 0, 0);
        }
      }
      store_a_from(a_store, stage ^ 1, true);
      __syncthreads();
      stage ^= 1;
    };
    // this workgroup's super-blocks: all of them, or slice `slice` of `nslices`
    const int sb_total = steps >> 2;  // steps is a multiple of 4 here
    const int sb_per = (sb_total + nslices - 1) / nslices;
    const int ks0 = min(slice * sb_per, sb_total) * 4;
    const int ks1 = min(ks0 + sb_per * 4, steps);
    load_a_sub(areg, ks0);
    issue_b(ks0 >> 2, bl);
    load_a_sub(areg1, ks0 + 1);
    store_a_from(areg, stage, true);
    __syncthreads();
    for (int ks = ks0; ks < ks1; ks += 4) {
      step(ks, 0, areg, areg1);
      step(ks + 1, 1, areg1, areg);
      step(ks + 2, 2, areg, areg1);
      step(ks + 3, 3, areg1, areg);
    }
  } else if constexpr (kQuant) {
    // quantised B: per step and column tile one 16-byte load of codes, one scale, one zero-point word.
    // Two register sets alternate (no copies), and the prefetch of the next step is unconditional (the
    // last step re-reads its own block): a uniform number of loads per step keeps the wait counts exact,
    // so the loads issued at the top of a step stay in flight under that step's MFMAs.
    struct WRegs {  // all members 32-bit wide: the struct stays in registers
      u32x4 w[kNT];
      uint32_t s[kNT];  // fp16 bits of the scale
      uint32_t z[kNT];
    };
    auto load_w = [&](int kb, WRegs& wr) {
      const int grp = (kb + 32 * lh) >> gs_shift;
#pragma unroll
      for (int tn = 0; tn < kNT; ++tn) {
        wr.w[tn] = *reinterpret_cast<const u32x4*>(a.qweight + (size_t)ncol[tn] * a.ldw + (kb >> 3) + 4 * lh);
        wr.s[tn] = reinterpret_cast<const unsigned short*>(a.scales)[(size_t)ncol[tn] * a.lds + grp];
        wr.z[tn] = (uint32_t)a.qzeros[(size_t)ncol[tn] * a.ldz + (grp >> 3)];
      }
    };
    // Step s: dequantise W(s) out of its register set, refill that set with W(s+2) and the matching
    // activation set with A(s+2), run the MFMAs of step s on LDS stage s%2, then move A(s+1) (loaded one
    // step ago, so it has had a whole step to arrive) into the other LDS stage.  Loads are unconditional
    // (clamped to the last block) so that every step issues the same number of them.
    auto step = [&](int ks, WRegs& wr, ARegs& a_fill, const ARegs& a_store) {
      const int kb = ks * kBK;
      h8 bfrag[kNT][4];
      const int grp = (kb + 32 * lh) >> gs_shift;
#pragma unroll
      for (int tn = 0; tn < kNT; ++tn) {
        const half_t z = (half_t)(float)nibble(wr.z[tn], grp & 7);
        const half_t zl = (half_t)(-1024.0f) - z, zh = (half_t)(-64.0f) - z;
        const h2 zb_lo = {zl, zl}, zb_hi = {zh, zh};
        const h2 s2 = bitcast_u32<h2>(wr.s[tn] | (wr.s[tn] << 16));
        bfrag[tn][0] = dequant_word(wr.w[tn].x, zb_lo, zb_hi, s2);
        bfrag[tn][1] = dequant_word(wr.w[tn].y, zb_lo, zb_hi, s2);
        bfrag[tn][2] = dequant_word(wr.w[tn].z, zb_lo, zb_hi, s2);
        bfrag[tn][3] = dequant_word(wr.w[tn].w, zb_lo, zb_hi, s2);
      }
      const int kb2 = min(ks + 2, steps - 1) * kBK;
      load_w(kb2, wr);
      load_a_to(a_fill, a.x, a.K, kb2);
      mma_step(stage, bfrag);
      store_a_from(a_store, stage ^ 1, true);
      __syncthreads();
      stage ^= 1;
    };
    WRegs w0, w1;
    load_a_to(areg, a.x, a.K, 0);
    load_w(0, w0);
    load_a_to(areg1, a.x, a.K, min(1, steps - 1) * kBK);
    load_w(min(1, steps - 1) * kBK, w1);
    store_a_from(areg, stage, true);
    __syncthreads();
    for (int ks = 0; ks < steps; ks += 2) {
      step(ks, w0, areg, areg1);
      if (ks + 1 >= steps) break;
      step(ks + 1, w1, areg1, areg);
    }
  } else {
    // plain fp16 B (the shared projection r = x R^T for many rows): same two-deep pipeline, the B
    // fragments are loaded as they are (4 x 16 bytes per lane, column tile and step)
    struct BRegs {
      u32x4 v[kNT][4];
    };
    auto load_b = [&](int kb, BRegs& br) {
#pragma unroll
      for (int tn = 0; tn < kNT; ++tn)
#pragma unroll
        for (int t = 0; t < 4; ++t)
          br.v[tn][t] = *reinterpret_cast<const u32x4*>(a.bmat + (size_t)ncol[tn] * a.ldb + kb + 32 * lh + 8 * t);
    };
    auto step = [&](int ks, BRegs& br, ARegs& a_fill, const ARegs& a_store) {
      h8 bfrag[kNT][4];
#pragma unroll
      for (int tn = 0; tn < kNT; ++tn)
#pragma unroll
        for (int t = 0; t < 4; ++t) bfrag[tn][t] = __builtin_bit_cast(h8, br.v[tn][t]);
      const int kb2 = min(ks + 2, steps - 1) * kBK;
      load_b(kb2, br);
      load_a_to(a_fill, a.x, a.K, kb2);
      mma_step(stage, bfrag);
      store_a_from(a_store, stage ^ 1, false);
      __syncthreads();
      stage ^= 1;
    };
    BRegs b0, b1;
    load_a_to(areg, a.x, a.K, 0);
    load_b(0, b0);
    load_a_to(areg1, a.x, a.K, min(1, steps - 1) * kBK);
    load_b(min(1, steps - 1) * kBK, b1);
    store_a_from(areg, stage, false);
    __syncthreads();
    for (int ks = 0; ks < steps; ks += 2) {
      step(ks, b0, areg, areg1);
      if (ks + 1 >= steps) break;
      step(ks + 1, b1, areg1, areg);
    }
  }

  // ---- epilogue: accumulator register i of a 32x32 tile is row 8*(i/4) + 4*lh + i%4, column ln ---------
  if constexpr (kQuant && kSuper) {
    if (nslices > 1) {
      float* part = gg.partials + ((size_t)slice * part_tiles + part_tile) * (BM * BN);
#pragma unroll
      for (int tm = 0; tm < kMT; ++tm)
#pragma unroll
        for (int tn = 0; tn < kNT; ++tn)
#pragma unroll
          for (int i = 0; i < 16; ++i) part[((tm * kNT + tn) * 16 + i) * 256 + tid] = acc[tm][tn][i];
      return;
    }
  }
#pragma unroll
  for (int tn = 0; tn < kNT; ++tn) {
    const int n = bn * BN + wave * (32 * kNT) + tn * 32 + ln;
    if (n >= a.N) continue;
    const float b = a.bias ? (float)a.bias[n] : 0.f;
#pragma unroll
    for (int tm = 0; tm < kMT; ++tm) {
#pragma unroll
      for (int i = 0; i < 16; ++i) {
        const int m = m0 + tm * 32 + 8 * (i >> 2) + 4 * lh + (i & 3);
        if (m < a.M) a.y[(size_t)m * a.ldy + n] = (half_t)(acc[tm][tn][i] + b);
      }
    }
  }
}

// ---- the same GEMM on the tiled copy of the weights (tiled.hpp) ---------------------------------------------------
// Same tiles, same workgroup -> tile map, same split of K, same partial tiles and epilogue as gemm_mfma_kernel's
// super-block form, same arithmetic (the weight is rounded to fp16 once).  What differs is how the operands arrive:
//   * B: a wave's 16-byte loads of a chunk of the tiled stream ARE the B operands of its 32 x 256 block, in lane order;
//     scale and zero-point ride in the same chunk (one 8-byte load per lane and super-block).  No pass of the weights
//     through LDS, no gathers of scales and zero-point words, no per-wave barriers around a staging tile.  One set of
//     registers holds a super-block; each 16-byte piece is refilled with the next super-block's as soon as its four
//     words have been dequantised, a whole super-block of matrix instructions ahead of its use.
//   * A: the tiled copy holds the nibbles of a code word in the order in which the masks deliver them, so the
//     activations need no permutation and go from memory straight into LDS (buffer_load ... lds: no registers, no
//     vector instructions, no ds_write).  Stages of 128 columns (one quantisation-group half of a super-block)
//     instead of 64: half the barriers per matrix instruction.  A load of a wave fills one contiguous kilobyte of
//     LDS -- four rows of 256 bytes, no padding -- so bank conflicts are avoided by the choice of what goes where:
//     slot c' of row r holds the 16-byte piece c' ^ (r % 16) of that row, and a fragment read of piece c looks in
//     slot c ^ (r % 16): sixteen consecutive rows land in sixteen different slots.
//   * The matrix instructions of a code word and the vector instructions that dequantise the next one are interleaved by hand
//     (order_word), and the correction runs behind the weights, its sum in registers of its own, r straight into LDS like the
//     activations: in front, its two round trips came before the first weights, and its staging registers made the 128 x 256
//     tile spill.  Together 1.04 times as fast in the mean over 15 groups of 1B to 14B shapes at 72 to 2048 rows (8B gate|up at 2048
//     rows 443 -> 430 us, down_proj at 333 rows 61.7 -> 55.8, 14B o_proj at 100 rows 21.2 -> 18.7, same cuts).
constexpr int kTRow = 256;  // bytes of a staged row: 128 halves, swizzled instead of padded

// The order of a word's instructions: behind every matrix instruction its share of the next word's kOps vector instructions per column tile,
// the next fragments from LDS in front (few matrix instructions a word) or as soon as a fragment has been used for the last time.
template <int kMT, int kNT, int kOps>
__device__ __forceinline__ void order_word() {
  constexpr int kShare = (kOps * kNT + kMT * kNT - 1) / (kMT * kNT);
  constexpr bool kReadsFirst = kMT * kNT <= 4;
  if constexpr (kReadsFirst) __builtin_amdgcn_sched_group_barrier(0x100, kMT, 0);
#pragma unroll
  for (int q = 0; q < kMT * kNT; ++q) {
    __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
    __builtin_amdgcn_sched_group_barrier(0x002, kShare, 0);
    if (!kReadsFirst && q % kNT == kNT - 1) __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
  }
  __builtin_amdgcn_sched_barrier(0);
}

// kWk = 2: eight waves on the same tile, the second four take the second half of the workgroup's K range with LDS stages
// of their own, and the two accumulator sets meet in LDS before the epilogue.  For launches with about one tile per
// compute unit: a SIMD then holds two waves of the one workgroup it has, instead of one wave with nothing to overlap its
// waits with, and the K loop of a tile takes half as many steps.
// One super-block of weights and one half-step of activations are ahead.  Four sets of registers and four stages measured the same or slower
// on every shape at 100 and 333 rows (8B gate|up at 100 rows 41.4 -> 42.2 us, down_proj 28.2 -> 28.9), but that says nothing of more activations in
// flight: in front of a barrier the compiler waits for every load to LDS (see proj_front.hpp), whatever the wait above it leaves.
// kProj: the launch computes r = x R^T itself.  The readers need r behind their K loop, which is when the workgroups in front of the grid are
// done as a rule; they wait for the words of their rows' tiles (bounded: a reader that gives up computes its r from x and R), and
// read r past the caches the stores of the workgroups in front have passed.
// kExact: up to 64 rows, the arithmetic of the kernel of skinny_tiled.hip: the matrix instructions multiply code - zero, and the sum over a
// half of 128 columns meets its scale in fp32, so the weight is never rounded (nine vector instructions a word and sixteen a
// half and tile against thirteen a word: as many at two row tiles).
template <int kMT, int kNT, int kWk, typename YT, bool kProj, bool kExact>
__global__ __launch_bounds__(256 * kWk) __attribute__((amdgpu_waves_per_eu((kMT * kNT <= 2 && !(kExact && kMT == 2) ? 4 : 2), 8)))
void gemm_tiled_kernel(const GemmGroup gg, const int m_blocks) {
  extern __shared__ __attribute__((aligned(16))) unsigned char smem_all[];
  const int front = kProj ? gg.front.front : 0;
  unsigned long long tag = 0;
  if constexpr (kProj) {
    tag = launch_tag();
    if ((int)blockIdx.x < front) {
      run_front<4 * kWk>(gg.front, (int)blockIdx.x, tag, smem_all);
      return;
    }
  }
  // (with workgroups in front the slices of K lie behind each other in x: in y every one of them would bring a front that only leaves again)
  const int across = kProj && gg.slices > 1 ? ((int)gridDim.x - front) / gg.slices : (int)gridDim.x - front;
  int wg = (int)blockIdx.x - front, slice = (int)blockIdx.y, nslices = gg.slices;
  if (kProj && gg.slices > 1) {
    slice = wg / across;
    wg -= slice * across;
  }
  int part_tile = wg, part_tiles = across;
  if (gg.tail_slices > 1) {
    nslices = 1;
    if (wg >= gg.full) {
      const int t = wg - gg.full;
      part_tile = t / gg.tail_slices;
      slice = t - part_tile * gg.tail_slices;
      wg = gg.full + part_tile;
      nslices = gg.tail_slices;
      part_tiles = ((int)gridDim.x - front - gg.full) / gg.tail_slices;
    }
  }
  GemmArgs a = gg.m[0];
  int blk_base = 0;
#define GLOWQ_PICK(i)                                         \
  if (gg.n > i && wg >= gg.blk_end[i - 1]) {                 \
    a = gg.m[i];                                              \
    blk_base = gg.blk_end[i - 1];                             \
  }
  GLOWQ_PICK(1)
  GLOWQ_PICK(2)
  GLOWQ_PICK(3)
#undef GLOWQ_PICK
  constexpr int BM = 32 * kMT;
  constexpr int BN = 128 * kNT;
  constexpr int kAL = 2 * kMT;  // 16-byte pieces of a stage (BM rows x 256 bytes) per thread
  static_assert(kWk == 1 || kWk == 2, "one or two K groups");
  const int gk = kWk > 1 ? __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 8) : 0;  // K group of this wave
  unsigned char* smem = smem_all + (size_t)gk * 2 * BM * kTRow;
  const int tid = (int)threadIdx.x & 255;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int blk = wg - blk_base;
  const int bm = blk % m_blocks;  // row blocks vary fastest: neighbouring workgroups share weight columns
  const int bn = blk / m_blocks;
  const int m0 = bm * BM;
  const int ln = lane & 31, lh = lane >> 5;

  const auto rsrc = [](const void* p, size_t bytes) {
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(p), 0, (int)(uint32_t)bytes, 0x00020000);
  };
  const int RB = (a.N + 31) >> 5;
  const int SB = a.K >> 8;
  // row block of column tile tn of this wave, clamped into the member (columns past N are computed and dropped)
  int rb[kNT];
#pragma unroll
  for (int tn = 0; tn < kNT; ++tn) rb[tn] = min(bn * (BN / 32) + wave * kNT + tn, RB - 1);

  // this workgroup's super-blocks: all of them, or slice `slice` of `nslices`; dealt to the K groups in contiguous halves.
  // Both groups run the same number of steps (they share the barriers): a step past a group's part reads past the end of
  // its descriptor -- zero codes at scale zero.
  const int sb_per = (SB + nslices - 1) / nslices;
  const int ws0 = min(slice * sb_per, SB), ws1 = min(ws0 + sb_per, SB);
  const int per_group = (ws1 - ws0 + kWk - 1) / kWk;
  const int sb0 = min(ws0 + gk * per_group, ws1), sb1 = min(sb0 + per_group, ws1);
  const int sb_end = sb0 + per_group;  // steps run up to here

  // The correction extends K: behind the last super-block of the last slice the walk goes on over the rank, in steps of 128 columns of
  // r, dealt to the K groups in turn, with the tiled left factor as B operand.
  const bool corr = a.r != nullptr && a.lt != nullptr && slice == nslices - 1;
  const int LB = (a.rank + 63) >> 6;
  const __amdgpu_buffer_rsrc_t rs_x = rsrc(a.x, (size_t)a.M * a.K * 2);
  const __amdgpu_buffer_rsrc_t rs_r = rsrc(corr ? a.r : a.x, corr ? (size_t)a.M * a.rank * 2 : 0);
  const __amdgpu_buffer_rsrc_t rs_w = rsrc(a.wt, (size_t)RB * sb1 * tiled::kChunk);
  const __amdgpu_buffer_rsrc_t rs_l = rsrc(corr ? a.lt : a.wt, corr ? (size_t)RB * LB * tiled::kLChunk : 0);
  constexpr uint32_t kPast = 0xFFFF0000u;  // a scalar offset past the end of any descriptor: zeros

  // ---- activations: piece q of thread t fills slot (t & 15) of row 16 q + (t >> 4) of the stage, which holds the
  // 16-byte piece (t & 15) ^ (row % 16) of that row's 256 bytes (row % 16 = (t >> 4) % 16 for every q); every wave fills the
  // four rows 16 q + 4 wave + [0, 4) of piece q, one contiguous kilobyte of LDS per load.  Rows past M lie past the end of the descriptor.
  const int srow = tid >> 4;                    // 0..15: the row within a block of sixteen
  const int spiece = (tid & 15) ^ srow;         // the piece of the row this thread moves
  const uint32_t x_lane = (uint32_t)srow * (uint32_t)a.K * 2u + (uint32_t)spiece * 16u;
  const uint32_t r_lane = (uint32_t)srow * (uint32_t)a.rank * 2u + (uint32_t)spiece * 16u;
  typedef __attribute__((address_space(3))) void* lds_ptr_t;
  // rank columns [128 st, 128 st + 128) of r into stage `stg`; pieces past the rank meet zeros of the left factor and are read as zeros
  auto load_r = [&](int st, int stg) __attribute__((always_inline)) {
    constexpr int kPastCaches = kProj ? 16 : 0;  // where the workgroups in front left it
    const uint32_t off = st * 128 + spiece * 8 < a.rank ? r_lane : kPast;
#pragma unroll
    for (int q = 0; q < kAL; ++q)
      __builtin_amdgcn_raw_ptr_buffer_load_lds(rs_r, (lds_ptr_t)(smem + (size_t)stg * BM * kTRow + (16 * q + 4 * wave) * kTRow), 16, (int)off,
                                               (int)((uint32_t)(m0 + 16 * q) * (uint32_t)a.rank * 2u + (uint32_t)st * 256u), 0, kPastCaches);
  };
  // the same without r: every thread computes the eight entries of its pieces
  auto compute_r = [&](int st, int stg) {
#pragma unroll 1
    for (int q = 0; q < kAL; ++q) {
      const int row = m0 + srow + 16 * q;
      h8 own;
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        const int j = st * 128 + spiece * 8 + e;
        float sum = 0.f;
        if (row < a.M && j < a.rank) {
          const h2* xv = reinterpret_cast<const h2*>(a.x + (size_t)row * a.K);
          const h2* rv = reinterpret_cast<const h2*>(gg.front.R + (size_t)j * a.K);
#pragma unroll 1
          for (int k = 0; k < a.K / 2; ++k) sum = __builtin_amdgcn_fdot2(xv[k], rv[k], sum, false);
        }
        own[e] = (half_t)sum;
      }
      *reinterpret_cast<h8*>(smem + (size_t)stg * BM * kTRow + (16 * q + srow) * kTRow + (tid & 15) * 16) = own;
    }
  };
  // half-step hs = 2 sb + g of the activations (clamped into the row) into stage `stg`
  auto load_x = [&](int hs, int stg) __attribute__((always_inline)) {
    const uint32_t col = (uint32_t)min(hs, 2 * SB - 1) * 256u;
#pragma unroll
    for (int q = 0; q < kAL; ++q)
      __builtin_amdgcn_raw_ptr_buffer_load_lds(rs_x, (lds_ptr_t)(smem + (size_t)stg * BM * kTRow + (16 * q + 4 * wave) * kTRow), 16, (int)x_lane,
                                               (int)((uint32_t)(m0 + 16 * q) * (uint32_t)a.K * 2u + col), 0, 0);
  };
  // A fragment of row tile tm, piece c of the staged row (which 16 columns: see the callers)
  auto read_a = [&](int stage, int tm, int c) __attribute__((always_inline)) {
    return *reinterpret_cast<const h8*>(smem + (size_t)stage * BM * kTRow + (tm * 32 + ln) * kTRow + ((c ^ (ln & 15)) << 4));
  };
  // The activations of the next stage have landed before the workgroup's barrier: loads return in order, so it is enough
  // to wait until no more loads are outstanding than were issued behind them.  The scheduling barriers keep the loads where
  // they are written: left alone, the compiler sinks the refills to the end of the half-step, where nothing hides them.
  auto wait_loads_but = [&](auto n_const) __attribute__((always_inline)) {
    constexpr int n = decltype(n_const)::value;
    // (a comment in the assembly: the build checks that the n loads in front of it are none of those that go to LDS, isa_lint.py)
    asm volatile("; loads to LDS are followed by %0 others" ::"n"(n));
    __builtin_amdgcn_s_waitcnt((n & 15) | 0x0F70 | ((n >> 4) << 14));  // vmcnt(n), nothing else
  };

  // ---- weights: two sets of registers take turns; while the pieces of one are dequantised, the same pieces of the other are
  // refilled with the next super-block (a set refilled in place would have to be copied at the loop's back edge, and a copy waits for
  // the load)
  struct BSet {
    u32x4 w[kNT][4];
    u32x2 side[kNT];
  };
  BSet b[2];
  const int w_lane = lane * 16;
  const uint32_t chunk_stride = (uint32_t)RB * (uint32_t)tiled::kChunk;
  auto load_w = [&](BSet& s, int sb, int piece) __attribute__((always_inline)) {
#pragma unroll
    for (int tn = 0; tn < kNT; ++tn)
      s.w[tn][piece] = __builtin_amdgcn_raw_buffer_load_b128(rs_w, w_lane + piece * 1024, (int)((uint32_t)rb[tn] * (uint32_t)tiled::kChunk + (uint32_t)sb * chunk_stride), 0);
  };
  auto load_side = [&](BSet& s, int sb) __attribute__((always_inline)) {
#pragma unroll
    for (int tn = 0; tn < kNT; ++tn)
      s.side[tn] = __builtin_bit_cast(u32x2, __builtin_amdgcn_raw_buffer_load_b64(rs_w, tiled::kCodeBytes + ln * 8, (int)((uint32_t)rb[tn] * (uint32_t)tiled::kChunk + (uint32_t)sb * chunk_stride), 0));
  };

  f16v acc[kMT][kNT];
#pragma unroll
  for (int tm = 0; tm < kMT; ++tm)
#pragma unroll
    for (int tn = 0; tn < kNT; ++tn)
#pragma unroll
      for (int i = 0; i < 16; ++i) acc[tm][tn][i] = 0.f;

  // ---- the quantised K loop, a half of a super-block (128 columns, one quantisation group) per stage --------
  // Half-step h = 2 sb + g requests the activations of half-step h + 1, then pieces 2 g and 2 g + 1 (and, with g = 0, scale and
  // zero-point) of super-block sb + 1; its last wait leaves in flight what was requested behind those activations.
  load_side(b[0], sb0);
  load_w(b[0], sb0, 0);
  load_w(b[0], sb0, 1);
  load_x(2 * sb0, 0);
  __builtin_amdgcn_sched_barrier(0);
  load_w(b[0], sb0, 2);
  load_w(b[0], sb0, 3);
  __builtin_amdgcn_sched_barrier(0);
  wait_loads_but(std::integral_constant<int, 2 * kNT>{});
  __syncthreads();

  // One code word of every column tile at a time: while the matrix instructions of word t run, the next word is dequantised between
  // them and its A fragments are on their way from LDS.  Written as word after word the compiler puts a word's thirteen vector
  // instructions and the wait for its fragments in front of its own matrix instructions, and the two pipes take turns.
  struct Zero {
    h2 lo[kNT], hi[kNT], s[kNT];
    float scale[kNT];  // kExact
  };
  auto zero_of = [&](const BSet& s, int g) __attribute__((always_inline)) {
    Zero z;
#pragma unroll
    for (int tn = 0; tn < kNT; ++tn) {
      const uint32_t sw = s.side[tn][g];
      const float nz = (float)__builtin_bit_cast(half_t, (uint16_t)(sw >> 16)) * 65536.0f;  // -zero
      const half_t zl = (half_t)(nz - 1024.0f), zh = (half_t)(nz - 64.0f);
      z.lo[tn] = h2{zl, zl};
      z.hi[tn] = h2{zh, zh};
      if constexpr (kExact) z.scale[tn] = (float)__builtin_bit_cast(half_t, (uint16_t)(sw & 0xFFFFu));
      else z.s[tn] = bitcast_u32<h2>(__builtin_amdgcn_perm(sw, sw, 0x01000100u));
    }
    return z;
  };
  int stage = 0;
  Zero zero = zero_of(b[0], 0);  // zero-points and scales of the half the next word lies in
  h8 bf[kNT];                    // the next word, dequantised
#pragma unroll
  for (int tn = 0; tn < kNT; ++tn) bf[tn] = dequant_word<!kExact>(b[0].w[tn][0][0], zero.lo[tn], zero.hi[tn], zero.s[tn]);
  // d (the set that holds super-block sb), g and whether another super-block follows are compile-time constants at every call site
  auto half_step = [&](int sb, auto d_const, auto g_const, auto more_const) __attribute__((always_inline)) {
    constexpr int d = decltype(d_const)::value, g = decltype(g_const)::value;
    constexpr bool kMore = decltype(more_const)::value;
    const BSet& cur = b[d];
    BSet& nxt = b[d ^ 1];
    f16v half_sum[kExact ? kMT : 1][kExact ? kNT : 1];
    float scale[kNT];
    h8 af[kMT];
#pragma unroll
    for (int u = 0; u < kMT; ++u) af[u] = read_a(stage, u, 8 * lh);
    if (g == 0 || kMore) load_x(2 * sb + g + 1, stage ^ 1);
    __builtin_amdgcn_sched_barrier(0);
    if (g == 0 && kMore) load_side(nxt, sb + 1);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int t = 0; t < 8; ++t) {
      if ((t & 3) == 0 && kMore) {
        load_w(nxt, sb + 1, 2 * g + t / 4);
        __builtin_amdgcn_sched_barrier(0);
      }
      h8 an[kMT], bn_[kNT];
      if (t < 7) {
#pragma unroll
        for (int u = 0; u < kMT; ++u) an[u] = read_a(stage, u, 8 * lh + t + 1);
      }
      if (t == 7) {
        if constexpr (kExact) {
#pragma unroll
          for (int tn = 0; tn < kNT; ++tn) scale[tn] = zero.scale[tn];
        }
        if (g == 0 || kMore) zero = zero_of(g == 0 ? cur : nxt, g ^ 1);
      }
#pragma unroll
      for (int tn = 0; tn < (t < 7 || g == 0 || kMore ? kNT : 0); ++tn) {
        const uint32_t w = t < 7 ? cur.w[tn][2 * g + (t + 1) / 4][(t + 1) & 3] : (g == 0 ? cur.w[tn][2][0] : nxt.w[tn][0][0]);
        bn_[tn] = dequant_word<!kExact>(w, zero.lo[tn], zero.hi[tn], zero.s[tn]);
      }
#pragma unroll
      for (int u = 0; u < kMT; ++u)
#pragma unroll
        for (int tn = 0; tn < kNT; ++tn) {
          f16v& sum = kExact ? half_sum[u][tn] : acc[u][tn];
          if (kExact && t == 0) sum = __builtin_amdgcn_mfma_f32_32x32x16_f16(af[u], bf[tn], f16v{}, 0, 0, 0);
          else sum = __builtin_amdgcn_mfma_f32_32x32x16_f16(af[u], bf[tn], sum, 0, 0, 0);
        }
      order_word<kMT, kNT, kExact ? 9 : 13>();
#pragma unroll
      for (int u = 0; u < kMT; ++u) af[u] = an[u];
#pragma unroll
      for (int tn = 0; tn < kNT; ++tn) bf[tn] = bn_[tn];
    }
    if constexpr (kExact) {
#pragma unroll
      for (int u = 0; u < kMT; ++u)
#pragma unroll
        for (int tn = 0; tn < kNT; ++tn)
#pragma unroll
          for (int e = 0; e < 16; ++e) acc[u][tn][e] = __builtin_fmaf(scale[tn], half_sum[u][tn][e], acc[u][tn][e]);
    }
    __builtin_amdgcn_sched_barrier(0);
    wait_loads_but(std::integral_constant<int, kMore ? 2 * kNT + (g == 0 ? kNT : 0) : 0>{});
    __syncthreads();
    stage ^= 1;
  };
  auto super_block = [&](int sb, auto d_const, auto more_const) __attribute__((always_inline)) {
    half_step(sb, d_const, std::integral_constant<int, 0>{}, more_const);
    half_step(sb, d_const, std::integral_constant<int, 1>{}, more_const);
  };

  int sb = sb0;
  for (; sb + 1 < sb_end; sb += 2) {
    super_block(sb, std::integral_constant<int, 0>{}, std::true_type{});
    super_block(sb + 1, std::integral_constant<int, 1>{}, std::true_type{});
  }
  // (nothing uses what an odd last one would request: the compiler drops those loads, and a count of them would leave the activations in flight)
  if (sb < sb_end) super_block(sb, std::integral_constant<int, 0>{}, std::false_type{});
  // requests past the end that are still on their way into the stages have to land before the stages are used for anything else
  wait_loads_but(std::integral_constant<int, 0>{});

  // ---- the correction, behind the weights: 128 rank columns (two blocks of the tiled left factor) per step, the steps dealt to the K
  // groups in turn.  Its sum is taken by itself, times alpha.  (The pairs at positions 2, 3, 6, 7 of every octet of the tiled left
  // factor are stored times 16: the fragments of r are divided by 16 there.)
  if (corr) {
    const int mine = (((a.rank + 127) >> 7) + kWk - 1) / kWk;  // (both K groups run the same number: past the rank they add zeros)
    bool have_r = true;
    if constexpr (kProj) {
      // the words of the tiles that cover this workgroup's rows
      const int side = 32 * gg.front.a, per_row = (a.rank + side - 1) / side * gg.front.slices;
      have_r = wait_words(gg.front.pub, m0 / side * per_row, (min(m0 + BM, a.M) + side - 1) / side * per_row, gg.front.slices, tag, gg.front.spin);
    }
    for (int i = 0; i < mine; ++i) {
      const int st = gk + kWk * i;
      __syncthreads();  // the fragment reads of the stage are done
      if (have_r) load_r(st, 0);  // (each wave's own affair: what it fetches or computes is its rows of the stage)
      else compute_r(st, 0);
      __builtin_amdgcn_sched_barrier(0);  // (the wait below counts the loads of the left factor behind those of r)
      u32x4 lf[8];
#pragma unroll
      for (int tn = 0; tn < kNT; ++tn) {
#pragma unroll
        for (int q = 0; q < 2; ++q)
#pragma unroll
          for (int t = 0; t < 4; ++t)
            lf[4 * q + t] = __builtin_amdgcn_raw_buffer_load_b128(rs_l, w_lane + t * 1024, 2 * st + q < LB ? (int)((uint32_t)(rb[tn] * LB + 2 * st + q) * (uint32_t)tiled::kLChunk) : (int)kPast, 0);
        if (tn == 0) {
          __builtin_amdgcn_sched_barrier(0);
          wait_loads_but(std::integral_constant<int, 8>{});
          __syncthreads();
        }
        constexpr int kPair = kMT > 1 && kMT * kNT < 8 ? 2 : 1;
        if (kMT * kNT >= 8) __builtin_amdgcn_sched_barrier(0);  // (registers: nothing of the next tile may start early)
#pragma unroll
        for (int u = 0; u < kMT; u += kPair) {
          f16v c[kPair];
#pragma unroll
          for (int v = 0; v < kPair; ++v)
#pragma unroll
            for (int e = 0; e < 16; ++e) c[v][e] = 0.f;
#pragma unroll
          for (int p = 0; p < 8; ++p)
#pragma unroll
            for (int v = 0; v < kPair; ++v) {
              u32x4 f = __builtin_bit_cast(u32x4, read_a(0, u + v, 8 * (p / 4) + 4 * lh + p % 4));
              const h2 k16 = {(half_t)0.0625f, (half_t)0.0625f};
              f.y = __builtin_bit_cast(uint32_t, bitcast_u32<h2>(f.y) * k16);
              f.w = __builtin_bit_cast(uint32_t, bitcast_u32<h2>(f.w) * k16);
              c[v] = __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(h8, f), __builtin_bit_cast(h8, lf[p]), c[v], 0, 0, 0);
            }
#pragma unroll
          for (int v = 0; v < kPair; ++v)
#pragma unroll
            for (int e = 0; e < 16; ++e) acc[u + v][tn][e] = __builtin_fmaf(a.alpha, c[v][e], acc[u + v][tn][e]);
          if (kMT * kNT >= 8) __builtin_amdgcn_sched_barrier(0);
        }
      }
    }
  }

  // ---- the second K group hands its accumulators over through LDS, once every wave is done with the stages
  if constexpr (kWk > 1) {
    __syncthreads();
    float* red = reinterpret_cast<float*>(smem_all);
    if (gk == 1) {
#pragma unroll
      for (int tm = 0; tm < kMT; ++tm)
#pragma unroll
        for (int tn = 0; tn < kNT; ++tn)
#pragma unroll
          for (int i = 0; i < 16; ++i) red[((tm * kNT + tn) * 16 + i) * 256 + tid] = acc[tm][tn][i];
    }
    __syncthreads();
    if (gk == 1) return;
#pragma unroll
    for (int tm = 0; tm < kMT; ++tm)
#pragma unroll
      for (int tn = 0; tn < kNT; ++tn)
#pragma unroll
        for (int i = 0; i < 16; ++i) acc[tm][tn][i] += red[((tm * kNT + tn) * 16 + i) * 256 + tid];
  }

  // ---- epilogue: accumulator register i of a 32x32 tile is row 8*(i/4) + 4*lh + i%4, column ln ---------
  if (nslices > 1) {
    float* part = gg.partials + ((size_t)slice * part_tiles + part_tile) * (BM * BN);
#pragma unroll
    for (int tm = 0; tm < kMT; ++tm)
#pragma unroll
      for (int tn = 0; tn < kNT; ++tn)
#pragma unroll
        for (int i = 0; i < 16; ++i) part[((tm * kNT + tn) * 16 + i) * 256 + tid] = acc[tm][tn][i];
    return;
  }
  if (m0 + BM <= a.M && (bn + 1) * BN <= a.N) {
    // A tile inside the output: no test per element, and a row's address is a scalar base plus one lane offset for all of them.
    // With a test and a 64-bit address per element the 16 kMT kNT stores of a wave are some twelve instructions each, 3 to 6 us of
    // a tile that takes 50 (Qwen2.5-7B layer at 2048 rows 965 -> 928 us, 8B o_proj at 2048 rows 74.5 -> 69.5).
    YT* corner = reinterpret_cast<YT*>(a.y) + (size_t)m0 * a.ldy + (bn * BN + wave * (32 * kNT));
    const uint32_t lane_off = (uint32_t)(4 * lh) * (uint32_t)a.ldy + (uint32_t)ln;
    float b[kNT];
#pragma unroll
    for (int tn = 0; tn < kNT; ++tn) b[tn] = a.bias ? (float)a.bias[bn * BN + wave * (32 * kNT) + tn * 32 + ln] : 0.f;
#pragma unroll
    for (int tm = 0; tm < kMT; ++tm)
#pragma unroll
      for (int i = 0; i < 16; ++i) {
        YT* row = corner + (size_t)(tm * 32 + 8 * (i >> 2) + (i & 3)) * a.ldy;
#pragma unroll
        for (int tn = 0; tn < kNT; ++tn) store_y(row + tn * 32 + lane_off, acc[tm][tn][i] + b[tn]);
      }
    return;
  }
#pragma unroll
  for (int tn = 0; tn < kNT; ++tn) {
    const int n = bn * BN + wave * (32 * kNT) + tn * 32 + ln;
    if (n >= a.N) continue;
    const float b = a.bias ? (float)a.bias[n] : 0.f;
#pragma unroll
    for (int tm = 0; tm < kMT; ++tm) {
#pragma unroll
      for (int i = 0; i < 16; ++i) {
        const int m = m0 + tm * 32 + 8 * (i >> 2) + 4 * lh + (i & 3);
        if (m < a.M) store_y(reinterpret_cast<YT*>(a.y) + (size_t)m * a.ldy + n, acc[tm][tn][i] + b);
      }
    }
  }
}

// y = fp16(sum over the slices, in slice order, of the partial tiles of gemm_mfma_kernel<kMT, kNT> + bias); same grid
// in x, same workgroup -> (member, row block, column block) map and accumulator-register order as the producer.
// gridDim.y = kMT * kNT: workgroup y of a tile sums one 32 x 32 accumulator tile of each wave (a tile per workgroup
// left the sum of 64 tail tiles to 64 workgroups: 20 us for 34 MB).
template <int kMT, int kNT, typename YT>
__global__ __launch_bounds__(256) void gemm_reduce_kernel(const GemmGroup gg, const int m_blocks) {
  // uniform split: one workgroup per tile of the producer; tail split: one per tail tile (tiles full, full + 1, ...)
  const bool tail = gg.tail_slices > 1;
  const int wg = (tail ? gg.full : 0) + (int)blockIdx.x;
  const int nslices = tail ? gg.tail_slices : gg.slices;
  GemmArgs a = gg.m[0];
  int blk_base = 0;
  for (int i = 1; i < gg.n; ++i)
    if (wg >= gg.blk_end[i - 1]) {
      a = gg.m[i];
      blk_base = gg.blk_end[i - 1];
    }
  constexpr int BM = 32 * kMT, BN = 128 * kNT;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, ln = lane & 31, lh = lane >> 5;
  const int blk = wg - blk_base;
  const int m0 = (blk % m_blocks) * BM, bn = blk / m_blocks;
  const size_t slice_stride = (size_t)gridDim.x * (BM * BN);
  const float* part = gg.partials + (size_t)blockIdx.x * (BM * BN) + tid;
  const int tn = (int)blockIdx.y % kNT, tm = (int)blockIdx.y / kNT;
  {
    const int n = bn * BN + wave * (32 * kNT) + tn * 32 + ln;
    const float b = (n < a.N && a.bias) ? (float)a.bias[n] : 0.f;
    {
      float v[16];
#pragma unroll
      for (int i = 0; i < 16; ++i) v[i] = 0.f;
      for (int z = 0; z < nslices; ++z) {
#pragma unroll
        for (int i = 0; i < 16; ++i) v[i] += part[(size_t)z * slice_stride + ((tm * kNT + tn) * 16 + i) * 256];
      }
#pragma unroll
      for (int i = 0; i < 16; ++i) {
        const int m = m0 + tm * 32 + 8 * (i >> 2) + 4 * lh + (i & 3);
        if (m < a.M && n < a.N) store_y(reinterpret_cast<YT*>(a.y) + (size_t)m * a.ldy + n, v[i] + b);
      }
    }
  }
}

// ---- host side ------------------------------------------------------------------------------------
template <int kMT, int kNT, bool kQuant, bool kSuper = false, bool kTiled = false, int kWk = 1, typename YT = half_t, bool kProj = false, bool kExact = false>
static hipError_t launch_gemm_t(GemmGroup& gg, hipStream_t stream) {
  static_assert(!kTiled || (kQuant && kSuper), "the tiled copy serves the super-block form");
  static_assert(kTiled || (kWk == 1 && std::is_same_v<YT, half_t>), "K groups inside a workgroup and fp32 outputs: the tiled-copy kernel");
  constexpr int BM = 32 * kMT, BN = 128 * kNT;
  auto kern = kTiled ? gemm_tiled_kernel<kMT, kNT, kWk, YT, kProj, kExact> : gemm_mfma_kernel<kMT, kNT, kQuant, kSuper>;
  size_t lds = kTiled ? (size_t)kWk * 2 * BM * kTRow
                      : (size_t)2 * BM * kARow * sizeof(half_t) + (kSuper ? (size_t)4 * (32 * kNT) * 144 : 0);
  if (kWk > 1 && lds < (size_t)BM * BN * sizeof(float)) lds = (size_t)BM * BN * sizeof(float);  // the hand-over of the accumulators
  if constexpr (kProj) lds = std::max(lds, front_lds(gg.front));
  static LdsLimit lds_limit;
  if (hipError_t e = ensure_dynamic_lds(reinterpret_cast<const void*>(kern), lds, lds_limit); e != hipSuccess) return e;
  const int m_blocks = (gg.m[0].M + BM - 1) / BM;
  int total = 0;
  for (int i = 0; i < gg.n; ++i) {
    total += m_blocks * ((gg.m[i].N + BN - 1) / BN);
    gg.blk_end[i] = total;
  }
  if (!(kQuant && kSuper)) gg.slices = 1;
  if (!(kQuant && kSuper) || gg.slices > 1 || gg.tail_slices < 2 || gg.full < 0 || gg.full >= total) gg.tail_slices = 0;
  const int front = kProj ? gg.front.front : 0;  // (the launch record names the grid of the tiles)
  const int tail_wgs = gg.tail_slices > 1 ? gg.full + (total - gg.full) * gg.tail_slices : 0;
  note_launch(tail_wgs > 0 ? tail_wgs : total, tail_wgs > 0 ? 1 : gg.slices, 256 * kWk, "%s<%d,%d,%d%s>",
              kTiled ? "gemm_tiled_kernel" : "gemm_mfma_kernel", kMT, kNT, kWk, kExact ? ",exact" : std::is_same_v<YT, float> ? ",float" : "");
  if (tail_wgs > 0) {
    const int tail_tiles = total - gg.full;
    hipLaunchKernelGGL(kern, dim3(front + tail_wgs, 1), dim3(256 * kWk), lds, stream, gg, m_blocks);
    if (hipError_t e = hipGetLastError(); e != hipSuccess) return e;
    hipLaunchKernelGGL((gemm_reduce_kernel<kMT, kNT, YT>), dim3(tail_tiles, kMT * kNT), dim3(256), 0, stream, gg, m_blocks);
    return hipGetLastError();
  }
  hipLaunchKernelGGL(kern, kProj ? dim3(front + total * gg.slices) : dim3(total, gg.slices), dim3(256 * kWk), lds, stream, gg, m_blocks);
  if (hipError_t e = hipGetLastError(); e != hipSuccess || gg.slices == 1) return e;
  hipLaunchKernelGGL((gemm_reduce_kernel<kMT, kNT, YT>), dim3(total, kMT * kNT), dim3(256), 0, stream, gg, m_blocks);
  return hipGetLastError();
}

// What a launch of gemm_tiled_kernel takes, in us: a fit over 250 (group, rows) pairs -- 21 groups of 1.5B to 14B shapes,
// 65 to 1024 rows, with and without slices of K, 8400 timings, 7 % rms -- used to compare ways to cut one product.  The timings are those of the
// loop before its instructions were interleaved, with the correction in front; of the present one, on the cuts it picks for 24 groups at 72 to 2048
// rows with r given and without, the sums are 9 % off (rms), 4 % too short in the mean (10 % of 32-row tiles and of K groups, 2 % of the others).  A half-step
// (128 columns of K) of a tile costs `step` on the first workgroup of a compute unit and `step_more` on every further one
// (they share its matrix cores, but fill each other's waits); a split of K pays the launch that adds the slices and the
// traffic of their fp32 tiles.
struct GemmCost {
  int mt, nt, wk;
  float fixed, rank_block, step, step_more, reduce, partial_mb, output_mb;
};
constexpr GemmCost kGemmCost[] = {
    {1, 1, 1, 1.6f, 1.9f, 0.45f, 0.27f, 1.7f, 0.50f, 0.80f}, {1, 2, 1, 2.1f, 3.3f, 0.69f, 0.53f, 2.3f, 0.28f, 0.65f},
    {2, 1, 1, 2.2f, 2.1f, 0.60f, 0.39f, 1.6f, 0.37f, 0.64f}, {2, 1, 2, 2.0f, 3.0f, 0.96f, 0.88f, 2.3f, 0.34f, 0.96f},
    {2, 2, 1, 2.9f, 3.3f, 0.90f, 0.77f, 1.6f, 0.29f, 0.52f}, {4, 1, 1, 3.1f, 2.8f, 1.00f, 0.73f, 1.9f, 0.24f, 0.59f},
    {4, 2, 1, 5.0f, 4.0f, 1.43f, 1.27f, 1.1f, 0.23f, 0.58f}, {4, 2, 2, 6.0f, 5.5f, 2.46f, 3.10f, 1.3f, 0.25f, 0.92f}};

// The same for the unrounded form at 33 to 64 rows: 558 timings of 19 groups of 1B to 14B shapes at 36 and 57 rows, 6 % rms.  Of 24 groups at 33, 48
// and 64 rows, with r given and without, with a workspace and without, the cut it picks takes 1.6 % longer than the fastest of twelve in the mean,
// 19 % at most (3584 x 3584 with r given).
constexpr GemmCost kGemmExactCost[] = {{1, 1, 1, 1.9f, 1.0f, 0.43f, 0.21f, 3.1f, 0.47f, 1.63f},
                                       {2, 1, 1, 1.5f, 1.9f, 0.52f, 0.32f, 3.1f, 0.35f, 1.65f},
                                       {2, 1, 2, 4.3f, 1.1f, 0.81f, 1.03f, 2.7f, 0.35f, 1.83f}};

static int gemm_tiles(const GemmGroup& gg, int mt, int nt) {
  int cols = 0;
  for (int i = 0; i < gg.n; ++i) cols += (gg.m[i].N + 128 * nt - 1) / (128 * nt);
  return (gg.m[0].M + 32 * mt - 1) / (32 * mt) * cols;
}

// The part of a launch's cost that no cut changes needs the group; the rest needs its tiles.  (Calls from Python are often bound by
// the host: the rule looks at some forty cuts in under a microsecond.)
static float gemm_cost_fixed(const GemmGroup& gg, const GemmCost& c) {
  int rank = 0;
  float cols = 0.f;
  for (int i = 0; i < gg.n; ++i) {
    if (gg.m[i].r != nullptr) rank = gg.m[i].rank;
    cols += (float)gg.m[i].N;
  }
  return c.fixed + c.rank_block * (float)((rank + 127) / 128) + c.output_mb * cols * (float)gg.m[0].M * 2e-6f;
}

// `tail_slices` > 1: the tiles past the last multiple of the compute-unit count are cut into that many (slices is then 1)
static float gemm_cost_cut(const GemmCost& c, int tiles, int sb, int slices, int tail_slices, int num_cus) {
  const auto half_steps = [&](int s) { return (float)(2 * (((sb + s - 1) / s + c.wk - 1) / c.wk)); };
  const float tile_mb = (float)(32 * c.mt) * (128 * c.nt) * 4e-6f;
  if (tail_slices > 1)
    return half_steps(1) * (c.step + (float)(tiles / num_cus - 1) * c.step_more) + half_steps(tail_slices) * c.step_more + c.reduce +
           c.partial_mb * tile_mb * (float)(tiles % num_cus * tail_slices);
  const float us = half_steps(slices) * (c.step + (float)((tiles * slices + num_cus - 1) / num_cus - 1) * c.step_more);
  return slices > 1 ? us + c.reduce + c.partial_mb * tile_mb * (float)(tiles * slices) : us;
}

// the super-block form: addresses its operands with 32-bit byte offsets
static bool gemm_super_form(const GemmGroup& gg) {
  static const int env_super = getenv("GLOWQ_GEMM_SUPER") ? atoi(getenv("GLOWQ_GEMM_SUPER")) : 1;
  bool fits32 = (size_t)gg.m[0].M * gg.m[0].K * 2 < (1ull << 32);
  for (int i = 0; i < gg.n; ++i) {
    const size_t rows = (size_t)gg.m[i].N;
    fits32 = fits32 && rows * gg.m[i].ldw * 4 < (1ull << 32) && rows * gg.m[i].lds * 2 < (1ull << 32) && rows * gg.m[i].ldz * 4 < (1ull << 32);
  }
  return env_super != 0 && (gg.m[0].K & 255) == 0 && gg.m[0].group_size >= 128 && fits32;
}

// the tiled copy of the weights where every member brings one (and its tiled left factor where it is corrected)
static bool gemm_tiled_form(const GemmGroup& gg) {
  static const int env_tiled = getenv("GLOWQ_GEMM_TILED") ? atoi(getenv("GLOWQ_GEMM_TILED")) : 1;
  bool ok = gemm_super_form(gg) && env_tiled != 0 && tiled::applies(gg.m[0].K, gg.m[0].group_size);
  for (int i = 0; i < gg.n; ++i)
    ok = ok && gg.m[i].wt != nullptr && (gg.m[i].r == nullptr || gg.m[i].lt != nullptr) && tiled::weight_bytes(gg.m[i].N, gg.m[i].K) < (1ull << 32);
  return ok;
}

static float proj_launch_us(int M, int K, int rank, int num_cus, size_t ws_bytes);
bool proj_on_small_kernel(int M, int K, int rank);  // abi.hip

// How a launch that computes r itself cuts it, given its own cut, and what that is predicted to cost it, in us; `f.count` 0: r comes from a
// launch of its own, which is predicted to cost less (that cost, then).
//  * Tiles of 32 x 32 with K in as many slices as keep six stages each and leave one workgroup a compute unit, or tiles of 64 x 64: 0.45 and
//    0.65 us a stage of 128 columns, 1.65 times that where every compute unit has work of the launch's own as well, about 2 us at the ends, 2.5
//    for the sum of slices: measured on launches that waited for r.  What that
//    costs the launch: what its first readers wait, the places that the workgroups in front keep from others where the launch takes more
//    than one round, and some of their time where they make it more than one (with fewer slices they may not).  8B q|k|v at 100 rows, us, with one / two / four slices
//    21.9 / 20.2 / 20.1, projection in front 26.2, r given 19.6; 8B down_proj at 100 rows 64 / 43 / 34, 29.8 with sixteen, 38.1, 27.8.
//  * Where the launch's own workgroups are no more than one a compute unit and do not all find an empty one beside those in front, the
//    front is filled up to one a compute unit with workgroups that only hold their places: the others then come out one a compute unit as well.
//    Otherwise some compute units get two, and the launch takes as long as those: 8B down_proj at 333 rows 72.3 with 220 in front, 57.6
//    with 264, projection in front 67.6, r given 55.8; 14B down_proj at 512 rows 134 with 128, 106 with 256, 118, 100.
// 24 groups of 1B to 14B shapes at 72 to 2048 rows: 1.14 times as fast in the mean with the rule as with the projection in front, 1.5 % slower at most.
static float plan_front(GemmGroup& gg, const GemmCost& c, bool exact, int num_cus, float launch_us) {
  FrontArgs& f = gg.front;
  const int tiles = gemm_tiles(gg, c.mt, c.nt), sb = f.K >> 8, stages = f.K >> 7;
  const int own = gg.tail_slices > 1 ? gg.full + (tiles - gg.full) * gg.tail_slices : tiles * gg.slices;
  float best = f.any_cost ? 1e30f : launch_us;
  f.count = 0;
  for (int a = 1; a <= 2; ++a) {
    // workgroups that a compute unit holds: registers, and the LDS that the workgroups in front want (48 or 64 KB of 160)
    const int per_cu = (c.mt == 4 && c.nt == 2 && c.wk == 2) || (exact && c.wk == 2) ? 1 : (c.mt * c.nt <= 2 && c.wk == 1 && a == 1 ? 3 : 2);
    const int slots = num_cus * per_cu, held = std::min((own + num_cus - 1) / num_cus, per_cu);
    if (a == 2 && per_cu == 2 && c.mt * c.nt <= 2 && own > slots) continue;  // (with 48 KB or less there were three)
    const float readers = gemm_cost_fixed(gg, c) + (float)(2 * (((sb + gg.slices - 1) / gg.slices + c.wk - 1) / c.wk)) * (c.step + (float)(held - 1) * c.step_more);
    const long r_tiles = (long)((f.M + 32 * a - 1) / (32 * a)) * ((f.rank + 32 * a - 1) / (32 * a));
    const long room = per_cu == 1 ? num_cus - own : std::min(num_cus, kMaxFront);
    if (r_tiles > room) continue;
    const int most = a == 1 ? std::max(1, std::min({stages / 6, (int)(room / r_tiles), 16})) : 1;
    const int fitting = std::min(most, (int)((slots - own) / r_tiles));  // slices with which everything is there at once
    for (const int slices : {most, fitting}) {
      if (slices < 1) continue;
      const int count = (int)r_tiles * slices;
      const float there = 2.f + (a == 1 ? 0.45f : 0.65f) * (own > num_cus ? 1.65f : 1.f) * (float)((stages + slices - 1) / slices) + (slices > 1 ? 2.5f : 0.f);
      float us = 1.5f + std::max(0.f, 1.25f * there + 1.f - readers);  // (a late r costs far more than the rest)
      if (own > slots) us += there * (float)count / (float)slots;
      else if (own + count > slots) us += 0.37f * there;
      if (us >= best) continue;
      best = us;
      f.a = a;
      f.slices = slices;
      f.count = count;
      f.front = own <= num_cus && count + own > num_cus && per_cu > 1 ? num_cus : count;
    }
  }
  return best;
}

// Up to 64 rows in the unrounded form: one row block of 64, or up to two of 32, K cut and dealt as the costs have it.  Group launches, us, this /
// the kernel of skinny_tiled.hip with 64 rows, which it replaced (consumer and producer waves, five of them on four SIMDs on the wide groups,
// and every workgroup's x through registers): 57 rows 8B q|k|v 14.5 / 18.3, o_proj 13.0 / 16.1, gate|up 26.2 / 32.4, down_proj 20.9 / 26.5; 14B
// gate|up 42.8 / 45.4, down_proj 25.2 / 31.5; 15 groups at 33 to 64 rows 1.25 times as fast in the mean.
static hipError_t launch_gemm_exact(GemmGroup& gg, int num_cus, size_t ws_bytes, hipStream_t stream) {
  const int sb_total = gg.m[0].K >> 8;
  const bool fused = gg.front.pub != nullptr;
  // (the projection launch of these rows: 3.4 us at 32 rows, K = 4096, rank 128, 4.3 at 64 rows, 7.5 at 57 rows, K = 5120, rank 256)
  const float macs = (float)gg.m[0].M * (float)gg.m[0].K * (float)gg.front.rank;
  const float launch_us = !fused ? 0.f : proj_on_small_kernel(gg.m[0].M, gg.m[0].K, gg.front.rank) ? 2.3f + 0.065e-6f * macs : proj_launch_us(gg.m[0].M, gg.m[0].K, gg.front.rank, num_cus, ws_bytes);
  const GemmCost* best = nullptr;
  float best_us = 0.f;
  GemmGroup cut = gg;
  // of each kind of cut (tiles; all of them in slices of K, or those of the last, partly filled round) the cheapest, with what r costs it
  for (const GemmCost& c : kGemmExactCost)
    for (const bool tail_only : {false, true}) {
      const int tiles = gemm_tiles(gg, c.mt, c.nt), tail = tiles % num_cus;
      if (tail_only && (tiles < num_cus || tail == 0)) continue;
      const size_t tile_bytes = (size_t)(32 * c.mt) * (128 * c.nt) * sizeof(float);
      float us = 0.f;
      int slices = 0;
      for (int s = tail_only ? 2 : 1; s <= 16 && s * 2 <= std::max(sb_total, 2); ++s) {
        const int per = (sb_total + s - 1) / s, cut_tiles = tail_only ? tail : tiles;
        if ((sb_total + per - 1) / per != s) continue;  // a slice without super-blocks
        if (s > 1 && (cut_tiles * s > (tail_only ? 1 : 3) * num_cus || (size_t)cut_tiles * s * tile_bytes > std::min(ws_bytes, (size_t)32 << 20))) break;
        const float t = gemm_cost_cut(c, tiles, sb_total, tail_only ? 1 : s, tail_only ? s : 0, num_cus);
        if (slices != 0 && t >= us) continue;
        us = t;
        slices = s;
      }
      if (slices == 0) continue;
      cut.slices = tail_only ? 1 : slices;
      cut.tail_slices = tail_only ? slices : 0;
      cut.full = tail_only ? tiles - tail : 0;
      us += gemm_cost_fixed(gg, c);
      if (fused) us += plan_front(cut, c, true, num_cus, launch_us);
      if (best != nullptr && us >= best_us) continue;
      best = &c;
      best_us = us;
      gg.slices = cut.slices;
      gg.tail_slices = cut.tail_slices;
      gg.full = cut.full;
      gg.front = cut.front;
    }
  if (fused && gg.front.count == 0) return hipErrorNotReady;
#define GLOWQ_GEMM_EXACT_CASE(MT, WK)                    \
  if (best->mt == MT && best->nt == 1 && best->wk == WK) \
    return fused ? launch_gemm_t<MT, 1, true, true, true, WK, half_t, true, true>(gg, stream) : launch_gemm_t<MT, 1, true, true, true, WK, half_t, false, true>(gg, stream);
  GLOWQ_GEMM_EXACT_CASE(1, 1) GLOWQ_GEMM_EXACT_CASE(2, 1) GLOWQ_GEMM_EXACT_CASE(2, 2)
#undef GLOWQ_GEMM_EXACT_CASE
  return hipErrorInvalidValue;
}

static hipError_t launch_gemm_group(GemmGroup& gg, int num_cus, size_t ws_bytes, bool y32, hipStream_t stream) {
  // Tile choice: the largest tile (most reuse of both operands) whose workgroup count still fills the chip; when
  // none does, the one with the most workgroups.  Row tiles are capped by M (and at 4: 8 spills), column tiles at
  // 2 per wave unless every member is narrow.
  int n_max = 0;
  for (int i = 0; i < gg.n; ++i) n_max = gg.m[i].N > n_max ? gg.m[i].N : n_max;
  const int nt_cap = n_max > 128 ? 2 : 1;
  const int M = gg.m[0].M;
  static const int mt_max = getenv("GLOWQ_GEMM_MT") ? atoi(getenv("GLOWQ_GEMM_MT")) : 4;
  int mt_cap = M > 128 ? 8 : (M > 64 ? 4 : (M > 32 ? 2 : 1));
  if (mt_cap > mt_max) mt_cap = mt_max;
  if (y32 && mt_cap > 4) mt_cap = 4;  // (256-row tiles are there for measurements, on the canonical buffers, which have no fp32 outputs)
  static const int order[6][2] = {{4, 2}, {2, 2}, {4, 1}, {2, 1}, {1, 2}, {1, 1}};
  int mt = 1, nt = 1;
  long best = -1;
  for (int c = 0; c < 6; ++c) {
    const int cmt = order[c][0], cnt = order[c][1];
    if (cmt > mt_cap || cnt > nt_cap) continue;
    long wgs = 0;
    for (int i = 0; i < gg.n; ++i) wgs += (long)((M + 32 * cmt - 1) / (32 * cmt)) * ((gg.m[i].N + 128 * cnt - 1) / (128 * cnt));
    if (wgs >= num_cus) {
      mt = cmt;
      nt = cnt;
      break;
    }
    if (wgs > best) {
      best = wgs;
      mt = cmt;
      nt = cnt;
    }
  }
  if (mt_cap == 8 && mt == 4 && mt_max >= 8) mt = 8;
  static const int force_mt = getenv("GLOWQ_GEMM_FORCE_MT") ? atoi(getenv("GLOWQ_GEMM_FORCE_MT")) : 0;
  static const int force_nt = getenv("GLOWQ_GEMM_FORCE_NT") ? atoi(getenv("GLOWQ_GEMM_FORCE_NT")) : 0;
  if (force_mt > 0 && force_mt <= mt_cap) mt = force_mt;
  if (force_nt > 0 && force_nt <= nt_cap) nt = force_nt;
  const bool super = gemm_super_form(gg);
  const bool tiled_ok = gemm_tiled_form(gg);
  // About one 128 x 256 tile per compute unit and a long K (where K would otherwise be cut into slices over workgroups,
  // with fp32 partial tiles through the workspace and a second launch for their sum): eight waves per tile, the K range
  // dealt to two groups of four inside the workgroup (gemm_tiled_kernel's kWk = 2), the sum in LDS.  Qwen2.5-7B down_proj at
  // 2048 rows (K = 18944, 224 tiles): 308 -> 294 us.  On short K it does not pay: o_proj (K = 3584, 224 tiles) 77.5 -> 78.6 us
  // against two co-resident 64 x 256 workgroups per compute unit, q|k|v (288 tiles) 100.6 -> 114.9 (its tail tiles, cut
  // along K, no longer fit beside a whole tile).
  static const int env_wk = getenv("GLOWQ_GEMM_WK") ? atoi(getenv("GLOWQ_GEMM_WK")) : 0;
  int wk = 1;
  if (tiled_ok && mt_cap >= 4 && nt_cap == 2 && env_wk != 1) {
    long tiles42 = 0;
    for (int i = 0; i < gg.n; ++i) tiles42 += (long)((M + 127) / 128) * ((gg.m[i].N + 255) / 256);
    if ((tiles42 * 2 >= num_cus && tiles42 < 2L * num_cus && (gg.m[0].K >> 8) >= 32) || env_wk == 2) {
      mt = 4;
      nt = 2;
      wk = 2;
    }
  }
  // Split K through the workspace: where even the largest tile the rows allow leaves CUs idle, that tile is kept and K
  // is cut into slices of at least sixteen super-blocks until the workgroups number about two per CU.
  static const int env_split = getenv("GLOWQ_GEMM_SPLIT") ? atoi(getenv("GLOWQ_GEMM_SPLIT")) : 1;
  const int ws_slices_fit = gg.slices;  // on entry: how many slices of the whole output the workspace holds
  gg.slices = 1;
  if (super && env_split != 0 && ws_slices_fit >= 2 && mt_cap >= 2 && nt_cap == 2 && wk == 1) {
    const int bmt = mt_cap >= 4 ? 4 : 2;
    long tiles = 0;
    for (int i = 0; i < gg.n; ++i) tiles += (long)((M + 32 * bmt - 1) / (32 * bmt)) * ((gg.m[i].N + 255) / 256);
    const int sb_total = gg.m[0].K >> 8;
    long want = (2L * num_cus) / tiles;
    // every slice writes the whole output once more in fp32, the reduction reads it back, and a short K loop is mostly
    // ramp: only slices of 16 super-blocks and more pay (measured: 2048 x 3584 outputs gain 8 % at K = 18944 in two
    // slices and lose 12 % at K = 3584; 128..512 rows of K = 4096 lose up to 40 % in slices of four super-blocks)
    // ... unless the output has so few tiles that most of the chip would otherwise sit idle for the whole of a long K
    // (4096 outputs of K = 14336 at 65..256 rows: 16 to 32 tiles, 97 -> 75..80 us with slices of four to eight)
    static const int env_depth = getenv("GLOWQ_GEMM_MIN_DEPTH") ? atoi(getenv("GLOWQ_GEMM_MIN_DEPTH")) : 0;
    const long min_depth = env_depth > 0 ? env_depth : (tiles >= 64 ? 16 : (tiles >= 32 ? 8 : 4));
    if (want > sb_total / min_depth) want = sb_total / min_depth;
    if (want > ws_slices_fit) want = ws_slices_fit;
    if (tiles < num_cus && want >= 2 && tiles * want * 2 >= num_cus) {
      mt = bmt;
      nt = 2;
      gg.slices = (int)want;
    }
  }
  // Tail split: the tiles beyond the last multiple of the CU count are cut along K so that the work they add is spread
  // over the whole chip (2368 tiles on 256 CUs: 9.25 tiles' worth of time instead of 10; 288 tiles: 1.125 instead of 2).
  // Only where that tail is at most 0.6 of a round, K leaves every slice two super-blocks or more, and the workspace
  // holds the partial tiles.
  static const int env_tail = getenv("GLOWQ_GEMM_TAIL") ? atoi(getenv("GLOWQ_GEMM_TAIL")) : 1;
  gg.full = 0;
  gg.tail_slices = 0;
  if (super && env_tail != 0 && gg.slices == 1 && ws_bytes > 0) {
    long tiles = 0;
    for (int i = 0; i < gg.n; ++i) tiles += (long)((M + 32 * mt - 1) / (32 * mt)) * ((gg.m[i].N + 128 * nt - 1) / (128 * nt));
    const long tail = tiles % num_cus;
    const int sb_total = gg.m[0].K >> 8;
    // (measured at 2048 rows, projection launch included: 2368 tiles 590 -> 573 us, 288 tiles 119 -> 107 us)
    if (tiles > num_cus && tail > 0 && tail * 10 <= (long)num_cus * 6) {
      long s_want = num_cus / tail;
      if (s_want > 8) s_want = 8;
      if (s_want > sb_total / 2) s_want = sb_total / 2;
      const size_t tile_bytes = (size_t)(32 * mt) * (128 * nt) * sizeof(float);
      while (s_want >= 2 && (size_t)tail * s_want * tile_bytes > ws_bytes) --s_want;
      if (s_want >= 2) {
        // (slices of equal depth: no more of them than leave none empty)
        const int per = (sb_total + (int)s_want - 1) / (int)s_want;
        gg.tail_slices = (sb_total + per - 1) / per;
        gg.full = (int)(tiles - tail);
      }
    }
  }
  // From 65 rows on the tiled copy the cut above stands unless another one is predicted 9 % faster: the choice above fills the
  // chip with tiles first and cuts K only where that leaves most of it idle, but up to about a thousand rows one round of
  // workgroups made of smaller tiles and slices of K is often the shorter way (8B o_proj at 100 rows 18.4 -> 15.1 us, down_proj
  // 35.7 -> 30.5, 14B q|k|v 31.6 -> 25.3, 14B down_proj at 512 rows 123 -> 108).  With and without this rule, 21 groups of 1.5B
  // to 14B shapes at 12 row counts: 82 of 189 pairs at 72 to 1024 rows get another cut, 1.25 times as fast in the mean and the
  // least of them 1.5 % faster; of 63 pairs at 1200 to 2048 rows, past the rows of the fit, 6 do (1.05 to 1.19 times).
  // Without the margin the rule costs more than 1 % on 30 pairs of the fit (all of these timed with the loop that the costs were fitted to).  Cuts that send more than 32 MB of fp32 tiles through
  // the workspace are not tried: from there the fit scatters by 7 to 11 % (standard deviation) instead of 3 to 5.
  if (tiled_ok && mt_cap >= 4 && nt_cap == 2 && force_mt == 0 && force_nt == 0 && env_wk == 0) {
    const int sb_total = gg.m[0].K >> 8;
    float best_us = 0.f;
    for (const GemmCost& c : kGemmCost)
      if (c.mt == mt && c.nt == nt && c.wk == wk)
        best_us = 0.91f * (gemm_cost_fixed(gg, c) + gemm_cost_cut(c, gemm_tiles(gg, mt, nt), sb_total, gg.slices, gg.tail_slices, num_cus));
    // a second launch where there was none also takes the host's time, which calls from Python at the small end wait for
    const float second = gg.slices > 1 || gg.tail_slices > 1 ? 0.f : 1.5f;
    for (const GemmCost& c : kGemmCost) {
      if (!((c.nt == 1 && c.mt <= 2) || (c.mt == 4 && c.nt == 2 && c.wk == 1))) continue;  // <1,1,1>, <2,1,1>, <2,1,2>, <4,2,1>
      const int tiles = gemm_tiles(gg, c.mt, c.nt);
      const float fixed = gemm_cost_fixed(gg, c);
      if (tiles > 64 * num_cus) continue;
      for (int s = 1; s <= 16 && s * 2 <= std::max(sb_total, 2); ++s) {  // two super-blocks and more to a slice, three rounds at most
        const size_t partial_bytes = (size_t)(tiles * s) * (32 * c.mt) * (128 * c.nt) * sizeof(float);
        if (s > 1 && (env_split == 0 || tiles * s > 3 * num_cus || partial_bytes > std::min(ws_bytes, (size_t)32 << 20))) break;
        const int per = (sb_total + s - 1) / s;
        if ((sb_total + per - 1) / per != s) continue;  // a slice without super-blocks
        const float us = fixed + gemm_cost_cut(c, tiles, sb_total, s, 0, num_cus) + (s > 1 ? second : 0.f);
        if (us >= best_us) continue;
        best_us = us;
        mt = c.mt;
        nt = c.nt;
        wk = c.wk;
        gg.slices = s;
        gg.full = gg.tail_slices = 0;
      }
    }
  }
  if (gg.front.pub != nullptr) {
    bool planned = false;
    for (const GemmCost& c : kGemmCost)
      if (tiled_ok && c.mt == mt && c.nt == nt && c.wk == wk) {
        plan_front(gg, c, false, num_cus, proj_launch_us(M, gg.m[0].K, gg.front.rank, num_cus, ws_bytes));
        planned = gg.front.count > 0;
      }
    if (!planned) return hipErrorNotReady;
  }
#define GLOWQ_GEMM_TILED_CASE(MT, NT, WK)                                                  \
  if (tiled_ok && mt == MT && nt == NT && wk == WK) {                                      \
    if (gg.front.pub != nullptr)                                                           \
      return y32 ? launch_gemm_t<MT, NT, true, true, true, WK, float, true>(gg, stream) : launch_gemm_t<MT, NT, true, true, true, WK, half_t, true>(gg, stream); \
    return y32 ? launch_gemm_t<MT, NT, true, true, true, WK, float>(gg, stream) : launch_gemm_t<MT, NT, true, true, true, WK>(gg, stream); \
  }
  GLOWQ_GEMM_TILED_CASE(4, 2, 1) GLOWQ_GEMM_TILED_CASE(2, 2, 1) GLOWQ_GEMM_TILED_CASE(1, 2, 1) GLOWQ_GEMM_TILED_CASE(4, 1, 1)
  GLOWQ_GEMM_TILED_CASE(2, 1, 1) GLOWQ_GEMM_TILED_CASE(1, 1, 1) GLOWQ_GEMM_TILED_CASE(4, 2, 2) GLOWQ_GEMM_TILED_CASE(2, 1, 2)
#undef GLOWQ_GEMM_TILED_CASE
  if (y32) return hipErrorInvalidValue;  // (gemm_widens said no)
#define GLOWQ_GEMM_CASE(MT, NT)                                                            \
  if (mt == MT && nt == NT) return super ? launch_gemm_t<MT, NT, true, true>(gg, stream) : launch_gemm_t<MT, NT, true>(gg, stream);
  GLOWQ_GEMM_CASE(8, 2) GLOWQ_GEMM_CASE(4, 2) GLOWQ_GEMM_CASE(2, 2) GLOWQ_GEMM_CASE(1, 2)
  GLOWQ_GEMM_CASE(8, 1) GLOWQ_GEMM_CASE(4, 1) GLOWQ_GEMM_CASE(2, 1) GLOWQ_GEMM_CASE(1, 1)
#undef GLOWQ_GEMM_CASE
  return hipErrorInvalidValue;
}

// The MFMA route needs 64-deep k blocks that stay inside one quantisation group per 32-column half and
// 16-byte aligned rows everywhere.
bool gemm_supported(const GroupDev& g) {
  if ((g.K % kBK) != 0 || (g.group_size % 32) != 0 || (g.group_size & (g.group_size - 1)) != 0) return false;
  // r is either given or still to be produced from R into r_out by the projection launch that goes ahead
  const half_t* r = g.r != nullptr ? g.r : (g.R != nullptr ? g.r_out : nullptr);
  if (r != nullptr && ((g.rank & 7) != 0 || g.rank < 8)) return false;
  if ((reinterpret_cast<uintptr_t>(g.x) & 15u) != 0) return false;
  if (r != nullptr && (reinterpret_cast<uintptr_t>(r) & 15u) != 0) return false;
  for (int i = 0; i < g.n_members; ++i) {
    const MemberDev& m = g.mem[i];
    if ((reinterpret_cast<uintptr_t>(m.qweight) & 15u) != 0 || (m.ldw & 3) != 0) return false;
    if (m.L != nullptr && (reinterpret_cast<uintptr_t>(m.L) & 15u) != 0) return false;
  }
  return true;
}

static void fill_gemm_group(const GroupDev& g, GemmGroup& gg) {
  gg.n = g.n_members;
  for (int i = 0; i < g.n_members; ++i) {
    const MemberDev& m = g.mem[i];
    GemmArgs& a = gg.m[i];
    a.x = g.x;
    a.r = (m.L != nullptr) ? (g.r != nullptr ? g.r : g.r_out) : nullptr;  // (given, or produced by the launch ahead)
    a.qweight = m.qweight;
    a.scales = m.scales;
    a.qzeros = m.qzeros;
    a.bmat = m.L;
    a.bias = m.bias;
    a.y = m.y;
    a.wt = static_cast<const unsigned char*>(m.tiled);
    a.lt = (m.L != nullptr && m.tiled_L != nullptr && m.tiled_rank == g.rank) ? static_cast<const unsigned char*>(m.tiled_L) : nullptr;
    a.M = g.M;
    a.N = m.N;
    a.K = g.K;
    a.group_size = g.group_size;
    a.rank = g.rank;
    a.ldw = m.ldw;
    a.lds = m.lds;
    a.ldz = m.ldz;
    a.ldb = g.rank;
    a.ldy = m.ldy;
    a.alpha = g.alpha;
  }
}

// whether a call can have fp32 outputs: the kernels on the tiled copy have them
bool gemm_widens(const GroupDev& g) {
  GemmGroup gg;
  fill_gemm_group(g, gg);
  for (int i = 1; i < g.n_members; ++i)
    if ((g.mem[i].y32 != 0) != (g.mem[0].y32 != 0)) return false;
  return gemm_supported(g) && gemm_tiled_form(gg);
}

size_t gemm_handover_bytes() { return kGemmHandoverBytes; }

hipError_t launch_gemm(GroupDev& g, int num_cus, hipStream_t stream, bool exact) {
  GemmGroup gg;
  fill_gemm_group(g, gg);
  // slices of the padded output (rows to a multiple of 128, columns of every member to a multiple of 256) that fit the
  // workspace; launch_gemm_group turns this into the slice count
  size_t padded = 0;
  for (int i = 0; i < g.n_members; ++i) padded += (size_t)((g.M + 127) / 128 * 128) * ((g.mem[i].N + 255) / 256 * 256);
  // a launch that computes r itself (run_group set g.pub) keeps its words in front of the partial tiles
  const bool ws_ok = g.ws != nullptr && (reinterpret_cast<uintptr_t>(g.ws) & 15u) == 0;
  const size_t words = g.pub != nullptr ? kGemmHandoverBytes : 0, ws_bytes = ws_ok && g.ws_bytes > words ? g.ws_bytes - words : 0;
  gg.slices = (int)std::min<size_t>(ws_bytes / (padded * sizeof(float)), 64);
  gg.partials = reinterpret_cast<float*>(static_cast<unsigned char*>(g.ws) + words);
  gg.front = FrontArgs{g.x, g.R, g.r_out, g.pub, nullptr, g.M, g.K, g.rank, 0, 0, 1, 1, g.pub_mute ? kNeverRaised : g.pub_spin, g.pub_any_cost};
  gg.front.partials = gg.partials == nullptr ? nullptr : reinterpret_cast<float*>(static_cast<unsigned char*>(g.ws) + kGemmWordBytes);
  if (exact) return launch_gemm_exact(gg, num_cus, ws_bytes, stream);
  return launch_gemm_group(gg, num_cus, ws_bytes, g.mem[0].y32 != 0, stream);
}

// ---- shared projection for many rows: r[M, rank] = fp16(x[M, K] . R[rank, K]^T) ---------------------------
// N = rank is tiny, so the parallelism has to come from M and K: a workgroup owns 32 rows of x and up to 128
// columns of r, and its four waves split K -- wave w takes the 64-deep slice w of every 256-deep block, with
// its own A fragments (x, staged in LDS for all four slices at once) and its own B fragments (R, straight
// from global memory, prefetched one block ahead).  There is no barrier-bound dependency between the waves
// inside a block beyond the staging of x; the four partial tiles meet in LDS once, at the end.
constexpr int kPK = 256;           // k depth of one block (4 waves x 64)
constexpr int kPRow = kPK + 8;     // padded LDS row in halves

//
// Split K (gridDim.z > 1): workgroup z of a tile takes a contiguous range of blocks and leaves its fp32 partial tile
// in the caller's workspace, [tile][slice][kNT * 1024] floats in accumulator-register order; proj_reduce_kernel then
// adds the partials in slice order and writes r.  (Finishing a tile in the workgroup that arrives last at a counter
// was measured first: the device-scope traffic it needs inside one launch costs 20 us and more, a second launch 4.)
struct ProjSplit {
  float* partials;
};

template <int kNT>
__global__ __launch_bounds__(256) void proj_mfma_kernel(const half_t* __restrict__ x, const half_t* __restrict__ R,
                                                        half_t* __restrict__ r, int M, int K, int rank, ProjSplit sp) {
  extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
  half_t* lds_x = reinterpret_cast<half_t*>(smem);  // [2][32][kPRow]; reused for the final reduction
  constexpr size_t kLdsX = (size_t)2 * 32 * kPRow * sizeof(half_t), kLdsRed = (size_t)4 * kNT * 16 * 64 * 4;
  constexpr size_t b_tile_offset = kLdsX > kLdsRed ? kLdsX : kLdsRed;  // the waves' B tiles lie behind both
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = tid >> 6;
  const int ln = lane & 31, lh = lane >> 5;
  const int m0 = blockIdx.x * 32;
  const int n0 = blockIdx.y * (32 * kNT);
  const int all_blocks = (K + kPK - 1) / kPK;  // K is a multiple of 64; the last block may be partial
  const int slices = gridDim.z;
  const int per_slice = (all_blocks + slices - 1) / slices;
  const int blk_begin = min((int)blockIdx.z * per_slice, all_blocks);
  const int blocks = min(blk_begin + per_slice, all_blocks);  // this workgroup walks blocks [blk_begin, blocks)

  f16v acc[kNT];
#pragma unroll
  for (int tn = 0; tn < kNT; ++tn)
#pragma unroll
    for (int i = 0; i < 16; ++i) acc[tn][i] = 0.f;

  // x tile of a block: 32 rows x 32 octets; thread t takes octets t, t+256, t+512, t+768
  struct XRegs {
    u32x4 v[4];
  };
  auto load_x = [&](int kb, XRegs& xr) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int q = tid + 256 * i;
      const int row = min(m0 + (q >> 5), M - 1);
      const int k = min(kb + (q & 31) * 8, K - 8);
      xr.v[i] = *reinterpret_cast<const u32x4*>(x + (size_t)row * K + k);
    }
  };
  auto store_x = [&](int stage, const XRegs& xr) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int q = tid + 256 * i;
      *reinterpret_cast<u32x4*>(lds_x + ((size_t)stage * 32 + (q >> 5)) * kPRow + (q & 31) * 8) = xr.v[i];
    }
  };
  // R reaches the B operand through a wave-private LDS tile: the wave's 128-byte row segments (its 64-column slice of
  // 32 kNT rows of R) are loaded in memory order, 8 lanes per segment, and read back in MFMA lane order.  Fragment
  // loads straight from memory put every lane of a request on a line of its own.
  constexpr int kSeg = 144;  // bytes per row segment in the tile: 128 + 16, conflict-free fragment reads
  unsigned char* btile = smem + b_tile_offset + (size_t)wave * (32 * kNT) * kSeg;
  struct BRegs {
    u32x4 w[kNT * 4];  // row 8 q + lane / 8 of the tile, piece lane % 8
  };
  // this wave's slice of a block: columns kb + 64*wave .. +63; a slice past the end of K is weighted by zero
  auto load_b = [&](int kb, BRegs& br) {
    const int ks = min(kb + 64 * wave, K - 64);
#pragma unroll
    for (int q = 0; q < kNT * 4; ++q)
      br.w[q] = *reinterpret_cast<const u32x4*>(R + (size_t)min(n0 + q * 8 + (lane >> 3), rank - 1) * K + ks + (lane & 7) * 8);
  };
  auto stage_b = [&](const BRegs& br) {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");  // fragment reads of the previous block are done
    __builtin_amdgcn_wave_barrier();
#pragma unroll
    for (int q = 0; q < kNT * 4; ++q)
      *reinterpret_cast<u32x4*>(btile + (q * 8 + (lane >> 3)) * kSeg + (lane & 7) * 16) = br.w[q];
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
  };
  auto mma_block = [&](int stage, int kb) {
    if (kb + 64 * wave >= K) return;  // wave-uniform: nothing of this slice lies inside K
#pragma unroll
    for (int t = 0; t < 4; ++t) {
      const h8 af = *reinterpret_cast<const h8*>(lds_x + ((size_t)stage * 32 + ln) * kPRow + 64 * wave + (4 * lh + t) * 8);
#pragma unroll
      for (int tn = 0; tn < kNT; ++tn) {
        const h8 bf = *reinterpret_cast<const h8*>(btile + (tn * 32 + ln) * kSeg + lh * 64 + t * 16);
        acc[tn] = __builtin_amdgcn_mfma_f32_32x32x16_f16(af, bf, acc[tn], 0, 0, 0);
      }
    }
  };

  int stage = 0;
  // Block s: move B(s) out of its register set into the wave's LDS tile, refill that set with B(s+2) and the matching x set with
  // x(s+2), run the MFMAs of block s on LDS stage s%2, then move x(s+1) (loaded one block ago) into the other
  // stage.  Two blocks of loads are in flight at any time.
  auto block = [&](int blk, BRegs& br, XRegs& x_fill, const XRegs& x_store) {
    stage_b(br);
    const int kn = min(blk + 2, all_blocks - 1) * kPK;
    load_b(kn, br);
    load_x(kn, x_fill);
    mma_block(stage, blk * kPK);
    store_x(stage ^ 1, x_store);
    __syncthreads();
    stage ^= 1;
  };
  XRegs x0, x1;
  BRegs b0, b1;
  load_x(min(blk_begin, all_blocks - 1) * kPK, x0);
  load_b(min(blk_begin, all_blocks - 1) * kPK, b0);
  load_x(min(blk_begin + 1, all_blocks - 1) * kPK, x1);
  load_b(min(blk_begin + 1, all_blocks - 1) * kPK, b1);
  store_x(0, x0);
  __syncthreads();
  for (int blk = blk_begin; blk < blocks; blk += 2) {
    block(blk, b0, x0, x1);
    if (blk + 1 >= blocks) break;
    block(blk + 1, b1, x1, x0);
  }

  // the four K slices meet in LDS: [wave][tile][16 regs][64 lanes] floats
  float* red = reinterpret_cast<float*>(smem);
  __syncthreads();
#pragma unroll
  for (int tn = 0; tn < kNT; ++tn)
#pragma unroll
    for (int i = 0; i < 16; ++i) red[((wave * kNT + tn) * 16 + i) * 64 + lane] = acc[tn][i];
  __syncthreads();
  // wave w finishes registers 4w .. 4w+3 of every tile
#pragma unroll
  for (int tn = 0; tn < kNT; ++tn) {
    const int n = n0 + tn * 32 + ln;
#pragma unroll
    for (int ii = 0; ii < 4; ++ii) {
      const int i = wave * 4 + ii;
      float v = 0.f;
#pragma unroll
      for (int w = 0; w < 4; ++w) v += red[((w * kNT + tn) * 16 + i) * 64 + lane];
      if (slices == 1) {
        const int m = m0 + 8 * (i >> 2) + 4 * lh + (i & 3);
        if (m < M && n < rank) r[(size_t)m * rank + n] = (half_t)v;
      } else {
        const size_t tile = (size_t)blockIdx.y * gridDim.x + blockIdx.x;
        sp.partials[(tile * slices + blockIdx.z) * (kNT * 1024) + (tn * 16 + i) * 64 + lane] = v;
      }
    }
  }
}

// r[m, n] = fp16(sum over the slices, in slice order, of the partial tiles of proj_mfma_kernel<kNT>).  One thread per
// accumulator element of a tile; m_blocks = gridDim.x of the producing launch.
__global__ __launch_bounds__(256) void proj_reduce_kernel(const float* __restrict__ partials, half_t* __restrict__ r, int M,
                                                          int rank, int nt, int slices, int m_blocks) {
  const int per_tile = nt * 1024;
  const int e = blockIdx.x * blockDim.x + threadIdx.x;  // element of the tile: (tn * 16 + i) * 64 + lane
  const int tile = blockIdx.y;
  if (e >= per_tile) return;
  const int lane = e & 63, i = (e >> 6) & 15, tn = e >> 10;
  const int m = (tile % m_blocks) * 32 + 8 * (i >> 2) + 4 * (lane >> 5) + (i & 3);
  const int n = (tile / m_blocks) * (32 * nt) + tn * 32 + (lane & 31);
  const float* src = partials + (size_t)tile * slices * per_tile + e;
  float v = 0.f;
  int z = 0;
  for (; z + 8 <= slices; z += 8) {
    float t[8];
#pragma unroll
    for (int u = 0; u < 8; ++u) t[u] = src[(size_t)(z + u) * per_tile];
#pragma unroll
    for (int u = 0; u < 8; ++u) v += t[u];
  }
  for (; z < slices; ++z) v += src[(size_t)z * per_tile];
  if (m < M && n < rank) r[(size_t)m * rank + n] = (half_t)v;
}

// ---- shared projection of many rows: tiles of 64 x 64 or 128 x 128, both operands through LDS --------------------
// proj_mfma_kernel's 32-row tiles read R once per 32 rows and x once per 32 or 64 columns, 16 or 8 products for every element
// that a compute unit pulls in, two blocks in flight.  Here a workgroup of four waves (two by two) takes 64 kA rows of x and 64 kB rows
// of R in stages of 128 columns that go from memory straight into LDS (kSt stages in a ring, swizzled like the activations of
// gemm_tiled_kernel: slot c' of row q holds the row's 16-byte piece c' ^ (q % 16)), and K is cut over gridDim.z workgroups
// whose fp32 tiles [slice][M][rank] meet in proj_sum_kernel, in slice order.
template <int kA>
__global__ __launch_bounds__(256) void proj_tile_kernel(const half_t* __restrict__ x, const half_t* __restrict__ R, half_t* __restrict__ r,
                                                        float* __restrict__ partials, int M, int K, int rank) {
  extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
  constexpr int kB = kA, kSt = 2;  // (three and four stages: never in flight, the barrier's wait is for all loads to LDS; a second workgroup of a compute unit fills the waits)
  constexpr int BM = 64 * kA, BN = 64 * kB;
  constexpr int kStage = (BM + BN) * kTRow;
  constexpr int kLoads = (BM + BN) / 16;  // 16-byte loads of a thread per stage
  const int tid = (int)threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int ln = lane & 31, lh = lane >> 5;
  const int m0 = (int)blockIdx.x * BM, n0 = (int)blockIdx.y * BN;
  const int all = K >> 7, per = (all + (int)gridDim.z - 1) / (int)gridDim.z;
  const int first = min((int)blockIdx.z * per, all), n = min(per, all - first);  // this workgroup's stages
  const auto rsrc = [](const void* p, size_t bytes) {
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(p), 0, (int)(uint32_t)bytes, 0x00020000);
  };
  const __amdgpu_buffer_rsrc_t rs_x = rsrc(x, (size_t)M * K * 2), rs_r = rsrc(R, (size_t)rank * K * 2);
  const int srow = tid >> 4, spiece = (tid & 15) ^ srow;
  uint32_t off[kLoads];
#pragma unroll
  for (int q = 0; q < kLoads; ++q) {
    const int row = q < BM / 16 ? min(m0 + 16 * q + srow, M - 1) : min(n0 + 16 * (q - BM / 16) + srow, rank - 1);  // past the end: dropped results
    off[q] = ((uint32_t)row * (uint32_t)K + (uint32_t)spiece * 8u) * 2u;
  }
  auto request = [&](int st) __attribute__((always_inline)) {
    typedef __attribute__((address_space(3))) void* lds_ptr_t;
    unsigned char* dst = smem + (size_t)(st % kSt) * kStage + 4 * wave * kTRow;
#pragma unroll
    for (int q = 0; q < kLoads; ++q)
      __builtin_amdgcn_raw_ptr_buffer_load_lds(q < BM / 16 ? rs_x : rs_r, (lds_ptr_t)(dst + 16 * q * kTRow), 16, (int)off[q], (first + st) * 256, 0, 0);
  };
  f16v acc[kA][kB];
#pragma unroll
  for (int a = 0; a < kA; ++a)
#pragma unroll
    for (int b = 0; b < kB; ++b)
#pragma unroll
      for (int i = 0; i < 16; ++i) acc[a][b][i] = 0.f;
#pragma unroll
  for (int st = 0; st < kSt - 1; ++st)
    if (st < n) request(st);
  const int wr = (wave >> 1) * (32 * kA), wc = (wave & 1) * (32 * kB);
  for (int st = 0; st < n; ++st) {
    __builtin_amdgcn_s_waitcnt(0x0F70);  // vmcnt(0): this wave's part of stage st has landed, behind the barrier everybody's
    __syncthreads();
    if (st + kSt - 1 < n) request(st + kSt - 1);  // into the stage that everybody is done with
    const unsigned char* base = smem + (size_t)(st % kSt) * kStage;
#pragma unroll
    for (int t = 0; t < 8; ++t) {
      const int slot = ((2 * t + lh) ^ (ln & 15)) << 4;
      h8 af[kA], bf[kB];
#pragma unroll
      for (int a = 0; a < kA; ++a) af[a] = *reinterpret_cast<const h8*>(base + (wr + 32 * a + ln) * kTRow + slot);
#pragma unroll
      for (int b = 0; b < kB; ++b) bf[b] = *reinterpret_cast<const h8*>(base + (BM + wc + 32 * b + ln) * kTRow + slot);
#pragma unroll
      for (int a = 0; a < kA; ++a)
#pragma unroll
        for (int b = 0; b < kB; ++b) acc[a][b] = __builtin_amdgcn_mfma_f32_32x32x16_f16(af[a], bf[b], acc[a][b], 0, 0, 0);
    }
  }
#pragma unroll
  for (int a = 0; a < kA; ++a)
#pragma unroll
    for (int b = 0; b < kB; ++b) {
      const int col = n0 + wc + 32 * b + ln;
#pragma unroll
      for (int i = 0; i < 16; ++i) {
        const int m = m0 + wr + 32 * a + 8 * (i >> 2) + 4 * lh + (i & 3);
        if (m >= M || col >= rank) continue;
        if (gridDim.z == 1) r[(size_t)m * rank + col] = (half_t)acc[a][b][i];
        else partials[((size_t)blockIdx.z * M + m) * rank + col] = acc[a][b][i];
      }
    }
}

// r = fp16(sum of the slices in slice order); four elements to a thread, one wave to a workgroup (rank 128 at 100 rows: 50
// of them, rank 256 at 1500 rows: 1500)
__global__ __launch_bounds__(64) void proj_sum_kernel(const float* __restrict__ partials, half_t* __restrict__ r, long n4, int slices) {
  const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n4) return;
  const f4* src = reinterpret_cast<const f4*>(partials) + i;
  f4 v = {0.f, 0.f, 0.f, 0.f};
  constexpr int kBatch = 8;  // slices in flight
  for (int z = 0; z < slices; z += kBatch) {
    f4 t[kBatch];
#pragma unroll
    for (int u = 0; u < kBatch; ++u) t[u] = src[(size_t)min(z + u, slices - 1) * n4];
#pragma unroll
    for (int u = 0; u < kBatch; ++u)
#pragma unroll
      for (int e = 0; e < 4; ++e) v[e] += z + u < slices ? t[u][e] : 0.f;
  }
  h4 o;
#pragma unroll
  for (int e = 0; e < 4; ++e) o[e] = (half_t)v[e];
  reinterpret_cast<h4*>(r)[i] = o;
}

template <int kA>
static hipError_t launch_proj_tile(const half_t* x, const half_t* R, half_t* r, int M, int K, int rank, int slices, float* ws, hipStream_t stream) {
  auto kern = proj_tile_kernel<kA>;
  constexpr size_t lds = (size_t)2 * (128 * kA) * kTRow;
  static LdsLimit lds_limit;
  if (hipError_t e = ensure_dynamic_lds(reinterpret_cast<const void*>(kern), lds, lds_limit); e != hipSuccess) return e;
  const int row_tiles = (M + 64 * kA - 1) / (64 * kA), col_tiles = (rank + 64 * kA - 1) / (64 * kA);
  note_launch(row_tiles * col_tiles, slices, 256, "proj_tile_kernel<%d>", kA);
  hipLaunchKernelGGL(kern, dim3(row_tiles, col_tiles, slices), dim3(256), lds, stream, x, R, r, ws, M, K, rank);
  if (hipError_t e = hipGetLastError(); e != hipSuccess || slices == 1) return e;
  const long n4 = (long)M * rank / 4;
  hipLaunchKernelGGL(proj_sum_kernel, dim3((unsigned)((n4 + 63) / 64)), dim3(64), 0, stream, ws, r, n4, slices);
  return hipGetLastError();
}

// How a projection is cut: columns per workgroup (32 * nt) and K slices.  The tile width follows the workgroup count
// (narrow tiles where 64 columns each would leave CUs idle; R is small, re-reading it is cheap).  K is split only with a
// workspace, where the tiles alone fill less than half the chip and K is long enough for the second launch to pay
// (from 4096 columns): then as many slices as bring the workgroup count to about two per CU, each at least two
// blocks deep, as far as the workspace reaches.
struct ProjPlan {
  int nt, slices;
};
static ProjPlan plan_proj(int M, int K, int rank, int num_cus, size_t ws_bytes) {
  const int m_blocks = (M + 31) / 32;
  const int blocks = (K + kPK - 1) / kPK;
  ProjPlan best;
  best.slices = 1;
  best.nt = (m_blocks * ((rank + 63) / 64) < num_cus && rank > 32) ? 1 : 2;
  if (blocks < 16) return best;
  long best_wgs = (long)m_blocks * ((rank + 32 * best.nt - 1) / (32 * best.nt));
  // with a workspace: the tile width whose split brings the most workgroups (up to two per CU); the wider tile on a
  // tie, since x is then read fewer times
  for (int nt : {2, 1}) {
    if (nt == 2 && rank <= 32) continue;
    const long tiles = (long)m_blocks * ((rank + 32 * nt - 1) / (32 * nt));
    if (tiles * 2 > num_cus || tiles > 65535) continue;
    long want = (2L * num_cus + tiles - 1) / tiles;
    const int min_depth = tiles >= 16 ? 4 : 2;  // blocks per slice: the partials of many tiles are traffic of their own
    if (want > blocks / min_depth) want = blocks / min_depth;
    const long fit = (long)(ws_bytes / sizeof(float) / ((size_t)tiles * nt * 1024));
    if (want > fit) want = fit;
    if (want < 2) continue;
    long wgs = tiles * want;
    if (wgs > 2L * num_cus) wgs = 2L * num_cus;
    if (wgs > best_wgs) {
      best_wgs = wgs;
      best.nt = nt;
      best.slices = (int)want;
    }
  }
  return best;
}

// Which of the two kernels, and how the tiles are cut: by what they are predicted to take, in us -- fits over 204 (M, K, rank),
// 65 to 2048 rows, 7 % rms, of the same form as kGemmCost: a block (256 columns) or stage (128) of K on the first workgroup of
// a compute unit, on every further one, the second launch, its walk over the slices, the traffic of the fp32 tiles, x.  The
// tile kernel has to be 7 % ahead.  With and without the rule, 12 (K, rank) at 65 to 2048 rows: it takes 87 of 132, 1.32 times as
// fast in the mean and the least of them 3 % faster.  The plan is also asked at 21 to 64 rows where the small kernel is not used
// (proj_on_small_kernel), which extrapolates the fit: at 48 rows 1.11 and 1.24 times as fast on the two shapes it gets
// there (K = 18944 rank 128, K = 17408 rank 256).  us, this / 32-row tiles:
// K = 18944, rank 128 at 100 / 333 / 2048 rows 11.1 / 14.7, 15.3 / 21.1, 30 / 37; K = 17408, rank 256 at 200 / 1500 rows 14.4 / 26.9,
// 34 / 78; K = 4096, rank 128 at 100 / 1500 rows 7.3 / 8.6, 12.0 / 17.1; K = 1536, rank 256 at 512 rows 8.9 / 6.9 (not taken).
struct ProjTilePlan {
  int a, slices;  // a = 0: the 32-row tiles
  float us;       // prediction
};
static ProjTilePlan plan_proj_tile(const ProjPlan& p, int M, int K, int rank, int num_cus, size_t ws_bytes) {
  const auto rounds_more = [&](long wgs) { return (float)((wgs + num_cus - 1) / num_cus - 1); };
  const float slice_mb = (float)M * (float)rank * 4e-6f;
  const int blocks = (K + kPK - 1) / kPK, stages = K >> 7;
  const float per = (float)((blocks + p.slices - 1) / p.slices);
  const long wgs = (long)((M + 31) / 32) * ((rank + 32 * p.nt - 1) / (32 * p.nt)) * p.slices;
  float best = 3.9f + per * (p.nt == 1 ? 0.48f : 0.81f) + per * 0.52f * rounds_more(wgs);
  if (p.slices > 1) best += 1.6f + 0.09f * (float)p.slices + 1.5f * slice_mb * (float)p.slices;
  best *= 0.93f;
  ProjTilePlan plan = {0, 1, best};
  for (int a = 1; a <= 2; ++a) {
    const long row_tiles = (M + 64 * a - 1) / (64 * a), col_tiles = (rank + 64 * a - 1) / (64 * a);
    if (row_tiles * col_tiles > 4L * num_cus) continue;
    const int tiles = (int)(row_tiles * col_tiles);
    for (const int s : {1, 2, 3, 4, 5, 6, 7, 8, 10, 12, 14, 16, 20, 24, 28, 32}) {
      if (s > stages || tiles * s > 4 * num_cus || (s > 1 && (size_t)s * M * rank * sizeof(float) > ws_bytes)) break;
      const int depth = (stages + s - 1) / s;
      float us = (a == 1 ? 2.1f : 5.4f) + (float)depth * ((a == 1 ? 0.62f : 1.05f) + (a == 1 ? 0.29f : 1.66f) * rounds_more(tiles * s)) +
                 0.07f * (float)M * (float)K * 2e-6f;
      if (s > 1) us += 2.5f + (a == 1 ? 0.074f : 0.043f) * (float)s + (a == 1 ? 0.56f : 0.43f) * slice_mb * (float)s;
      if (s > 1 && p.slices == 1) us += 1.5f;  // a second launch where there was none also takes the host's time
      if (us >= best) continue;
      best = us;
      plan = {a, (stages + depth - 1) / depth, us};  // no slice without stages
    }
  }
  return plan;
}

static float proj_launch_us(int M, int K, int rank, int num_cus, size_t ws_bytes) {
  return plan_proj_tile(plan_proj(M, K, rank, num_cus, ws_bytes), M, K, rank, num_cus, ws_bytes).us;
}

size_t proj_workspace_bytes(int M, int K, int rank, int num_cus) {
  if (M <= 16 || (K % kBK) != 0) return 0;
  const ProjPlan p = plan_proj(M, K, rank, num_cus, ~(size_t)0 >> 8);
  if (p.slices < 2) return 0;
  const long tiles = (long)((M + 31) / 32) * ((rank + 32 * p.nt - 1) / (32 * p.nt));
  return (size_t)tiles * p.slices * p.nt * 1024 * sizeof(float);
}

template <int NT>
static hipError_t launch_proj_t(const half_t* x, const half_t* R, half_t* r, int M, int K, int rank, int slices, void* ws,
                                hipStream_t stream) {
  const int m_blocks = (M + 31) / 32;
  const size_t lds_x = (size_t)2 * 32 * kPRow * sizeof(half_t);
  const size_t lds_red = (size_t)4 * NT * 16 * 64 * 4;
  const size_t lds = (lds_x > lds_red ? lds_x : lds_red) + (size_t)4 * (32 * NT) * 144;  // + the four waves' B tiles
  static LdsLimit lds_limit;
  if (hipError_t e = ensure_dynamic_lds(reinterpret_cast<const void*>(proj_mfma_kernel<NT>), lds, lds_limit); e != hipSuccess) return e;
  ProjSplit sp = {slices > 1 ? static_cast<float*>(ws) : nullptr};
  const int col_blocks = (rank + 32 * NT - 1) / (32 * NT);
  hipLaunchKernelGGL(proj_mfma_kernel<NT>, dim3(m_blocks, col_blocks, slices), dim3(256), lds, stream, x, R, r, M, K, rank, sp);
  if (hipError_t e = hipGetLastError(); e != hipSuccess || slices == 1) return e;
  hipLaunchKernelGGL(proj_reduce_kernel, dim3(NT * 4, m_blocks * col_blocks), dim3(256), 0, stream, sp.partials, r, M, rank, NT,
                     slices, m_blocks);
  return hipGetLastError();
}

hipError_t launch_shared_proj_mfma(const half_t* x, const half_t* R, half_t* r, int M, int K, int rank, int num_cus,
                                   hipStream_t stream, void* ws, size_t ws_bytes) {
  if ((K % kBK) != 0 || K < kBK) return hipErrorInvalidValue;
  if (ws == nullptr || (reinterpret_cast<uintptr_t>(ws) & 15u) != 0) ws_bytes = 0;
  const ProjPlan p = plan_proj(M, K, rank, num_cus, ws_bytes);
  const bool tiles_ok = (K & 127) == 0 && (rank & 3) == 0 && (size_t)M * K * 2 < (1ull << 32) && (size_t)rank * K * 2 < (1ull << 32) &&
                        (reinterpret_cast<uintptr_t>(x) & 15u) == 0 && (reinterpret_cast<uintptr_t>(R) & 15u) == 0 &&
                        (reinterpret_cast<uintptr_t>(r) & 7u) == 0;
  if (tiles_ok) {
    const ProjTilePlan t = plan_proj_tile(p, M, K, rank, num_cus, ws_bytes);
    if (t.a == 1) return launch_proj_tile<1>(x, R, r, M, K, rank, t.slices, static_cast<float*>(ws), stream);
    if (t.a == 2) return launch_proj_tile<2>(x, R, r, M, K, rank, t.slices, static_cast<float*>(ws), stream);
  }
  note_launch((M + 31) / 32 * ((rank + 32 * p.nt - 1) / (32 * p.nt)), p.slices, 256, "proj_mfma_kernel<%d>", p.nt);
  if (p.nt == 2) return launch_proj_t<2>(x, R, r, M, K, rank, p.slices, ws, stream);
  return launch_proj_t<1>(x, R, r, M, K, rank, p.slices, ws, stream);
}

}  // namespace glowq
