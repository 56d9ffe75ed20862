// 8B-class linear layers at draft / verify row counts on gfx950, FP8 (e4m3fn)
// or bf16 weights: y = x W^T with a bias or SwiGLU epilogue.
//
// The weight-streaming kernel (linear.hip) reads x again for every 16 - 32
// output columns; at hidden 4096 and 64 rows that is 524 KB of x per 16 KB -
// 131 KB of FP8 weights, and the L1s, not HBM, set the time (gate/up 57 us,
// down 44 us for 117 / 59 MB).  Here a workgroup takes 128 rows of W -- for
// SwiGLU 64 gate rows and their 64 up rows -- and all (up to 160) rows of x,
// and moves both through an LDS ring filled by DMA:
//
// * eight waves: four column groups of two 16-column W tiles (SwiGLU: a gate
//   tile and its up tile, so a pair sits in one lane) times all MT x tiles
//   (v_mfma_f32_16x16x32_bf16, A = W, B = x^T), twice: the two waves of a
//   column group (two per SIMD, so that one's LDS reads and conversions run
//   beside the other's MFMAs: FP8 gate/up at 64 rows 31.0 -> 29.3 us) take
//   the first and the second MFMA of every 64 k, and add up at the end;
// * KS k-elements per ring step: whole 128-byte lines of FP8 rows (KS 128),
//   64 for bf16 rows and above 128 rows, where the ring would hold two slots
//   (80 - 96 rows 46 -> 36 us with KS 128);
// * FP8 weights stay bytes in LDS and become bf16(float(w8) * scale[row]) in
//   registers; MFMA h of 64 k takes k = 16 g + 8 h + j (g = lane / 16) from W
//   and x alike, for bf16 weights too, so that both forms add up in the same
//   order and agree bit for bit;
// * few output columns (down_proj, o_proj) would leave most CUs idle: K is
//   then split over workgroups, which write fp32 partials to the caller's
//   workspace, and a second launch adds them in split order.
//
// Measured (graph replay, weights cold): bf16 gate/up 28672 x 4096 at 64 rows
// 40 us (5.9 TB/s of weight; 68.6 before); FP8 29.3 us (57), where the chain of
// a step -- LDS reads, conversion, MFMAs behind one barrier -- sets the pace,
// not the stream: at 32 rows 24.6 us, and slots for more W in flight (x in a
// shallow ring of its own) changed nothing at 64.  (Torch callers reach the bf16
// form at up to 32 rows: above, kernels.linear takes the library, with which it
// has not been compared.)
#include <algorithm>

#include "lm_head.hpp"

namespace nsg {
namespace {

typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));

constexpr int kRlWaves = 8;
constexpr int kRlWRows = 128;  // W rows per workgroup
constexpr int kRlLds = 160 * 1024;

template <int MT, int KS, bool W8>
constexpr int rl_stage_bytes() {
  return MT * 16 * KS * 2 + kRlWRows * KS * (W8 ? 1 : 2);
}
template <int MT, int KS, bool W8>
constexpr int rl_stages() {
  return kRlLds / rl_stage_bytes<MT, KS, W8>() < 8 ? kRlLds / rl_stage_bytes<MT, KS, W8>() : 8;
}

__device__ __forceinline__ void dma16(uint32_t lds, const void* src) {
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, off"
               :
               : "s"(lds), "v"(src)
               : "memory", "m0");
}
__device__ __forceinline__ void dma16_nt(uint32_t lds, const void* src) {
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, off nt"
               :
               : "s"(lds), "v"(src)
               : "memory", "m0");
}

// bf16(float(w8) * s) of 8 e4m3fn bytes (linear.hip's dequantisation).
__device__ __forceinline__ bf16x8 dequant8(uint32_t a, uint32_t b, float s) {
  const floatx2_t f0 = __builtin_amdgcn_cvt_pk_f32_fp8((int)a, false);
  const floatx2_t f1 = __builtin_amdgcn_cvt_pk_f32_fp8((int)a, true);
  const floatx2_t f2 = __builtin_amdgcn_cvt_pk_f32_fp8((int)b, false);
  const floatx2_t f3 = __builtin_amdgcn_cvt_pk_f32_fp8((int)b, true);
  return __builtin_bit_cast(
      bf16x8, u32x4{pack_bf16x2(f0[0] * s, f0[1] * s), pack_bf16x2(f1[0] * s, f1[1] * s),
                    pack_bf16x2(f2[0] * s, f2[1] * s), pack_bf16x2(f3[0] * s, f3[1] * s)});
}

// Physical 16-byte segment of logical segment s in row r of a tile whose rows
// hold BYTES bytes: the 16 rows of a fragment read then fall on distinct
// banks (rows of 256 bytes: one per bank row; of 128: two; of 64: four, which
// are contiguous for a fragment and need no swizzle).
template <int BYTES>
__device__ __forceinline__ int rl_swz(int r, int s) {
  if constexpr (BYTES == 256) return s ^ (r & 15);
  if constexpr (BYTES == 128) return s ^ ((r >> 1) & 7);
  return s;
}

template <int MT, int KS, bool SILU, bool W8>
__global__ __launch_bounds__(kRlWaves * 64) void ring_linear_kernel(RingLinearParams p) {
  constexpr int XB = KS * 2;               // bytes of an x row per step
  constexpr int WB = KS * (W8 ? 1 : 2);    // bytes of a W row per step
  constexpr int XI = MT * 16 * XB / 1024;  // x copies per step
  constexpr int WI = kRlWRows * WB / 1024; // W copies per step
  constexpr int kX = (XI + kRlWaves - 1) / kRlWaves;
  constexpr int kW = WI / kRlWaves;
  constexpr int NI = kX + kW;
  constexpr int SB = rl_stage_bytes<MT, KS, W8>();
  constexpr int kStages = rl_stages<MT, KS, W8>();
  static_assert(WI % kRlWaves == 0, "whole W copies per wave");
  static_assert(kStages >= 3 && (kStages - 2) * NI <= 63, "vmcnt counts to 63");
  static_assert(kStages * SB >= 8 * MT * 1024, "the partial sums of one wave group fit the ring");
  __shared__ __attribute__((aligned(1024))) uint8_t ring[kStages * SB];

  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int cw = wave & 3, h = wave >> 2;  // column group; which MFMA of every 64 k
  const int r16 = lane & 15;
  const int g4 = lane >> 4;
  const int tile = blockIdx.x, split = blockIdx.y;
  // splits start at multiples of 128 k whatever KS is
  const int n128 = p.K / 128;
  const int s0 = n128 * split / p.splits * (128 / KS);
  const int nst = n128 * (split + 1) / p.splits * (128 / KS) - s0;
  // Workgroups sweep K from different places (in units of 128 k): rows of a
  // power-of-two length put one k of every row on one L2 channel, and in step
  // all workgroups would queue there, for x as well (gate/up at 16 rows 31.7
  // -> 23.5 us).
  const int rot = (int)((blockIdx.x >> 3) + 4 * (blockIdx.x & 7)) % (nst / (128 / KS)) * (128 / KS);
  const uint32_t ring_lds = lds_addr(ring);

  // W row r of the workgroup's 128: column group r / 32, its tile r / 16 % 2
  auto w_row = [&](int r) {
    const int rr = r & 31;
    if constexpr (SILU)
      return (rr < 16 ? 0 : p.N) + min(tile * 64 + (r >> 5) * 16 + (rr & 15), p.N - 1);
    return min(tile * kRlWRows + r, p.N - 1);
  };

  // DMA sources (rows past M repeat row M - 1, columns past N the last one)
  const bf16* xsrc[kX];
  uint32_t x_lds[kX];
#pragma unroll
  for (int i = 0; i < kX; ++i) {
    const int copy = min(wave * kX + i, XI - 1);  // surplus copies repeat the last
    x_lds[i] = ring_lds + copy * 1024;
    const int r = (copy * 1024 + lane * 16) / XB;
    const int seg = rl_swz<XB>(r, lane % (XB / 16));
    xsrc[i] = p.x + (int64_t)min(r, p.M - 1) * p.ldx + (int64_t)s0 * KS + seg * 8;
  }
  const uint8_t* wsrc[kW];
#pragma unroll
  for (int i = 0; i < kW; ++i) {
    const int r = ((wave * kW + i) * 1024 + lane * 16) / WB;
    const int seg = rl_swz<WB>(r, lane % (WB / 16));
    wsrc[i] = static_cast<const uint8_t*>(p.w) +
              ((int64_t)w_row(r) * p.ldw + (int64_t)s0 * KS) * (W8 ? 1 : 2) + seg * 16;
  }
  const uint32_t w_lds = ring_lds + MT * 16 * XB + wave * kW * 1024;
  float wsc[2] = {1.f, 1.f};
  if constexpr (W8) {
    wsc[0] = p.w_scale[w_row(cw * 32 + r16)];
    wsc[1] = p.w_scale[w_row(cw * 32 + 16 + r16)];
  }
  // (the scales have landed before the first copy is issued: the compiler,
  // which does not see the copies, would drain them with its own wait)
  asm volatile("" ::"v"(wsc[0]), "v"(wsc[1]));

  int issued = 0, i_slot = 0, i_k = rot;
  auto issue = [&]() {
    const uint32_t sb = (uint32_t)i_slot * SB;
    i_slot = i_slot + 1 == kStages ? 0 : i_slot + 1;
#pragma unroll
    for (int i = 0; i < kW; ++i) {
      if constexpr (WB >= 128)
        dma16_nt(w_lds + sb + i * 1024, wsrc[i] + (int64_t)i_k * WB);
      else  // half a line per step: the other half should still be in L2
        dma16(w_lds + sb + i * 1024, wsrc[i] + (int64_t)i_k * WB);
    }
#pragma unroll
    for (int i = 0; i < kX; ++i) dma16(x_lds[i] + sb, xsrc[i] + (int64_t)i_k * KS);
    i_k = i_k + 1 == nst ? 0 : i_k + 1;
    ++issued;
  };
  for (int s = 0; s < kStages - 1 && s < nst; ++s) issue();

  floatx4 acc[2][MT];
#pragma unroll
  for (int nt = 0; nt < 2; ++nt)
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) acc[nt][mt] = floatx4{0.f, 0.f, 0.f, 0.f};

  int c_slot = 0;
  for (int s = 0; s < nst; ++s) {
    // step s landed for this wave, then for every wave; the slot of step
    // s - 1 is free
    wait_steps<NI, kStages - 2>(issued - 1 - s);
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    if (issued < nst) issue();
    const uint8_t* st = ring + c_slot * SB;
    c_slot = c_slot + 1 == kStages ? 0 : c_slot + 1;
    const uint8_t* ws = st + MT * 16 * XB + cw * 32 * WB;
#pragma unroll
    for (int u = 0; u < KS / 64; ++u) {
      bf16x8 wf[2], xf[MT];
#pragma unroll
      for (int nt = 0; nt < 2; ++nt) {
        const int r = nt * 16 + r16;  // (the swizzles repeat every 16 rows)
        if constexpr (W8) {
          const u32x2 v = *reinterpret_cast<const u32x2*>(
              ws + r * WB + 16 * rl_swz<WB>(r, 4 * u + g4) + 8 * h);
          wf[nt] = dequant8(v[0], v[1], wsc[nt]);
        } else {
          wf[nt] = *reinterpret_cast<const bf16x8*>(ws + r * WB +
                                                    16 * rl_swz<WB>(r, 8 * u + 2 * g4 + h));
        }
      }
#pragma unroll
      for (int mt = 0; mt < MT; ++mt)
        xf[mt] = *reinterpret_cast<const bf16x8*>(st + (mt * 16 + r16) * XB +
                                                  16 * rl_swz<XB>(r16, 8 * u + 2 * g4 + h));
#pragma unroll
      for (int nt = 0; nt < 2; ++nt)
#pragma unroll
        for (int mt = 0; mt < MT; ++mt)
          acc[nt][mt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wf[nt], xf[mt], acc[nt][mt], 0, 0,
                                                                0);
    }
  }

  // The two wave groups' sums meet in LDS (every copy has landed, every
  // read is done): each group finishes the x tiles of its own parity.
  __syncthreads();
  auto slot = [&](int nt, int mt) {
    return reinterpret_cast<floatx4*>(ring) + ((cw * 2 + nt) * MT + mt) * 64 + lane;
  };
#pragma unroll
  for (int mt = 0; mt < MT; ++mt)
    if ((mt & 1) != h) {
#pragma unroll
      for (int nt = 0; nt < 2; ++nt) *slot(nt, mt) = acc[nt][mt];
    }
  __syncthreads();

  // lane l of (nt, mt) holds row 16 mt + l % 16, columns 4 (l / 16) + i of W
  // tile nt
  const int c0 = SILU ? tile * 64 + cw * 16 : tile * kRlWRows + cw * 32;
#pragma unroll
  for (int mt = 0; mt < MT; ++mt) {
    const int m = mt * 16 + r16;
    if ((mt & 1) != h || m >= p.M) continue;
    floatx4 sum[2];
#pragma unroll
    for (int nt = 0; nt < 2; ++nt) sum[nt] = acc[nt][mt] + *slot(nt, mt);
    if constexpr (SILU) {
      const int n = c0 + 4 * g4;
      if (n >= p.N) continue;
      float v[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const float g = bf16_bits_to_float(float_to_bf16_bits(sum[0][i]));
        const float u = bf16_bits_to_float(float_to_bf16_bits(sum[1][i]));
        v[i] = bf16_bits_to_float(float_to_bf16_bits(g / (1.f + __expf(-g)))) * u;
      }
      *reinterpret_cast<uint2*>(p.y + (int64_t)m * p.ldy + n) =
          uint2{pack_bf16x2(v[0], v[1]), pack_bf16x2(v[2], v[3])};
    } else {
#pragma unroll
      for (int nt = 0; nt < 2; ++nt) {
        const int n = c0 + nt * 16 + 4 * g4;
        if (n >= p.N) continue;
        if (p.splits > 1) {
          *reinterpret_cast<floatx4*>(p.partials +
                                      ((int64_t)split * p.M + m) * p.N + n) = sum[nt];
        } else {
          floatx4 v = sum[nt];
          if (p.bias) {
            const uint2 b = *reinterpret_cast<const uint2*>(p.bias + n);
            v += floatx4{bf16_bits_to_float(b.x & 0xffffu), bf16_bits_to_float(b.x >> 16),
                         bf16_bits_to_float(b.y & 0xffffu), bf16_bits_to_float(b.y >> 16)};
          }
          *reinterpret_cast<uint2*>(p.y + (int64_t)m * p.ldy + n) =
              uint2{pack_bf16x2(v[0], v[1]), pack_bf16x2(v[2], v[3])};
        }
      }
    }
  }
}

// y = bf16(sum of the K splits, in split order, + bias): 4 columns per thread.
__global__ __launch_bounds__(256) void split_sum_kernel(RingLinearParams p) {
  const int64_t q = (int64_t)blockIdx.x * 256 + threadIdx.x;
  const int64_t total = (int64_t)p.M * p.N / 4;
  if (q >= total) return;
  const int64_t e = q * 4;
  const int m = (int)(e / p.N), n = (int)(e - (int64_t)m * p.N);
  floatx4 part[kRlMaxSplits];
#pragma unroll
  for (int s = 0; s < kRlMaxSplits; ++s)  // all loads in flight; splits past the last repeat it
    part[s] = *reinterpret_cast<const floatx4*>(
        p.partials + (int64_t)min(s, p.splits - 1) * p.M * p.N + e);
  floatx4 v = part[0];
#pragma unroll
  for (int s = 1; s < kRlMaxSplits; ++s)
    if (s < p.splits) v += part[s];
  if (p.bias) {
    const uint2 b = *reinterpret_cast<const uint2*>(p.bias + n);
    v += floatx4{bf16_bits_to_float(b.x & 0xffffu), bf16_bits_to_float(b.x >> 16),
                 bf16_bits_to_float(b.y & 0xffffu), bf16_bits_to_float(b.y >> 16)};
  }
  *reinterpret_cast<uint2*>(p.y + (int64_t)m * p.ldy + n) =
      uint2{pack_bf16x2(v[0], v[1]), pack_bf16x2(v[2], v[3])};
}

template <int MT, int KS>
int32_t launch_ks(const RingLinearParams& p, bool silu, hipStream_t s) {
  const int cols = silu ? 64 : kRlWRows;
  const dim3 g((p.N + cols - 1) / cols, p.splits), b(kRlWaves * 64);
  if (silu && p.w_scale) {
    hipLaunchKernelGGL((ring_linear_kernel<MT, KS, true, true>), g, b, 0, s, p);
  } else if (silu) {
    hipLaunchKernelGGL((ring_linear_kernel<MT, 64, true, false>), g, b, 0, s, p);
  } else if (p.w_scale) {
    hipLaunchKernelGGL((ring_linear_kernel<MT, KS, false, true>), g, b, 0, s, p);
  } else {
    // (bf16 rows are twice as long: 64 k per step)
    hipLaunchKernelGGL((ring_linear_kernel<MT, 64, false, false>), g, b, 0, s, p);
  }
  if (int32_t rc = launch_status("ring_linear_kernel")) return rc;
  if (p.splits == 1) return NSG_OK;
  const int64_t quads = (int64_t)p.M * p.N / 4;
  hipLaunchKernelGGL(split_sum_kernel, dim3((unsigned)((quads + 255) / 256)), dim3(256), 0, s, p);
  return launch_status("split_sum_kernel");
}

}  // namespace

int ring_linear_splits(int N, int K) {
  const int tiles = (N + kRlWRows - 1) / kRlWRows;
  // whole ring steps per split, at least four
  return std::max(1, std::min({kRlMaxSplits, 256 / tiles, K / (4 * 128)}));
}

bool ring_linear_fits(int M, int N, int K) {
  return M >= 1 && M <= kHeadMaxRows && N % 4 == 0 && N >= 4 && K % 128 == 0 && K >= 512;
}

int32_t launch_ring_linear(const RingLinearParams& p, bool silu, hipStream_t s) {
  if (p.M <= 16) return launch_ks<1, 128>(p, silu, s);
  if (p.M <= 32) return launch_ks<2, 128>(p, silu, s);
  if (p.M <= 48) return launch_ks<3, 128>(p, silu, s);
  if (p.M <= 64) return launch_ks<4, 128>(p, silu, s);
  if (p.M <= 96) return launch_ks<6, 128>(p, silu, s);
  if (p.M <= 128) return launch_ks<8, 128>(p, silu, s);
  return launch_ks<10, 64>(p, silu, s);
}

}  // namespace nsg
