// Prefill attention for gfx950: the work items of a plan whose query tiles
// are full (prompts: every position is a query), same semantics and inputs
// as the verify kernel (verify_attention.hip): ragged multi-query attention
// over the NHD paged KV cache, GQA, bottom-right causal rule
// (nano_sglang/model/causal_lm.py:359-471).
//
// What bounds it: the matrix cores and, beside them, one exponential per
// score.  A wave therefore owns 32 query rows (v_mfma_f32_32x32x16_bf16): a
// K or V fragment read from LDS feeds 32 rows instead of the verify kernel's
// 16, and a workgroup of NW waves (32 NW rows of one request and KV head)
// shares each K / V step, so LDS and L2 reads per flop are halved and
// quartered.  No KV split: the planner takes this kernel only for enough well
// filled tiles, so there is no merge launch either.
//
// Per workgroup, in 64-token steps through an LDS ring filled by DMA:
//   * S^T = K Q^T (M = 32 tokens, N = 32 query rows): lane l holds row l % 32
//     and 16 tokens 8 a + 4 (l / 32) + b of each 32-token half, so a row's max
//     and sum need one swap between the wave's halves;
//   * P^T in bf16 is directly the B operand of O^T += V^T P^T: the MFMA's k
//     slots (l / 32, j) stand for tokens 4 (l / 32) + j and 8 + 4 (l / 32) +
//     j - 4 of 16, and the V^T fragments are read in that order by
//     ds_read_b64_tr_b16;
//   * online softmax in base 2 with lazy rescaling, as in the verify kernel;
//     steps wholly above a wave's causal limits are skipped, steps wholly
//     below them run without the mask.
//
// Measured (eager calls, the verify kernel before): two prompts of 2048 - 8192
// tokens, 32 / 8 heads of 128: 1092 -> 607 us (0.92 PFLOP/s of the causal
// products; all waves in step 671 - 696, raised wave priority in the matrix
// phase 631); 32 prompts of 100 - 512, 14 / 2 heads of 64: 37.1 -> 20.1 us.
// At head dim 128 the counters show the matrix cores busy 36 % and the vector
// ALU 47 % of the time, LDS 28 %, a third of its cycles bank conflicts.
#include "attention.hpp"

namespace nsg {
namespace {

typedef float floatx16 __attribute__((ext_vector_type(16)));

constexpr int kStep = 64;  // KV tokens per ring step

// One LDS DMA copy of 16 bytes per lane (lane l lands at lds + 16 l), in asm:
// through the builtin the compiler's wait-count pass would wait for every
// copy in flight before each LDS read; the ring's own waits order them.
__device__ __forceinline__ void dma16(uint32_t lds, const void* src) {
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, off"
               :
               : "s"(lds), "v"(src)
               : "memory", "m0");
}

__device__ __forceinline__ float max_xor32(float x) {
  const auto b = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false,
                                                  false);
  return fmaxf(__uint_as_float(b[0]), __uint_as_float(b[1]));
}
__device__ __forceinline__ float sum_xor32(float x) {
  const auto b = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false,
                                                  false);
  return __uint_as_float(b[0]) + __uint_as_float(b[1]);
}

// Ring slots.  Head dim 128: four with the two wave groups (a slot is read over
// four phases), two for 128 rows (68 KB: two workgroups a CU).  Head dim 64:
// three (52 KB: three workgroups of four waves a CU, at 168 registers).
template <int D, int NW>
constexpr int prefill_ring() {
  return D == 64 ? 3 : NW == 4 ? 2 : 4;
}

template <int D, int NW>
__global__ __launch_bounds__(NW * 64, D == 64 ? 3 : 2) void prefill_attn_kernel(AttnParams p) {
  constexpr int KC = D / 16;              // k chunks of S^T = K Q^T
  constexpr int DT = D / 32;              // d tiles of O^T
  constexpr int CPR = D / 8;              // 16-byte chunks per token row
  constexpr int TILE = kStep * D;         // bf16 per K (or V) tile
  constexpr int TPI = 64 / CPR;           // token rows per 1 KB copy
  constexpr int NR = kStep / TPI / NW;    // row blocks a wave copies per step (K and V each)
  constexpr int NI = 2 * NR;              // copies per wave per step
  constexpr int kNBuf = prefill_ring<D, NW>();
  constexpr bool PP = NW == 8;              // (head dim 128 only) two wave groups half a step apart
  static_assert(NR >= 1 && (kNBuf - 1) * NI <= 63, "vmcnt counts to 63");
  __shared__ __attribute__((aligned(1024))) bf16 ring[kNBuf][2][TILE];
  __shared__ int s_pages[kMaxItemPages];

  const int wi = blockIdx.y;
  const int h = blockIdx.x;
  const int* wk = p.work + (size_t)wi * NSG_ATTN_WORK_INTS;
  const int qs = wk[0], qn = wk[1], lim0 = wk[2], pb = wk[3], kve = wk[5];
  if (qn == 0) return;
  const int P = 1 << p.log2P;
  const int G = p.G;
  const int nrows = qn * G;
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int r32 = lane & 31;
  const int g = lane >> 5;

  // page ids of the item (from token 0: items are not split)
  const int npages = min(((kve - 1) >> p.log2P) + 1, kMaxItemPages);
  bool bad_page = false;
  for (int i = tid; i < npages; i += NW * 64) {
    int pg = p.kv_indices[pb + i];
    if ((unsigned)pg >= (unsigned)p.num_pages) {
      bad_page = true;  // reads the pool's first page instead
      pg = 0;
    }
    s_pages[i] = pg;
  }

  // this lane's query row and its causal limit; the wave's smallest and
  // largest limit (rows past the tile's end load its first row, masked out)
  const int row = wave * 32 + r32;
  const bool row_ok = row < nrows;
  const int tau = row / G;
  const int gam = row - tau * G;
  const int lim = row_ok ? lim0 + (p.causal ? tau : 0) : -1;
  const int w_lo = lim0 + (p.causal ? (wave * 32) / G : 0);
  const int w_hi = wave * 32 >= nrows ? -1
                   : lim0 + (p.causal ? min(wave * 32 + 31, nrows - 1) / G : 0);
  bf16x8 qf[KC];
  {
    const bf16* qrow = p.q + (row_ok ? ((size_t)(qs + tau) * p.Hq + h * G + gam) * D
                                     : ((size_t)qs * p.Hq + h * G) * D);
#pragma unroll
    for (int c = 0; c < KC; ++c) qf[c] = load_bf16x8(qrow + 16 * c + 8 * g);
  }
  // Q has landed before the first copy is issued (the compiler does not see
  // the copies: its own wait for Q would drain them)
#pragma unroll
  for (int c = 0; c < KC; ++c) asm volatile("" ::"v"(__builtin_bit_cast(u32x4, qf[c])));
  __syncthreads();  // page ids visible

  floatx16 oacc[DT];
#pragma unroll
  for (int dt = 0; dt < DT; ++dt)
#pragma unroll
    for (int i = 0; i < 16; ++i) oacc[dt][i] = 0.f;
  float m_run = kMaskVal, l_run = 0.f;

  // LDS read offsets (bytes inside a K or V tile).  K fragment c of half s:
  // token 32 s + r32, logical chunk 2 c + g (the swizzle repeats every 16
  // rows).  V^T fragment (dt, m, hh): lane i of a 16-lane group addresses
  // token 16 m + 8 hh + 4 g + i / 4, columns 32 dt + 16 dh + 4 (i % 4) .. + 3,
  // and receives column i of the group's 16 for tokens j = 0..3.
  // (Offsets of the other fragments differ from these by an XOR of bits the
  // swizzles leave alone: chunk 2 c + g is (2 c) ^ g, d tile dt is chunk 4 dt
  // ^ the tile's own, so they cost one instruction and no register.)
  const int koff = 2 * (r32 * D + ((g ^ swz_k<D>(r32)) * 8));  // fragment c: koff ^ 32 c
  int voff[2];  // fragment (dt, hh): voff[hh] ^ 64 dt; the swizzle repeats every 8 rows
#pragma unroll
  for (int hh = 0; hh < 2; ++hh) {
    const int i = lane & 15, dh = (lane >> 4) & 1;
    const int t = 8 * hh + 4 * g + (i >> 2);
    const int c = 16 * dh + 4 * (i & 3);
    voff[hh] = 2 * (t * D + (((c >> 3) ^ swz_v<D>(t)) << 3) + (c & 7));
  }

  // DMA: row block i of this wave holds token rows (wave + NW i) TPI .. + TPI
  // of a step, for K and for V; lane: row lane / CPR, physical chunk lane % CPR
  const size_t tok_bytes = (size_t)p.Hkv * D * 2;
  const char* kbase = reinterpret_cast<const char*>(p.kc + (size_t)h * D);
  const char* vbase = reinterpret_cast<const char*>(p.vc + (size_t)h * D);
  const uint32_t ring_lds = lds_addr(&ring[0][0][0]);
  int d_t[NR];
  uint32_t d_k[NR], d_v[NR], d_lds[NR];
#pragma unroll
  for (int i = 0; i < NR; ++i) {
    const int t0 = (wave + NW * i) * TPI;
    const int t = t0 + lane / CPR;
    const int pc = lane % CPR;
    d_t[i] = t;
    d_k[i] = (pc ^ swz_k<D>(t)) * 16;
    d_v[i] = (pc ^ swz_v<D>(t)) * 16;
    d_lds[i] = t0 * D * 2;
  }
  const int n_it = (kve + kStep - 1) / kStep;
  const int last_tok = kve - 1;
  auto issue = [&](int it, int slot) {
    const uint32_t sb = ring_lds + (uint32_t)slot * (2 * TILE * 2);
#pragma unroll
    for (int i = 0; i < NR; ++i) {
      // tokens past the item's end repeat its last one (masked out)
      const int tok = min(it * kStep + d_t[i], last_tok);
      const int page = s_pages[min(tok >> p.log2P, kMaxItemPages - 1)];
      const size_t off = ((size_t)(uint32_t)page * P + (tok & (P - 1))) * tok_bytes;
      dma16(sb + d_lds[i], kbase + off + d_k[i]);
      dma16(sb + 2 * TILE + d_lds[i], vbase + off + d_v[i]);
    }
  };

  floatx16 sacc[2];  // S^T of the current step
  u32x4 pf[4];       // P^T of it in bf16: one B operand per 16 tokens
  auto qk = [&](int slot) {
    const char* Kt = reinterpret_cast<const char*>(&ring[slot][0][0]);
#pragma unroll
    for (int s = 0; s < 2; ++s) {
      floatx16 acc;
#pragma unroll
      for (int i = 0; i < 16; ++i) acc[i] = 0.f;
#pragma unroll
      for (int c = 0; c < KC; ++c) {
        const bf16x8 kf = *reinterpret_cast<const bf16x8*>(Kt + 32 * s * D * 2 + (koff ^ (32 * c)));
        acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(kf, qf[c], acc, 0, 0, 0);
      }
      sacc[s] = acc;
    }
  };
  // online softmax over a step's 64 tokens (this lane: 32 of them)
  auto softmax_of = [&](auto masked, int t0) {
    constexpr bool MASKED = decltype(masked)::value;
    float mx = kMaskVal;
#pragma unroll
    for (int s = 0; s < 2; ++s)
#pragma unroll
      for (int i = 0; i < 16; ++i) {
        if constexpr (MASKED) {
          const int j = t0 + 32 * s + 8 * (i >> 2) + 4 * g + (i & 3);
          if (j > lim || j >= kve) sacc[s][i] = kMaskVal;
        }
        mx = fmaxf(mx, sacc[s][i]);
      }
    mx = max_xor32(mx);
    mx = (MASKED && mx == kMaskVal) ? kMaskVal : mx * p.scale_log2;
    const bool grow = mx > m_run + kLazyRescale;
    if (__builtin_amdgcn_ballot_w64(grow)) {
      const float mnew = grow ? mx : m_run;
      const float alpha = __builtin_amdgcn_exp2f(m_run - mnew);
      m_run = mnew;
      l_run *= alpha;
#pragma unroll
      for (int dt = 0; dt < DT; ++dt) oacc[dt] *= alpha;
    }
    float ps = 0.f;
#pragma unroll
    for (int s = 0; s < 2; ++s) {
      float pv[16];
#pragma unroll
      for (int i = 0; i < 16; ++i) {
        const float e = __builtin_amdgcn_exp2f(fmaf(sacc[s][i], p.scale_log2, -m_run));
        pv[i] = MASKED && sacc[s][i] == kMaskVal ? 0.f : e;
        ps += pv[i];
      }
#pragma unroll
      for (int m = 0; m < 2; ++m)
        pf[2 * s + m] = u32x4{cvt_pk_bf16(pv[8 * m], pv[8 * m + 1]),
                              cvt_pk_bf16(pv[8 * m + 2], pv[8 * m + 3]),
                              cvt_pk_bf16(pv[8 * m + 4], pv[8 * m + 5]),
                              cvt_pk_bf16(pv[8 * m + 6], pv[8 * m + 7])};
    }
    l_run += ps;
  };
  auto softmax = [&](int t0) {
    if (t0 + kStep - 1 <= w_lo && t0 + kStep <= kve)
      softmax_of(std::false_type{}, t0);
    else
      softmax_of(std::true_type{}, t0);
  };
  auto pv_mul = [&](int slot) {  // O^T += V^T P^T
    const char* Vt = reinterpret_cast<const char*>(&ring[slot][1][0]);
#pragma unroll
    for (int m = 0; m < 4; ++m) {
#pragma unroll
      for (int dt = 0; dt < DT; ++dt) {
        const v4i16 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
            (__attribute__((address_space(3))) v4i16*)(Vt + 16 * m * D * 2 + (voff[0] ^ (64 * dt))));
        const v4i16 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
            (__attribute__((address_space(3))) v4i16*)(Vt + 16 * m * D * 2 + (voff[1] ^ (64 * dt))));
        const v8i16 w = __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7);
        oacc[dt] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(
            __builtin_bit_cast(bf16x8, w), __builtin_bit_cast(bf16x8, pf[m]), oacc[dt], 0, 0, 0);
      }
    }
  };
  // A workgroup-wide phase boundary: every LDS read of this wave has
  // returned, nothing moves across.
  auto phase = [&]() {
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_sched_barrier(0);
    asm volatile("" ::: "memory");
  };

  if constexpr (PP) {
    // Two wave groups half a step apart: a SIMD holds one wave of each, and
    // while one runs its matrix phase (O += P V of step i - 1, S = K Q of
    // step i) the other runs its softmax phase, so the matrix cores and the
    // vector ALU work side by side.  Phase n of the workgroup: group 0 is in
    // the matrix phase of step n / 2 (n even) or the softmax of n / 2 (odd),
    // group 1 one phase behind.  Slot i % 4 is read in phases 2 i .. 2 i + 3
    // (K by both groups, then V), so from phase 2 i + 4 on it takes step
    // i + 4; a step's copies go out three phases ahead or more.
    const int grp = wave >> 2;
    issue(0, 0);
    if (1 < n_it) issue(1, 1);
    wait_steps<NI, 1>(min(n_it - 1, 1));
    phase();  // phase 0 begins: step 0 in LDS
    if (grp == 1) {
      if (2 < n_it) issue(2, 2);
      wait_steps<NI, 1>(min(max(n_it - 2, 0), 1));  // step 1 (if any) landed
      phase();
    }
    bool had = false;  // the previous step's P is pending
    for (int it = 0; it < n_it; ++it) {
      const int t0 = it * kStep;
      const bool vis = t0 <= w_hi;  // something visible to this wave's rows
      if (had) pv_mul((it - 1) & 3);
      if (vis) qk(it & 3);
      had = vis;
      if (grp == 1) wait_steps<NI, 1>(min(max(n_it - 2 - it, 0), 1));
      phase();
      const int nx = it + 2 + grp;
      if (nx < n_it) issue(nx, nx & 3);
      if (vis) softmax(t0);
      if (grp == 0) wait_steps<NI, 1>(min(max(n_it - 2 - it, 0), 1));
      phase();
    }
    if (had) pv_mul((n_it - 1) & 3);
    if (grp == 0) phase();  // group 1's last softmax phase
  } else {
#pragma unroll
    for (int it = 0; it < kNBuf - 1; ++it)
      if (it < n_it) issue(it, it);
    int slot = 0;
    for (int it = 0; it < n_it; ++it) {
      // step `it` landed for this wave (the later issued steps stay in
      // flight), and for every wave; slot (it - 1) is free
      wait_steps<NI, kNBuf - 2>(min(n_it - 1 - it, kNBuf - 2));
      phase();
      const int cur = slot;
      if (it + kNBuf - 1 < n_it) issue(it + kNBuf - 1, slot == 0 ? kNBuf - 1 : slot - 1);
      slot = slot + 1 == kNBuf ? 0 : slot + 1;
      const int t0 = it * kStep;
      if (t0 > w_hi) continue;  // nothing visible to this wave's rows
      qk(cur);
      softmax(t0);
      pv_mul(cur);
    }
  }

  if (bad_page) atomicOr(p.flags, 1);
  const float l = sum_xor32(l_run);
  if (!row_ok) return;
  const float inv = l > 0.f ? 1.f / l : 0.f;
  bf16* orow = p.out + ((size_t)(qs + tau) * p.Hq + h * G + gam) * D + 4 * g;
#pragma unroll
  for (int dt = 0; dt < DT; ++dt)
#pragma unroll
    for (int a = 0; a < 4; ++a) {
      const floatx16 o = oacc[dt];
      *reinterpret_cast<u32x2*>(orow + 32 * dt + 8 * a) =
          u32x2{cvt_pk_bf16(o[4 * a] * inv, o[4 * a + 1] * inv),
                cvt_pk_bf16(o[4 * a + 2] * inv, o[4 * a + 3] * inv)};
    }
}

}  // namespace

int32_t launch_prefill_attn(int head_dim, int waves, int num_work, const AttnParams& prm,
                            hipStream_t stream) {
  const dim3 grid(prm.Hkv, num_work), block(waves * 64);
  if (head_dim == 64 && waves == 4)
    hipLaunchKernelGGL((prefill_attn_kernel<64, 4>), grid, block, 0, stream, prm);
  else if (head_dim == 128 && waves == 4)
    hipLaunchKernelGGL((prefill_attn_kernel<128, 4>), grid, block, 0, stream, prm);
  else if (head_dim == 128 && waves == 8)
    hipLaunchKernelGGL((prefill_attn_kernel<128, 8>), grid, block, 0, stream, prm);
  else {
    set_error("prefill attention: head_dim %d, %d waves", head_dim, waves);
    return NSG_ERR_ARG;
  }
  return launch_status("prefill_attn_kernel");
}

}  // namespace nsg
