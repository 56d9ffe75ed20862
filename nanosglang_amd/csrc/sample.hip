// Temperature / top-k / top-p sampling of one token per logits row on gfx950.
//
// Reference: nano_sglang/engine/sampling.py:25-50 (sample_token: argmax when
// T < 1e-6) and :71-88 (_sample_pytorch):
//   logits / T;
//   top-k: mask logits < the k-th largest (ties with it are kept);
//   top-p: sort descending, p = softmax; mask sorted position i when
//     sum_{j<i} p_j >= top_p (the exclusive cumulative);
//   softmax, multinomial.
// Here the rule is evaluated exactly: every token's weight
// w = 2^(x*log2(e)/T - max*log2(e)/T) is held in 2^-40 fixed point (uint64),
// so every mass is an exact integer sum, independent of summation order; the
// top-p comparison is (double)prefix < top_p * (double)Z.  Among equal logits
// at the top-p boundary, the lowest vocabulary indices come first (torch's
// sort leaves that order unspecified).  The token is drawn by inverse CDF in
// vocabulary order: the first index whose inclusive kept-mass prefix exceeds
// floor(u * Z_kept).
//
// No sort: thresholds are found by radix selection over an order-preserving
// integer key of the logit (16 bits for bf16, 32 for fp32), one byte per
// level, most significant first.  Launches (the grid covers every row and
// chunk of the vocabulary; no workgroup waits on another inside a launch):
//   max_kernel   (chunks, rows): chunk max key and its first index; clears the
//                row's histograms.
//   hist_kernel  (chunks, rows), once per stage (top-k levels, then top-p
//                levels): resolves the previous stage from its histogram
//                (every workgroup, identically), then adds its chunk's
//                counts (top-k) or masses (top-p) per key byte into the row's
//                256-bin histogram (four LDS copies per wave, then
//                device-scope atomics).
//   sums_kernel  (chunks, rows): resolves the last stage -> the boundary key
//                v*, how many of its ties are kept (m*) and their weight; per
//                chunk: mass of keys > v* and count of keys == v*.
//   select_kernel (rows): kept mass per chunk (ties ranked in vocabulary
//                order), the chunk holding the draw, then a block scan of that
//                chunk.
// Greedy rows use max_kernel and select_kernel only.
#include <climits>
#include <cstring>
#include <type_traits>

#include "common.hpp"

namespace nsg {
namespace {

constexpr int kSThreads = 256;
constexpr int kSWaves = kSThreads / 64;
constexpr int kSMaxChunks = 64;
constexpr int kSTargetWgs = 1024;
constexpr int kBins = 256;
constexpr int kMaxStages = 8;   // 4 levels (fp32 keys) x 2 filters
constexpr int kMaxRows = 1 << 16;
constexpr int kPreTiles = 3;    // tiles of 8 x 256 elements loaded before a stage resolves
constexpr float kFix = 1099511627776.f;  // 2^40: fixed-point scale of the weights
constexpr float kLog2eS = 1.4426950408889634f;

typedef unsigned long long u64;
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

// Per-row state after a stage has been resolved (written by the first
// workgroup of the launch that resolved it, read by later launches).
struct SmpState {
  uint32_t prefix;  // key bits fixed so far for the current filter
  uint32_t tk;      // top-k threshold key (every key >= tk is kept by top-k)
  uint32_t vs;      // final: boundary key v*
  uint32_t ms;      // final: how many tokens with key == v* are kept (lowest indices)
  u64 above_c;      // count of keys above the current prefix range
  u64 above_m;      // mass of keys above the current prefix range
  u64 ws;           // final: weight of one token with key == v*
  double pz;        // top_p * Z_k
};

struct SmpParams {
  const void* x;
  int64_t stride;
  int rows, V;
  float c;  // log2(e) / T
  int greedy;
  int K;    // top-k (0 = off)
  double P; // top-p (>= 1 = off)
  const float* u;
  int64_t u_stride;
  int64_t* out;
  int nch, cs;
  int levels;  // key bytes
  int nk, np;  // stages of each filter (0 or levels)
  uint2* cmax;        // [rows][nch] (max key, first index)
  uint32_t* hcnt;     // [rows][kMaxStages][256]
  u64* hmass;         // [rows][kMaxStages][256]
  SmpState* st;       // [rows][kMaxStages + 1]
  uint32_t* todo;     // [rows]: 1 for a row left to the staged launches; null: all rows
  u64* csum;          // [rows][nch]
  uint32_t* ceq;      // [rows][nch]
};

template <typename T>
struct SKey;
template <>
struct SKey<bf16> {
  static constexpr int kBits = 16;
  static __device__ __forceinline__ uint32_t key(uint32_t b) {
    if (b == 0x8000u) b = 0;  // -0 == +0
    return (b & 0x8000u) ? (~b & 0xFFFFu) : (b | 0x8000u);
  }
  static __device__ __forceinline__ float val(uint32_t b) { return __uint_as_float(b << 16); }
  static __device__ __forceinline__ uint32_t bits_of_key(uint32_t k) {
    return (k & 0x8000u) ? (k & 0x7FFFu) : (~k & 0xFFFFu);
  }
  // raw bits of 8 consecutive elements e .. e+7 (those >= end are unused)
  static __device__ __forceinline__ void load8(const void* row, int e, int end, bool vec,
                                               uint32_t* r) {
    const uint16_t* p = reinterpret_cast<const uint16_t*>(row);
    if (vec && e + 8 <= end) {
      const u32x4 v = *reinterpret_cast<const u32x4*>(p + e);
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        r[2 * i] = v[i] & 0xFFFFu;
        r[2 * i + 1] = v[i] >> 16;
      }
    } else {
#pragma unroll
      for (int i = 0; i < 8; ++i) r[i] = e + i < end ? p[e + i] : 0u;
    }
  }
};
template <>
struct SKey<float> {
  static constexpr int kBits = 32;
  static __device__ __forceinline__ uint32_t key(uint32_t b) {
    if (b == 0x80000000u) b = 0;
    return (b & 0x80000000u) ? ~b : (b | 0x80000000u);
  }
  static __device__ __forceinline__ float val(uint32_t b) { return __uint_as_float(b); }
  static __device__ __forceinline__ uint32_t bits_of_key(uint32_t k) {
    return (k & 0x80000000u) ? (k & 0x7FFFFFFFu) : ~k;
  }
  static __device__ __forceinline__ void load8(const void* row, int e, int end, bool vec,
                                               uint32_t* r) {
    const uint32_t* p = reinterpret_cast<const uint32_t*>(row);
    if (vec && e + 8 <= end) {
      const u32x4 a = *reinterpret_cast<const u32x4*>(p + e);
      const u32x4 b = *reinterpret_cast<const u32x4*>(p + e + 4);
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        r[i] = a[i];
        r[4 + i] = b[i];
      }
    } else {
#pragma unroll
      for (int i = 0; i < 8; ++i) r[i] = e + i < end ? p[e + i] : 0u;
    }
  }
};

__device__ __forceinline__ u64 weight_of(float v, float c, float mc) {
  const float w = __builtin_amdgcn_exp2f(__builtin_fmaf(v, c, -mc));
  return (u64)(w * kFix);
}

template <typename T>
__device__ __forceinline__ const void* row_ptr(const SmpParams& p, int row) {
  return reinterpret_cast<const T*>(p.x) + (int64_t)row * p.stride;
}

__device__ __forceinline__ u64 shfl_u64(u64 v, int src) {
  const uint32_t lo = __shfl((uint32_t)v, src, 64);
  const uint32_t hi = __shfl((uint32_t)(v >> 32), src, 64);
  return ((u64)hi << 32) | lo;
}
__device__ __forceinline__ u64 shfl_up_u64(u64 v, int d) {
  const uint32_t lo = __shfl_up((uint32_t)v, d, 64);
  const uint32_t hi = __shfl_up((uint32_t)(v >> 32), d, 64);
  return ((u64)hi << 32) | lo;
}
__device__ __forceinline__ u64 wave_incl_scan_u64(u64 x, int lane) {
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    const u64 y = shfl_up_u64(x, o);
    if (lane >= o) x += y;
  }
  return x;
}

// Row max key (and its first index) from the chunk records; one wave.
__device__ __forceinline__ uint2 row_max(const SmpParams& p, int row, int lane) {
  uint2 best = make_uint2(0u, 0x7FFFFFFFu);
  for (int c = lane; c < p.nch; c += 64) {
    const uint2 v = p.cmax[(int64_t)row * p.nch + c];
    if (v.x > best.x || (v.x == best.x && v.y < best.y)) best = v;
  }
#pragma unroll
  for (int o = 32; o >= 1; o >>= 1) {
    const uint32_t kx = __shfl_xor(best.x, o, 64);
    const uint32_t ky = __shfl_xor(best.y, o, 64);
    if (kx > best.x || (kx == best.x && ky < best.y)) best = make_uint2(kx, ky);
  }
  return best;
}

template <typename T>
__device__ __forceinline__ float max_c(const SmpParams& p, uint32_t maxkey) {
  return SKey<T>::val(SKey<T>::bits_of_key(maxkey)) * p.c;
}

// Resolves stage s of a row from its histogram, given the state before it,
// and returns the state after it.  Top-k stages hold counts, top-p stages
// masses.  Executed by one whole wave; lane l holds bins 4l .. 4l+3.
template <typename T>
__device__ SmpState resolve_stage(const SmpParams& p, int row, int s, SmpState in, float mc) {
  const int lane = threadIdx.x & 63;
  const bool topk = s < p.nk;
  const int level = topk ? s : s - p.nk;
  const int64_t h0 = ((int64_t)row * kMaxStages + s) * kBins + 4 * lane;
  u64 h[4];
#pragma unroll
  for (int j = 0; j < 4; ++j) h[j] = topk ? (u64)p.hcnt[h0 + j] : p.hmass[h0 + j];
  SmpState o = in;
  const u64 incl = wave_incl_scan_u64(h[0] + h[1] + h[2] + h[3], lane);
  const u64 tot = shfl_u64(incl, 63);
  if (!topk && level == 0) {  // Z_k: every key >= tk, which this histogram holds
    o.pz = p.P * (double)tot;
    o.above_m = 0;
  }
  // cumulative from the top bin down; a = everything above this lane's bins
  u64 a = (topk ? o.above_c : o.above_m) + (tot - incl);
  int hit = -1;
  u64 ha = 0;
#pragma unroll
  for (int j = 3; j >= 0; --j) {
    const u64 n = a + h[j];
    const bool reach = topk ? n >= (u64)p.K : (double)n >= o.pz;
    if (hit < 0 && reach) {
      hit = 4 * lane + j;
      ha = a;
    }
    a = n;
  }
  // lanes below the crossing reach too: the crossing is the highest lane hit
  const uint64_t bal = __builtin_amdgcn_ballot_w64(hit >= 0);
  int src = bal ? 63 - (int)__builtin_clzll(bal) : -1;
  if (src < 0) {
    // unreachable for exact integer counts and masses (a level's bins always
    // hold the crossing); keep a defined result: the lowest bin
    src = 0;
    if (lane == 0) {
      hit = 0;
      ha = (topk ? o.above_c : o.above_m) + (tot - incl) + h[3] + h[2] + h[1];
    }
  }
  const int bin = __shfl(hit, src, 64);
  const u64 above = shfl_u64(ha, src);
  if (topk) o.above_c = above;
  else o.above_m = above;
  o.prefix = (in.prefix << 8) | (uint32_t)bin;
  if (level == p.levels - 1) {
    const uint32_t key = o.prefix;
    const u64 W = weight_of(SKey<T>::val(SKey<T>::bits_of_key(key)), p.c, mc);
    if (topk) {
      // every key >= tk is kept by top-k; without top-p that is the boundary
      o.tk = key;
      o.vs = key;
      o.ms = UINT_MAX;
      o.ws = W;
      o.prefix = 0;
      o.above_c = 0;
      o.above_m = 0;
    } else {
      // ties of v* kept: the m with (double)(S + m W) < pz, lowest indices
      // first (m = 0 always is); past their count every tie is kept
      const u64 S = o.above_m;
      u64 m0 = UINT_MAX;
      if (W > 0) {
        const double need = (o.pz - (double)S) / (double)W;
        m0 = need <= 1.0 ? 1 : (need >= (double)p.V ? (u64)p.V : (u64)ceil(need));
        while (m0 < (u64)p.V && (double)(S + m0 * W) < o.pz) ++m0;
        while (m0 > 1 && !((double)(S + (m0 - 1) * W) < o.pz)) --m0;
      }
      o.vs = key;
      o.ms = (uint32_t)m0;
      o.ws = W;
    }
  }
  return o;
}

template <typename T>
__device__ SmpState initial_state(const SmpParams& p) {
  SmpState s;
  s.prefix = 0;
  s.tk = 0;
  s.vs = 0;
  s.ms = UINT_MAX;
  s.above_c = 0;
  s.above_m = 0;
  s.ws = 0;
  s.pz = 0.0;
  return s;
}

// State before stage s (s = 0: initial; else the record stage s-1's launch
// left, resolved with histogram s-1).  One wave; the first workgroup of the
// row stores it for the next launch.
template <typename T>
__device__ SmpState state_before(const SmpParams& p, int row, int s, bool store, float mc) {
  SmpState st = initial_state<T>(p);
  if (s > 0)
    st = resolve_stage<T>(p, row, s - 1, p.st[(int64_t)row * (kMaxStages + 1) + s - 1], mc);
  if (store && (threadIdx.x & 63) == 0) p.st[(int64_t)row * (kMaxStages + 1) + s] = st;
  return st;
}

// ---- launch 1: chunk max key (first index) and histogram clearing ----
template <typename T>
__global__ __launch_bounds__(kSThreads) void max_kernel(SmpParams p, bool vec) {
  const int ch = blockIdx.x, row = blockIdx.y, tid = threadIdx.x;
  if (p.todo && p.todo[row] == 0) return;
  const int nst = p.nk + p.np;
  for (int i = ch * kSThreads + tid; i < nst * kBins; i += p.nch * kSThreads) {
    p.hcnt[(int64_t)row * kMaxStages * kBins + i] = 0;
    p.hmass[(int64_t)row * kMaxStages * kBins + i] = 0;
  }
  const void* x = row_ptr<T>(p, row);
  const int c0 = ch * p.cs, c1 = min(p.V, c0 + p.cs);
  uint32_t bk = 0, bi = 0x7FFFFFFFu;
  for (int e = c0 + 8 * tid; e < c1; e += 8 * kSThreads) {
    uint32_t r[8];
    SKey<T>::load8(x, e, c1, vec, r);
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const uint32_t k = SKey<T>::key(r[i]);
      if (e + i < c1 && (k > bk || bi == 0x7FFFFFFFu)) {
        bk = k;
        bi = e + i;
      }
    }
  }
  __shared__ uint2 sh[kSWaves];
  const int lane = tid & 63, wave = tid >> 6;
#pragma unroll
  for (int o = 32; o >= 1; o >>= 1) {
    const uint32_t kx = __shfl_xor(bk, o, 64), ix = __shfl_xor(bi, o, 64);
    if (ix != 0x7FFFFFFFu && (bi == 0x7FFFFFFFu || kx > bk || (kx == bk && ix < bi))) {
      bk = kx;
      bi = ix;
    }
  }
  if (lane == 0) sh[wave] = make_uint2(bk, bi);
  __syncthreads();
  if (tid == 0) {
    uint2 b = sh[0];
    for (int w = 1; w < kSWaves; ++w) {
      const uint2 v = sh[w];
      if (v.y != 0x7FFFFFFFu && (b.y == 0x7FFFFFFFu || v.x > b.x || (v.x == b.x && v.y < b.y)))
        b = v;
    }
    p.cmax[(int64_t)row * p.nch + ch] = b;
  }
}

// ---- launch 2..: one histogram stage (counts for top-k, masses for top-p) ----
template <typename T, bool kCount>
__global__ __launch_bounds__(kSThreads) void hist_kernel(SmpParams p, int s, bool vec) {
  constexpr int kCopies = 4;  // per wave, by lane & 3: a quarter of the same-bin conflicts
  typedef typename std::conditional<kCount, uint32_t, u64>::type H;
  const int ch = blockIdx.x, row = blockIdx.y, tid = threadIdx.x;
  if (p.todo && p.todo[row] == 0) return;
  const int lane = tid & 63, wave = tid >> 6;
  __shared__ H lh[kSWaves * kCopies][kBins];
  __shared__ SmpState s_st;
  __shared__ float s_mc;
  const void* x = row_ptr<T>(p, row);
  const int c0 = ch * p.cs, c1 = min(p.V, c0 + p.cs);
  // the chunk's first tiles are loaded while wave 0 resolves the stage
  uint32_t pre[kPreTiles][8];
#pragma unroll
  for (int t = 0; t < kPreTiles; ++t) {
    const int e = c0 + 8 * tid + t * 8 * kSThreads;
    if (e < c1) SKey<T>::load8(x, e, c1, vec, pre[t]);
  }
  for (int i = tid; i < kSWaves * kCopies * kBins; i += kSThreads) (&lh[0][0])[i] = 0;
  if (wave == 0) {
    const uint2 mk = row_max(p, row, lane);
    const float mc = max_c<T>(p, mk.x);
    const SmpState st = state_before<T>(p, row, s, ch == 0, mc);
    if (lane == 0) {
      s_st = st;
      s_mc = mc;
    }
  }
  __syncthreads();
  const SmpState st = s_st;
  const float mc = s_mc;
  const int level = kCount ? s : s - p.nk;
  const int shift = SKey<T>::kBits - 8 * (level + 1);
  const uint32_t lo_key = kCount ? 0u : st.tk;
  H* mine = lh[wave * kCopies + (lane & 3)];
  auto tile = [&](int e, const uint32_t* r) {
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const uint32_t k = SKey<T>::key(r[i]);
      const bool match = e + i < c1 && k >= lo_key &&
                         (level == 0 || (k >> (shift + 8)) == st.prefix);
      if (match) {
        const uint32_t bin = (k >> shift) & 0xFFu;
        if (kCount) atomicAdd(&mine[bin], (H)1);
        else atomicAdd(&mine[bin], (H)weight_of(SKey<T>::val(r[i]), p.c, mc));
      }
    }
  };
#pragma unroll
  for (int t = 0; t < kPreTiles; ++t) {
    const int e = c0 + 8 * tid + t * 8 * kSThreads;
    if (e < c1) tile(e, pre[t]);
  }
  for (int e = c0 + 8 * tid + kPreTiles * 8 * kSThreads; e < c1; e += 8 * kSThreads) {
    uint32_t r[8];
    SKey<T>::load8(x, e, c1, vec, r);
    tile(e, r);
  }
  __syncthreads();
  H t = 0;
#pragma unroll
  for (int w = 0; w < kSWaves * kCopies; ++w) t += lh[w][tid];
  if (t) {
    const int64_t o = ((int64_t)row * kMaxStages + s) * kBins + tid;
    if (kCount) atomicAdd(p.hcnt + o, (uint32_t)t);
    else atomicAdd(p.hmass + o, (u64)t);
  }
}

// ---- per-chunk kept mass above v* and ties at v* ----
template <typename T>
__global__ __launch_bounds__(kSThreads) void sums_kernel(SmpParams p, bool vec) {
  const int ch = blockIdx.x, row = blockIdx.y, tid = threadIdx.x;
  if (p.todo && p.todo[row] == 0) return;
  const int lane = tid & 63, wave = tid >> 6;
  __shared__ SmpState s_st;
  __shared__ float s_mc;
  __shared__ u64 sm[kSWaves];
  __shared__ uint32_t sc[kSWaves];
  const void* x = row_ptr<T>(p, row);
  const int c0 = ch * p.cs, c1 = min(p.V, c0 + p.cs);
  uint32_t pre[kPreTiles][8];
#pragma unroll
  for (int t = 0; t < kPreTiles; ++t) {
    const int e = c0 + 8 * tid + t * 8 * kSThreads;
    if (e < c1) SKey<T>::load8(x, e, c1, vec, pre[t]);
  }
  if (wave == 0) {
    const uint2 mk = row_max(p, row, lane);
    const float mc = max_c<T>(p, mk.x);
    const SmpState st = state_before<T>(p, row, p.nk + p.np, ch == 0, mc);
    if (lane == 0) {
      s_st = st;
      s_mc = mc;
    }
  }
  __syncthreads();
  const uint32_t vs = s_st.vs;
  const float mc = s_mc;
  u64 m = 0;
  uint32_t n = 0;
  auto tile = [&](int e, const uint32_t* r) {
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      if (e + i >= c1) continue;
      const uint32_t k = SKey<T>::key(r[i]);
      if (k > vs) m += weight_of(SKey<T>::val(r[i]), p.c, mc);
      n += k == vs;
    }
  };
#pragma unroll
  for (int t = 0; t < kPreTiles; ++t) {
    const int e = c0 + 8 * tid + t * 8 * kSThreads;
    if (e < c1) tile(e, pre[t]);
  }
  for (int e = c0 + 8 * tid + kPreTiles * 8 * kSThreads; e < c1; e += 8 * kSThreads) {
    uint32_t r[8];
    SKey<T>::load8(x, e, c1, vec, r);
    tile(e, r);
  }
  m = shfl_u64(wave_incl_scan_u64(m, lane), 63);
#pragma unroll
  for (int o = 32; o >= 1; o >>= 1) n += __shfl_xor(n, o, 64);
  if (lane == 0) {
    sm[wave] = m;
    sc[wave] = n;
  }
  __syncthreads();
  if (tid == 0) {
    u64 tm = 0;
    uint32_t tn = 0;
    for (int w = 0; w < kSWaves; ++w) {
      tm += sm[w];
      tn += sc[w];
    }
    p.csum[(int64_t)row * p.nch + ch] = tm;
    p.ceq[(int64_t)row * p.nch + ch] = tn;
  }
}

// Block exclusive scan of one uint64 per thread (fixed order); returns the
// exclusive prefix and writes the block total to *total.
__device__ u64 block_excl_scan_u64(u64 x, u64* sh, u64* total) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const u64 incl = wave_incl_scan_u64(x, lane);
  if (lane == 63) sh[wave] = incl;
  __syncthreads();
  u64 pre = 0, tot = 0;
#pragma unroll
  for (int w = 0; w < kSWaves; ++w) {
    if (w < wave) pre += sh[w];
    tot += sh[w];
  }
  __syncthreads();
  *total = tot;
  return pre + incl - x;
}

// ---- the draw: one workgroup per row ----
template <typename T>
__global__ __launch_bounds__(kSThreads) void select_kernel(SmpParams p, bool vec) {
  const int row = blockIdx.x, tid = threadIdx.x;
  if (p.todo && p.todo[row] == 0) return;
  const int lane = tid & 63, wave = tid >> 6;
  __shared__ u64 sh[kSWaves];
  __shared__ int s_ch;
  __shared__ u64 s_target, s_base;
  __shared__ uint32_t s_eq0;
  __shared__ float s_mc;
  __shared__ int s_tok;
  if (p.greedy) {
    if (wave == 0) {
      const uint2 mk = row_max(p, row, lane);
      if (lane == 0) p.out[row] = mk.y;
    }
    return;
  }
  const SmpState st = p.st[(int64_t)row * (kMaxStages + 1) + p.nk + p.np];
  if (wave == 0) {
    const uint2 mk = row_max(p, row, lane);
    // kept mass per chunk: everything above v*, then the lowest-index ties
    u64 km = 0;
    uint32_t eq = 0;
    if (lane < p.nch) {
      km = p.csum[(int64_t)row * p.nch + lane];
      eq = p.ceq[(int64_t)row * p.nch + lane];
    }
    uint32_t ie = eq;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
      const uint32_t y = __shfl_up(ie, o, 64);
      if (lane >= o) ie += y;
    }
    const uint32_t before = ie - eq;
    const uint32_t kept = st.ms > before ? min(eq, st.ms - before) : 0u;
    km += (u64)kept * st.ws;
    const u64 incl = wave_incl_scan_u64(km, lane);
    const u64 Z = shfl_u64(incl, 63);
    const float u = p.u[(int64_t)row * p.u_stride];
    u64 target = (u64)((double)u * (double)Z);
    if (Z > 0 && target >= Z) target = Z - 1;
    const uint64_t hit = __builtin_amdgcn_ballot_w64(lane < p.nch && km > 0 && incl > target);
    const int ch = hit ? (int)__builtin_ctzll(hit) : -1;
    if (lane == 0) {
      s_ch = Z > 0 ? ch : -1;
      s_target = target;
      s_mc = max_c<T>(p, mk.x);
    }
    if (ch >= 0 && lane == ch) {
      s_base = incl - km;
      s_eq0 = before;
    }
  }
  __syncthreads();
  const int ch = s_ch;
  if (ch < 0) {  // no positive weight (all logits -inf)
    if (tid == 0) p.out[row] = -1;
    return;
  }
  if (tid == 0) s_tok = -1;
  const u64 target = s_target;
  const float mc = s_mc;
  u64 run = s_base;          // kept mass before the current block
  uint32_t eq_run = s_eq0;   // ties at v* before the current block
  const void* x = row_ptr<T>(p, row);
  const int c0 = ch * p.cs, c1 = min(p.V, c0 + p.cs);
  int last_kept = -1;
  for (int e0 = c0; e0 < c1; e0 += 8 * kSThreads) {
    const int e = e0 + 8 * tid;
    uint32_t r[8];
    if (e < c1) SKey<T>::load8(x, e, c1, vec, r);
    uint32_t key[8];
    uint32_t neq = 0;
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      key[i] = e + i < c1 ? SKey<T>::key(r[i]) : 0u;
      neq += (e + i < c1) && key[i] == st.vs;
    }
    u64 tot_eq;
    const uint32_t eq_before = eq_run + (uint32_t)block_excl_scan_u64(neq, sh, &tot_eq);
    u64 w[8];
    u64 tw = 0;
    uint32_t rank = eq_before;
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      w[i] = 0;
      if (e + i < c1) {
        bool kept = key[i] > st.vs;
        if (key[i] == st.vs) {
          kept = rank < st.ms;
          ++rank;
        }
        if (kept) {
          w[i] = weight_of(SKey<T>::val(r[i]), p.c, mc);
          if (w[i]) last_kept = e + i;
        }
      }
      tw += w[i];
    }
    u64 tot_w;
    const u64 pre = run + block_excl_scan_u64(tw, sh, &tot_w);
    if (pre <= target && target < pre + tw) {
      u64 acc = pre;
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        acc += w[i];
        if (w[i] && acc > target) {
          s_tok = e + i;
          break;
        }
      }
    }
    __syncthreads();
    if (s_tok >= 0) break;
    run += tot_w;
    eq_run += (uint32_t)tot_eq;
  }
  // rounding guard: the last kept token of the chunk (the chunk's kept mass
  // is the exact sum scanned here, so this is not reached)
  if (s_tok < 0) {
    int lk = last_kept;
#pragma unroll
    for (int o = 32; o >= 1; o >>= 1) lk = max(lk, __shfl_xor(lk, o, 64));
    __shared__ int s_lk[kSWaves];
    if (lane == 0) s_lk[wave] = lk;
    __syncthreads();
    if (tid == 0) {
      int b = -1;
      for (int w2 = 0; w2 < kSWaves; ++w2) b = max(b, s_lk[w2]);
      p.out[row] = b;
    }
    return;
  }
  if (tid == 0) p.out[row] = s_tok;
}

// ---- top-k draws (with or without top-p) of K <= kTkMaxK: one launch ----
// A row's K-th largest logit needs no histogram of the whole row: K of the
// largest logits lie above the smallest of 16 numbers, wave w's ceil(K / 16)-th
// largest lane maximum.  So one workgroup per row (1024 threads) reads the
// row once -- bf16 rows of up to 155,640 logits stay in registers, longer and
// fp32 rows are read a second time, from L2 --, collects the few hundred
// logits at or above that bound in LDS, and evaluates the rule on them: the
// K-th largest key by radix selection, then, over the tokens kept by top-k,
// each one's mass above it (top-p) and its mass prefix in vocabulary order (the
// draw), by direct sums of the same 2^-40 integers as the staged launches, so
// the token is the same.  The staged form took a launch per key byte and
// filter and three more, 7 - 10 us each whatever its work.  Eager calls, us,
// staged -> this: 32 rows x 151,936 bf16, top-k 50 and top-p 0.9 57.2 -> 28.5,
// top-k alone 41.3 -> 23.7, fp32 83 -> 41 / 56 -> 32; 32 x 32,000 bf16 41 -> 27;
// top-k 200 and top-p 0.95 57 -> 39 (topk_ahead says where it is not ahead).
// About 10 us of that are the marked rows' launches, which return at once.
// Rows with so many ties that the lists overflow (more than 8192 logits at the
// bound, or 1024 kept) are marked (todo), and the staged launches that follow do
// those rows only: every other row's workgroups return at once.  Such rows pay
// for both: 32 rows of one value, 151,936 bf16, top-k 50: 50 -> 69 us, with
// top-p 0.9 78 -> 98.
constexpr int kTkThreads = 1024;
constexpr int kTkWaves = kTkThreads / 64;
constexpr int kTkMaxK = 256;
constexpr int kTkSlotCap = 2048;  // slots of 8 logits that hold one to collect
constexpr int kTkCap = 8192;   // collected logits
constexpr int kTkKeep = 1024;  // tokens kept by top-k
constexpr int kTkSlots = 19;   // slots of 8 bf16 logits a thread holds

typedef short v2i16 __attribute__((ext_vector_type(2)));

// Signed order-preserving integers of raw logit bits (-0 is -1 until
// tk_key): missing elements (all bits set) are the lowest.
template <typename T>
struct TkBits;
template <>
struct TkBits<bf16> {
  static constexpr int kDwords = 4;  // of 8 elements
  static __device__ __forceinline__ uint32_t order(uint32_t packed) {
    v2i16 x = __builtin_bit_cast(v2i16, packed);
    x ^= (x >> 15) & (short)0x7FFF;
    return __builtin_bit_cast(uint32_t, x);
  }
  static __device__ __forceinline__ int at(const uint32_t* d, int i) {  // i unrolled
    return (int)(short)(i & 1 ? d[i >> 1] >> 16 : d[i >> 1] & 0xFFFFu);
  }
  static __device__ __forceinline__ int max8(const uint32_t* d) {
    v2i16 m = __builtin_bit_cast(v2i16, d[0]);
#pragma unroll
    for (int i = 1; i < 4; ++i)
      m = __builtin_elementwise_max(m, __builtin_bit_cast(v2i16, d[i]));
    return max((int)m[0], (int)m[1]);
  }
};
template <>
struct TkBits<float> {
  static constexpr int kDwords = 8;
  static __device__ __forceinline__ uint32_t order(uint32_t b) {
    return b ^ ((uint32_t)((int)b >> 31) & 0x7FFFFFFFu);
  }
  static __device__ __forceinline__ int at(const uint32_t* d, int i) { return (int)d[i]; }
  static __device__ __forceinline__ int max8(const uint32_t* d) {
    int m = (int)d[0];
#pragma unroll
    for (int i = 1; i < 8; ++i) m = max(m, (int)d[i]);
    return m;
  }
};
// SKey's unsigned key of an order integer.
template <typename T>
__device__ __forceinline__ uint32_t tk_key(int order) {
  if (order == -1) order = 0;  // -0 == +0
  return (uint32_t)order + (SKey<T>::kBits == 16 ? 0x8000u : 0x80000000u);
}

// A row in slots of 8 elements: slot s holds elements head - 8 + 8 s .. + 8,
// head (1 .. 8) chosen so that whole slots are 16-byte aligned whatever the
// row's address; the elements outside the row (of the first and the last
// slot) are missing.
template <typename T>
struct TkRow {
  const T* x;
  int V, head, slots;
  __device__ __forceinline__ TkRow(const SmpParams& p, int row) {
    x = reinterpret_cast<const T*>(row_ptr<T>(p, row));
    V = p.V;
    head = (int)((0u - (uint32_t)reinterpret_cast<uintptr_t>(x)) % 16u / sizeof(T));
    if (head == 0) head = 8;
    slots = 1 + (max(V - head, 0) + 7) / 8;
  }
  __device__ __forceinline__ int first(int s) const { return head - 8 + 8 * s; }
  // raw bits, packed as they lie in memory
  __device__ __forceinline__ void load(int s, uint32_t* d) const {
    const int e0 = first(s);
    if (e0 >= 0 && e0 + 8 <= V) {
#pragma unroll
      for (int i = 0; i < TkBits<T>::kDwords; i += 4) {
        const u32x4 v = *reinterpret_cast<const u32x4*>(x + e0 + i * (4 / sizeof(T)));
#pragma unroll
        for (int k = 0; k < 4; ++k) d[i + k] = v[k];
      }
      return;
    }
#pragma unroll
    for (int i = 0; i < TkBits<T>::kDwords; ++i) d[i] = 0xFFFFFFFFu;
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      if (e0 + i < 0 || e0 + i >= V) continue;
      if constexpr (sizeof(T) == 2) {
        const uint32_t b = reinterpret_cast<const uint16_t*>(x)[e0 + i];
        d[i >> 1] = i & 1 ? (d[i >> 1] & 0xFFFFu) | (b << 16) : (d[i >> 1] & 0xFFFF0000u) | b;
      } else {
        d[i] = reinterpret_cast<const uint32_t*>(x)[e0 + i];
      }
    }
  }
  __device__ __forceinline__ void load_ordered(int s, uint32_t* d) const {
    load(s, d);
#pragma unroll
    for (int i = 0; i < TkBits<T>::kDwords; ++i) d[i] = TkBits<T>::order(d[i]);
  }
};

template <typename T, bool HELD>
__global__ __launch_bounds__(kTkThreads) void topk_kernel(SmpParams p) {
  constexpr int DW = TkBits<T>::kDwords;
  constexpr int kBatch = 4;  // slots in flight when the row is not held
  __shared__ __attribute__((aligned(16))) uint32_t s_key[kTkCap], s_idx[kTkCap];
  __shared__ __attribute__((aligned(16))) u64 s_w[kTkKeep];
  __shared__ __attribute__((aligned(16))) uint32_t s_raw[kTkSlotCap][DW];
  __shared__ uint32_t s_slot[kTkSlotCap];
  __shared__ uint32_t s_hist[kBins];
  __shared__ uint32_t s_wmax[kTkWaves], s_wthr[kTkWaves];
  __shared__ uint32_t s_n, s_ns, s_n2, s_bin, s_above;
  const int row = blockIdx.x, tid = threadIdx.x;
  const int lane = tid & 63, wave = tid >> 6;
  const TkRow<T> r(p, row);
  if (tid == 0) p.todo[row] = 0;
  const float u = p.u[(int64_t)row * p.u_stride];  // (used last: lands meanwhile)

  // ---- the row, and each thread's largest logit ----
  constexpr int kMissing = SKey<T>::kBits == 16 ? -32768 : INT_MIN;
  uint32_t held[HELD ? kTkSlots : 1][DW];
  int mx = kMissing;
  if constexpr (HELD) {
#pragma unroll
    for (int j = 0; j < kTkSlots; ++j) {
      if (j * kTkThreads < r.slots) {  // wave-uniform
        if (tid + j * kTkThreads < r.slots) {
          r.load(tid + j * kTkThreads, held[j]);
        } else {
#pragma unroll
          for (int i = 0; i < DW; ++i) held[j][i] = 0xFFFFFFFFu;
        }
      }
    }
#pragma unroll
    for (int j = 0; j < kTkSlots; ++j) {
      if (j * kTkThreads < r.slots) {
#pragma unroll
        for (int i = 0; i < DW; ++i) held[j][i] = TkBits<T>::order(held[j][i]);
        mx = max(mx, TkBits<T>::max8(held[j]));
      }
    }
  } else {
    for (int s0 = tid; s0 < r.slots; s0 += kBatch * kTkThreads) {
      uint32_t d[kBatch][DW];
#pragma unroll
      for (int b = 0; b < kBatch; ++b) r.load(min(s0 + b * kTkThreads, r.slots - 1), d[b]);
#pragma unroll
      for (int b = 0; b < kBatch; ++b) {
        if (s0 + b * kTkThreads >= r.slots) break;  // each slot counts for one thread only
#pragma unroll
        for (int i = 0; i < DW; ++i) d[b][i] = TkBits<T>::order(d[b][i]);
        mx = max(mx, TkBits<T>::max8(d[b]));
      }
    }
  }

  // ---- row maximum, and a bound with at least K logits at or above it ----
  const uint32_t mk = tk_key<T>(mx);
  {
    uint32_t wm = mk;
#pragma unroll
    for (int o = 32; o >= 1; o >>= 1) wm = max(wm, (uint32_t)__shfl_xor((int)wm, o, 64));
    const int m = (p.K + kTkWaves - 1) / kTkWaves;  // 1 .. 16
    uint32_t t = 0;  // the wave's m-th largest lane maximum
    for (int b = SKey<T>::kBits - 1; b >= 0; --b) {
      const uint32_t c = t | (1u << b);
      if (__builtin_popcountll(__builtin_amdgcn_ballot_w64(mk >= c)) >= m) t = c;
    }
    if (lane == 0) {
      s_wmax[wave] = wm;
      s_wthr[wave] = t;
    }
    if (tid == 0) s_n = s_ns = s_n2 = 0;
  }
  __syncthreads();
  uint32_t maxkey = 0, bound = 0xFFFFFFFFu;
#pragma unroll
  for (int w = 0; w < kTkWaves; ++w) {
    maxkey = max(maxkey, s_wmax[w]);
    bound = min(bound, s_wthr[w]);
  }
  const float mc = max_c<T>(p, maxkey);
  auto weight = [&](uint32_t key) {
    return weight_of(SKey<T>::val(SKey<T>::bits_of_key(key)), p.c, mc);
  };
  const u64 wmax = weight(maxkey);  // 2^40 up to the rounding of max * c
  if (wmax == 0) {  // no positive weight (an infinite or NaN maximum)
    if (tid == 0) p.out[row] = -1;
    return;
  }
  if (wmax > 1ull << 41) {  // that rounding is no longer small: sums might wrap
    if (tid == 0) p.todo[row] = 1;
    return;
  }

  // ---- collect the logits at or above the bound: first the slots that hold
  //      any (places by ballots, one counter update per wave), then, a thread
  //      per element of those, the logits ----
  auto collect = [&](uint32_t key0) {
    const int o0 = (int)(key0 - (SKey<T>::kBits == 16 ? 0x8000u : 0x80000000u));
    const int thr = o0 == 0 ? -1 : o0;  // both zeros
    auto place = [&](uint32_t* counter, uint32_t count) {  // wave-uniform count > 0
      uint32_t at = 0;
      if (lane == 0) at = atomicAdd(counter, count);
      return (uint32_t)__builtin_amdgcn_readfirstlane((int)at);
    };
    auto below = [&](uint64_t bits) {  // bits of lanes before this one
      return __builtin_amdgcn_mbcnt_hi((uint32_t)(bits >> 32),
                                       __builtin_amdgcn_mbcnt_lo((uint32_t)bits, 0u));
    };
    auto keep_slots = [&](auto n_slots, int s_first, auto&& data) {  // slots s_first + 1024 j
      constexpr int N = decltype(n_slots)::value;
      uint64_t hit[N];
      uint32_t count = 0;
#pragma unroll
      for (int j = 0; j < N; ++j) {
        const bool in = s_first + j * kTkThreads < r.slots;
        hit[j] = __builtin_amdgcn_ballot_w64(in && TkBits<T>::max8(data(j)) >= thr);
        count += (uint32_t)__builtin_popcountll(hit[j]);
      }
      if (count == 0) return;
      uint32_t at = place(&s_ns, count);
#pragma unroll
      for (int j = 0; j < N; ++j) {
        if (hit[j] == 0) continue;
        const uint32_t mine = at + below(hit[j]);
        if ((hit[j] >> lane & 1) && mine < kTkSlotCap) {
          s_slot[mine] = (uint32_t)(s_first + j * kTkThreads);
#pragma unroll
          for (int i = 0; i < DW; i += 4)
            *reinterpret_cast<u32x4*>(&s_raw[mine][i]) =
                u32x4{data(j)[i], data(j)[i + 1], data(j)[i + 2], data(j)[i + 3]};
        }
        at += (uint32_t)__builtin_popcountll(hit[j]);
      }
    };
    if constexpr (HELD) {
      keep_slots(std::integral_constant<int, kTkSlots>{}, tid,
                 [&](int j) -> const uint32_t* { return held[j]; });
    } else {
      for (int s0 = tid; s0 - tid < r.slots; s0 += kBatch * kTkThreads) {
        uint32_t d[kBatch][DW];
#pragma unroll
        for (int b = 0; b < kBatch; ++b)
          r.load_ordered(min(s0 + b * kTkThreads, r.slots - 1), d[b]);
        keep_slots(std::integral_constant<int, kBatch>{}, s0,
                   [&](int j) -> const uint32_t* { return d[j]; });
      }
    }
    __syncthreads();
    const int elems = 8 * (int)min(s_ns, (uint32_t)kTkSlotCap);
    for (int q0 = wave * 64; q0 < elems; q0 += kTkThreads) {
      const int q = q0 + lane;
      const int sl = min(q, elems - 1) >> 3;
      const int i = q & 7;
      int o;
      if constexpr (sizeof(T) == 2) {
        const uint32_t d = s_raw[sl][i >> 1];
        o = (int)(short)(i & 1 ? d >> 16 : d & 0xFFFFu);
      } else {
        o = (int)s_raw[sl][i];
      }
      const int e = r.first((int)s_slot[sl]) + i;
      const uint64_t hit =
          __builtin_amdgcn_ballot_w64(q < elems && o >= thr && e >= 0 && e < r.V);
      if (hit == 0) continue;
      const uint32_t at = place(&s_n, (uint32_t)__builtin_popcountll(hit)) + below(hit);
      if ((hit >> lane & 1) && at < kTkCap) {
        s_key[at] = tk_key<T>(o);
        s_idx[at] = (uint32_t)e;
      }
    }
    __syncthreads();
  };
  collect(bound);
  if (s_ns > kTkSlotCap || s_n > kTkCap) {
    // leave out what has no weight (masked logits): a key whose exponent is
    // below -41 weighs less than 2^-40
    uint32_t lo = 0, hi = maxkey;
    while (hi - lo > 1) {
      const uint32_t mid = lo + (hi - lo) / 2;
      const float v = SKey<T>::val(SKey<T>::bits_of_key(mid));
      if (__builtin_fmaf(v, p.c, -mc) >= -41.f) hi = mid;
      else lo = mid;
    }
    if (hi <= bound) {  // nothing to leave out
      if (tid == 0) p.todo[row] = 1;
      return;
    }
    __syncthreads();
    if (tid == 0) s_n = s_ns = 0;
    __syncthreads();
    collect(hi);
    if (s_ns > kTkSlotCap || s_n > kTkCap) {
      if (tid == 0) p.todo[row] = 1;
      return;
    }
  }
  const int n = (int)s_n;

  // ---- the K-th largest key (fewer than K collected: all are kept) ----
  uint32_t tk = 0;
  if (n > p.K) {
    uint32_t need = (uint32_t)p.K;
    for (int shift = SKey<T>::kBits - 8; shift >= 0; shift -= 8) {
      if (tid < kBins) s_hist[tid] = 0;
      __syncthreads();
      for (int i = tid; i < n; i += kTkThreads) {
        const uint32_t k = s_key[i];
        if (shift == SKey<T>::kBits - 8 || (k >> (shift + 8)) == tk)
          atomicAdd(&s_hist[(k >> shift) & 0xFFu], 1u);
      }
      __syncthreads();
      if (wave == 0) {
        uint32_t h[4], sum = 0;
#pragma unroll
        for (int j = 0; j < 4; ++j) sum += h[j] = s_hist[4 * lane + j];
        uint32_t incl = sum;
#pragma unroll
        for (int o = 1; o < 64; o <<= 1) {
          const uint32_t y = __shfl_up(incl, o, 64);
          if (lane >= o) incl += y;
        }
        uint32_t above = __shfl(incl, 63, 64) - incl;  // in bins above this lane's
        const uint64_t reach = __builtin_amdgcn_ballot_w64(above + sum >= need);
        if (lane == 63 - __builtin_clzll(reach)) {  // the highest lane that reaches (one does)
          int j = 3;
          while (j > 0 && above + h[j] < need) above += h[j--];
          s_bin = 4 * lane + j;
          s_above = above;
        }
      }
      __syncthreads();
      tk = (tk << 8) | s_bin;
      need -= s_above;
    }
  }

  // ---- the tokens kept by top-k, in place at the front of the lists ----
  uint32_t ck[kTkCap / kTkThreads], ci[kTkCap / kTkThreads];
#pragma unroll
  for (int j = 0; j < kTkCap / kTkThreads; ++j) {
    const int i = tid + j * kTkThreads;
    ck[j] = i < n ? s_key[i] : 0u;
    ci[j] = i < n ? s_idx[i] : 0u;
  }
  __syncthreads();
#pragma unroll
  for (int j = 0; j < kTkCap / kTkThreads; ++j) {
    if (tid + j * kTkThreads < n && ck[j] >= tk) {
      const uint32_t at = atomicAdd(&s_n2, 1u);
      if (at < kTkKeep) {
        s_key[at] = ck[j];
        s_idx[at] = ci[j];
        s_w[at] = weight(ck[j]);
      }
    }
  }
  __syncthreads();
  const int n2 = (int)s_n2;
  if (n2 > kTkKeep) {
    if (tid == 0) p.todo[row] = 1;
    return;
  }
  __syncthreads();  // (s_n2 is read before anything below)

  // The sums over the kept tokens: 2^lg threads per token (adjacent lanes),
  // each a share of the tokens, so that every thread works on a few terms.
  int lg = 0;
  while (lg < 6 && n2 << (lg + 1) <= kTkThreads) ++lg;
  const int tok = tid >> lg, part = tid & ((1 << lg) - 1), step = 1 << lg;
  uint32_t key = 0, idx = 0;
  u64 w = 0;
  if (tok < n2) {
    key = s_key[tok];
    idx = s_idx[tok];
    w = s_w[tok];
  }
  auto group_sum = [&](u64 v) {
    for (int o = 1; o < step; o <<= 1)
      v += ((u64)(uint32_t)__shfl_xor((int)(uint32_t)(v >> 32), o, 64) << 32) +
           (uint32_t)__shfl_xor((int)(uint32_t)v, o, 64);
    return v;
  };

  // ---- top-p: a token stays while the mass before it, in order of falling
  //      key, then index, is below top_p Z ----
  if (p.P < 1.0) {
    u64 z = 0, above = 0;
    if (tok < n2) {
#pragma unroll 4
      for (int j = part; j < n2; j += step) {
        const uint32_t kj = s_key[j];
        const u64 wj = s_w[j];
        z += wj;
        // (a tie weighs the same: the ties before this token as mass too)
        above += kj > key || (kj == key && s_idx[j] < idx) ? wj : 0;
      }
    }
    z = group_sum(z);
    above = group_sum(above);
    __syncthreads();
    if (tok < n2) {
      if (!((double)above < p.P * (double)z)) w = 0;
      if (part == 0) s_w[tok] = w;
    }
    __syncthreads();
  }

  // ---- the draw: inverse CDF in vocabulary order ----
  u64 z = 0, pre = 0;
  if (tok < n2) {
#pragma unroll 4
    for (int j = part; j < n2; j += step) {
      const u64 wj = s_w[j];
      z += wj;
      pre += s_idx[j] < idx ? wj : 0;
    }
  }
  z = group_sum(z);
  pre = group_sum(pre);
  if (tok < n2 && part == 0) {
    u64 target = (u64)((double)u * (double)z);
    if (target >= z) target = z - 1;  // (z > 0: the largest logit is kept)
    if (w > 0 && pre <= target && target < pre + w) p.out[row] = idx;
  }
}

// Where topk_kernel is ahead of the staged launches (graph replay, both sides,
// 10 vocabularies of 1000 - 200,000, 1 - 1024 rows, eight settings): its
// workgroups take a CU each and their sums grow with K^2, while the staged
// launches grow with the elements.
// * K to 128 (fp32, whose staged form has four levels a filter instead of two:
//   200): 0.7 - 1.0 of the staged time at few elements, 0.26 at 128 x 151,936.
//   More rows than CUs take a second round, which pays from about 8000 columns
//   (512 x 1000 bf16, top-k 50: 26.5 -> 29 us; 1024 x 5000: 44 -> 62).
// * K to 200 (fp32 256) from 2^20 elements: 1 x 128,256 bf16, top-k 200: 36 -> 37,
//   16 x 128,256: 44 -> 38; K to 256 from 2^22 (4 x 151,936: 41 -> 51, 32 x
//   151,936: 57 -> 52).
// * bf16 without top-p from 2^19: that staged form has five launches, and an
//   eager call is bound by their number, one more here (2 x 128,256: 25.4 ->
//   26.5 - 28.4, 4 x 151,936: 0.96 of the time; in a graph 0.8 - 0.9 at both).
bool topk_ahead(int rows, int V, int K, int esz, bool top_p) {
  if (K <= 0 || K > kTkMaxK) return false;
  constexpr int kCus = 256;
  const int64_t elements = (int64_t)rows * V;
  if (esz == 2 && !top_p && elements < 1 << 19) return false;
  if (K <= (esz == 4 ? 200 : 128)) return rows <= kCus || V >= 8192;
  if (K <= 200 || esz == 4)
    return elements >= 1 << 20 && (rows <= kCus || V >= 16384);
  return elements >= 1 << 22 && (rows <= kCus || V >= 32768);
}

struct SLayout {
  int nch, cs;
  int64_t cmax_off, hcnt_off, hmass_off, st_off, csum_off, ceq_off;
  int64_t staged;  // bytes of the staged launches; then the row marks of topk_kernel
  int64_t total;
};

SLayout slayout(int rows, int V) {
  SLayout L;
  const int max_ch = std::max(1, std::min(kSMaxChunks, (V + 1023) / 1024));
  L.nch = std::max(1, std::min(max_ch, (kSTargetWgs + rows - 1) / std::max(1, rows)));
  L.cs = ((V + L.nch - 1) / L.nch + 7) / 8 * 8;
  L.nch = (V + L.cs - 1) / L.cs;
  auto al = [](int64_t x) { return (x + 255) / 256 * 256; };
  L.cmax_off = kWorkspaceHeaderBytes;  // the acceptance header stays untouched
  L.hcnt_off = L.cmax_off + al((int64_t)rows * kSMaxChunks * 8);
  L.hmass_off = L.hcnt_off + al((int64_t)rows * kMaxStages * kBins * 4);
  L.st_off = L.hmass_off + al((int64_t)rows * kMaxStages * kBins * 8);
  L.csum_off = L.st_off + al((int64_t)rows * (kMaxStages + 1) * sizeof(SmpState));
  L.ceq_off = L.csum_off + al((int64_t)rows * kSMaxChunks * 8);
  L.staged = L.ceq_off + al((int64_t)rows * kSMaxChunks * 4);
  L.total = L.staged + al((int64_t)rows * 4);
  return L;
}

template <typename T>
int32_t launch_sample(const SmpParams& p, bool vec, hipStream_t s) {
  if (p.todo) {
    // (a bf16 row of 8 head elements at most and whole slots after them)
    if (sizeof(T) == 2 && p.V <= 8 * (kTkThreads * kTkSlots - 1))
      hipLaunchKernelGGL((topk_kernel<T, sizeof(T) == 2>), dim3(p.rows), dim3(kTkThreads), 0, s, p);
    else
      hipLaunchKernelGGL((topk_kernel<T, false>), dim3(p.rows), dim3(kTkThreads), 0, s, p);
    if (int32_t rc = launch_status("sample topk_kernel")) return rc;
  }
  const dim3 g(p.nch, p.rows);
  hipLaunchKernelGGL((max_kernel<T>), g, dim3(kSThreads), 0, s, p, vec);
  int32_t rc = launch_status("sample max_kernel");
  if (rc || p.greedy) {
    if (rc) return rc;
    hipLaunchKernelGGL((select_kernel<T>), dim3(p.rows), dim3(kSThreads), 0, s, p, vec);
    return launch_status("sample select_kernel");
  }
  for (int st = 0; st < p.nk + p.np; ++st) {
    if (st < p.nk) hipLaunchKernelGGL((hist_kernel<T, true>), g, dim3(kSThreads), 0, s, p, st, vec);
    else hipLaunchKernelGGL((hist_kernel<T, false>), g, dim3(kSThreads), 0, s, p, st, vec);
    rc = launch_status("sample hist_kernel");
    if (rc) return rc;
  }
  hipLaunchKernelGGL((sums_kernel<T>), g, dim3(kSThreads), 0, s, p, vec);
  rc = launch_status("sample sums_kernel");
  if (rc) return rc;
  hipLaunchKernelGGL((select_kernel<T>), dim3(p.rows), dim3(kSThreads), 0, s, p, vec);
  return launch_status("sample select_kernel");
}

}  // namespace
}  // namespace nsg

using namespace nsg;

extern "C" int64_t nsg_sample_workspace_bytes(int32_t rows, int32_t vocab) {
  if (rows < 0 || vocab <= 0) return -1;
  return slayout(rows, vocab).total;
}

extern "C" int32_t nsg_sample(const void* logits, int64_t row_stride, int32_t logits_dtype,
                              int32_t rows, int32_t vocab, float temperature, int32_t top_k,
                              float top_p, const float* uniforms, int64_t uniform_stride,
                              int64_t* tokens, void* workspace, int64_t workspace_bytes,
                              nsg_stream_t stream) {
  NSG_CHECK_ARG(rows >= 0 && rows <= kMaxRows, "rows %d outside [0, %d]", rows, kMaxRows);
  NSG_CHECK_ARG(vocab > 0, "vocab %d", vocab);
  NSG_CHECK_ARG(logits_dtype == 0 || logits_dtype == 1, "logits_dtype %d (0 bf16, 1 fp32)",
                logits_dtype);
  const bool greedy = temperature < 1e-6f;
  NSG_CHECK_ARG(greedy || (top_p > 0.f && top_p == top_p),
                "top_p %g must be in (0, 1] (1 = off)", (double)top_p);
  if (rows == 0) {
    clear_error();
    return NSG_OK;
  }
  NSG_CHECK_ARG(logits && tokens && workspace, "null pointer argument");
  NSG_CHECK_ARG(greedy || uniforms, "uniforms required when temperature > 0");
  NSG_CHECK_ARG(row_stride >= vocab, "row_stride %lld < vocab %d", (long long)row_stride, vocab);
  const SLayout L = slayout(rows, vocab);
  if (workspace_bytes < L.staged) {
    set_error("workspace has %lld bytes, needs %lld", (long long)workspace_bytes,
              (long long)L.staged);
    return NSG_ERR_WORKSPACE;
  }
  SmpParams p{};
  p.x = logits;
  p.stride = row_stride;
  p.rows = rows;
  p.V = vocab;
  p.greedy = greedy ? 1 : 0;
  p.c = greedy ? 0.f : kLog2eS / temperature;
  p.K = (!greedy && top_k > 0 && top_k < vocab) ? top_k : 0;
  p.P = (!greedy && top_p < 1.f) ? (double)top_p : 1.0;
  p.u = uniforms;
  p.u_stride = uniform_stride;
  p.out = tokens;
  p.nch = L.nch;
  p.cs = L.cs;
  const int esz = logits_dtype == 0 ? 2 : 4;
  p.levels = esz;  // one key byte per level
  p.nk = p.K > 0 ? p.levels : 0;
  p.np = p.P < 1.0 ? p.levels : 0;
  char* ws = static_cast<char*>(workspace);
  p.cmax = reinterpret_cast<uint2*>(ws + L.cmax_off);
  p.hcnt = reinterpret_cast<uint32_t*>(ws + L.hcnt_off);
  p.hmass = reinterpret_cast<u64*>(ws + L.hmass_off);
  p.st = reinterpret_cast<SmpState*>(ws + L.st_off);
  p.csum = reinterpret_cast<u64*>(ws + L.csum_off);
  p.ceq = reinterpret_cast<uint32_t*>(ws + L.ceq_off);
  // (a workspace without room for the marks: the staged launches alone)
  p.todo = topk_ahead(rows, vocab, p.K, esz, p.P < 1.0) && workspace_bytes >= L.total
               ? reinterpret_cast<uint32_t*>(ws + L.staged)
               : nullptr;
  const bool vec = (reinterpret_cast<uintptr_t>(logits) % 16 == 0) &&
                   ((row_stride * esz) % 16 == 0);
  hipStream_t s = static_cast<hipStream_t>(stream);
  return logits_dtype == 0 ? launch_sample<bf16>(p, vec, s) : launch_sample<float>(p, vec, s);
}
