// What the attention kernels share: their parameters, the LDS tile swizzles
// and the small device helpers.
#pragma once

#include <type_traits>

#include "common.hpp"

namespace nsg {

constexpr float kMaskVal = -1.0e30f; // finite "minus infinity" (no inf - inf)
constexpr float kLazyRescale = 8.f;  // rescale O only when a row max grows by > 2^8
constexpr int kMaxItemPages = 1024;  // page ids one work item may span

typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
typedef short v4i16 __attribute__((ext_vector_type(4)));
typedef short v8i16 __attribute__((ext_vector_type(8)));

struct AttnParams {
  const bf16* q;
  const bf16* kc;
  const bf16* vc;
  bf16* out;
  const int* qo_indptr;
  const int* kv_indptr;
  const int* kv_indices;
  const int* kv_last;
  const int* work;
  int num_work;
  int Hq, Hkv, G, log2P, num_pages, causal;
  float scale_log2;
  int* flags;
  float* partials;
};

__device__ __forceinline__ bf16x8 load_bf16x8(const bf16* p) {
  u32x4 v = *reinterpret_cast<const u32x4*>(p);
  return __builtin_bit_cast(bf16x8, v);
}

typedef float floatx2 __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));

// Two floats -> packed bf16 pair (v_cvt_pk_bf16_f32, round to nearest even).
__device__ __forceinline__ uint32_t cvt_pk_bf16(float lo, float hi) {
  return __builtin_bit_cast(uint32_t, __builtin_convertvector(floatx2{lo, hi}, bf16x2));
}

// Transposing LDS reads of the V^T fragments, in asm.  Written through the
// builtin, every such read after a global_load_lds gets a conservative
// vmcnt(0) from the compiler (it cannot tell the read from the ring slots
// still being filled), which stalls each step until every copy in flight has
// landed; the ring's own waits (vmcnt per step plus the barrier) already
// order these reads.  tr_issue starts the two reads of one d tile; tr_wait
// waits until at most N LDS operations are outstanding, after which the
// tile's registers (tied operands, so that the compiler reads them only
// after the wait) hold the data.  LDS operations complete in order, so the
// reads of tile dt are done once those of tile dt + 1 are the only ones left.
__device__ __forceinline__ void tr_issue(v4i16& lo, v4i16& hi, uint32_t a0, uint32_t a1) {
  asm volatile("ds_read_b64_tr_b16 %0, %2\n\tds_read_b64_tr_b16 %1, %3"
               : "=&v"(lo), "=&v"(hi)
               : "v"(a0), "v"(a1)
               : "memory");
}
template <int N>
__device__ __forceinline__ void tr_wait(v4i16& lo, v4i16& hi) {
  asm volatile("s_waitcnt lgkmcnt(%2)" : "+v"(lo), "+v"(hi) : "n"(N) : "memory");
}


// LDS tile swizzles: 16-byte chunk c of token row t is stored at physical
// chunk c ^ swz(t).  K fragments read one logical chunk of 16 consecutive
// tokens (needs distinct banks across t).  A V^T transposing read takes one
// 32-byte chunk pair from each of 16 rows t = 4g + j (g, j < 4): the pair
// index is XORed with a function of t that spreads those 16 rows over every
// 32-byte bank window (with 256-byte bank rows: 2 rows per window, the
// minimum).
template <int D>
__device__ __forceinline__ int swz_k(int t) {
  if constexpr (D == 64) return (t >> 1) & 7;  // 128-byte rows: two rows per bank cycle
  return t & 15;                               // 256-byte rows: one row per bank cycle
}
template <int D>
__device__ __forceinline__ int swz_v(int t) {
  if constexpr (D == 64) return 2 * ((t >> 1) & 3);  // odd rows sit in the other half-row
  return 2 * (t & 7);
}


// The prefill kernel (prefill_attention.hip): unsplit work items of up to
// 32 * waves query rows, waves = 4, or 8 at head dim 128.
int32_t launch_prefill_attn(int head_dim, int waves, int num_work, const AttnParams& prm,
                            hipStream_t stream);

}  // namespace nsg
