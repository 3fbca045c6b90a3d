// What the gfx950 attention kernels share: argument block, LDS tile layout, matrix instruction and fp8 packing.
#ifndef FA8_DEVICE_H_
#define FA8_DEVICE_H_
#include <hip/hip_runtime.h>

#include <cstdint>

#include "fa8_api.h"

namespace fa8 {

typedef int v2i __attribute__((ext_vector_type(2)));
typedef int v4i __attribute__((ext_vector_type(4)));
typedef int v8i __attribute__((ext_vector_type(8)));
typedef unsigned v4u __attribute__((ext_vector_type(4)));
typedef float v4f __attribute__((ext_vector_type(4)));
typedef float v16f __attribute__((ext_vector_type(16)));
typedef _Float16 v4h __attribute__((ext_vector_type(4)));

#define LDS_PTR(T, p) ((__attribute__((address_space(3))) T*)(p))

constexpr int kQBlock = 128;   // query rows per workgroup
constexpr int kQWave = 32;     // query rows per wavefront
constexpr int kKvBlock = 64;   // kv rows per online-softmax step
constexpr int kThreads = 256;  // 4 wavefronts
constexpr int kVersion = 7;
// main loops (template parameter LOOP of the kernel)
constexpr int kLoopRolling = 0, kLoopPipelined = 1, kLoopDense = 2, kLoopDenseRagged = 3;

struct KernelArgs {
  const uint8_t* q;
  const uint8_t* k;
  const uint8_t* v;
  void* o;
  float* lse;  // optional
  int heads, seqlen_q, seqlen_k, n_qblocks, bh_total;
  int kv_group;      // q heads per k/v head
  int interleave;    // causal: how many heads deal their q blocks alternately (see decode_block)
  int causal_shift;  // key j is visible to query i when j <= i + causal_shift
  float scale_log2;  // softmax_scale * log2(e)
  int whole_lines;   // O leaves as whole lines
  long long q_bs, q_hs, q_rs;
  long long k_bs, k_hs, k_rs;
  long long v_bs, v_hs, v_rs;
  long long o_bs, o_hs, o_rs;
  long long lse_bs, lse_hs;
};

// Arguments of the kernels for small launches, packed: an argument block of more than 112 bytes makes the launch itself slower on the
// host (2.75 us up to 112 bytes, 3.4 - 3.6 us from 120 on; an empty kernel in a loop).  Strides are 32-bit, in units of 16 elements
// (q, k, v) and of 4 elements (o); `mode` holds flags, log2 of the number of q heads per k/v head (31: no power of two) and the number
// itself.
constexpr unsigned kSharedCausal = 1, kSharedBottomRight = 2, kSharedFp8Out = 4, kSharedLines = 8;
constexpr unsigned kSharedShift = 8;  // bits 8..12: log2 of the group, 31 if it is no power of two
constexpr unsigned kSharedGroup = 16;

inline bool packable(const Fa8FwdParams* p) {
  const long long most16 = 16LL << 32, most4 = 4LL << 32;
  const long long in[] = {p->q_batch_stride, p->q_head_stride, p->q_row_stride, p->k_batch_stride, p->k_head_stride, p->k_row_stride,
                          p->v_batch_stride, p->v_head_stride, p->v_row_stride};
  for (long long s : in)
    if (s >= most16) return false;
  if (p->o_batch_stride >= most4 || p->o_head_stride >= most4 || p->o_row_stride >= most4) return false;
  if (p->lse_batch_stride >= 1LL << 32 || p->lse_head_stride >= 1LL << 32) return false;
  const int group = p->heads_k > 0 ? p->heads / p->heads_k : 1;
  return group < 1 << 16 && (long long)group * p->seqlen_q < 1LL << 30;
}
inline unsigned pack_mode(const Fa8FwdParams* p) {
  const int group = p->heads_k > 0 ? p->heads / p->heads_k : 1;
  unsigned shift = 31;
  for (unsigned i = 0; i < 16; ++i)
    if (group == 1 << i) shift = i;
  return (p->is_causal ? kSharedCausal : 0) | (p->causal_align == FA8_CAUSAL_BOTTOM_RIGHT ? kSharedBottomRight : 0) |
         (p->out_dtype != FA8_OUT_FP16 ? kSharedFp8Out : 0) | shift << kSharedShift | (unsigned)group << kSharedGroup;
}

#if defined(__HIP_DEVICE_COMPILE__)
// 16 bytes of a row of o (8-byte aligned), written through the L2 at once.  Left dirty there they are written back when the kernel ends; asked not to
// be kept anywhere (non-temporal) they leave the sooner, but the kernel that reads o next finds them in HBM instead of the memory-side cache: its
// loss is more than the call's gain.  us, dirty -> not kept -> through, the call and the call with a copy of o after it: 8 x 32 heads, 1024 keys, head dim 128, causal
// 69.2, 89.7 -> 63.7, 93.8 -> 69.0, 88.2; 4 x 16 heads, 1024 keys, head dim 64 20.5, 24.0 -> 19.4, 24.5 -> 19.5, 23.3; 2 x 32 heads, 4096 keys 300.0, 322.7 ->
// 298.5, 329.0 -> 299.4, 324.0; 16 heads, 2048 keys, head dim 256, causal 38.8, 44.6 -> 37.0, 47.3 -> 38.5, 44.8.
__device__ __forceinline__ void store_row_chunk(uint8_t* at, v4i x) {
  __builtin_amdgcn_global_store_b128((__attribute__((address_space(1))) v4u*)at, (v4u)x, "agent");
}
#endif

// LDS row r (0..63) of a K tile holds kv row kv_of_lds_row(r) of the block.  With this order the 16
// accumulator registers a lane gets from S^T sub-tile t (rows 8a+4h+b of the 32x32 result, h = lane/32)
// are kv rows 32h+16t+(4a+b): exactly the bytes 16t..16t+15 of the lane's B operand in the PV MFMA.
__device__ __forceinline__ int kv_of_lds_row(int r) {
  const int t = r >> 5, a = (r >> 3) & 3, h = (r >> 2) & 1, b = r & 3;
  return 32 * h + 16 * t + 4 * a + b;
}

// Swizzle: a tile is an array of 128-byte lines of eight 16-byte chunks.  A row of D bytes is two lines (D = 256),
// one line (128), half a line (64) or a quarter (32).  The chunk position inside its line is XORed with a key
// taken from the row (line) number, chosen so that the eight lanes the LDS serves together (eight consecutive
// rows, same chunk) fall on eight different positions, for the K reads and for the transposing V reads alike.
template <int D, bool IS_V>
__device__ __forceinline__ int tile_offset(int row, int chunk) {
  if constexpr (D == 256) {
    const int key = IS_V ? (row & 7) : ((row & 7) ^ ((row >> 3) & 1));
    return row * 256 + ((chunk >> 3) << 7) + (((chunk & 7) ^ key) << 4);
  } else if constexpr (D == 128) {
    const int key = IS_V ? (row & 7) : ((row & 7) ^ ((row >> 3) & 1));
    return row * 128 + ((chunk ^ key) << 4);
  } else if constexpr (D == 64) {
    const int line = row >> 1;
    const int key = IS_V ? (line & 3) : ((line & 3) ^ ((line >> 2) & 1));
    return line * 128 + ((((row & 1) << 2) | (chunk ^ key)) << 4);
  } else {
    static_assert(D == 32, "head dims: 32, 64, 128, 256");
    const int line = row >> 2;
    return line * 128 + ((((row & 3) << 1) | (chunk ^ (line & 1))) << 4);
  }
}

// Inverse of tile_offset for the copy engine: which (row, chunk) lives at 16-byte slot `slot`.
template <int D, bool IS_V>
__device__ __forceinline__ void tile_slot_decode(int slot, int& row, int& chunk) {
  if constexpr (D == 256) {
    row = slot >> 4;
    const int key = IS_V ? (row & 7) : ((row & 7) ^ ((row >> 3) & 1));
    chunk = (slot & 8) | ((slot & 7) ^ key);
  } else if constexpr (D == 128) {
    row = slot >> 3;
    const int key = IS_V ? (row & 7) : ((row & 7) ^ ((row >> 3) & 1));
    chunk = (slot & 7) ^ key;
  } else if constexpr (D == 64) {
    const int line = slot >> 3, w = slot & 7;
    const int key = IS_V ? (line & 3) : ((line & 3) ^ ((line >> 2) & 1));
    row = line * 2 + (w >> 2);
    chunk = (w & 3) ^ key;
  } else {
    const int line = slot >> 3, w = slot & 7;
    row = line * 4 + (w >> 1);
    chunk = (w & 1) ^ (line & 1);
  }
}

// v_permlane32_swap exchanges lanes 32-63 of its first operand with lanes 0-31 of its second.  Fed the same
// value x twice it returns {x of the low half-lane, x of the high half-lane} in every lane of a query.
typedef unsigned v2u __attribute__((ext_vector_type(2)));
__device__ __forceinline__ float lane32_max(float x) {
  const v2u r = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  // median(a, b, +inf) = max(a, b) in one instruction (fmaxf would first quiet both operands); the +inf is made opaque to
  // the optimiser, which would otherwise turn the median back into that max
  float inf = INFINITY;
  asm("" : "+v"(inf));
  return __builtin_amdgcn_fmed3f(__uint_as_float(r[0]), __uint_as_float(r[1]), inf);
}
__device__ __forceinline__ float lane32_sum(float x) {
  const v2u r = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}

// max of two floats that are no signalling NaN (fmaxf first quiets operands that come from memory, an instruction each)
__device__ __forceinline__ float max2(float a, float b) {
  float r;
  asm("v_max_f32 %0, %1, %2" : "=v"(r) : "v"(a), "v"(b));
  return r;
}

// max of three floats; the compiler fuses the pair into one v_max3_f32.
__device__ __forceinline__ float max3(float a, float b, float c) { return __builtin_fmaxf(__builtin_fmaxf(a, b), c); }

template <bool E5M2>
__device__ __forceinline__ v16f mfma_fp8(const v8i& a, const v8i& b, const v16f& c) {
  if constexpr (E5M2)
    return __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(a, b, c, 1, 1, 0, 0, 0, 0);
  else
    return __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(a, b, c, 0, 0, 0, 0, 0, 0);
}

template <bool E5M2>
__device__ __forceinline__ int pack4_fp8(float a, float b, float c, float d) {
  int r;
  asm volatile("" : "=v"(r));  // any value will do (both 16-bit halves are overwritten below): defines r, emits nothing
  if constexpr (E5M2) {
    r = __builtin_amdgcn_cvt_pk_bf8_f32(a, b, r, false);
    r = __builtin_amdgcn_cvt_pk_bf8_f32(c, d, r, true);
  } else {
    r = __builtin_amdgcn_cvt_pk_fp8_f32(a, b, r, false);
    r = __builtin_amdgcn_cvt_pk_fp8_f32(c, d, r, true);
  }
  return r;
}

}  // namespace fa8
#endif  // FA8_DEVICE_H_
