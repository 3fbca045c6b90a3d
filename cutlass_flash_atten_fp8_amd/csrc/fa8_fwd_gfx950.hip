// FP8 flash-attention forward for gfx950 (MI355X): kernels and the C-ABI launcher (libfa8.so).
//
// One workgroup = 4 wavefronts = 128 query rows of one (batch, head); every wavefront owns 32 query
// rows and the whole head dimension (a multiple of 32 up to 256: the bucket sizes of the reference's
// dispatch, csrc/static_switch.h:50-77).  KV is walked in ascending blocks of 64 rows, the block size
// the reference instantiates (kBlockM = kBlockN = 64, reference csrc/flash_attention.cu:624), so the
// running max that P is quantised against evolves exactly as in the reference loop
// (csrc/flash_attention.cu:468-534).
//
// Formulation (different from the reference, which computes S = Q K^T with m16n8k32 atoms,
// csrc/mma_sm89.hpp:10-35):
//   * S^T = K Q^T with v_mfma_f32_32x32x64_f8f6f4 (A = K tile from LDS, B = Q held in registers).
//     In the 32x32 accumulator layout a lane owns ONE query column and 16 kv rows, so the online
//     softmax row max / row sum (reference csrc/utils.h:22-98 quad butterflies) are in-register
//     reductions plus one v_permlane32_swap.
//   * O^T = V^T P^T with the same instruction (A = V^T, B = P^T).  The fp32 -> fp8 P registers of a
//     lane already are a valid B operand when the K tile rows are stored in LDS in a permuted order
//     (kv_of_lds_row below); this replaces the reference's accumulator-to-A-operand reshuffle
//     (csrc/reg2reg.h:31-96).  V^T fragments come from the row-major V tile in LDS through the
//     transposing LDS read ds_read_b64_tr_b8, so V is consumed as [B,H,N,d] with no extra pass.
//   * K and V tiles go HBM -> LDS with buffer_load_dwordx4 ... lds (no register staging), two or three
//     stages, one barrier per KV block; 16-byte chunks are XOR-swizzled against bank conflicts,
//     the swizzle being applied on the global-address side of the copy.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <atomic>
#include <cmath>
#include <cstdint>
#include <cstdlib>
#include <type_traits>

#include "fa8_device.h"
#include "fa8_launch.h"

// wavefronts per SIMD the kernels are compiled for: 3 (at most 168 VGPRs per lane) up to head dim 128, 2 (256 VGPRs:
// the output accumulators alone take 128) for head dim 256; the pipelined loop 2; the dense loop 3 (head dim 64: 4)
#define FA8_WAVES_PER_EU(D, LOOP) ((LOOP) == 1 ? 2 : ((LOOP) >= 2 ? ((D) == 64 ? 4 : 3) : ((D) > 128 ? 2 : 3)))

namespace {

using namespace fa8;

// Workgroup id -> (batch*head, q block).  Workgroups are dealt to the 8 XCDs round-robin by id; when
// batch*heads is a multiple of 8 all q blocks of one head are kept on one XCD so its K/V stay in that
// XCD's L2.  Workgroups start in id order.  Full attention: head after head.  Causal: workgroups differ in length
// (q block i walks i+1 of the n q blocks' worth of keys), so the longest come first and `interleave` heads of the XCD
// take turns at every q block: the workgroups that run side by side then have about the same length and the
// short ones fill the end of the launch (head after head, a late head's longest workgroup would start when the
// rest of the chip is already draining).
template <bool CAUSAL>
__device__ __forceinline__ void decode_block(const KernelArgs& a, int id, int& bh, int& qb) {
  int qi;
  if ((a.bh_total & 7) == 0) {
    const int xcd = id & 7, s = id >> 3;
    int hl;  // head index inside this XCD's share of bh_total / 8 heads
    if (CAUSAL) {
      // groups of `interleave` heads (the last group takes what is left)
      const int per_group = a.interleave * a.n_qblocks;
      const int grp = s / per_group, r = s - grp * per_group;
      const int g = min(a.interleave, (a.bh_total >> 3) - grp * a.interleave);
      qi = r / g;
      hl = grp * a.interleave + (r - qi * g);
    } else {
      hl = s / a.n_qblocks;
      qi = s - hl * a.n_qblocks;
    }
    // grouped-query attention: an XCD takes a contiguous range of q heads, so the heads that share a k/v head follow
    // each other on one XCD
    bh = a.kv_group > 1 ? xcd * (a.bh_total >> 3) + hl : hl * 8 + xcd;
  } else if (CAUSAL) {
    qi = id / a.bh_total;  // no head stays on one XCD anyway: all heads take turns
    bh = id - qi * a.bh_total;
  } else {
    bh = id / a.n_qblocks;
    qi = id - bh * a.n_qblocks;
  }
  qb = CAUSAL ? (a.n_qblocks - 1 - qi) : qi;
}

// LOOP selects the main loop; all three perform the same arithmetic in the same order, their results are bitwise equal.
// kLoopRolling: one KV block after the other (S^T, softmax, PV), three wavefronts per SIMD hide each other's latencies.
// kLoopPipelined: software-pipelined for launches that leave a SIMD with two wavefronts or fewer (short sequences, few
// heads): the matrix instructions of the neighbouring blocks (PV of block j-1, S^T of block j+1) are issued between the
// chunks of the softmax of block j, so that one wavefront alone keeps the matrix and the vector pipe busy; about 180
// VGPRs (two wavefronts per SIMD), four LDS stages; every block may be masked.
// kLoopDense: the same pipeline squeezed into 168 VGPRs (three wavefronts per SIMD, three LDS stages) for launches
// in which no block needs a mask (full attention over a whole number of KV blocks): one logits buffer, whose halves are
// refilled by the S^T products of block j+1 as soon as the softmax of block j has turned them into weights.
// kLoopDenseRagged: the same for full attention over keys that end inside a block: the last steps mask.  (A form of its own: as a
// branch of the dense loop's last steps it cost launches of whole blocks 0.5 - 1 %.)
template <int D, bool CAUSAL, bool E5M2, int OUT, bool VT, int LOOP>
__global__ __launch_bounds__(kThreads) __attribute__((amdgpu_waves_per_eu(FA8_WAVES_PER_EU(D, LOOP)))) void fa8_fwd_kernel(
    const KernelArgs a) {
#if defined(__HIP_DEVICE_COMPILE__)  // the body uses device-only types (buffer resources); the host pass only needs the stub
  static_assert(D % 32 == 0 && D >= 32 && D <= 256, "head dims: multiples of 32 up to 256");
  constexpr bool PIPE = LOOP == kLoopPipelined, RAGGED = LOOP == kLoopDenseRagged, DENSE = LOOP == kLoopDense || RAGGED;
  static_assert(LOOP == kLoopRolling || D == 64 || D == 128, "the pipelined loops are built for head dims 64 and 128");
  static_assert(!DENSE || !CAUSAL, "the dense loop masks nothing but the keys past the end");
  // LDS tiles are laid out for the next power of two: rows of DP bytes, of which the first D are used
  constexpr int DP = D <= 32 ? 32 : (D <= 64 ? 64 : (D <= 128 ? 128 : 256));
  constexpr int kTileBytes = kKvBlock * DP;  // one K or V tile
  // copy passes per tile: one pass is 256 lanes x 16 bytes.  A 32-wide tile is half a pass: there wavefronts 0-1 copy
  // K and wavefronts 2-3 copy V in one common pass.
  constexpr bool kSplitPass = kTileBytes < kThreads * 16;
  constexpr int kPasses = kSplitPass ? 1 : kTileBytes / (kThreads * 16);
  constexpr int kKSteps = (D + 63) / 64;  // MFMA k-steps over the head dim for S^T (D % 64 == 32: the last one is half zeros)
  constexpr int kMTiles = D / 32;         // 32-row tiles of O^T
  // LDS stages per operand: three (copies issued two KV blocks ahead) where three workgroups then still fit in the
  // 160 KB of a CU, two for head dims above 128 (2 x 32 KB per workgroup, two workgroups per CU)
  // (the pipelined loop: four, copies issued up to four blocks ahead; the dense loop: three)
  constexpr int kStages = PIPE ? 4 : (D > 128 ? 2 : 3);
  // One LDS object per (stage, operand): the compiler then knows that the asynchronous HBM -> LDS copy into one
  // stage cannot alias the reads of the other stage and does not wait for the copy before those reads.
  __shared__ __attribute__((aligned(1024))) uint8_t k_lds0[kTileBytes];
  __shared__ __attribute__((aligned(1024))) uint8_t k_lds1[kTileBytes];
  __shared__ __attribute__((aligned(1024))) uint8_t k_lds2[kStages >= 3 ? kTileBytes : 16];
  __shared__ __attribute__((aligned(1024))) uint8_t k_lds3[kStages >= 4 ? kTileBytes : 16];
  __shared__ __attribute__((aligned(1024))) uint8_t v_lds0[kTileBytes];
  __shared__ __attribute__((aligned(1024))) uint8_t v_lds1[kTileBytes];
  __shared__ __attribute__((aligned(1024))) uint8_t v_lds2[kStages >= 3 ? kTileBytes : 16];
  __shared__ __attribute__((aligned(1024))) uint8_t v_lds3[kStages >= 4 ? kTileBytes : 16];

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);  // wave-uniform: keep it (and all it feeds) in scalar registers
  const int qn = lane & 31, h = lane >> 5;

  int bh, qb;
  decode_block<CAUSAL>(a, blockIdx.x, bh, qb);
  const int b = bh / a.heads, hd = bh - b * a.heads;
  const int q0 = qb * kQBlock;
  const int q_wave0 = q0 + wave * kQWave;
  const int q_row = q_wave0 + qn;  // this lane's query row
  const uint8_t* qp = a.q + b * a.q_bs + hd * a.q_hs;
  const int hd_kv = a.kv_group == 1 ? hd : hd / a.kv_group;  // grouped-query attention: several q heads per k/v head
  const uint8_t* kp = a.k + b * a.k_bs + hd_kv * a.k_hs;
  const uint8_t* vp = a.v + b * a.v_bs + hd_kv * a.v_hs;
  const float c = a.scale_log2;

  // ---- Q fragment (B operand of S^T = K Q^T): row q_row, bytes [64ks + 32h, +32) ----
  // (D % 64 == 32: the upper half of the last k-step does not exist; those lanes hold zeros and load nothing)
  v8i qf[kKSteps];
  {
    const int qr = min(q_row, a.seqlen_q - 1);
    const uint8_t* src = qp + (long long)qr * a.q_rs;
#pragma unroll
    for (int ks = 0; ks < kKSteps; ++ks) {
      const bool upper_exists = 64 * ks + 32 < D;
      const uint8_t* s8 = src + 64 * ks + (upper_exists ? 32 * h : 0);
      const v4i lo = *(const v4i*)(s8);
      const v4i hi = *(const v4i*)(s8 + 16);
      qf[ks] = {lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
      if (!upper_exists && h) qf[ks] = v8i{0, 0, 0, 0, 0, 0, 0, 0};
    }
  }

  // ---- HBM -> LDS copy: buffer_load_dwordx4 ... lds ----
  // In pass p wavefront w fills LDS bytes [(4p+w)*1024, +1024) of the tile, lane l the 16 bytes at +16l; which
  // (kv row, 16-byte chunk) belongs there follows from the swizzle.  (A 32-wide tile is 2 KB: wavefronts 0-1 fill the K
  // tile, wavefronts 2-3 the V tile.)  The source address is the head's base (buffer resource) + a per-lane byte
  // offset that never changes (VGPR) + the block's byte offset (SGPR): no vector ALU work per block.  The resource
  // ends with the last kv row, so rows past the end of a ragged last block read 0.  LDS chunks that lie past the
  // head dim (D < DP) get an offset beyond any resource and read 0 as well: the K fragments of a half k-step rely on it.
  constexpr unsigned kNoSource = 0x80000000u;
  auto copy_segment = [&](int p) __attribute__((always_inline)) { return kSplitPass ? (wave & 1) : (p * 4 + wave); };
  unsigned k_src[kPasses], v_src[kPasses];
#pragma unroll
  for (int p = 0; p < kPasses; ++p) {
    const int slot = copy_segment(p) * 64 + lane;
    int r, ch;
    tile_slot_decode<DP, false>(slot, r, ch);
    k_src[p] = ch * 16 < D ? (unsigned)(kv_of_lds_row(r) * (int)a.k_rs + ch * 16) : kNoSource;
    if constexpr (VT) {
      // v is [d, Nk]: the tile is D rows of 64 kv bytes (4 chunks), laid out like a 64-byte-row K tile
      tile_slot_decode<64, false>(slot, r, ch);
      v_src[p] = r < D ? (unsigned)(r * (int)a.v_rs + ch * 16) : kNoSource;
    } else {
      tile_slot_decode<DP, true>(slot, r, ch);
      v_src[p] = ch * 16 < D ? (unsigned)(r * (int)a.v_rs + ch * 16) : kNoSource;
    }
  }
  const int kv_last = a.seqlen_k - 1;
  constexpr int kRsrcFlags = 0x00020000;  // raw buffer, 32-bit data format
  // Start the asynchronous copy of the K rows / the V rows of KV block j into the LDS buffer kb / vb.  The pipelined loops
  // start two tile copies in every step, also when the block no longer exists (so that one s_waitcnt constant fits every
  // step): such a copy (exists = false, wave-uniform) goes through a resource of length 0, every lane of it is out of range,
  // zeros land in LDS and no memory is touched.  Its scalar offset is 0: a lane is out of range if its own offset is not below
  // length - scalar offset, a difference that must not be negative.
  // (Dense loop: the second pass of a copy differs from the first by a whole number of rows, 16 kv rows of K and 32 (64) rows
  // of V (V^T): the difference sits in the scalar offset and both passes share one vector register.  In a ragged last block that
  // scalar offset may lie past the last row: it stops at the resource's length, where every lane is out of range.)
  const int k_bytes = (int)(kv_last * a.k_rs + D);
  const int v_bytes = VT ? (int)((D - 1) * a.v_rs + a.seqlen_k) : (int)(kv_last * a.v_rs + D);
  auto segment_offset = [&](int base, int rows, int length) __attribute__((always_inline)) {
    return RAGGED ? (int)min((unsigned)base + (unsigned)rows, (unsigned)length) : base + rows;
  };
  auto issue_k = [&](int j, uint8_t* kb, bool exists) __attribute__((always_inline)) {
    const __amdgpu_buffer_rsrc_t rsrc = __builtin_amdgcn_make_buffer_rsrc((void*)kp, 0, exists ? k_bytes : 0, kRsrcFlags);
    const int k_rs = exists ? (int)a.k_rs : 0;
    const int k_base = (int)((unsigned)j * kKvBlock * (unsigned)k_rs);  // below 2^32 (fa8_fwd_validate)
#pragma unroll
    for (int p = 0; p < kPasses; ++p)
      if (!kSplitPass || wave < 2)
        __builtin_amdgcn_raw_ptr_buffer_load_lds(rsrc, LDS_PTR(void, kb + copy_segment(p) * 1024), 16, DENSE ? k_src[0] : k_src[p],
                                                 DENSE ? segment_offset(k_base, p * 16 * k_rs, k_bytes) : k_base, 0, 0);
  };
  auto issue_v = [&](int j, uint8_t* vb, bool exists) __attribute__((always_inline)) {
    const __amdgpu_buffer_rsrc_t rsrc = __builtin_amdgcn_make_buffer_rsrc((void*)vp, 0, exists ? v_bytes : 0, kRsrcFlags);
    const int v_rs = exists ? (int)a.v_rs : 0;
    const int v_base = VT ? (exists ? j * kKvBlock : 0) : (int)((unsigned)j * kKvBlock * (unsigned)v_rs);
    // transposed v, ragged last block: the 16-byte chunks past the last kv column would read the start of the next
    // head-dim row (or run off the tensor); they are pulled back onto the last chunk instead (and masked later)
    const bool v_clamp = VT && (j + 1) * kKvBlock > a.seqlen_k;
#pragma unroll
    for (int p = 0; p < kPasses; ++p) {
      const int seg = copy_segment(p) * 1024;
      if (!kSplitPass || wave >= 2) {
        if (v_clamp) {
          int r, ch;
          tile_slot_decode<64, false>(copy_segment(p) * 64 + lane, r, ch);
          const unsigned off = r < D ? (unsigned)(r * (int)a.v_rs + min(v_base + ch * 16, a.seqlen_k - 16)) : kNoSource;
          __builtin_amdgcn_raw_ptr_buffer_load_lds(rsrc, LDS_PTR(void, vb + seg), 16, off, 0, 0, 0);
        } else {
          __builtin_amdgcn_raw_ptr_buffer_load_lds(rsrc, LDS_PTR(void, vb + seg), 16, DENSE ? v_src[0] : v_src[p],
                                                   DENSE ? segment_offset(v_base, p * (VT ? 64 : 32) * v_rs, v_bytes) : v_base, 0, 0);
        }
      }
    }
  };
  auto issue_tile = [&](int j, uint8_t* kb, uint8_t* vb) __attribute__((always_inline)) {
    issue_k(j, kb, true);
    issue_v(j, vb, true);
  };

  // ---- per-lane LDS read offsets ----
  // K fragment (A operand of S^T): the lane's row inside the 32-row MFMA tile is lane % 32 and its k-group
  // lane / 32: chunks 4ks+2h and 4ks+2h+1 of LDS row 32t + lane % 32.  (Head dim 32: both k-groups read chunks 0
  // and 1; the upper group meets the zeros of the Q fragment.  Head dims 96, 160, 224: the upper group of the last
  // k-step reads zero-filled chunks.)
  int k_off[kKSteps][2];
#pragma unroll
  for (int ks = 0; ks < kKSteps; ++ks)
#pragma unroll
    for (int e = 0; e < 2; ++e) k_off[ks][e] = tile_offset<DP, false>(qn, DP >= 64 ? 4 * ks + 2 * h + e : e);
  constexpr int kSubTileStride = 32 * DP;  // LDS bytes between S^T sub-tiles (32 rows)
  // V^T fragment (A operand of O^T = V^T P^T) through ds_read_b64_tr_b8: inside a group of 16 lanes, lanes
  // 2j and 2j+1 address the two 8-byte halves of kv row j of an 8 x 16 byte block, and lane i receives
  // byte i of each of the 8 rows: 8 consecutive kv for one head-dim column.
  const int tr_j = (lane & 15) >> 1, tr_e = lane & 1, tr_g1 = (lane >> 4) & 1;
  // (transposed v: the tile already is V^T, [d][64 kv]: plain 16-byte reads of row 32mt + lane % 32, chunks 2h, 2h+1)
  int v_off[kMTiles], vt_off[2];
#pragma unroll
  for (int mt = 0; mt < kMTiles; ++mt) v_off[mt] = tile_offset<DP, true>(32 * h + tr_j, 2 * mt + tr_g1) + 8 * tr_e;
#pragma unroll
  for (int e = 0; e < 2; ++e) vt_off[e] = tile_offset<64, false>(qn, 2 * h + e);
  constexpr int kVtTileStride = 32 * 64;  // LDS bytes between 32-row groups of the [d][64] tile
  constexpr int kTrStride = 8 * DP;  // LDS bytes between successive groups of 8 kv rows

  // Causal: key j is visible to query i when j <= i + shift (shift 0: the reference's rule, csrc/flash_attention.cu:62-64;
  // shift = Nk - Nq aligns the diagonal with the bottom right corner).  At least block 0 is always walked (fully
  // masked if need be), so a query that sees no key ends with l = 0 and an all-zero output row.
  const int shift = CAUSAL ? a.causal_shift : 0;
  const int n_tiles = CAUSAL ? max(1, (min(a.seqlen_k, q0 + kQBlock + shift) + kKvBlock - 1) / kKvBlock)
                             : (a.seqlen_k + kKvBlock - 1) / kKvBlock;
  // Leading blocks that need no mask for any row of the workgroup: they end at or before the first query row's
  // last visible key (causal) and inside the kv range.  They are processed by the mask-free copy of the loop body.
  const int n_plain = (CAUSAL ? max(0, min(q0 + shift, a.seqlen_k)) : a.seqlen_k) / kKvBlock;

  v16f o_acc[kMTiles];
#pragma unroll
  for (int mt = 0; mt < kMTiles; ++mt)
#pragma unroll
    for (int i = 0; i < 16; ++i) o_acc[mt][i] = 0.f;
  // running row max of raw S (both half-lanes of a query hold the same value).  The loops that mask without a special case start it at a finite value
  // below every possible logit (|s| <= 57344^2 * 256 < 1e12) instead of -inf: a row that has not seen a key yet then needs no
  // special case (its rescale factor exp2((m_run - m_new) * c) is 0 or multiplies zeros, m_new * c stays finite, and a masked
  // logit -inf still gives exp2(-inf) = 0 for the positive scales these loops run with); the results are the same bit for bit.
  float m_run = PIPE || RAGGED ? -1.0e30f : -INFINITY;
  float l_run = 0.f;        // this lane's share of the running row sum

  // K fragment of S^T sub-tile t, k-step ks, and V^T fragment of O^T tile mt, from the tiles in kb / vb
  auto load_kf = [&](const uint8_t* kb, int t, int ks) __attribute__((always_inline)) {
    const v4i lo = *LDS_PTR(const v4i, kb + t * kSubTileStride + k_off[ks][0]);
    const v4i hi = *LDS_PTR(const v4i, kb + t * kSubTileStride + k_off[ks][1]);
    return v8i{lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
  };
  auto load_vf = [&](const uint8_t* vb, int mt) __attribute__((always_inline)) {
    v8i vf;
    if constexpr (VT) {
      const v4i lo = *LDS_PTR(const v4i, vb + mt * kVtTileStride + vt_off[0]);
      const v4i hi = *LDS_PTR(const v4i, vb + mt * kVtTileStride + vt_off[1]);
      vf = {lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
    } else {
#pragma unroll
      for (int g = 0; g < 4; ++g) {
        const v2i r = __builtin_amdgcn_ds_read_tr8_b64_v2i32(LDS_PTR(v2i, vb + v_off[mt] + g * kTrStride));
        vf[2 * g] = r[0];
        vf[2 * g + 1] = r[1];
      }
    }
    return vf;
  };

  // S^T, online softmax and PV for KV block j held in kb / vb.
  auto compute_tile = [&](int j, const uint8_t* kb, const uint8_t* vb, auto masked_c) __attribute__((always_inline)) {
    // kMasked also marks the general path (first block, diagonal, tail): only there can the running max still be -inf
    constexpr bool kMasked = decltype(masked_c)::value;
    const int kv0 = j * kKvBlock;
    // ---- S^T = K Q^T : two 32(kv) x 32(q) sub-tiles ----
    v16f s[2];
#pragma unroll
    for (int t = 0; t < 2; ++t) {
#pragma unroll
      for (int i = 0; i < 16; ++i) s[t][i] = 0.f;
#pragma unroll
      for (int ks = 0; ks < kKSteps; ++ks) {
        s[t] = mfma_fp8<E5M2>(load_kf(kb, t, ks), qf[ks], s[t]);
      }
    }
    // ---- causal / tail mask: register i of sub-tile t is kv row kv0 + 32h + 16t + i ----
    const int kv_limit = CAUSAL ? min(q_row + shift, kv_last) : kv_last;  // last kv this query attends to
    if constexpr (kMasked) {
#pragma unroll
      for (int t = 0; t < 2; ++t)
#pragma unroll
        for (int i = 0; i < 16; ++i)
          if (kv0 + 32 * h + 16 * t + i > kv_limit) s[t][i] = -INFINITY;
    }
    // ---- online softmax (reference softmax_rescale_o, csrc/flash_attention.cu:233-273) ----
    // 33 values (32 logits and the running max) in 16 three-input maxima: four independent chains over sub-tile 0
    // (it is ready first), then sub-tile 1
    float mx[4];
#pragma unroll
    for (int ch = 0; ch < 4; ++ch) mx[ch] = max3(s[0][4 * ch], s[0][4 * ch + 1], s[0][4 * ch + 2]);
#pragma unroll
    for (int ch = 0; ch < 4; ++ch) mx[ch] = max3(mx[ch], s[0][4 * ch + 3], s[1][4 * ch]);
#pragma unroll
    for (int ch = 0; ch < 4; ++ch) mx[ch] = max3(mx[ch], s[1][4 * ch + 1], s[1][4 * ch + 2]);
    const float m_new = lane32_max(max3(max3(mx[0], s[1][3], s[1][7]), max3(mx[1], s[1][11], s[1][15]), max3(mx[2], mx[3], m_run)));
    if (__any(m_new != m_run)) {
      float alpha = __builtin_amdgcn_exp2f((m_run - m_new) * c);
      if constexpr (kMasked) alpha = (m_run == -INFINITY) ? 0.f : alpha;
      l_run *= alpha;
      // only the lanes of the queries whose max moved multiply (the others would multiply by exactly 1): the instructions are
      // issued either way, but idle lanes draw no power, and this kernel runs at the board's power limit
      if (alpha != 1.f) {
#pragma unroll
        for (int mt = 0; mt < kMTiles; ++mt)
#pragma unroll
          for (int i = 0; i < 16; ++i) o_acc[mt][i] *= alpha;
      }
      m_run = m_new;
    }
    float mc = m_new * c;
    if constexpr (kMasked) mc = (m_new == -INFINITY) ? 0.f : mc;
    float sum0, sum1;  // row sum of this block in two chains, started from the first two weights
    v8i p8;
#pragma unroll
    for (int t = 0; t < 2; ++t) {
#pragma unroll
      for (int i = 0; i < 16; ++i) s[t][i] = __builtin_amdgcn_exp2f(__builtin_fmaf(s[t][i], c, -mc));
      if constexpr (kMasked) {
        // a masked logit is -inf; force its weight to 0 even when scale <= 0 would give NaN or 1
#pragma unroll
        for (int i = 0; i < 16; ++i)
          if (kv0 + 32 * h + 16 * t + i > kv_limit) s[t][i] = 0.f;
      }
#pragma unroll
      for (int i = 0; i < 16; i += 2) {
        sum0 = (t == 0 && i == 0) ? s[t][i] : sum0 + s[t][i];
        sum1 = (t == 0 && i == 0) ? s[t][i + 1] : sum1 + s[t][i + 1];
      }
#pragma unroll
      for (int w = 0; w < 4; ++w)
        p8[4 * t + w] = pack4_fp8<E5M2>(s[t][4 * w], s[t][4 * w + 1], s[t][4 * w + 2], s[t][4 * w + 3]);
    }
    l_run += sum0 + sum1;
    // ---- O^T += V^T P^T : the V^T fragment of tile mt+1 is fetched while the MFMA of tile mt runs ----
    v8i vf_cur = load_vf(vb, 0);
#pragma unroll
    for (int mt = 0; mt < kMTiles; ++mt) {
      v8i vf_next;
      if (mt + 1 < kMTiles) vf_next = load_vf(vb, mt + 1);
      o_acc[mt] = mfma_fp8<E5M2>(vf_cur, p8, o_acc[mt]);
      if (mt + 1 < kMTiles) vf_cur = vf_next;
    }
  };
  // Three LDS stages: copies issued two KV blocks ahead.  At the end of the step for block j the copy of block
  // j+1 (issued one step earlier) must have landed while the copy of block j+2 (issued in this step: kLoadsPerTile
  // loads per lane) may stay in flight; vmcnt counts this lane's loads in issue order.  The barrier then tells every
  // wavefront that all shares of block j+1 are in LDS and that block j's stage may be overwritten.  It is a bare
  // s_barrier: __syncthreads() would also wait for the copy that is meant to stay in flight.
  constexpr int kLoadsPerTile = kSplitPass ? 1 : 2 * kPasses;
  auto stage_sync = [&](bool next_in_flight) __attribute__((always_inline)) {
    // s_waitcnt immediate (gfx9 layout): vmcnt[3:0], expcnt[6:4] = 7 (no wait on those), lgkmcnt[11:8] = 0: the reads of block j have returned.  The
    // compiler may move the last product of a step, and its wait for its operands, behind the barrier; a copy into the stage, one of nothing above
    // all, could then overtake the read.
    if (next_in_flight)
      __builtin_amdgcn_s_waitcnt(0x0070 | kLoadsPerTile);
    else
      __builtin_amdgcn_s_waitcnt(0x0070);
    __builtin_amdgcn_s_barrier();
  };
  static_assert(kLoadsPerTile < 16, "vmcnt immediate above");

  if constexpr (DENSE) {
    // ---- dense loop: the software pipeline in 168 VGPRs ----
    // Iteration j is the softmax of block j in 8 chunks of 4 weights.  In front of chunks 0-3 go the PV products of block j-1
    // (head dim 64: chunks 0 and 2), in front of chunks 4-5 the S^T products of sub-tile 0 of block j+1, written over sub-tile 0
    // of block j, which is all weights by then; the S^T products of sub-tile 1 follow the last chunk and run under the rescale
    // of O.  LDS operands are fetched one matrix instruction ahead.  K(t) and V(t) live in stage t % 3.  Step j starts the
    // copies of K(j+3) (its stage held K(j), last read in step j-1) and V(j+1) (its stage held V(j-2), last read in step j-1)
    // in front of chunks 1 and 2, reads K(j+1) and V(j-1), and ends when K(j+2) and V(j), started in step j-1, have landed.
    v16f s[2];
    v8i p8;
    constexpr int kPvEvery = 4 / kMTiles;  // the PV product of tile mt goes in front of chunk mt * kPvEvery
    constexpr int kSEvery = 2 / kKSteps;   // the S^T product (sub-tile 0, k-step ks) in front of chunk 4 + ks * kSEvery
    auto iteration = [&](auto first_c, auto tail_c, int j, const uint8_t* kb_next, const uint8_t* vb_prev, uint8_t* k_dst, uint8_t* v_dst)
                         __attribute__((always_inline)) {
      constexpr bool kFirst = decltype(first_c)::value;
      constexpr bool kTail = RAGGED && decltype(tail_c)::value;  // block j may be the last one, with keys that do not exist
      v8i vfrag[kMTiles];
      v8i kfrag[2][kKSteps];
      if constexpr (!kFirst) vfrag[0] = load_vf(vb_prev, 0);
      if constexpr (kTail) {
        if (j >= n_plain) {  // wave-uniform; the block has a key, so the row max stays finite
          const int left = kv_last - j * kKvBlock - 32 * h;
#pragma unroll
          for (int t = 0; t < 2; ++t)
#pragma unroll
            for (int i = 0; i < 16; ++i)
              if (16 * t + i > left) s[t][i] = -INFINITY;
        }
      }
      float mx[4];
#pragma unroll
      for (int ch = 0; ch < 4; ++ch) mx[ch] = max3(s[0][4 * ch], s[0][4 * ch + 1], s[0][4 * ch + 2]);
#pragma unroll
      for (int ch = 0; ch < 4; ++ch) mx[ch] = max3(mx[ch], s[0][4 * ch + 3], s[1][4 * ch]);
#pragma unroll
      for (int ch = 0; ch < 4; ++ch) mx[ch] = max3(mx[ch], s[1][4 * ch + 1], s[1][4 * ch + 2]);
      const float m_new = lane32_max(max3(max3(mx[0], s[1][3], s[1][7]), max3(mx[1], s[1][11], s[1][15]), max3(mx[2], mx[3], m_run)));
      bool changed = false;
      float alpha = 1.f;
      const float mc = m_new * c;
      if constexpr (kFirst) {
        m_run = m_new;  // O and l are still zero
      } else {
        changed = __any(m_new != m_run);
        if (changed) {
          alpha = __builtin_amdgcn_exp2f((m_run - m_new) * c);
          l_run *= alpha;
          m_run = m_new;
        }
      }
      float sum0, sum1;
      v8i p8_cur;
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int u = 0; u < 8; ++u) {
        if (u == 1) issue_k(min(j + 3, n_tiles), k_dst, j + 3 < n_tiles);
        if (u == 2) issue_v(min(j + 1, n_tiles), v_dst, j + 1 < n_tiles);
        // LDS operands of the matrix instructions in front of the next chunk
        if constexpr (!kFirst) {
#pragma unroll
          for (int mt = 1; mt < kMTiles; ++mt)
            if (mt * kPvEvery - 1 == u) vfrag[mt] = load_vf(vb_prev, mt);
        }
#pragma unroll
        for (int ks = 0; ks < kKSteps; ++ks)
          if (4 + ks * kSEvery - 1 == u) kfrag[0][ks] = load_kf(kb_next, 0, ks);
        if (u >= 8 - kKSteps) kfrag[1][u - (8 - kKSteps)] = load_kf(kb_next, 1, u - (8 - kKSteps));
        // one matrix instruction in front of the chunk
        if (u < 4 && u % kPvEvery == 0) {
          if constexpr (!kFirst) o_acc[u / kPvEvery] = mfma_fp8<E5M2>(vfrag[u / kPvEvery], p8, o_acc[u / kPvEvery]);
        }
        if (u >= 4 && (u - 4) % kSEvery == 0 && (u - 4) / kSEvery < kKSteps) {
          // (after the last block this is the product of a stale tile: never used)
          const int ks = (u - 4) / kSEvery;
          if (ks == 0) {
            v16f z;
#pragma unroll
            for (int i = 0; i < 16; ++i) z[i] = 0.f;
            s[0] = mfma_fp8<E5M2>(kfrag[0][ks], qf[ks], z);
          } else {
            s[0] = mfma_fp8<E5M2>(kfrag[0][ks], qf[ks], s[0]);
          }
        }
        __builtin_amdgcn_sched_barrier(0);
        // chunk u of the softmax: weights 4w .. 4w+3 of sub-tile t
        const int t = u >> 2, w = u & 3;
        float x[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) x[i] = __builtin_amdgcn_exp2f(__builtin_fmaf(s[t][4 * w + i], c, -mc));
        sum0 = (u == 0) ? x[0] : sum0 + x[0];
        sum1 = (u == 0) ? x[1] : sum1 + x[1];
        sum0 += x[2];
        sum1 += x[3];
        int packed = pack4_fp8<E5M2>(x[0], x[1], x[2], x[3]);
        // the weights are only read in the next iteration; without this pin the compiler sinks the conversions there
        asm volatile("" : "+v"(packed));
        p8_cur[u] = packed;
        __builtin_amdgcn_sched_barrier(0);
      }
#pragma unroll
      for (int ks = 0; ks < kKSteps; ++ks) {
        if (ks == 0) {
          v16f z;
#pragma unroll
          for (int i = 0; i < 16; ++i) z[i] = 0.f;
          s[1] = mfma_fp8<E5M2>(kfrag[1][ks], qf[ks], z);
        } else {
          s[1] = mfma_fp8<E5M2>(kfrag[1][ks], qf[ks], s[1]);
        }
      }
      l_run += sum0 + sum1;
      asm volatile("" : "+v"(l_run));  // keeps the additions above where they are written
      // O now holds the PV product of block j-1: bring it to the new row max (in the lanes whose max moved, see compute_tile)
      if (changed) {
        if (alpha != 1.f) {
#pragma unroll
          for (int mt = 0; mt < kMTiles; ++mt)
#pragma unroll
            for (int i = 0; i < 16; ++i) o_acc[mt][i] *= alpha;
        }
      }
      p8 = p8_cur;
    };
    // Waits until at most `tiles` tile copies (kPasses loads each) are in flight, then the barrier: it publishes the landed
    // tiles and frees the stages read before it.  vmcnt counts this lane's loads in issue order.
    auto wait_in_flight = [&](auto tiles_c) __attribute__((always_inline)) {
      constexpr int n = decltype(tiles_c)::value * kPasses;
      static_assert(n < 16, "vmcnt immediate");
      __builtin_amdgcn_s_waitcnt(0x0070 | n);  // (and its LDS reads have returned, see stage_sync)
      __builtin_amdgcn_s_barrier();
    };
    using T = std::true_type;
    using F = std::false_type;
    issue_k(0, k_lds0, true);
    issue_k(min(1, n_tiles), k_lds1, 1 < n_tiles);
    issue_k(min(2, n_tiles), k_lds2, 2 < n_tiles);
    issue_v(0, v_lds0, true);
    wait_in_flight(std::integral_constant<int, 2>());  // K(0) and K(1) landed
#pragma unroll
    for (int t = 0; t < 2; ++t) {
#pragma unroll
      for (int i = 0; i < 16; ++i) s[t][i] = 0.f;
#pragma unroll
      for (int ks = 0; ks < kKSteps; ++ks) s[t] = mfma_fp8<E5M2>(load_kf(k_lds0, t, ks), qf[ks], s[t]);
    }
    __builtin_amdgcn_s_waitcnt(0xC07F);
    __builtin_amdgcn_s_barrier();  // every wavefront has read K(0): step 0 may overwrite its stage
    // One step with compile-time LDS stages (PH = j % 3).
    auto step = [&](auto first_c, auto tail_c, auto ph_c, int j) __attribute__((always_inline)) {
      constexpr int PH = decltype(ph_c)::value;
      uint8_t* const kst[3] = {k_lds0, k_lds1, k_lds2};
      uint8_t* const vst[3] = {v_lds0, v_lds1, v_lds2};
      iteration(first_c, tail_c, j, kst[(PH + 1) % 3], vst[(PH + 2) % 3], kst[PH], vst[(PH + 1) % 3]);
      wait_in_flight(std::integral_constant<int, 2>());  // the two copies of this step may stay in flight
    };
    constexpr std::integral_constant<int, 0> ph0{};
    constexpr std::integral_constant<int, 1> ph1{};
    constexpr std::integral_constant<int, 2> ph2{};
    step(T(), T(), ph0, 0);
    int j = 1;
    for (; j + 2 < (RAGGED ? n_plain : n_tiles); j += 3) {
      step(F(), F(), ph1, j);
      step(F(), F(), ph2, j + 1);
      step(F(), F(), ph0, j + 2);
    }
    // up to two more whole blocks, and a ragged one
    if (j < n_tiles) {
      step(F(), T(), ph1, j);
      if (j + 1 < n_tiles) {
        step(F(), T(), ph2, j + 1);
        if (RAGGED && j + 2 < n_tiles) step(F(), T(), ph0, j + 2);
      }
    }
    __builtin_amdgcn_s_waitcnt(0x0F70);  // the last copies (of nothing) must not outlive the workgroup's LDS
    // the PV product of the last block
    {
      const int st = (n_tiles - 1) % 3;
      const uint8_t* vb = st == 0 ? v_lds0 : (st == 1 ? v_lds1 : v_lds2);
#pragma unroll
      for (int mt = 0; mt < kMTiles; ++mt) o_acc[mt] = mfma_fp8<E5M2>(load_vf(vb, mt), p8, o_acc[mt]);
    }
  } else if constexpr (PIPE) {
    // ---- software-pipelined loop ----
    // Iteration j is the softmax of block j in 8 chunks of 4 weights with a matrix instruction in front of the chunks: first
    // the PV products of block j-1, then the S^T products of block j+1 (head dim 128: one per chunk, 64: every second
    // chunk), their LDS operands fetched two instructions ahead.  K(t) lives in K stage t % 4, V(t) in V stage t % 4.  Step j
    // starts the copies of K(j+4) and V(j+2) (their stages held K(j) and V(j-2), last read in iteration j-1), reads K(j+1)
    // and V(j-1), and ends when K(j+2) and V(j) have landed.  Every block takes this path, masked blocks included (their
    // weights become exact zeros), so the loop needs no second form.
    constexpr int kSlots = kMTiles + 2 * kKSteps;  // matrix instructions per iteration
    constexpr int kChunksPerSlot = 8 / kSlots;     // 1 (head dim 128) or 2 (64)
    v16f sbuf[2][2];
    v8i p8buf[2];
    const int kv_limit = CAUSAL ? min(q_row + shift, kv_last) : kv_last;  // last kv this query attends to
    auto iteration = [&](auto first_c, int j, const uint8_t* kb_next, const uint8_t* vb_prev, v16f(&s)[2], v16f(&sn)[2],
                         const v8i& p8_prev, v8i& p8_cur) __attribute__((always_inline)) {
      constexpr bool kFirst = decltype(first_c)::value;
      const bool masked = j >= n_plain;  // wave-uniform
      v8i frag[kSlots];
      if constexpr (!kFirst) {
        frag[0] = load_vf(vb_prev, 0);
        frag[1] = load_vf(vb_prev, 1);
      }
      if (masked) {
        // a masked logit becomes -inf and its weight exp2(-inf) = 0 (the launcher takes this loop only for scale > 0)
        const int kv0 = j * kKvBlock;
#pragma unroll
        for (int t = 0; t < 2; ++t)
#pragma unroll
          for (int i = 0; i < 16; ++i)
            if (kv0 + 32 * h + 16 * t + i > kv_limit) s[t][i] = -INFINITY;
      }
      float mx[4];
#pragma unroll
      for (int ch = 0; ch < 4; ++ch) mx[ch] = max3(s[0][4 * ch], s[0][4 * ch + 1], s[0][4 * ch + 2]);
#pragma unroll
      for (int ch = 0; ch < 4; ++ch) mx[ch] = max3(mx[ch], s[0][4 * ch + 3], s[1][4 * ch]);
#pragma unroll
      for (int ch = 0; ch < 4; ++ch) mx[ch] = max3(mx[ch], s[1][4 * ch + 1], s[1][4 * ch + 2]);
      const float m_new = lane32_max(max3(max3(mx[0], s[1][3], s[1][7]), max3(mx[1], s[1][11], s[1][15]), max3(mx[2], mx[3], m_run)));
      bool changed = false;
      float alpha = 1.f;
      float mc = m_new * c;
      if constexpr (kFirst) {
        m_run = m_new;  // O and l are still zero
      } else {
        changed = __any(m_new != m_run);
        if (changed) {
          alpha = __builtin_amdgcn_exp2f((m_run - m_new) * c);
          l_run *= alpha;
          m_run = m_new;
        }
      }
      float sum0, sum1;
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int u = 0; u < 8; ++u) {
        if (u % kChunksPerSlot == 0) {
          const int slot = u / kChunksPerSlot;
          // operands of the matrix instruction two slots ahead
          if (slot + 2 < kSlots) {
            const int sl = slot + 2;
            if (sl < kMTiles) {
              if constexpr (!kFirst) frag[sl] = load_vf(vb_prev, sl);
            } else {
              frag[sl] = load_kf(kb_next, (sl - kMTiles) / kKSteps, (sl - kMTiles) % kKSteps);
            }
          }
          if (slot < kMTiles) {
            if constexpr (!kFirst) o_acc[slot] = mfma_fp8<E5M2>(frag[slot], p8_prev, o_acc[slot]);
          } else {
            // (after the last block this is the product of a stale tile: never used)
            const int t = (slot - kMTiles) / kKSteps, ks = (slot - kMTiles) % kKSteps;
            if (ks == 0) {
              v16f z;
#pragma unroll
              for (int i = 0; i < 16; ++i) z[i] = 0.f;
              sn[t] = mfma_fp8<E5M2>(frag[slot], qf[ks], z);
            } else {
              sn[t] = mfma_fp8<E5M2>(frag[slot], qf[ks], sn[t]);
            }
          }
          __builtin_amdgcn_sched_barrier(0);
        }
        // chunk u of the softmax: weights 4w .. 4w+3 of sub-tile t
        const int t = u >> 2, w = u & 3;
#pragma unroll
        for (int i = 4 * w; i < 4 * w + 4; ++i) s[t][i] = __builtin_amdgcn_exp2f(__builtin_fmaf(s[t][i], c, -mc));
        sum0 = (u == 0) ? s[t][4 * w] : sum0 + s[t][4 * w];
        sum1 = (u == 0) ? s[t][4 * w + 1] : sum1 + s[t][4 * w + 1];
        sum0 += s[t][4 * w + 2];
        sum1 += s[t][4 * w + 3];
        int packed = pack4_fp8<E5M2>(s[t][4 * w], s[t][4 * w + 1], s[t][4 * w + 2], s[t][4 * w + 3]);
        // the weights are only read in the next iteration; without this pin the compiler sinks the conversions there, in
        // one clump in front of the PV products that wait for them
        asm volatile("" : "+v"(packed));
        p8_cur[u] = packed;
        __builtin_amdgcn_sched_barrier(0);
      }
      l_run += sum0 + sum1;
      asm volatile("" : "+v"(l_run));  // keeps the additions above where they are written (sunk to the end they cost registers)
      // O now holds the PV product of block j-1 (issued four or more chunks ago): bring it to the new row max (in the lanes
      // whose max moved, see compute_tile)
      if (changed) {
        if (alpha != 1.f) {
#pragma unroll
          for (int mt = 0; mt < kMTiles; ++mt)
#pragma unroll
            for (int i = 0; i < 16; ++i) o_acc[mt][i] *= alpha;
        }
      }
    };
    // Every step starts two tile copies, also past the last block this workgroup walks (those copy nothing, see issue_k), so the
    // number of loads in flight is the same at every step.  vmcnt counts this lane's loads in issue order.
    // Waits until at most `tiles` tile copies (kPasses loads each) are in flight, then the barrier: it publishes the landed
    // tiles and frees the stages read before it.
    auto wait_in_flight = [&](auto tiles_c) __attribute__((always_inline)) {
      constexpr int n = decltype(tiles_c)::value * kPasses;
      static_assert(n < 16, "vmcnt immediate");
      __builtin_amdgcn_s_waitcnt(0x0070 | n);  // (and its LDS reads have returned, see stage_sync)
      __builtin_amdgcn_s_barrier();
    };
    // Ends step j: K(j+2) and V(j) must have landed; the copies of steps j-1 and j (K(j+3), V(j+1), K(j+4), V(j+2)) may stay
    // in flight.
    auto end_step = [&]() __attribute__((always_inline)) { wait_in_flight(std::integral_constant<int, 4>()); };
    // The PV product of the last block (its weights are in p8), V in stage vb.
    auto finish = [&](const uint8_t* vb, const v8i& p8) __attribute__((always_inline)) {
#pragma unroll
      for (int mt = 0; mt < kMTiles; ++mt) o_acc[mt] = mfma_fp8<E5M2>(load_vf(vb, mt), p8, o_acc[mt]);
    };
    using T = std::true_type;
    using F = std::false_type;
    // the copies of steps -4 .. -1
    issue_k(0, k_lds0, true);
    issue_k(min(1, n_tiles), k_lds1, 1 < n_tiles);
    issue_k(min(2, n_tiles), k_lds2, 2 < n_tiles);
    issue_v(0, v_lds0, true);
    issue_k(min(3, n_tiles), k_lds3, 3 < n_tiles);
    issue_v(min(1, n_tiles), v_lds1, 1 < n_tiles);
    wait_in_flight(std::integral_constant<int, 5>());  // K(0) landed
#pragma unroll
    for (int t = 0; t < 2; ++t) {
#pragma unroll
      for (int i = 0; i < 16; ++i) sbuf[0][t][i] = 0.f;
#pragma unroll
      for (int ks = 0; ks < kKSteps; ++ks) sbuf[0][t] = mfma_fp8<E5M2>(load_kf(k_lds0, t, ks), qf[ks], sbuf[0][t]);
    }
    end_step();  // K(1) landed, and every wavefront has read K(0): step 0 may overwrite its stage
    // One step with compile-time LDS stages (PH = j % 4) and buffers (j % 2); the mask-free form for the leading blocks.
    auto step = [&](auto first_c, auto ph_c, int j) __attribute__((always_inline)) {
      constexpr int PH = decltype(ph_c)::value;
      constexpr bool kFirst = decltype(first_c)::value;
      uint8_t* const kst[4] = {k_lds0, k_lds1, k_lds2, k_lds3};
      uint8_t* const vst[4] = {v_lds0, v_lds1, v_lds2, v_lds3};
      issue_k(min(j + 4, n_tiles), kst[PH], j + 4 < n_tiles);
      issue_v(min(j + 2, n_tiles), vst[(PH + 2) % 4], j + 2 < n_tiles);
      iteration(first_c, j, kst[(PH + 1) % 4], vst[(PH + 3) % 4], sbuf[PH % 2], sbuf[(PH + 1) % 2], p8buf[(PH + 1) % 2],
                p8buf[PH % 2]);
      end_step();
      (void)kFirst;
    };
    constexpr std::integral_constant<int, 0> ph0{};
    constexpr std::integral_constant<int, 1> ph1{};
    constexpr std::integral_constant<int, 2> ph2{};
    constexpr std::integral_constant<int, 3> ph3{};
    step(T(), ph0, 0);
    int j = 1;
    for (; j + 3 < n_tiles; j += 4) {
      step(F(), ph1, j);
      step(F(), ph2, j + 1);
      step(F(), ph3, j + 2);
      step(F(), ph0, j + 3);
    }
    // up to three more blocks; the weights of the last block end in p8buf[0]
    if (j < n_tiles) {
      step(F(), ph1, j);
      if (j + 1 < n_tiles) {
        step(F(), ph2, j + 1);
        if (j + 2 < n_tiles) {
          step(F(), ph3, j + 2);
          p8buf[0] = p8buf[1];
        }
      } else {
        p8buf[0] = p8buf[1];
      }
    }
    __builtin_amdgcn_s_waitcnt(0x0F70);  // the copies past the last block must not outlive the workgroup's LDS
    {
      const int st = (n_tiles - 1) & 3;
      finish(st == 0 ? v_lds0 : (st == 1 ? v_lds1 : (st == 2 ? v_lds2 : v_lds3)), p8buf[0]);
    }
  } else if constexpr (kStages == 3) {
    issue_tile(0, k_lds0, v_lds0);
    if (n_tiles > 1) issue_tile(1, k_lds1, v_lds1);
    stage_sync(n_tiles > 1);
    // Block 0 takes the general path: it is the only block that can meet a running max of -inf.
    if (n_tiles > 2) issue_tile(2, k_lds2, v_lds2);
    compute_tile(0, k_lds0, v_lds0, std::true_type());
    stage_sync(n_tiles > 2);
    int j = 1;
    // Mask-free blocks, three per trip so that every third reads one fixed LDS stage (the compiler can then tell
    // that the copies in flight go to other stages and need not be waited for before the reads).
    // Inside this loop every copy is issued unconditionally (block j+4 exists), which lets the compiler see that each
    // s_waitcnt below always leaves exactly one block in flight.
    for (; j + 2 < n_plain && j + 4 < n_tiles; j += 3) {
      issue_tile(j + 2, k_lds0, v_lds0);
      compute_tile(j, k_lds1, v_lds1, std::false_type());
      stage_sync(true);
      issue_tile(j + 3, k_lds1, v_lds1);
      compute_tile(j + 1, k_lds2, v_lds2, std::false_type());
      stage_sync(true);
      issue_tile(j + 4, k_lds2, v_lds2);
      compute_tile(j + 2, k_lds0, v_lds0, std::false_type());
      stage_sync(true);
    }
    // The last few mask-free blocks: same arithmetic, LDS stage chosen at run time, copies issued while blocks remain.
    for (; j < n_plain; ++j) {
      const int st = j % 3, st2 = (j + 2) % 3;
      if (j + 2 < n_tiles)
        issue_tile(j + 2, st2 == 0 ? k_lds0 : (st2 == 1 ? k_lds1 : k_lds2), st2 == 0 ? v_lds0 : (st2 == 1 ? v_lds1 : v_lds2));
      compute_tile(j, st == 0 ? k_lds0 : (st == 1 ? k_lds1 : k_lds2), st == 0 ? v_lds0 : (st == 1 ? v_lds1 : v_lds2),
                   std::false_type());
      stage_sync(j + 2 < n_tiles);
    }
    // The remaining blocks (the blocks on the diagonal, the kv tail) take the masking copy.
    for (; j < n_tiles; ++j) {
      const int st = j % 3, st2 = (j + 2) % 3;
      if (j + 2 < n_tiles)
        issue_tile(j + 2, st2 == 0 ? k_lds0 : (st2 == 1 ? k_lds1 : k_lds2), st2 == 0 ? v_lds0 : (st2 == 1 ? v_lds1 : v_lds2));
      // a wavefront whose 32 query rows all lie before this kv block has nothing to add (causal)
      if (!CAUSAL || j * kKvBlock <= q_wave0 + kQWave - 1 + shift)
        compute_tile(j, st == 0 ? k_lds0 : (st == 1 ? k_lds1 : k_lds2), st == 0 ? v_lds0 : (st == 1 ? v_lds1 : v_lds2),
                     std::true_type());
      stage_sync(j + 2 < n_tiles);
    }
  } else {
    // Two stages: the copy of block j+1 is issued at the start of the step for block j and must have landed at its end.
    issue_tile(0, k_lds0, v_lds0);
    stage_sync(false);
    if (n_tiles > 1) issue_tile(1, k_lds1, v_lds1);
    compute_tile(0, k_lds0, v_lds0, std::true_type());
    stage_sync(false);
    int j = 1;
    for (; j + 1 < n_plain && j + 2 < n_tiles; j += 2) {
      issue_tile(j + 1, k_lds0, v_lds0);
      compute_tile(j, k_lds1, v_lds1, std::false_type());
      stage_sync(false);
      issue_tile(j + 2, k_lds1, v_lds1);
      compute_tile(j + 1, k_lds0, v_lds0, std::false_type());
      stage_sync(false);
    }
    for (; j < n_plain; ++j) {  // the last mask-free blocks
      const bool odd = j & 1;
      if (j + 1 < n_tiles) issue_tile(j + 1, odd ? k_lds0 : k_lds1, odd ? v_lds0 : v_lds1);
      compute_tile(j, odd ? k_lds1 : k_lds0, odd ? v_lds1 : v_lds0, std::false_type());
      stage_sync(false);
    }
    for (; j < n_tiles; ++j) {
      const bool odd = j & 1;
      if (j + 1 < n_tiles) issue_tile(j + 1, odd ? k_lds0 : k_lds1, odd ? v_lds0 : v_lds1);
      if (!CAUSAL || j * kKvBlock <= q_wave0 + kQWave - 1 + shift)
        compute_tile(j, odd ? k_lds1 : k_lds0, odd ? v_lds1 : v_lds0, std::true_type());
      stage_sync(false);
    }
  }

  // ---- epilogue: O / l, convert, store (reference csrc/flash_attention.cu:542-582) ----
  const float l_tot = lane32_sum(l_run);
  const float inv = (l_tot == 0.f || l_tot != l_tot) ? 1.f : 1.f / l_tot;
  // log-sum-exp of the scaled logits of the row (natural log), -inf for a row that saw no key; the reference reserves
  // the output but never writes it (csrc/flash.h:56, csrc/flash_attention.cu:658-659)
  if (a.lse != nullptr && h == 0 && q_row < a.seqlen_q) {
    const float lse = l_tot > 0.f ? (m_run * c + __builtin_amdgcn_logf(l_tot)) * 0.6931471805599453f : (l_tot == 0.f ? -INFINITY : l_tot);
    a.lse[b * a.lse_bs + hd * a.lse_hs + q_row] = lse;
  }
  // A lane holds pieces of 8 bytes (fp8: 4) of its row, 16 (8) bytes apart: stored as they are, a wavefront's store touches 32 rows with 16
  // bytes each, and at the end of a launch whose workgroups all run at once the 16-byte writes are what the L2s wait for.  There they go through LDS, 128
  // bytes of the 32 rows at a time, and leave as whole lines, eight lanes a row (store_row_chunk).  us, pieces -> lines: 16 x 32 heads, 256 keys, head dim 128,
  // causal 27.6 -> 22.4; 8 x 32 heads, 1024 keys, causal 77.1 -> 69.0; 4 x 16 heads, 1024 keys, head dim 64 21.3 -> 19.5; 2 x 16 heads, 2999 keys 99.2 -> 95.5;
  // 2 x 32 heads, 4096 keys 309.3 -> 299.4.  Smaller launches keep the pieces: whole_lines has the line between the two.
  constexpr int kElem = OUT == FA8_OUT_FP16 ? 2 : 1;
  // register i = 4a2 + b2 of tile mt is head-dim column 32mt + 8a2 + 4h + b2: a lane's piece a2 of tile mt in the output type
  auto piece = [&](int mt, int a2) __attribute__((always_inline)) {
    if constexpr (OUT == FA8_OUT_FP16) {
      v4h x;
#pragma unroll
      for (int b2 = 0; b2 < 4; ++b2) x[b2] = (_Float16)(o_acc[mt][4 * a2 + b2] * inv);
      return x;
    } else {
      float x[4];
      constexpr float kMaxFinite = OUT == FA8_OUT_E5M2 ? 57344.f : 448.f;
#pragma unroll
      for (int b2 = 0; b2 < 4; ++b2) {
        const float y = o_acc[mt][4 * a2 + b2] * inv;
        x[b2] = (y != y) ? y : fminf(fmaxf(y, -kMaxFinite), kMaxFinite);  // saturate to finite, keep NaN
      }
      return pack4_fp8<OUT == FA8_OUT_E5M2>(x[0], x[1], x[2], x[3]);
    }
  };
  using Piece = decltype(piece(0, 0));
  // (the pieces follow in line: a launch of few workgroups has none of this in the instruction cache, and a jump costs it 0.2 us)
  if (__builtin_expect(!a.whole_lines, 1)) {
    if (q_row < a.seqlen_q) {
      uint8_t* const at = (uint8_t*)a.o + ((long long)b * a.o_bs + (long long)hd * a.o_hs + (long long)q_row * a.o_rs + 4 * h) * kElem;
#pragma unroll
      for (int mt = 0; mt < kMTiles; ++mt)
#pragma unroll
        for (int a2 = 0; a2 < 4; ++a2) *(Piece*)(at + (32 * mt + 8 * a2) * kElem) = piece(mt, a2);
    }
    return;
  }
  // (head dims 32 and 256: the lane's number taken anew; with transposed v, keeping it over the loop for these addresses spilled eight registers of
  // head dim 256 and cost head dim 32 the fifth workgroup of a compute unit.  Head dim 224 spilled ten the other way round.)
  const int lane_o = D == 32 || D == 256 ? (int)__builtin_amdgcn_mbcnt_hi(~0u, __builtin_amdgcn_mbcnt_lo(~0u, 0u)) : lane, row_o = lane_o & 31, half_o = lane_o >> 5;
  uint8_t* const op = (uint8_t*)a.o + ((long long)b * a.o_bs + (long long)hd * a.o_hs + (long long)q_wave0 * a.o_rs) * kElem;
  __builtin_amdgcn_s_waitcnt(0x0070);  // every wavefront has read its last tiles, and its copies (also those of nothing) have landed
  __builtin_amdgcn_s_barrier();
  constexpr int kRowBytes = D * kElem <= 32 ? 32 : (D * kElem <= 64 ? 64 : 128), kSlab = 32 * kRowBytes;  // of a wavefront
  constexpr int kChunks = kRowBytes / 16, kRoundTiles = kRowBytes / (32 * kElem), kRounds = (kMTiles + kRoundTiles - 1) / kRoundTiles;
  constexpr int kPerTile = kTileBytes / kSlab < 4 ? kTileBytes / kSlab : 4;  // slabs that a K or V tile has room for
  static_assert(kPerTile >= 1 && kStages * kPerTile >= 3, "four slabs in K stages and a V stage");
  uint8_t* const slab = kPerTile == 4 ? k_lds0 + wave * kSlab
                        : kPerTile >= 2 ? (wave < 2 ? k_lds0 : k_lds1) + (wave & 1) * kSlab
                                        : (wave == 0 ? k_lds0 : wave == 1 ? k_lds1 : wave == 2 ? k_lds2 : v_lds0);
  constexpr int kRowsAtOnce = 64 / kChunks;
  // 16-byte chunk ch of row r: neighbouring rows start in different banks
  auto slab_at = [](int r, int ch) __attribute__((always_inline)) { return r * kRowBytes + ((ch ^ (kChunks == 8 ? r & 7 : kChunks == 4 ? (r >> 1) & 3 : (r >> 2) & 1)) << 4); };
#pragma unroll
  for (int n = 0; n < kRounds; ++n) {
#pragma unroll
    for (int m = 0; m < kRoundTiles; ++m) {
      if (n * kRoundTiles + m >= kMTiles) break;
#pragma unroll
      for (int a2 = 0; a2 < 4; ++a2) {
        const int ch = 2 * kElem * m + (kElem == 2 ? a2 : a2 >> 1), byte = kElem == 2 ? 8 * half_o : 8 * (a2 & 1) + 4 * half_o;
        *LDS_PTR(Piece, slab + slab_at(row_o, ch) + byte) = piece(n * kRoundTiles + m, a2);
      }
    }
    const int ch = lane_o % kChunks;
#pragma unroll
    for (int p = 0; p < 32 / kRowsAtOnce; ++p) {
      const int r = p * kRowsAtOnce + lane_o / kChunks;
      const v4i x = *LDS_PTR(const v4i, slab + slab_at(r, ch));
      if (q_wave0 + r < a.seqlen_q && n * kRowBytes + 16 * ch < D * kElem)
        store_row_chunk(op + (long long)r * a.o_rs * kElem + n * kRowBytes + 16 * ch, x);
    }
  }
#endif  // __HIP_DEVICE_COMPILE__
}

template <int D, bool CAUSAL, bool E5M2, int OUT>
int launch(const KernelArgs& a, bool v_transposed, int loop, hipStream_t stream) {
  const dim3 grid((unsigned)(a.bh_total * a.n_qblocks));
  // hipLaunchKernel returns the status of this launch itself; the thread's sticky "last error" (which an earlier,
  // unrelated call may have left behind) is neither read nor cleared.
  KernelArgs args = a;
  void* argv[] = {&args};
  const void* fn = v_transposed ? (const void*)&fa8_fwd_kernel<D, CAUSAL, E5M2, OUT, true, kLoopRolling>
                                : (const void*)&fa8_fwd_kernel<D, CAUSAL, E5M2, OUT, false, kLoopRolling>;
  if constexpr (D == 64 || D == 128) {
    if (loop == FA8_SCHEDULE_PIPELINED)
      fn = v_transposed ? (const void*)&fa8_fwd_kernel<D, CAUSAL, E5M2, OUT, true, kLoopPipelined>
                        : (const void*)&fa8_fwd_kernel<D, CAUSAL, E5M2, OUT, false, kLoopPipelined>;
    if constexpr (!CAUSAL) {
      if (loop == FA8_SCHEDULE_DENSE)
        fn = v_transposed ? (const void*)&fa8_fwd_kernel<D, false, E5M2, OUT, true, kLoopDense>
                          : (const void*)&fa8_fwd_kernel<D, false, E5M2, OUT, false, kLoopDense>;
      if (loop == FA8_SCHEDULE_DENSE && a.seqlen_k % kKvBlock != 0)
        fn = v_transposed ? (const void*)&fa8_fwd_kernel<D, false, E5M2, OUT, true, kLoopDenseRagged>
                          : (const void*)&fa8_fwd_kernel<D, false, E5M2, OUT, false, kLoopDenseRagged>;
    }
  }
  return (int)hipLaunchKernel(fn, grid, dim3(kThreads), argv, 0, stream);
}

template <int D, bool CAUSAL>
int launch_types(const Fa8FwdParams* p, const KernelArgs& a, int loop, hipStream_t stream) {
  const bool e5m2 = p->in_dtype == FA8_DTYPE_E5M2, vt = p->v_layout == FA8_V_TRANSPOSED;
  if (p->out_dtype == FA8_OUT_FP16)
    return e5m2 ? launch<D, CAUSAL, true, FA8_OUT_FP16>(a, vt, loop, stream)
                : launch<D, CAUSAL, false, FA8_OUT_FP16>(a, vt, loop, stream);
  // fp8 output: the reference stores O in the input element type (csrc/flash_attention.cu:557, :655-656); the two
  // mixed combinations are not built
  if (e5m2)
    return p->out_dtype == FA8_OUT_E5M2 ? launch<D, CAUSAL, true, FA8_OUT_E5M2>(a, vt, loop, stream) : FA8_ERR_UNSUPPORTED;
  return p->out_dtype == FA8_OUT_E4M3 ? launch<D, CAUSAL, false, FA8_OUT_E4M3>(a, vt, loop, stream) : FA8_ERR_UNSUPPORTED;
}

// KV blocks walked by all workgroups of a launch together.
long long launch_kv_blocks(const Fa8FwdParams* p) {
  const long long bh = (long long)p->batch * p->heads, nq = (p->seqlen_q + kQBlock - 1) / kQBlock;
  const long long tk = (p->seqlen_k + kKvBlock - 1) / kKvBlock;
  if (!p->is_causal) return bh * nq * tk;
  // q block i walks clamp(base + 2 i, 1, tk) blocks: one block up to i = n1 - 1, all tk blocks from i = first
  const long long s64 = p->causal_align == FA8_CAUSAL_BOTTOM_RIGHT ? (long long)p->seqlen_k - p->seqlen_q : 0;
  const long long base = 2 + (s64 >= 0 ? (s64 + kKvBlock - 1) / kKvBlock : -((-s64) / kKvBlock));
  long long n1 = base <= 1 ? (1 - base) / 2 + 1 : 0;
  if (n1 > nq) n1 = nq;
  long long first = tk > base ? (tk - base + 1) / 2 : 0;
  if (first < n1) first = n1;
  if (first > nq) first = nq;
  const long long cnt = first - n1;
  return bh * (n1 + cnt * base + (n1 + first - 1) * cnt + (nq - first) * tk);
}

// Compute units of the current device (0 if the runtime cannot tell), asked once per device.  The current device must be the
// one that owns the stream and the tensors of the call (the PyTorch binding and the ctypes mirror see to it).
int compute_units() {
  static std::atomic<int> cached[64];  // zero-initialised; racing first calls store the same value
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) return 0;
  int n = cached[dev].load(std::memory_order_relaxed);
  if (n == 0) {
    if (hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || n < 1) return 0;
    cached[dev].store(n, std::memory_order_relaxed);
  }
  return n;
}

// Which main loop a valid call runs (see fa8_fwd_kernel): FA8_SCHEDULE_ROLLING, _PIPELINED or _DENSE.
// The pipelined loops exist for head dims 64 and 128 and for a softmax scale in (0, 1e6) (the pipelined loop relies on
// exp2(-inf * scale) = 0 for masked logits and on its finite stand-in for a row max of -inf times the scale staying finite);
// elsewhere every hint is ignored and the rolling loop runs.
// Dense: full (non-causal) attention.  Over a whole number of KV blocks no logit is ever masked: measured 1 - 2 % faster than the rolling
// loop on launches that fill the chip and 3 - 5 % faster than the pipelined loop on small ones, so it is the choice wherever it applies.
// Over keys that end inside a block (kLoopDenseRagged) head dim 128, new / old time: 0.87 - 0.98 where the pipelined loop ran (2 sequences,
// 16 heads, 2999 keys 96.0 -> 91.8 us; 8, 40, 777: 102 -> 92), 0.90 - 1.0 where the rolling one did (2, 32, 4097: 346 -> 336), 1.01 - 1.04 up to
// one workgroup a compute unit (1, 4, 8096: 93.7 -> 96.6), where the pipelined loop stays; head dim 64 0.91 - 1.0 above three workgroups a compute
// unit, 1.00 - 1.02 below, where it stays too.  A hint for the dense loop under a mask falls back to the automatic choice.
// Pipelined: launches that cannot keep three wavefronts on every SIMD for most of their run: at most four workgroups per
// compute unit (two resident at a time), or little work per compute unit (then filling and draining the chip, and for
// causal launches the thinning out of the workgroups, is a large share of the run).  Measured 5 - 15 % faster than the
// rolling loop there; the rolling loop is equal or up to 5 % faster elsewhere.
int choose_loop(const Fa8FwdParams* p) {
  if ((p->head_dim != 64 && p->head_dim != 128) || !(p->softmax_scale > 0.f && p->softmax_scale < 1.0e6f)) return FA8_SCHEDULE_ROLLING;
  if (p->schedule == FA8_SCHEDULE_ROLLING || p->schedule == FA8_SCHEDULE_PIPELINED) return p->schedule;
  if (!p->is_causal && (p->schedule == FA8_SCHEDULE_DENSE || p->seqlen_k % kKvBlock == 0)) return FA8_SCHEDULE_DENSE;
  const long long cus = compute_units();
  const long long wgs = (long long)p->batch * p->heads * ((p->seqlen_q + kQBlock - 1) / kQBlock);
  if (!p->is_causal && cus > 0 && wgs > (p->head_dim == 128 ? 1 : 3) * cus) return FA8_SCHEDULE_DENSE;
  // KV blocks per compute unit below which the pipelined loop was measured to win (head dim 64 has half the matrix work
  // per block)
  const long long few_blocks = p->head_dim == 64 ? 264 : 144;
  const bool small = cus > 0 && (wgs <= 4 * cus || (wgs <= few_blocks * cus && launch_kv_blocks(p) <= few_blocks * cus));
  return small ? FA8_SCHEDULE_PIPELINED : FA8_SCHEDULE_ROLLING;
}

// How the work of a call is cut (see fa8_fwd_kernel, fa8_shared_rows_kernel, fa8_split_logits_kernel).
struct Plan {
  int tiles_per_workgroup;  // of 32 query rows
  int waves_per_tile;       // 1: the loops of this file; 2, 4: wavefronts share a row tile
  int splits;               // > 1: the keys of a row tile dealt to this many workgroups (needs a workspace)
  int stages = 1;           // LDS stages of sharing wavefronts
  bool apart = false;       // sharing wavefronts each keep the sums of their own blocks
};
constexpr long long kMaxWorkspace = 256LL << 20;  // bytes that a call may ask for

// The rule, from 18 500 shapes drawn over all head dims, 1 - 10000 row tiles, 1 - 20000 keys, full and causal, grouped or not, every plan
// timed on every shape, and 9000 of `draw` in perf/cases.py.  A SIMD with one wavefront issues a vector instruction every 6 - 9 cycles, with three every 3: a launch of few
// rows is faster if several wavefronts share a row tile, up to the point where the unshared loops have about two wavefronts on every
// SIMD themselves; from there on sharing costs (a launch that fills the chip: 1.1 - 1.6x with two wavefronts a tile, 1.5 - 4x with
// four), unless the unshared launch, whose workgroups have 128 rows of one q head each, would be mostly idle.  `tiles` counts 32-row
// tiles and `pairs` workgroups of two of them (the query rows of a k/v head together), `wgs` the workgroups of the unshared launch;
// `longest` is the longest tile's KV blocks, `even` the pairs of that length that hold the same work (causal square: about half as
// many): what counts for a launch that starts its longest tiles first.  In brackets the median of shared / unshared time.
//   tiles <= CUs (head dim <= 64: 2 CUs), the most that run at once, and 3 blocks: four wavefronts a tile, one tile a workgroup
//     (0.75 at 6 blocks, 0.55 from 33 on).  At 2 blocks the exchange costs what it saves, unless the head dim is at most 128 and the
//     unshared workgroups are well filled (0.95).  Head dim <= 64, a single tile per k/v head, 12 blocks: any number, bound by HBM
//   More of them where the tiles differ in length (shortest < 3/5 longest), so that two or three share a CU with one LDS stage each and do not
//     wait for each other's barriers.  Work of the tiles / (CUs x longest): head dim <= 64 from 6 blocks on up to 1.5 (0.85 - 0.97), 16 blocks
//     1.75 (0.84 - 0.94), 24 blocks 2 (0.9); head dim 65 - 128 8 blocks 1 (0.90 - 0.93), 24 blocks 1.25 (0.86), 32 blocks 1.5 (0.82).  Equal
//     tiles: head dim <= 64, 16 blocks, up to the three a CU that run at once (0.85 - 0.97).  (13 400 drawn launches; beyond these lines 1.0 - 1.4)
//   LDS stages of one tile, four wavefronts: with one workgroup a CU (head dim <= 64: two) one stage takes 0.94 - 0.98 of the time of two below 16
//     blocks, the same at 16 - 24, 1.0 - 1.3 above (head dim 32: 0.98 at every length).  Where K and V come from memory for a tile or two alone
//     (decode steps), it takes more from fewer blocks on: head dims 96, 128 1.01 - 1.25 from 4 blocks a CU (of all k/v heads together), head dim 64 1.03 -
//     1.08 from 12 with a tile a CU at most (0.95 - 1.0 with more, below 24 blocks a head), head dim 32 1.07 - 1.26 from 32 (more than two tiles a
//     k/v head: 64).  192 heads, 42244 keys, head dim 32: 176 us with two, 222 with one; 128 heads, 1457 keys, head dim 128: 13.4, 16.9.  Two
//     stages of head dim 128 have no room for a second workgroup (0.7 - 0.8), of 64 and 32 for a third (0.8 - 0.88, up to the 4 a CU that take
//     two rounds either way: 1.02 - 1.13 from 24 blocks)
//   head dim 65 - 128, pairs <= CUs (one a CU) and 4 blocks: four wavefronts a tile, two tiles a workgroup, which share the copies of K
//     and V (0.6 - 0.85)
//   head dim above 128: the same from 16 blocks on (one LDS stage; 1.0 - 1.1 at 6 - 12 blocks, 0.95 at 16 - 24, 0.86 from 64 on, against two
//     wavefronts a tile).  Tiles of unequal length: also more pairs, from 24 blocks and even <= 3/4 CUs on (0.85 - 0.95; 1.0 - 1.1 at even = CUs)
//   no more rounds of the CUs with pairs than with unshared workgroups (full and causal, every head dim and number of rounds): two
//     wavefronts a tile, two tiles a workgroup (0.8 - 0.95; 0.2 - 0.75 where few queries of grouped heads leave half of the unshared
//     workgroups idle).  One round more costs 1.05 - 1.4, except: rounds of unequal length, even <= CUs (causal: a quarter more; head
//     dim <= 64: twice as many) and 5 blocks (head dim 32: 2) (0.8 - 1.0); head dim 32 up to 4/3 wgs (0.85 - 1.0); head dim 64 up to
//     half as many rounds more from 8 blocks on if the tiles are about equally long (0.85 - 0.95)
//   LDS stages of two tiles, two wavefronts a tile (423 drawn launches, head dims 64 - 128): with one stage a CU holds four workgroups of head dim
//     64 instead of three, three of 96 and 128 instead of two.  Where there are as many, one stage takes 0.90 - 0.96 of the time of
//     two (head dim 64) and 0.82 - 0.95 (96, 128); where there are fewer, 0.97 below 16 (8) blocks, 1.0 - 1.03 above, where two stay
//     (head dim 64, tiles of unequal length: from 8 blocks on; 40 heads, 704 keys: 9.0 us with two, 9.7 - 10.0 with one)
//     (head dims 96, 128, tiles of unequal length: 17 blocks up to 2.4 pairs a CU and even <= 5/4 CUs, 24 blocks 7/5 CUs, 28 blocks 2.5 pairs; one
//     stage takes 1.02 - 1.13 there, 0.9 - 0.93 beyond; a pair a k/v head, 10 blocks: also the 3 - 4 pairs a CU that take two rounds either way,
//     1.02 - 1.13: 1024 heads, 2097 keys, head dim 96, 80.8 us with two, 91.7 with one)
//   head dim 65 - 128, 8 blocks, more than two pairs a CU and up to the three that one stage lets run at once (causal, 16 blocks: 3.5, if
//     even <= 2 CUs): two wavefronts a tile, two tiles, though the unshared launch has fewer rounds (median 0.92, 0.82 - 1.0; beyond 1.02 - 1.4,
//     as with a mask aligned to the last key: 64 heads, 895 queries on 1841 keys, even 2.7 CUs, head dim 128: 36.9 us, 43.0 shared)
//   A single block leaves nothing to share but the products (1.05 - 1.3): only where the rows of grouped q heads fill the tiles that
//     they would leave idle, 2 pairs <= wgs, and on a full chip (0.2 - 0.8), and under the mask at head dim 32, whose unshared loop is
//     the rolling one (v as rows: 0.75 - 0.95, transposed 1.0 - 1.4)
// Splitting the keys as well costs an exchange of maxima and a reduction (where the logits do not fit in LDS a second kernel and their way
// through memory), and spreads the copies over all compute units: taken where the estimate of its time is below that of four sharing
// wavefronts, and then as fine as the compute units allow, down to one block a wavefront.  The estimates are fits (shared rows: 3003 drawn
// launches whose K and V come from HBM and 1725 whose K and V the Infinity Cache still holds; split: 1663 pairs of 306 drawn launches and a
// number of splits, K and V mostly from HBM): a start, a step per block of a wavefront's range, K and V, the parts of O, and the logits
// written and read; neither is below the rate at which it moves its bytes.  On the 306 launches the choice takes 0.5 % longer than
// the best of all numbers of splits on average; two blocks a wavefront at least, and the estimate for two kernels, took 6.5 % longer.  Of 5700 more
// launches, each measured with and without splitting, the choice is the slower one by more than 3 % in 2 of 100.  They set three things: head
// dims above 128 (one LDS stage) take K and V at 3.6 - 4.4 TB/s, from 24 blocks on added to the steps (at the 5.6 of the others 128 tiles of head dim 192, 7695 keys,
// were not split: 105 us, 82 in two parts), and two kernels 5 - 10 % longer than the fit; head dims 32 and 64 take 0.255 us a block from 56 on; and below 20 blocks head dims up to 128 are not
// split (4 heads, 974 keys, head dim 128: 8.8 us, 9.9 in four parts; 16 - 19 blocks 1.03 - 1.11).  One head, 32
// queries on 1121 keys, d128: 10.0 us shared, 19.3 split; one sequence of 32768 keys: 151 and 18; 2 sequences of 6881 keys, 8 queries of 3 k/v heads,
// group of 4, d128: 25.2 in 13 parts, 16.1 in 27.
// Sums apart (fa8_shared_rows_kernel with APART, head dims up to 128), where the caller leaves the order of the sums open: it replaces what the rules above
// give from the number of blocks on where its groups, with half the exchange, repay a longer start and the sum of the parts at the end.  24 000 drawn
// launches, K and V from HBM, median and 95th percentile of its time / theirs:
//   four wavefronts a tile, one tile: head dim 32 0.80, 0.96 and 64 0.85, 0.97 from 12 blocks on, up to two tiles a CU (below 12: 0.97 - 1.02; up to three a
//     CU 0.79 - 0.88 at head dim 32, 0.93 from 48 blocks on at 64, unless a k/v head has few rows and its bytes bound both: 1.1 - 1.3); head dim 96 0.89,
//     0.98 from 12 blocks and 128 0.94, 1.0 from 20 on, up to a tile a CU and more than one tile a k/v head (one: 0.98 - 1.05, bytes)
//   four wavefronts a tile, two tiles: 0.88, 1.0 (head dim 96, 12 blocks), 0.90, 0.99 (128, 20 blocks)
//   two wavefronts a tile, two tiles, instead of the same with sums together or of the unshared loops: head dim 32 0.90, 0.97 and 0.80, 0.92 (12 blocks, unequal
//     tiles 24; up to three pairs a CU); head dim 64 0.94, 0.99 instead of the former alone (16 blocks up to two pairs a CU, 32 up to three); head
//     dim 96 0.86, 0.95 and 0.87, 0.96 (12 blocks), 128 0.92, 0.98 and 0.90, 1.0 (24 blocks, instead of the unshared loops 32), up to the two pairs a CU that run
//     at once, k/v heads of more than 128 rows (fewer: up to 1.23, bytes); unequal tiles, 48 blocks: up to three pairs (head dim 32 from 24
//     blocks eight, 64 five), 0.87 - 0.93
void keep_sums_apart(const Fa8FwdParams* p, long long cus, long long rows, long long tiles, long long pairs, long long longest, bool unequal, Plan& n) {
  const int d = p->head_dim;
  // An fp8 output moves by a whole step of its type where the last bit of a sum carries it over a rounding boundary, 2^-9 in the range of the long
  // averages of small v, a quarter of their size: fp8 outputs keep the order of fa8_fwd, and its bits.
  if (n.splits > 1 || d > 128 || p->out_dtype != FA8_OUT_FP16) return;
  const bool many_rows = rows > 128;
  bool apart;
  if (n.waves_per_tile == 4 && n.tiles_per_workgroup == 1) {
    apart = d <= 64 ? longest >= 12 && (tiles <= 2 * cus || (tiles <= 3 * cus && many_rows && (d == 32 || longest >= 48)))
                    : longest >= (d == 96 ? 12 : 20) && tiles <= cus && rows > 32;
  } else if (n.waves_per_tile == 4) {
    apart = longest >= (d == 96 ? 12 : 20);
  } else {
    const bool shared = n.waves_per_tile == 2;
    const long long least = d == 32 ? (unequal ? 24 : 12) : (d == 64 ? (pairs <= 2 * cus ? 16 : 32) : (d == 96 ? 12 : (shared ? 24 : 32)));
    const long long most_unequal = d == 32 ? 8 : (d == 64 ? 5 : 3);
    apart = (d != 64 || shared) && longest >= least && pairs <= (d <= 64 ? 3 : 2) * cus && (d == 64 ? rows > 32 : many_rows);
    apart |= unequal && longest >= (d == 32 ? 24 : 48) && pairs <= most_unequal * cus && many_rows;
    if (apart) n = {2, 2, 1};
  }
  if (apart) {
    n.stages = 2;
    n.apart = true;
  }
}

Plan choose_plan(const Fa8FwdParams* p, bool workspace, bool any_order) {
  const Plan unshared = {kQBlock / 32, 1, 1};
  // the sharing kernels rely on exp2(-inf * scale) = 0 and a finite start of the row max, like the pipelined loop; a schedule hint
  // asks for a loop of the unshared kernel
  if (p->schedule != FA8_SCHEDULE_AUTO || !(p->softmax_scale > 0.f && p->softmax_scale < 1.0e6f) || !packable(p)) return unshared;
  const long long cus = compute_units();
  const long long group = p->heads_k > 0 ? p->heads / p->heads_k : 1, kv_heads = (long long)p->batch * (p->heads / group);
  const long long rows = group * p->seqlen_q, tiles = kv_heads * ((rows + 31) / 32);
  if (cus == 0 || p->batch > 65535 || rows > 32 * 65535LL) return unshared;
  const long long shift = p->causal_align == FA8_CAUSAL_BOTTOM_RIGHT ? (long long)p->seqlen_k - p->seqlen_q : 0;
  auto blocks_of = [&](long long q_last) {  // KV blocks that query q_last sees, at least one
    const long long keys = p->is_causal ? std::min<long long>(p->seqlen_k, q_last + 1 + shift) : p->seqlen_k;
    return std::max(1LL, (keys + kKvBlock - 1) / kKvBlock);
  };
  const long long longest = blocks_of(p->seqlen_q - 1), shortest = blocks_of(std::min<long long>(31 / group, p->seqlen_q - 1));
  const int d = p->head_dim;
  const long long pairs = kv_heads * ((rows + 63) / 64), wgs = (long long)p->batch * p->heads * ((p->seqlen_q + kQBlock - 1LL) / kQBlock);
  // mean length of the tiles: half way between the first and the last one, but for rows that see every key or none
  const long long even = pairs * (longest + shortest) / (2 * longest);
  // the same for workgroups of one tile, in quarters of the compute units; only lengths that differ make room for more than run at once
  const bool unequal = 5 * shortest < 3 * longest;
  const long long quarters = (tiles * (longest + shortest) / (2 * longest) * 4 + cus - 1) / cus;
  const long long most_quarters = d <= 64 ? (longest < 16 ? 6 : (longest < 24 ? 7 : 8)) : (d > 128 ? 0 : (longest < 24 ? 4 : (longest < 32 ? 5 : 6)));
  const long long pair_rounds = (pairs + cus - 1) / cus, wg_rounds = (wgs + cus - 1) / cus;
  const bool no_more_rounds = pair_rounds <= wg_rounds || (d == 32 && 3 * pairs <= 4 * wgs) ||
                              (d == 64 && longest >= 8 && 5 * shortest > 3 * longest && 2 * pair_rounds <= 3 * wg_rounds);
  const bool few_pairs = (longest >= 5 || d == 32) && 4 * even <= (p->is_causal ? 5 : 4) * (d <= 64 ? 2 : 1) * cus;
  const bool three_a_cu = d > 64 && d <= 128 && longest >= 8 && pairs > 2 * cus &&
                          (pairs <= 3 * cus || (unequal && longest >= 16 && 2 * pairs <= 7 * cus && even <= 2 * cus));
  const bool unequal_pairs = unequal && (longest >= 24 ? 5 * even <= 7 * cus : longest >= 17 && 4 * even <= 5 * cus) &&
                             (longest >= 28 ? 2 * pairs < 5 * cus : 5 * pairs <= 12 * cus);
  const bool two_rounds = rows <= 64 && longest >= 10 && pairs > 3 * cus && pairs <= 4 * cus;
  const bool one_block = (2 * pairs <= wgs && wgs > 2 * cus) || (d == 32 && p->is_causal && p->v_layout == FA8_V_ROWS && pairs <= wgs);
  // one tile a workgroup, two LDS stages: they run at once, or in no more rounds than with one stage; and K and V come from memory for a tile or two
  const bool two_fit = d <= 128 && (tiles <= (d <= 64 ? 2 : 1) * cus || (d <= 64 && longest >= 24 && tiles > 3 * cus && tiles <= 4 * cus));
  const long long own_blocks = d == 32 ? (rows <= 64 ? 32 : 64) : (rows > 64 || (d == 64 && tiles > cus) ? 1LL << 40 : (d == 64 ? 12 : 4));
  const bool own_kv = kv_heads * longest >= own_blocks * cus;
  Plan n = unshared;
  if ((longest >= 3 && tiles <= (d <= 64 ? 2 : 1) * cus) || (longest >= 12 && d <= 64 && rows <= 32) ||
      (longest == 2 && d <= 128 && tiles <= cus && 8 * wgs < 5 * tiles))
    n = {1, 4, 1, two_fit && ((longest >= 24 && d > 32) || own_kv) ? 2 : 1};
  else if (longest >= (d <= 64 ? 6 : 8) && (unequal ? quarters <= most_quarters : d <= 64 && tiles <= 3 * cus && longest >= 16))
    n = {1, 4, 1};
  else if (d > 64 && rows > 32 && ((pairs <= cus && longest >= (d <= 128 ? 4 : 16)) || (d > 128 && 4 * even <= 3 * cus && longest >= 24)))
    n = {2, 4, 1, d <= 128 ? 2 : 1};
  else if (longest >= 2 ? no_more_rounds || few_pairs || three_a_cu : one_block)
    n = {2, 2, 1, d == 32 || (d == 64 && longest >= (unequal ? 8 : 16) && pairs <= 3 * cus) ||
                          (d > 64 && d <= 128 && longest >= 8 && (pairs <= 2 * cus || unequal_pairs || two_rounds)) ? 2 : 1};
  if (workspace && n.waves_per_tile == 4 && n.tiles_per_workgroup == 1 && longest >= (d <= 128 ? 20 : 16)) {
    const long long most = std::max(1LL, std::min({32LL, cus / tiles, longest / 4}));  // one workgroup more than CUs takes twice as long
    const SplitForm form = split_form(p, (int)most);
    const long long splits = form.splits;
    const double range = form.blocks_per_range, row_bytes = d <= 32 ? 32 : (d <= 64 ? 64 : (d <= 128 ? 128 : 256));  // of an LDS tile
    const double kv_bytes = 2.0 * kv_heads * longest * kKvBlock * d, live = rows < 32 ? (double)rows : 32.0;
    const double s_bytes = 8.0 * tiles * live * longest * kKvBlock;
    const double shared_us = std::max({5.4 + (d <= 64 ? 0.23 : (d <= 128 ? 0.30 : 0.63)) * longest, 5.4 + kv_bytes / 5.6e6,
                                       d <= 64 ? 4.0 + 0.255 * longest : (d <= 128 || longest < 24 ? 0.0 : 4.1 + (d <= 192 ? 0.59 : 0.65) * longest + kv_bytes / 13.6e6)});
    const double split_us =
        form.one_kernel
            ? std::max(7.7 + (0.53 + 0.0057 * row_bytes) * range + kv_bytes / 23.5e6 + 1.34e-3 * d * live + 0.07 * splits, 5.4 + kv_bytes / 5.6e6)
            : (d <= 128 ? 1.0 : (d <= 192 ? 1.05 : 1.1)) *
                  std::max(7.5 + (0.6 + 0.0054 * row_bytes) * range + kv_bytes / 9.3e6 + 0.9e-3 * d * live + 0.16 * splits +
                               0.063 * range * live + s_bytes / 11e6, 2.3 + (kv_bytes + s_bytes) / 5.8e6);
    if (splits > 1 && split_us < shared_us && tiles * splits < 65536 && longest / (4 * splits) < 65535 &&
        split_workspace(p, (int)splits) <= kMaxWorkspace)
      n.splits = (int)splits;
  }
  if (any_order) keep_sums_apart(p, cus, rows, tiles, pairs, longest, unequal, n);
  return n;
}

// Tuning aid for measurements only: FA8_CAUSAL_INTERLEAVE=n in the environment (read once) replaces the number of heads of an
// XCD that take turns at every q block of a causal launch (see decode_block; the results do not depend on it).  0: unset.
int env_causal_interleave() {
  static std::atomic<int> cached{-1};
  int v = cached.load(std::memory_order_relaxed);
  if (v < 0) {
    const char* e = std::getenv("FA8_CAUSAL_INTERLEAVE");
    v = e ? std::atoi(e) : 0;
    if (v < 0 || v > 64) v = 0;
    cached.store(v, std::memory_order_relaxed);
  }
  return v;
}

bool span_ok(long long outer_stride, long long inner_extent) { return outer_stride >= inner_extent; }

}  // namespace

extern "C" int fa8_fwd_validate(const Fa8FwdParams* p) {
  if (p == nullptr || p->q == nullptr || p->k == nullptr || p->v == nullptr || p->o == nullptr) return FA8_ERR_NULL;
  if (p->batch < 1 || p->heads < 1 || p->seqlen_q < 1 || p->seqlen_k < 1 || p->head_dim < 1) return FA8_ERR_SHAPE;
  if (p->is_causal != 0 && p->is_causal != 1) return FA8_ERR_SHAPE;
  if (p->heads_k < 0 || (p->heads_k > 0 && p->heads % p->heads_k != 0)) return FA8_ERR_SHAPE;
  if (p->causal_align != FA8_CAUSAL_TOP_LEFT && p->causal_align != FA8_CAUSAL_BOTTOM_RIGHT) return FA8_ERR_DTYPE;
  if (p->schedule < FA8_SCHEDULE_AUTO || p->schedule > FA8_SCHEDULE_DENSE) return FA8_ERR_DTYPE;
  if (p->reserved0 != 0) return FA8_ERR_UNSUPPORTED;  // a field of a later version of the parameter block
  if ((long long)p->batch * p->heads > 0x7fffffffLL / ((p->seqlen_q + kQBlock - 1) / kQBlock)) return FA8_ERR_SHAPE;
  if (p->in_dtype != FA8_DTYPE_E4M3 && p->in_dtype != FA8_DTYPE_E5M2) return FA8_ERR_DTYPE;
  if (p->out_dtype != FA8_OUT_FP16 && p->out_dtype != FA8_OUT_E4M3 && p->out_dtype != FA8_OUT_E5M2) return FA8_ERR_DTYPE;
  if (p->v_layout != FA8_V_ROWS && p->v_layout != FA8_V_TRANSPOSED) return FA8_ERR_DTYPE;
  if (p->head_dim % 32 != 0 || p->head_dim > 256) return FA8_ERR_HEAD_DIM;
  if (!(p->softmax_scale == p->softmax_scale) || std::isinf(p->softmax_scale)) return FA8_ERR_SCALE;
  const long long d = p->head_dim;
  const long long v_rows = p->v_layout == FA8_V_ROWS ? p->seqlen_k : d;
  const long long v_cols = p->v_layout == FA8_V_ROWS ? d : p->seqlen_k;
  if (!span_ok(p->q_row_stride, d) || !span_ok(p->q_head_stride, 1) || !span_ok(p->q_batch_stride, 1)) return FA8_ERR_STRIDE;
  if (!span_ok(p->k_row_stride, d) || !span_ok(p->k_head_stride, 1) || !span_ok(p->k_batch_stride, 1)) return FA8_ERR_STRIDE;
  if (!span_ok(p->v_row_stride, v_cols) || !span_ok(p->v_head_stride, 1) || !span_ok(p->v_batch_stride, 1)) return FA8_ERR_STRIDE;
  if (!span_ok(p->o_row_stride, d) || !span_ok(p->o_head_stride, 1) || !span_ok(p->o_batch_stride, 1)) return FA8_ERR_STRIDE;
  // 16-byte vector loads of q/k/v rows; o is stored in pieces of 8 (fp8: 4) bytes or in 16-byte chunks that need no more than this alignment
  const long long in_strides[] = {p->q_batch_stride, p->q_head_stride, p->q_row_stride, p->k_batch_stride, p->k_head_stride,
                                  p->k_row_stride,   p->v_batch_stride, p->v_head_stride, p->v_row_stride};
  for (long long s : in_strides)
    if (s % 16 != 0) return FA8_ERR_ALIGN;
  if (((uintptr_t)p->q | (uintptr_t)p->k | (uintptr_t)p->v) % 16 != 0) return FA8_ERR_ALIGN;
  const long long o_elem = p->out_dtype == FA8_OUT_FP16 ? 2 : 1;
  const long long o_strides[] = {p->o_batch_stride, p->o_head_stride, p->o_row_stride};
  for (long long s : o_strides)
    if ((s * o_elem) % 8 != 0) return FA8_ERR_ALIGN;
  if ((uintptr_t)p->o % 8 != 0) return FA8_ERR_ALIGN;
  if (p->lse != nullptr) {
    if (!span_ok(p->lse_head_stride, p->seqlen_q) || !span_ok(p->lse_batch_stride, 1)) return FA8_ERR_STRIDE;
    if ((uintptr_t)p->lse % 4 != 0) return FA8_ERR_ALIGN;
  }
  // the kernels address k and v of one head with 32-bit byte offsets; a tile copy forms offsets for all 64 rows of a
  // block (rows past the end are not read, but their offsets are computed), hence at least 64 rows here
  const long long k_rows_addr = p->seqlen_k > kKvBlock ? p->seqlen_k : kKvBlock;
  const long long v_rows_addr = v_rows > kKvBlock ? v_rows : kKvBlock;
  if (k_rows_addr * p->k_row_stride > 0x7fffffffLL || v_rows_addr * p->v_row_stride > 0x7fffffffLL) return FA8_ERR_SHAPE;
  // ... and the offsets of a whole block just past the last row (block offset + row offset of its 64th row) must not wrap
  // around 32 bits, or the buffer's range check would take them for rows of the tensor (matters only for a few rows with a
  // row stride of tens of megabytes)
  if ((p->seqlen_k + 126LL) * p->k_row_stride + 256 > 0xffffffffLL || (v_rows + 126LL) * p->v_row_stride + 256 > 0xffffffffLL)
    return FA8_ERR_SHAPE;
  // transposed v is read in 16-byte chunks along kv
  if (p->v_layout == FA8_V_TRANSPOSED && p->seqlen_k % 16 != 0) return FA8_ERR_ALIGN;
  // an fp8 output has the element type of the inputs
  if ((p->out_dtype == FA8_OUT_E4M3 && p->in_dtype != FA8_DTYPE_E4M3) || (p->out_dtype == FA8_OUT_E5M2 && p->in_dtype != FA8_DTYPE_E5M2))
    return FA8_ERR_UNSUPPORTED;
  return FA8_OK;
}

namespace {

// Whether O leaves as whole lines, through LDS (the epilogues; the same bits either way).  The way costs a workgroup a barrier, an LDS round trip and
// instructions that are not in the cache yet, the pieces cost the L2s when many rows leave together.  2049 unshared and 3685 two-tile launches, drawn; time of lines / of
// pieces, median (95th percentile), with 256 compute units:
//   unshared, O above 1.8 MB: 0.94 (0.995), below: 1.07 (1.17); up to 32 queries: 1.06 (1.10) also above
//   two tiles a workgroup: a k/v head with no more than 32 rows, that is with one tile: 1.05
//     head dims 192 and 256 0.967 (1.013) whatever the size
//     128, and fp16 of 64: 0.964 (0.997) above 8192 rows, 1.06 (1.12) below
//     fp16 of 96, 160 and 224: 0.98 (1.01) above 16384 rows, 1.0 (1.06) from 8192 on, 1.08 below
//     fp8 of 64, 96, 160 and 224: 1.0 (1.04 - 1.12) above, 1.02 - 1.07 below; head dim 32: 1.0 - 1.02 (1.06) above, 1.07 below
// (Launches that keep the pieces take 0.99 - 1.01 of the time that they took in a library without lines.)
bool whole_lines(const Fa8FwdParams* p, bool shared) {
  const bool fp16 = p->out_dtype == FA8_OUT_FP16;
  const long long cus = compute_units(), rows = (long long)p->batch * p->heads * p->seqlen_q;
  const int d = p->head_dim, group = p->heads_k > 0 ? p->heads / p->heads_k : 1;
  if (!shared) return p->seqlen_q > 32 && rows * d * (fp16 ? 2 : 1) > 7168 * cus;
  if ((long long)group * p->seqlen_q <= 32) return false;
  if (d == 192 || d == 256) return true;
  if (d == 128 || (d == 64 && fp16)) return rows > 32 * cus;
  return fp16 && d > 32 && rows > 64 * cus;
}

// One wavefront per 32 query rows: the kernel of this file.
int launch_rows(const Fa8FwdParams* p, hipStream_t stream) {
  KernelArgs a;
  a.q = (const uint8_t*)p->q;
  a.k = (const uint8_t*)p->k;
  a.v = (const uint8_t*)p->v;
  a.o = p->o;
  a.lse = (float*)p->lse;
  a.lse_bs = p->lse_batch_stride; a.lse_hs = p->lse_head_stride;
  a.kv_group = p->heads_k > 0 ? p->heads / p->heads_k : 1;
  a.causal_shift = p->causal_align == FA8_CAUSAL_BOTTOM_RIGHT ? p->seqlen_k - p->seqlen_q : 0;
  a.heads = p->heads;
  a.seqlen_q = p->seqlen_q;
  a.seqlen_k = p->seqlen_k;
  a.n_qblocks = (p->seqlen_q + kQBlock - 1) / kQBlock;
  a.bh_total = p->batch * p->heads;
  a.interleave = a.bh_total / 8 < 8 ? (a.bh_total / 8 > 0 ? a.bh_total / 8 : 1) : 8;  // causal launches, see decode_block
  if (env_causal_interleave() > 0) a.interleave = env_causal_interleave();
  a.scale_log2 = p->softmax_scale * 1.4426950408889634f;
  a.whole_lines = whole_lines(p, false);
  a.q_bs = p->q_batch_stride; a.q_hs = p->q_head_stride; a.q_rs = p->q_row_stride;
  a.k_bs = p->k_batch_stride; a.k_hs = p->k_head_stride; a.k_rs = p->k_row_stride;
  a.v_bs = p->v_batch_stride; a.v_hs = p->v_head_stride; a.v_rs = p->v_row_stride;
  a.o_bs = p->o_batch_stride; a.o_hs = p->o_head_stride; a.o_rs = p->o_row_stride;
  const int loop = choose_loop(p);
  switch (p->head_dim) {
#define FA8_HEAD_DIM_CASE(D_) \
  case D_: return p->is_causal ? launch_types<D_, true>(p, a, loop, stream) : launch_types<D_, false>(p, a, loop, stream)
    FA8_HEAD_DIM_CASE(32);  // the head-dim buckets of the reference (csrc/static_switch.h:50-77)
    FA8_HEAD_DIM_CASE(64);
    FA8_HEAD_DIM_CASE(96);
    FA8_HEAD_DIM_CASE(128);
    FA8_HEAD_DIM_CASE(160);
    FA8_HEAD_DIM_CASE(192);
    FA8_HEAD_DIM_CASE(224);
    FA8_HEAD_DIM_CASE(256);
#undef FA8_HEAD_DIM_CASE
    default: return FA8_ERR_HEAD_DIM;
  }
}

int run(const Fa8FwdParams* p, void* workspace, long long bytes, unsigned late, bool any_order, hipStream_t stream) {
  Plan n = choose_plan(p, workspace != nullptr, any_order);
  if (n.splits > 1 && bytes < split_workspace(p, n.splits)) n = choose_plan(p, false, any_order);
  if (n.splits > 1) return (uintptr_t)workspace % 16 != 0 ? FA8_ERR_ALIGN : launch_split(p, n.splits, workspace, late, stream);
  return n.waves_per_tile > 1 ? launch_shared(p, n.tiles_per_workgroup, n.waves_per_tile, n.stages, n.apart, n.tiles_per_workgroup > 1 && whole_lines(p, true), stream)
                              : launch_rows(p, stream);
}

}  // namespace

extern "C" int fa8_fwd(const Fa8FwdParams* p, void* hip_stream) {
  const int rc = fa8_fwd_validate(p);
  return rc != FA8_OK ? rc : run(p, nullptr, 0, 0, false, (hipStream_t)hip_stream);
}

extern "C" int fa8_fwd_ws(const Fa8FwdParams* p, void* workspace, int64_t bytes, void* hip_stream) {
  const int rc = fa8_fwd_validate(p);
  return rc != FA8_OK ? rc : run(p, workspace, bytes, 0, false, (hipStream_t)hip_stream);
}

extern "C" int fa8_fwd_ws_late(const Fa8FwdParams* p, void* workspace, int64_t bytes, uint32_t late_parts, void* hip_stream) {
  const int rc = fa8_fwd_validate(p);
  return rc != FA8_OK ? rc : run(p, workspace, bytes, late_parts, false, (hipStream_t)hip_stream);
}

extern "C" int fa8_fwd_any_order(const Fa8FwdParams* p, void* workspace, int64_t bytes, void* hip_stream) {
  const int rc = fa8_fwd_validate(p);
  return rc != FA8_OK ? rc : run(p, workspace, bytes, 0, true, (hipStream_t)hip_stream);
}

extern "C" int fa8_fwd_apart(const Fa8FwdParams* p) {
  const int rc = fa8_fwd_validate(p);
  return rc != FA8_OK ? rc : (int)choose_plan(p, true, true).apart;
}

extern "C" int fa8_fwd_workspace(const Fa8FwdParams* p, int64_t* bytes) {
  const int rc = fa8_fwd_validate(p);
  if (rc != FA8_OK) return rc;
  if (bytes == nullptr) return FA8_ERR_NULL;
  const Plan n = choose_plan(p, true, false);  // (the same bytes for fa8_fwd_any_order: it changes no call that splits its keys)
  *bytes = n.splits > 1 ? split_workspace(p, n.splits) : 0;
  return FA8_OK;
}

extern "C" int fa8_fwd_plan(const Fa8FwdParams* p, int with_workspace, int32_t* rows_per_workgroup, int32_t* wavefronts_per_tile,
                            int32_t* kv_splits) {
  const int rc = fa8_fwd_validate(p);
  if (rc != FA8_OK) return rc;
  if (rows_per_workgroup == nullptr || wavefronts_per_tile == nullptr || kv_splits == nullptr) return FA8_ERR_NULL;
  const Plan n = choose_plan(p, with_workspace != 0, with_workspace == FA8_PLAN_ANY_ORDER);
  *rows_per_workgroup = 32 * n.tiles_per_workgroup;
  *wavefronts_per_tile = n.waves_per_tile;
  *kv_splits = n.splits;
  return FA8_OK;
}

extern "C" int fa8_fwd_form(const Fa8FwdParams* p, int with_workspace, int32_t* lds_stages, int32_t* kernels) {
  const int rc = fa8_fwd_validate(p);
  if (rc != FA8_OK) return rc;
  if (lds_stages == nullptr || kernels == nullptr) return FA8_ERR_NULL;
  const Plan n = choose_plan(p, with_workspace != 0, with_workspace == FA8_PLAN_ANY_ORDER);
  *lds_stages = n.waves_per_tile > 1 && n.splits == 1 ? n.stages : 0;
  *kernels = n.splits > 1 && !split_form(p, n.splits).one_kernel ? 2 : 1;
  return FA8_OK;
}

extern "C" int fa8_fwd_schedule(const Fa8FwdParams* p) {
  const int rc = fa8_fwd_validate(p);
  if (rc != FA8_OK) return rc;
  return choose_loop(p);
}

extern "C" int fa8_query(int what) {
  switch (what) {
    case FA8_QUERY_VERSION: return kVersion;
    case FA8_QUERY_KV_BLOCK: return kKvBlock;
    case FA8_QUERY_Q_BLOCK: return kQBlock;
    case FA8_QUERY_KV_ASCENDING: return 1;
    case FA8_QUERY_THREADS: return kThreads;
    case FA8_QUERY_PARAMS_SIZE: return (int)sizeof(Fa8FwdParams);
    default: return -1;
  }
}

extern "C" const char* fa8_error_string(int code) {
  switch (code) {
    case FA8_OK: return "ok";
    case FA8_ERR_NULL: return "a required pointer is NULL";
    case FA8_ERR_SHAPE: return "bad shape (a size < 1, too many workgroups, heads not a multiple of heads_k, or k/v of one head spanning 2 GiB or more)";
    case FA8_ERR_HEAD_DIM: return "head_dim must be a multiple of 32, at most 256";
    case FA8_ERR_STRIDE: return "a stride is smaller than the extent it spans";
    case FA8_ERR_ALIGN: return "q/k/v rows and a workspace must be 16-byte aligned and o rows 8-byte aligned";
    case FA8_ERR_DTYPE: return "unknown in_dtype / out_dtype / v_layout / causal_align code";
    case FA8_ERR_UNSUPPORTED: return "this build has no kernel for the requested combination";
    case FA8_ERR_SCALE: return "softmax_scale must be finite";
    default: return code > 0 ? hipGetErrorString((hipError_t)code) : "unknown fa8 error code";
  }
}
