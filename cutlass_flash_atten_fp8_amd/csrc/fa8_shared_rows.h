// Attention for launches with few query rows per compute unit: R tiles of 32 query rows per workgroup, each tile shared by W
// wavefronts (the kernels of fa8_fwd_gfx950.hip give a tile to one wavefront).
//
// W KV blocks of 64 rows are in work at a time.  Wavefront w of a tile computes S^T, the row max and the weights of block w; the
// row maxima of the W blocks meet in LDS, so every wavefront follows the running max block by block, exactly as one wavefront
// walking the blocks would.  The fp8 weights go through LDS too, and wavefront w then adds the W blocks, in order, to ITS
// 32-column tiles of O^T (tiles w, w + W, ...).  Every logit, weight and sum is formed by the same instructions in the same order
// as in the other kernels: the results are equal bit for bit.
//
// One iteration, one group of W blocks (STAGES == 2; the copies fly for an iteration or more):
//   row max of the group's S -> LDS | barrier 1 | running max; weights of sub-tile 0, PV products of the group before between their
//   chunks, copy of K two groups ahead | barrier 2 | weights of sub-tile 1, S^T products of the next group between their chunks, copy of
//   V of the next group; weights and row sums -> LDS
// One stage (STAGES == 1): the copies of the next group's K and this group's V fly for half an iteration.  Head dims above 128 have LDS for no more;
// up to 128 it lets two to four workgroups share a compute unit, each with barriers of its own: the one works while the other waits (16
// heads, 1024 keys, head dim 128, causal: 12.98 us with two tiles a workgroup, 11.73 with one and one stage).  Half an iteration is too short a
// flight where K and V come from memory for a tile or two alone.  choose_plan has the lines between the two and both sides of each.
//
// What bounds it: the one or two wavefronts of a SIMD walk one chain (row max - LDS - barrier - weights - LDS - barrier), about 310
// instructions a wavefront and iteration, each 5 cycles or more apart within a wavefront whatever its kind; 3500 cycles at R = 2, W = 4.
// Not the LDS (its reads run at 29 % of the cycles), not the copies alone (10 % without them), not the exponentials (10 %).
// With fewer stages or all copies of a half iteration started at its beginning the copies are the limit (4100 - 4700).
// S^T of the next group is formed also where no group follows (a stale tile, never used): behind a branch, the wait counts of the
// two paths met at every chunk and each one waited for the LDS reads just issued; with the additions of the row sums pinned to their
// chunks (the compiler moved all 32 to the end, with the weights alive until then) the registers went from 194 to 153 (R 2, W 4, head dim
// 128) and from 255 to 215 (R 2, W 2, head dim 256).  16 sequences of 8191 keys, K and V from the cache, 42.9 -> 41.1 us; 512 queries on 16384
// keys 102.1 -> 100.5; 16 heads, 2048 keys, head dim 256, causal 39.2 -> 38.4 (in a captured graph).  Measured (us, one wavefront a tile -> shared):
// 16 heads, 1024 keys, causal: head dim 64 13.3 -> 8.9 (R 1, W 4), 128 17.2 -> 12.4 (2, 4); 8 heads of 2048 keys, head dim 128, full: 28.5 ->
// 19.5 (2, 4); 512 queries on 16384 keys, 32 heads on 8 k/v heads: 176 -> 100 (2, 4); 8 heads, 3000 keys, head dim 160, causal: (2, 2) 43.5 -> (2, 4) 37.1; 16 heads, 2048 keys, head dim 256, causal: 47.1 ->
// 36.4 (2, 2); 1 query of 32 heads on 8 k/v heads, 16 sequences of 8191 keys: 137 -> 52, the rate of a plain copy (1, 4).
// Registers: two wavefronts a SIMD leave a lane 256, of which head dims 224 and 256 with two tiles take about 220.  (Transposed v: copies and
// fragments take their row differences from scalar and immediate offsets; with a register for each, 31 - 42 were once spilled there:
// 16 heads, 2048 keys, causal 76.4 us instead of 36.8, against 51.7 of the unshared loop.)
//
// APART (two LDS stages, head dims up to 128): the wavefronts of a tile exchange row maxima only.  Wavefront w takes every W-th block, its weights against
// the running max after that block as before, and adds the products to an O and an l of its own, brought to its own running max; at the end the W
// O's meet in the LDS of K and V and are added in order.  Logits and weights are the same bit for bit, the fp32 sums are taken in another order.
//   softmax of group g, chunks 0 - 5: S^T products of group g + 1 between them, copy of V of group g; row max of group g + 1 -> LDS | barrier 1 |
//   O to the max of group g - 1; chunks 6 and 7: PV products of group g - 1 between them, copy of K of group g + 3 | R > 1: barrier 2
// No weights go through LDS, no wavefront is without a column tile (head dims 32 and 64), every wavefront reads one block of K and V, and the latency of
// the exchange lies under chunks 6 and 7: without the barriers it takes 0.98 of the time.  What bounds it: the 211 vector instructions of a block (64 of them
// the rescaling of O, needed in two thirds of the groups, four blocks apart: 5 % of the time) at the rate of two wavefronts a SIMD, and the tile copies
// (8 KB a block and wavefront, twice the unshared loops': 10 %).  Copies spread over the chunks with an iteration or more of flight: started together after
// barrier 1 they took 102 us on the 512 queries below, the form with the sums together 99, this 91.  Prefetching into the L2 gives nothing,
// operands fetched two products ahead neither.  Measured (us, sums together -> apart, calls in a captured graph over rotating inputs): 512 queries on 16384 keys, 32 heads on 8 k/v heads, head
// dim 128: 98.8 -> 89.4; on 4096 keys 29.2 -> 27.0; 64 heads, 128 queries on 8192 keys, head dim 64: 39.4 -> 29.8; 4 heads, 4096 keys, causal, head dim 64: 21.5 -> 16.9; 4 heads,
// 4096 keys, full, head dim 96: 29.3 -> 25.7; 16 heads, 1024 keys, causal, head dim 64: 8.7 -> 7.8.  The lines of the rule: keep_sums_apart.
#ifndef FA8_SHARED_ROWS_H_
#define FA8_SHARED_ROWS_H_
#include <type_traits>

#include "fa8_device.h"

namespace fa8 {

constexpr float kMaxStart = -1.0e30f;  // below every possible logit, finite: see m_run in fa8_fwd_kernel

// 112 bytes: a larger argument block makes the launch itself slower on the host (2.75 us up to 112 bytes, 3.4 - 3.6 us from 120 on,
// an empty kernel in a loop).  Strides are in units of 16 elements (q, k, v) and 4 elements (o); see packable and pack_mode.
// The kernel takes the fields one by one in this order: the first 14 dwords then are in scalar registers when a wavefront starts
// (-amdgpu-kernarg-preload-count), and the first loads need not wait the 800 cycles that the arguments take from host memory.
#define FA8_SHARED_FIELDS(X)                                                                                                       \
  X(const uint8_t*, q) X(unsigned, k_hs) X(unsigned, k_rs) X(unsigned, k_bs) X(unsigned, q_hs) X(unsigned, q_rs) X(unsigned, q_bs) \
  X(int, seqlen_q) X(int, seqlen_k) X(unsigned, mode) X(float, scale_log2) X(const uint8_t*, v) X(void*, o) X(float*, lse)         \
  X(unsigned, v_bs) X(unsigned, v_hs) X(unsigned, v_rs) X(unsigned, o_bs) X(unsigned, o_hs) X(unsigned, o_rs)                      \
  X(unsigned, lse_bs) X(unsigned, lse_hs)
struct SharedArgs {
  const uint8_t* k;
#define FA8_FIELD(type, name) type name;
  FA8_SHARED_FIELDS(FA8_FIELD)
#undef FA8_FIELD
};
static_assert(sizeof(SharedArgs) == 112, "see above");

template <int D, bool E5M2, bool VT, int R, int W, int STAGES, bool APART>
__global__ __launch_bounds__(64 * R * W) __attribute__((amdgpu_waves_per_eu(2))) void fa8_shared_rows_kernel(
    const uint8_t* k_
#define FA8_FIELD(type, name) , type name##_
    FA8_SHARED_FIELDS(FA8_FIELD)
#undef FA8_FIELD
) {
#if defined(__HIP_DEVICE_COMPILE__)
  const SharedArgs a = {k_
#define FA8_FIELD(type, name) , name##_
                        FA8_SHARED_FIELDS(FA8_FIELD)
#undef FA8_FIELD
  };
  constexpr int DP = D <= 32 ? 32 : (D <= 64 ? 64 : (D <= 128 ? 128 : 256));
  constexpr int kTileBytes = kKvBlock * DP;
  constexpr int kKSteps = (D + 63) / 64;
  constexpr int kMTiles = D / 32;
  constexpr int kOut = (kMTiles + W - 1) / W;     // O^T tiles that a wavefront writes (the last wavefronts may have one less, or none)
  constexpr int kOwn = APART ? kMTiles : kOut;    // ... and adds products to: tiles kFirst + m * kStep
  constexpr int kStep = APART ? 1 : W;
  constexpr int kSegs = kTileBytes / 1024;        // 1 KB copy segments per K or V tile, shared by the R wavefronts of a block
  static_assert(!APART || STAGES == 2, "sums apart: two stages");
  static_assert(kSegs % R == 0, "a block's copy is split evenly over the row tiles");
  constexpr int kPasses = kSegs / R;
  // two stages each, separate objects: the compiler then knows that copies in flight do not alias the reads (see fa8_fwd_kernel)
  __shared__ __attribute__((aligned(1024))) uint8_t k_lds0[W * kTileBytes];
  __shared__ __attribute__((aligned(1024))) uint8_t k_lds1[STAGES == 2 ? W * kTileBytes : 16];
  __shared__ __attribute__((aligned(1024))) uint8_t v_lds0[W * kTileBytes];
  __shared__ __attribute__((aligned(1024))) uint8_t v_lds1[STAGES == 2 ? W * kTileBytes : 16];
  __shared__ __attribute__((aligned(1024))) uint8_t p_lds[APART ? 16 : R * W * 2048];
  __shared__ float max_lds[(APART ? 2 : 1) * R * W * 32];
  __shared__ float sum_lds[R * W * 64];

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int r = wave / W, w = wave - r * W;  // row tile of the workgroup, block of the group
  const int qn = lane & 31, h = lane >> 5;

  // grid: k/v heads x batches x row tiles.  Workgroups start in that order (x fastest) and go to the XCDs in turn, so a k/v head
  // stays on one XCD when there is a multiple of 8 of them; causal: the longest tiles of all heads first.
  const bool causal = a.mode & kSharedCausal;
  const int group = (int)(a.mode >> kSharedGroup), group_shift = (int)(a.mode >> kSharedShift) & 31;
  const int hk = blockIdx.x, b = blockIdx.y;
  // (gridDim would have to be loaded from memory)
  const int tiles = (group * a.seqlen_q + 32 * R - 1) / (32 * R);
  const int tile = causal ? tiles - 1 - (int)blockIdx.z : (int)blockIdx.z;
  // The query rows of a k/v head: row x is query x / group of q head x % group of the group.
  auto query_of = [&](int x) __attribute__((always_inline)) { return group_shift < 31 ? x >> group_shift : x / group; };
  const int last_row = group * a.seqlen_q - 1;
  const int row0 = (tile * R + r) * 32;  // first row of this wavefront's tile
  const int row = row0 + qn;
  const int k_rs = (int)a.k_rs * 16, v_rs = (int)a.v_rs * 16;
  const uint8_t* kp = a.k + ((unsigned long long)a.k_bs * b + (unsigned long long)a.k_hs * hk) * 16;
  const uint8_t* vp = a.v + ((unsigned long long)a.v_bs * b + (unsigned long long)a.v_hs * hk) * 16;
  const float c = a.scale_log2;

  // ---- HBM -> LDS copies (see fa8_fwd_kernel): wavefront (r, w) copies segments r, r + R, ... of block w of a group ----
  constexpr unsigned kNoSource = 0x80000000u;
  // A lane's offset in a segment depends on the segment number through few of its bits (the swizzle) and otherwise by whole rows:
  // segments that are kKVar (kVVar) apart differ by a multiple of the row stride.
  constexpr int kKVar = DP == 256 ? 4 : (DP == 128 ? 2 : 1);
  constexpr int kVVar = DP == 256 && !VT ? 2 : 1;  // (transposed v: all segments share one offset, see issue_v)
  // row of the block that a segment's rows count from
  auto k_row0 = [](int seg) {
    if (DP == 256) return 16 * (seg >> 3) + 4 * ((seg >> 1) & 3) + 32 * (seg & 1);
    if (DP == 128) return 16 * (seg >> 2) + 4 * (seg & 3);
    return DP == 64 ? 16 * (seg >> 1) + 8 * (seg & 1) : 16 * seg;
  };
  auto v_row0 = [](int seg) { return seg * (1024 / DP); };
  unsigned k_src[kPasses], v_src[VT ? 1 : kPasses];
  int v_chunk = 0;  // transposed v: the lane's first key of a block
#pragma unroll
  for (int p = 0; p < kPasses; ++p) {
    const int seg = p * R + r;
    constexpr int nk = kKVar > R ? kKVar / R : 1, nv = kVVar > R ? kVVar / R : 1;
    if (p < nk) {
      int tr, ch;
      tile_slot_decode<DP, false>(seg * 64 + lane, tr, ch);
      k_src[p] = ch * 16 < D ? (unsigned)(kv_of_lds_row(tr) * k_rs + ch * 16) : kNoSource;
    } else {
      k_src[p] = k_src[p % nk] + (unsigned)((k_row0(seg) - k_row0(p % nk * R + r)) * k_rs);
    }
    if (p < nv) {
      int tr, ch;
      tile_slot_decode<VT ? 64 : DP, !VT>(seg * 64 + lane, tr, ch);
      v_src[p] = VT || ch * 16 < D ? (unsigned)(tr * v_rs + ch * 16) : kNoSource;
      if (VT) v_chunk = ch * 16;
    } else if constexpr (!VT) {
      v_src[p] = v_src[p % nv] + (unsigned)((v_row0(seg) - v_row0(p % nv * R + r)) * v_rs);
    }
  }
  const int kv_last = a.seqlen_k - 1;
  constexpr int kRsrcFlags = 0x00020000;
  // Every step starts its copies, also of blocks that do not exist (through a resource of length 0), so that the number of loads
  // in flight is the same at every step.
  const int k_bytes = kv_last * k_rs + D;
  const int v_bytes = VT ? (D - 1) * v_rs + a.seqlen_k : kv_last * v_rs + D;
  auto issue_k = [&](int j, uint8_t* dst, bool exists, int from, int to) __attribute__((always_inline)) {
    const __amdgpu_buffer_rsrc_t rsrc = __builtin_amdgcn_make_buffer_rsrc((void*)kp, 0, exists ? k_bytes : 0, kRsrcFlags);
    const int base = (int)((unsigned)(exists ? j : 0) * kKvBlock * (unsigned)k_rs);
#pragma unroll
    for (int p = from; p < to; ++p)
      __builtin_amdgcn_raw_ptr_buffer_load_lds(rsrc, LDS_PTR(void, dst + w * kTileBytes + (p * R + r) * 1024), 16, k_src[p], base, 0, 0);
  };
  auto issue_v = [&](int j, uint8_t* dst, bool exists, int from, int to) __attribute__((always_inline)) {
    const __amdgpu_buffer_rsrc_t rsrc = __builtin_amdgcn_make_buffer_rsrc((void*)vp, 0, exists ? v_bytes : 0, kRsrcFlags);
    const int v_base = !exists ? 0 : (int)((unsigned)j * kKvBlock * (unsigned)v_rs);
    // transposed v, ragged last block: chunks past the last key are pulled back onto the last chunk (see fa8_fwd_kernel)
    const unsigned v_from = VT ? v_src[0] + (unsigned)min(exists ? j * kKvBlock : 0, a.seqlen_k - 16 - v_chunk) : 0;
#pragma unroll
    for (int p = from; p < to; ++p) {
      uint8_t* at = dst + w * kTileBytes + (p * R + r) * 1024;
      if constexpr (VT) {
        // Segments are 16 rows apart, in the scalar offset.  A lane is out of range if its offset is not below length - scalar offset,
        // which must not be negative: rows of the tile past the head dim, like blocks that do not exist, take length 0 and scalar offset 0.
        const bool there = exists && (16 * (p * R + R - 1) < D || 16 * (p * R + r) < D);
        const __amdgpu_buffer_rsrc_t rows = __builtin_amdgcn_make_buffer_rsrc((void*)vp, 0, there ? v_bytes : 0, kRsrcFlags);
        __builtin_amdgcn_raw_ptr_buffer_load_lds(rows, LDS_PTR(void, at), 16, v_from, there ? (int)((unsigned)(p * R * 16) * (unsigned)v_rs) : 0, 0, 0);
      } else {
        __builtin_amdgcn_raw_ptr_buffer_load_lds(rsrc, LDS_PTR(void, at), 16, v_src[p], v_base, 0, 0);
      }
    }
  };

  // ---- KV blocks: of this row tile (blocks), of the workgroup (all_blocks), and the leading ones without a mask ----
  const int shift = (a.mode & kSharedBottomRight) ? a.seqlen_k - a.seqlen_q : 0;
  auto blocks_of = [&](int first_row) __attribute__((always_inline)) {  // of the 32-row tile that starts at first_row
    if (!causal) return (a.seqlen_k + kKvBlock - 1) / kKvBlock;
    return max(1, (min(a.seqlen_k, query_of(min(first_row + 31, last_row)) + 1 + shift) + kKvBlock - 1) / kKvBlock);
  };
  const int blocks = blocks_of(row0);
  const int all_blocks = R == 1 ? blocks : blocks_of((tile * R + R - 1) * 32);
  const int n_plain = (causal ? max(0, min(query_of(min(row0, last_row)) + shift, a.seqlen_k)) : a.seqlen_k) / kKvBlock;
  const int rc = min(row, last_row);
  const int qi = query_of(rc);
  const int hd = hk * group + (rc - qi * group);
  const int kv_limit = causal ? min(qi + shift, kv_last) : kv_last;

  // ---- Q fragment ----
  v8i qf[kKSteps];
  {
    const uint8_t* src = a.q + ((unsigned long long)a.q_bs * b + (unsigned long long)a.q_hs * hd + (unsigned long long)a.q_rs * qi) * 16;
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
  issue_k(w, k_lds0, w < all_blocks, 0, kPasses);
  if constexpr (STAGES == 2) issue_k(w + W, k_lds1, w + W < all_blocks, 0, kPasses);
  if constexpr (!APART) issue_v(w, v_lds0, w < all_blocks, 0, kPasses);
  // ---- LDS read offsets (see fa8_fwd_kernel) ----
  int k_off[kKSteps][2];
#pragma unroll
  for (int ks = 0; ks < kKSteps; ++ks)
#pragma unroll
    for (int e = 0; e < 2; ++e) k_off[ks][e] = w * kTileBytes + tile_offset<DP, false>(qn, DP >= 64 ? 4 * ks + 2 * h + e : e);
  constexpr int kSubTileStride = 32 * DP, kVtTileStride = 32 * 64, kTrStride = 8 * DP;
  const int tr_j = (lane & 15) >> 1, tr_e = lane & 1, tr_g1 = (lane >> 4) & 1;
  // (transposed v: the tiles of a wavefront lie W tiles apart, its two offsets serve them all)
  int v_off[VT ? 2 : kOwn];
  if constexpr (VT) {
#pragma unroll
    for (int e = 0; e < 2; ++e) v_off[e] = w * (APART ? kTileBytes : kVtTileStride) + tile_offset<64, false>(qn, 2 * h + e);
  } else {
#pragma unroll
    for (int m = 0; m < kOwn; ++m)
      v_off[m] = (APART ? w * kTileBytes : 0) + tile_offset<DP, true>(32 * h + tr_j, 2 * min((APART ? 0 : w) + m * kStep, kMTiles - 1) + tr_g1) + 8 * tr_e;
  }
  auto load_vf = [&](const uint8_t* v_lds, int i, int m) __attribute__((always_inline)) {
    const uint8_t* vb = v_lds + i * kTileBytes;
    v8i vf;
    if constexpr (VT) {
      const v4i lo = *LDS_PTR(const v4i, vb + m * kStep * kVtTileStride + v_off[0]);
      const v4i hi = *LDS_PTR(const v4i, vb + m * kStep * kVtTileStride + v_off[VT ? 1 : 0]);
      vf = {lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
    } else {
#pragma unroll
      for (int g = 0; g < 4; ++g) {
        const v2i x = __builtin_amdgcn_ds_read_tr8_b64_v2i32(LDS_PTR(v2i, vb + v_off[VT ? 0 : m] + g * kTrStride));
        vf[2 * g] = x[0];
        vf[2 * g + 1] = x[1];
      }
    }
    return vf;
  };

  v16f o_acc[kOwn];
#pragma unroll
  for (int m = 0; m < kOwn; ++m)
#pragma unroll
    for (int i = 0; i < 16; ++i) o_acc[m][i] = 0.f;
  float m_run = kMaxStart, l_run = 0.f;
  auto load_kf = [&](const uint8_t* k_lds, int t, int ks) __attribute__((always_inline)) {
    const v4i lo = *LDS_PTR(const v4i, k_lds + t * kSubTileStride + k_off[ks][0]);
    const v4i hi = *LDS_PTR(const v4i, k_lds + t * kSubTileStride + k_off[ks][1]);
    return v8i{lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
  };
  auto s_product = [&](v16f& acc, int ks, const v8i& kf) __attribute__((always_inline)) {
    if (ks == 0) {
      v16f z;
#pragma unroll
      for (int i = 0; i < 16; ++i) z[i] = 0.f;
      acc = mfma_fp8<E5M2>(kf, qf[ks], z);
    } else {
      acc = mfma_fp8<E5M2>(kf, qf[ks], acc);
    }
  };
  const int groups = (all_blocks + W - 1) / W;

  if constexpr (APART) {
    v16f sbuf[2][2];
    v8i p8;
    float m_own = 0.f;              // running max after this wavefront's block of the group: what its weights are taken against
    float alpha = 1.f, o_alpha = 1.f;  // from m_own of the group before to m_own; of the two groups before, for O
    bool changed = false, o_changed = false;
    // logits of keys that a row does not see, then the row max of a block, with all blocks before the group -> LDS
    auto publish_max = [&](auto parity_c, v16f(&s)[2], int j) __attribute__((always_inline)) {
      constexpr int PH = decltype(parity_c)::value;
      if (j >= n_plain) {
#pragma unroll
        for (int t = 0; t < 2; ++t)
#pragma unroll
          for (int i = 0; i < 16; ++i)
            if (j * kKvBlock + 32 * h + 16 * t + i > kv_limit) s[t][i] = -INFINITY;
      }
      float mx[4];
#pragma unroll
      for (int ch = 0; ch < 4; ++ch) mx[ch] = max3(s[0][4 * ch], s[0][4 * ch + 1], s[0][4 * ch + 2]);
#pragma unroll
      for (int ch = 0; ch < 4; ++ch) mx[ch] = max3(mx[ch], s[0][4 * ch + 3], s[1][4 * ch]);
#pragma unroll
      for (int ch = 0; ch < 4; ++ch) mx[ch] = max3(mx[ch], s[1][4 * ch + 1], s[1][4 * ch + 2]);
      const float bm = lane32_max(max3(max3(mx[0], s[1][3], s[1][7]), max3(mx[1], s[1][11], s[1][15]), max3(mx[2], mx[3], m_run)));
      if (h == 0) max_lds[(PH * R * W + wave) * 32 + qn] = bm;
    };
    float maxima[W];
    auto read_maxima = [&](auto parity_c) __attribute__((always_inline)) {
      constexpr int PH = decltype(parity_c)::value;
#pragma unroll
      for (int i = 0; i < W; ++i) maxima[i] = max_lds[(PH * R * W + r * W + i) * 32 + qn];
    };
    // from the maxima of a group: m_own and m_run after it
    auto follow_max = [&](bool first) __attribute__((always_inline)) {
      float m = m_run, own = m_run;
#pragma unroll
      for (int i = 0; i < W; ++i) {
        m = max2(m, maxima[i]);
        own = i <= w ? m : own;
      }
      o_alpha = alpha;
      o_changed = changed;
      changed = !first && __any(own != m_own);
      alpha = changed ? __builtin_amdgcn_exp2f((m_own - own) * c) : 1.f;
      m_own = own;
      m_run = m;
    };
    auto rescale = [&]() __attribute__((always_inline)) {
      if (o_changed) {
        if (o_alpha != 1.f) {
#pragma unroll
          for (int m = 0; m < kOwn; ++m)
#pragma unroll
            for (int e = 0; e < 16; ++e) o_acc[m][e] *= o_alpha;
        }
      }
    };
    // Waits until all but the latest `copies` tile copies of this wavefront have landed and its LDS operations are done: with one tile a workgroup K and V of
    // a block are the wavefront's own, and its next copy may go where it has just read.
    auto wait = [&](auto copies_c) __attribute__((always_inline)) {
      constexpr int n = decltype(copies_c)::value * kPasses;
      static_assert(n < 64, "vmcnt has six bits");
      __builtin_amdgcn_s_waitcnt(0x0070 | (n & 15) | (n >> 4 << 14));
    };
    auto barrier = [&](auto copies_c) __attribute__((always_inline)) {
      wait(copies_c);
      __builtin_amdgcn_s_barrier();
    };
    constexpr std::integral_constant<int, 0> none{};
    constexpr std::integral_constant<int, 1> one{};
    constexpr std::integral_constant<int, 2> two{};
    constexpr int kS = 2 * kKSteps;
    constexpr int kCut = 6;  // chunks in front of barrier 1 (512 queries on 16384 keys: 5 92.1 us, 6 90.7, 7 94)
    auto iteration = [&](auto first_c, auto parity_c, int g) __attribute__((always_inline)) {
      constexpr int PH = decltype(parity_c)::value;
      constexpr bool kFirst = decltype(first_c)::value;
      v16f(&s)[2] = sbuf[PH];
      v16f(&sn)[2] = sbuf[PH ^ 1];
      uint8_t* const k_next = PH ? k_lds0 : k_lds1;
      uint8_t* const v_this = PH ? v_lds1 : v_lds0;
      uint8_t* const v_prev = PH ? v_lds0 : v_lds1;
      const int j = g * W + w;
      const float mc = m_own * c;
      float sum0, sum1, y[2][4], x[2][4];
      v8i p8_cur;
#pragma unroll
      for (int i = 0; i < 4; ++i) y[0][i] = __builtin_fmaf(s[0][i], c, -mc);
      auto pack = [&](int u) __attribute__((always_inline)) {
        int packed = pack4_fp8<E5M2>(x[u & 1][0], x[u & 1][1], x[u & 1][2], x[u & 1][3]);
        asm volatile("" : "+v"(packed));
        p8_cur[u] = packed;
      };
      auto add = [&](int u, int i) __attribute__((always_inline)) {
        float& sum = i & 1 ? sum1 : sum0;
        sum = (u == 0 && i < 2) ? x[u & 1][i] : sum + x[u & 1][i];
      };
      auto chunk = [&](int u) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          x[u & 1][i] = __builtin_amdgcn_exp2f(y[u & 1][i]);
          if (u < 7) y[(u + 1) & 1][i] = __builtin_fmaf(s[(u + 1) >> 2][4 * ((u + 1) & 3) + i], c, -mc);
          if (u > 0) add(u - 1, i);
          __builtin_amdgcn_sched_barrier(0);
        }
        if (u > 0) {
          pack(u - 1);
          asm volatile("" : "+v"(sum0), "+v"(sum1));
        }
        if (u == 7) {
#pragma unroll
          for (int i = 0; i < 4; ++i) add(7, i);
          pack(7);
        }
        __builtin_amdgcn_sched_barrier(0);
      };
      v8i kfrag[kS], vfrag[kOwn];
      kfrag[0] = load_kf(k_next, 0, 0);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int u = 0; u < kCut; ++u) {
        if (u < 4) {
#pragma unroll
          for (int n = (u * kS + 3) / 4; n < ((u + 1) * kS + 3) / 4; ++n) {
            if (n + 1 < kS) kfrag[n + 1] = load_kf(k_next, (n + 1) / kKSteps, (n + 1) % kKSteps);
            s_product(sn[n / kKSteps], n % kKSteps, kfrag[n]);
          }
          __builtin_amdgcn_sched_barrier(0);
          issue_v(j, v_this, j < all_blocks, u * kPasses / 4, (u + 1) * kPasses / 4);
        }
        chunk(u);
      }
      publish_max(std::integral_constant<int, PH ^ 1>(), sn, j + W);
      barrier(two);  // barrier 1: row maxima of group g + 1; V of group g - 1 has landed; K of group g + 1 has been read
      read_maxima(std::integral_constant<int, PH ^ 1>());
      if constexpr (!kFirst) vfrag[0] = load_vf(v_prev, 0, 0);
      __builtin_amdgcn_sched_barrier(0);
      if constexpr (!kFirst) rescale();
#pragma unroll
      for (int u = kCut; u < 8; ++u) {
        if constexpr (!kFirst) {
          constexpr int kIn = 8 - kCut;
#pragma unroll
          for (int m = (u - kCut) * kOwn / kIn; m < (u - kCut + 1) * kOwn / kIn; ++m) {
            if (m + 1 < kOwn) vfrag[m + 1] = load_vf(v_prev, 0, m + 1);
            o_acc[m] = mfma_fp8<E5M2>(vfrag[m], p8, o_acc[m]);
          }
          __builtin_amdgcn_sched_barrier(0);
        }
        issue_k(j + 3 * W, k_next, j + 3 * W < all_blocks, (u - kCut) * kPasses / (8 - kCut), (u - kCut + 1) * kPasses / (8 - kCut));
        chunk(u);
      }
      l_run = l_run * alpha + (sum0 + sum1);
      p8 = p8_cur;
      follow_max(false);
      // K of group g + 2 has landed; barrier 2 (a tile that two wavefronts read): for both, and V of group g - 1 has been read
      if constexpr (R > 1)
        barrier(two);
      else
        wait(two);
    };
    using T = std::true_type;
    using F = std::false_type;
    constexpr std::integral_constant<int, 0> even{};
    constexpr std::integral_constant<int, 1> odd{};
    // K of group 0 has landed
    if constexpr (R > 1)
      barrier(one);
    else
      wait(one);
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
      for (int ks = 0; ks < kKSteps; ++ks) s_product(sbuf[0][t], ks, load_kf(k_lds0, t, ks));
    publish_max(even, sbuf[0], w);
    barrier(none);
    read_maxima(even);
    issue_k(w + 2 * W, k_lds0, w + 2 * W < all_blocks, 0, kPasses);
    follow_max(true);
    iteration(T(), even, 0);
    int g = 1;
    for (; g + 1 < groups; g += 2) {
      iteration(F(), odd, g);
      iteration(F(), even, g + 1);
    }
    if (g < groups) iteration(F(), odd, g);
    barrier(none);
    // the products of the last group; then m_own is the max over all keys (the group after the last one shows none)
    rescale();
    // (a block behind the tile's last one is one that the workgroup's other tile sees: weights of zero, which an infinity or a NaN in v would turn into NaN)
    if ((groups - 1) * W + w < blocks) {
#pragma unroll
      for (int m = 0; m < kOwn; ++m) o_acc[m] = mfma_fp8<E5M2>(load_vf((groups & 1) ? v_lds0 : v_lds1, 0, m), p8, o_acc[m]);
    }
    o_alpha = alpha;
    o_changed = changed;
    rescale();
    l_run *= alpha;
    // The wavefronts of a tile add up their O and l, in their order: tiles of 4 KB through the LDS of K and V.
    constexpr int kUnits = W * kTileBytes / 4096;
    static_assert(R * W * kMTiles <= 4 * kUnits, "all tiles of O at once");
    auto unit = [&](int u) __attribute__((always_inline)) {
      const int at = u / kUnits;
      uint8_t* const base = at == 0 ? k_lds0 : (at == 1 ? v_lds0 : (at == 2 ? k_lds1 : v_lds1));
      return base + (u - at * kUnits) * 4096 + lane * 16;
    };
    sum_lds[wave * 64 + lane] = l_run;
    barrier(none);  // V has been read
#pragma unroll
    for (int m = 0; m < kMTiles; ++m)
#pragma unroll
      for (int e = 0; e < 4; ++e)
        *LDS_PTR(v4f, unit(wave * kMTiles + m) + e * 1024) = v4f{o_acc[m][4 * e], o_acc[m][4 * e + 1], o_acc[m][4 * e + 2], o_acc[m][4 * e + 3]};
    barrier(none);
#pragma unroll
    for (int m = 0; m < kOut; ++m) {
      if (w + m * W >= kMTiles) break;
#pragma unroll
      for (int i = 0; i < W; ++i)
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const v4f part = *LDS_PTR(const v4f, unit((r * W + i) * kMTiles + w + m * W) + e * 1024);
#pragma unroll
          for (int b2 = 0; b2 < 4; ++b2) o_acc[m][4 * e + b2] = i == 0 ? part[b2] : o_acc[m][4 * e + b2] + part[b2];
        }
    }
    l_run = sum_lds[r * W * 64 + lane];
#pragma unroll
    for (int i = 1; i < W; ++i) l_run += sum_lds[(r * W + i) * 64 + lane];
    if constexpr (R == 2 && D > 32) barrier(none);  // the parts have been read, O's lines may go there
  } else {
    // rescale factors of the group whose PV products are due, and whether any row of the tile needs them
    float alpha[W];
    bool changed[W];
    auto load_pf = [&](int i) __attribute__((always_inline)) {
      const v4i lo = *LDS_PTR(const v4i, p_lds + (r * W + i) * 2048 + lane * 16);
      const v4i hi = *LDS_PTR(const v4i, p_lds + (r * W + i) * 2048 + 1024 + lane * 16);
      return v8i{lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
    };
    // brings O and l to the running max after block i of the group and adds the block's row sums
    auto rescale = [&](int i, float sum) __attribute__((always_inline)) {
  #pragma clang fp contract(off)
      if (changed[i]) {
        l_run = l_run * alpha[i];
        if (alpha[i] != 1.f) {
#pragma unroll
          for (int m = 0; m < kOwn; ++m)
#pragma unroll
            for (int e = 0; e < 16; ++e) o_acc[m][e] *= alpha[i];
        }
      }
      l_run = l_run + sum;
    };
    // Barrier once this wavefront's LDS operations are done and all but its latest `copies` tile copies have landed (vmcnt counts a
    // lane's loads in issue order).  Bare s_barrier: __syncthreads() would wait for all copies.
    auto sync = [&](auto copies_c) __attribute__((always_inline)) {
      constexpr int n = decltype(copies_c)::value * kPasses;
      static_assert(n < 64, "vmcnt has six bits");
      __builtin_amdgcn_s_waitcnt(0x0070 | (n & 15) | (n >> 4 << 14));
      __builtin_amdgcn_s_barrier();
    };
    constexpr std::integral_constant<int, 0> none{};
    constexpr bool kAllOwn = kMTiles % W == 0;  // every wavefront has kOwn tiles of O^T
    auto owns = [&](int m) __attribute__((always_inline)) { return kAllOwn || w + m * W < kMTiles; };
    constexpr int kPv = W * kOwn, kS = 2 * kKSteps;  // matrix instructions of an iteration
    v16f sbuf[2][2];
    v8i p8;

    auto iteration = [&](auto first_c, auto parity_c, int g) __attribute__((always_inline)) {
      constexpr int PH = decltype(parity_c)::value;
      v16f(&s)[2] = sbuf[PH];
      v16f(&sn)[2] = sbuf[PH ^ 1];
      constexpr bool kTwo = STAGES == 2;
      uint8_t* const k_this = kTwo && PH ? k_lds1 : k_lds0;
      uint8_t* const k_next = kTwo && !PH ? k_lds1 : k_lds0;
      uint8_t* const v_prev = kTwo && !PH ? v_lds1 : v_lds0;
      constexpr bool kFirst = decltype(first_c)::value;
      const int j = g * W + w;
      const bool more = (g + 1) * W < all_blocks;  // workgroup-uniform
      if (j >= n_plain) {
#pragma unroll
        for (int t = 0; t < 2; ++t)
#pragma unroll
          for (int i = 0; i < 16; ++i)
            if (j * kKvBlock + 32 * h + 16 * t + i > kv_limit) s[t][i] = -INFINITY;
      }
      float mx[4];
#pragma unroll
      for (int ch = 0; ch < 4; ++ch) mx[ch] = max3(s[0][4 * ch], s[0][4 * ch + 1], s[0][4 * ch + 2]);
#pragma unroll
      for (int ch = 0; ch < 4; ++ch) mx[ch] = max3(mx[ch], s[0][4 * ch + 3], s[1][4 * ch]);
#pragma unroll
      for (int ch = 0; ch < 4; ++ch) mx[ch] = max3(mx[ch], s[1][4 * ch + 1], s[1][4 * ch + 2]);
      const float bm = lane32_max(max3(max3(mx[0], s[1][3], s[1][7]), max3(mx[1], s[1][11], s[1][15]), max3(mx[2], mx[3], m_run)));
      if (h == 0) max_lds[wave * 32 + qn] = bm;
      sync(std::integral_constant<int, kTwo || kFirst ? 1 : 0>());  // barrier 1: row maxima; weights, row sums and V of group g - 1; K of group g + 1; K of group g has been read
      v8i vfrag[kPv], pfrag[W], kfrag[kS];
      float sums[W], maxima[W];
#pragma unroll
      for (int i = 0; i < W; ++i) maxima[i] = max_lds[(r * W + i) * 32 + qn];
      if constexpr (!kFirst) {
        pfrag[0] = load_pf(0);
        if (owns(0)) vfrag[0] = load_vf(v_prev, 0, 0);
#pragma unroll
        for (int i = 0; i < W; ++i) sums[i] = sum_lds[(r * W + i) * 64 + lane];
      }
      float m_after[W], m_own = m_run;
#pragma unroll
      for (int i = 0; i < W; ++i) {
        m_after[i] = max2(i == 0 ? m_run : m_after[i - 1], maxima[i]);
        if (i == w) m_own = m_after[i];
      }
      const float mc = m_own * c;
      float sum0, sum1;
      __builtin_amdgcn_sched_barrier(0);
      // The softmax of 4 weights a chunk, three stages deep so that no instruction waits for the one before it: exponentials of
      // chunk u, their arguments for chunk u + 1, row sum and fp8 packing of chunk u - 1.  The scheduling barriers keep that order.
      float y[2][4], x[2][4];
#pragma unroll
      for (int i = 0; i < 4; ++i) y[0][i] = __builtin_fmaf(s[0][i], c, -mc);
      auto pack = [&](int u) __attribute__((always_inline)) {
        int packed = pack4_fp8<E5M2>(x[u & 1][0], x[u & 1][1], x[u & 1][2], x[u & 1][3]);
        asm volatile("" : "+v"(packed));
        p8[u] = packed;
      };
      auto add = [&](int u, int i) __attribute__((always_inline)) {
        float& sum = i & 1 ? sum1 : sum0;
        sum = (u == 0 && i < 2) ? x[u & 1][i] : sum + x[u & 1][i];
      };
      auto chunk = [&](int u) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          x[u & 1][i] = __builtin_amdgcn_exp2f(y[u & 1][i]);
          if (u < 7) y[(u + 1) & 1][i] = __builtin_fmaf(s[(u + 1) >> 2][4 * ((u + 1) & 3) + i], c, -mc);
          if (u > 0) add(u - 1, i);
          __builtin_amdgcn_sched_barrier(0);
        }
        if (u > 0) {
          pack(u - 1);
          asm volatile("" : "+v"(sum0), "+v"(sum1));  // keeps the additions in their chunk
        }
        if (u == 7) {
#pragma unroll
          for (int i = 0; i < 4; ++i) add(7, i);
          pack(7);
        }
        __builtin_amdgcn_sched_barrier(0);
      };
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        if constexpr (kTwo)
          issue_k(j + 2 * W, k_this, j + 2 * W < all_blocks, u * kPasses / 4, (u + 1) * kPasses / 4);
        else if (u == 0)
          issue_k(j + W, k_this, more && j + W < all_blocks, 0, kPasses);
        chunk(u);
        if constexpr (!kFirst) {
#pragma unroll
          for (int n = u * kPv / 4; n < (u + 1) * kPv / 4; ++n) {
            const int i = n / kOwn, m = n % kOwn;
            if (n + 1 < kPv) {  // operands of the next product
              if ((n + 1) % kOwn == 0) pfrag[(n + 1) / kOwn] = load_pf((n + 1) / kOwn);
              if (owns((n + 1) % kOwn)) vfrag[n + 1] = load_vf(v_prev, (n + 1) / kOwn, (n + 1) % kOwn);
            }
            if (m == 0) rescale(i, sums[i]);
            if (owns(m)) o_acc[m] = mfma_fp8<E5M2>(vfrag[n], pfrag[i], o_acc[m]);
          }
        }
        if (kTwo && u == 3) kfrag[0] = load_kf(k_next, 0, 0);
        __builtin_amdgcn_sched_barrier(0);
      }
#pragma unroll
      for (int i = 0; i < W; ++i) {
        const float before = i == 0 ? m_run : m_after[i - 1];
        changed[i] = __any(m_after[i] != before);
        alpha[i] = changed[i] ? __builtin_amdgcn_exp2f((before - m_after[i]) * c) : 1.f;
      }
      m_run = m_after[W - 1];
      // barrier 2: weights, row sums and V of group g - 1 have been read (LDS operations only; one stage: K of group g + 1 has landed)
      __builtin_amdgcn_s_waitcnt(kTwo ? 0xC07F : 0x0070);
      __builtin_amdgcn_s_barrier();
      if constexpr (!kTwo) {
        if constexpr (!kFirst) issue_v(j, v_prev, j < all_blocks, 0, kPasses);
        kfrag[0] = load_kf(k_next, 0, 0);
      }
#pragma unroll
      for (int u = 4; u < 8; ++u) {
        // (after the last group this is the product of a stale tile: never used)
#pragma unroll
        for (int n = ((u - 4) * kS + 3) / 4; n < ((u - 3) * kS + 3) / 4; ++n) {
          if (n + 1 < kS) kfrag[n + 1] = load_kf(k_next, (n + 1) / kKSteps, (n + 1) % kKSteps);
          s_product(sn[n / kKSteps], n % kKSteps, kfrag[n]);
        }
        __builtin_amdgcn_sched_barrier(0);
        if constexpr (kTwo) issue_v(j + W, v_prev, j + W < all_blocks, (u - 4) * kPasses / 4, (u - 3) * kPasses / 4);
        chunk(u);
        if (u == 4) *LDS_PTR(v4i, p_lds + wave * 2048 + lane * 16) = v4i{p8[0], p8[1], p8[2], p8[3]};
      }
      *LDS_PTR(v4i, p_lds + wave * 2048 + 1024 + lane * 16) = v4i{p8[4], p8[5], p8[6], p8[7]};
      sum_lds[wave * 64 + lane] = sum0 + sum1;
    };

    using T = std::true_type;
    using F = std::false_type;
    constexpr std::integral_constant<int, 0> even{};
    constexpr std::integral_constant<int, 1> odd{};
    sync(std::integral_constant<int, STAGES>());  // K of group 0 landed
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
      for (int ks = 0; ks < kKSteps; ++ks) s_product(sbuf[0][t], ks, load_kf(k_lds0, t, ks));
    iteration(T(), even, 0);
    int g = 1;
    for (; g + 1 < groups; g += 2) {
      iteration(F(), odd, g);
      iteration(F(), even, g + 1);
    }
    if (g < groups) iteration(F(), odd, g);
    sync(none);
    // the PV products of the last group
#pragma unroll
    for (int i = 0; i < W; ++i) {
      if ((groups - 1) * W + i < blocks) {
        rescale(i, sum_lds[(r * W + i) * 64 + lane]);
        const v8i pf = load_pf(i);
#pragma unroll
        for (int m = 0; m < kOwn; ++m)
          if (owns(m)) o_acc[m] = mfma_fp8<E5M2>(load_vf(STAGES == 1 || (groups & 1) ? v_lds0 : v_lds1, i, m), pf, o_acc[m]);
      }
    }
  }

  // ---- epilogue (see fa8_fwd_kernel) ----
  // Two tiles a workgroup: where many rows leave together (whole_lines) the rows of a tile meet in LDS, in the first K stage, and leave as whole lines.
  // One tile: there are fewer rows to write, and another barrier costs as much as it saves or more (16 heads, 1024 keys, head dim 64, causal
  // 7.73 -> 8.00 us).  us, pieces -> lines: 32 heads, 1000 keys, head dim 128, causal 15.5 -> 14.9; 16 heads, 2048 keys, head dim 256, causal 39.8 ->
  // 38.5; 512 queries on 4096 keys, 32 heads on 8 k/v heads 28.7 -> 28.1.
  const float l_tot = lane32_sum(l_run);
  const float inv = (l_tot == 0.f || l_tot != l_tot) ? 1.f : 1.f / l_tot;
  if (a.lse != nullptr && h == 0 && w == 0 && row <= last_row) {
    const float lse = l_tot > 0.f ? (m_run * c + __builtin_amdgcn_logf(l_tot)) * 0.6931471805599453f : (l_tot == 0.f ? -INFINITY : l_tot);
    a.lse[(unsigned long long)a.lse_bs * b + (unsigned long long)a.lse_hs * hd + qi] = lse;
  }
  // a lane's piece a2 of its m-th O^T tile, 4 columns in the output type
  auto piece = [&](auto elem_c, int m, int a2) __attribute__((always_inline)) {
    if constexpr (decltype(elem_c)::value == 2) {
      v4h x;
#pragma unroll
      for (int b2 = 0; b2 < 4; ++b2) x[b2] = (_Float16)(o_acc[m][4 * a2 + b2] * inv);
      return x;
    } else {
      constexpr float kMaxFinite = E5M2 ? 57344.f : 448.f;
      float x[4];
#pragma unroll
      for (int b2 = 0; b2 < 4; ++b2) {
        const float y = o_acc[m][4 * a2 + b2] * inv;
        x[b2] = (y != y) ? y : fminf(fmaxf(y, -kMaxFinite), kMaxFinite);
      }
      return pack4_fp8<E5M2>(x[0], x[1], x[2], x[3]);
    }
  };
  constexpr std::integral_constant<int, 1> fp8{};
  constexpr std::integral_constant<int, 2> fp16{};
  const bool fp8_out = !APART && (a.mode & kSharedFp8Out);  // (keep_sums_apart takes fp16 outputs only)
  constexpr bool kLines16 = R == 2 && D > 32, kLines8 = R == 2 && !APART && D % 64 == 0 && D >= 128;
  if (__builtin_expect(!kLines16 || !(a.mode & kSharedLines), D != 192 && D != 256)) {  // (what most calls take follows in line)
    if (row > last_row) return;
    const unsigned long long o_at = ((unsigned long long)a.o_bs * b + (unsigned long long)a.o_hs * hd + (unsigned long long)a.o_rs * qi) * 4 + 4 * h;
#pragma unroll
    for (int m = 0; m < kOut; ++m) {
      const int mt = w + m * W;
      if (kMTiles % W != 0 && mt >= kMTiles) break;
      if (!fp8_out) {
#pragma unroll
        for (int a2 = 0; a2 < 4; ++a2) *(v4h*)((_Float16*)a.o + o_at + 32 * mt + 8 * a2) = piece(fp16, m, a2);
      } else {
#pragma unroll
        for (int a2 = 0; a2 < 4; ++a2) *(int*)((uint8_t*)a.o + o_at + 32 * mt + 8 * a2) = piece(fp8, m, a2);
      }
    }
    return;
  }
  auto lines = [&](auto elem_c) __attribute__((always_inline)) {
    static_assert(R <= W, "the rows of the workgroup fit in one K stage");
    constexpr int kElem = decltype(elem_c)::value, kChunks = D * kElem / 16;  // 16-byte chunks of a row
    using Piece = decltype(piece(elem_c, 0, 0));
    // (the lane's number taken anew; kept over the loop for these addresses it cost head dim 64 the fourth workgroup of a compute unit)
    const int lane_o = (int)__builtin_amdgcn_mbcnt_hi(~0u, __builtin_amdgcn_mbcnt_lo(~0u, 0u)), row_o = lane_o & 31, half_o = lane_o >> 5;
    uint8_t* const tile_lds = k_lds0 + r * 32 * D * kElem;
    auto chunk_at = [](int rr, int ch) __attribute__((always_inline)) {  // neighbouring rows start in different banks
      const int key = kChunks % 8 == 0 ? rr & 7 : (kChunks % 4 == 0 ? (rr >> 1) & 3 : (rr >> 2) & 1);
      return rr * D * kElem + ((ch ^ key) << 4);
    };
#pragma unroll
    for (int m = 0; m < kOut; ++m) {
      const int mt = w + m * W;
      if (kMTiles % W != 0 && mt >= kMTiles) break;
#pragma unroll
      for (int a2 = 0; a2 < 4; ++a2) {
        const int ch = 2 * kElem * mt + (kElem == 2 ? a2 : a2 >> 1), byte = kElem == 2 ? 8 * half_o : 8 * (a2 & 1) + 4 * half_o;
        *LDS_PTR(Piece, tile_lds + chunk_at(row_o, ch) + byte) = piece(elem_c, m, a2);
      }
    }
    __builtin_amdgcn_s_waitcnt(0xC07F);
    __builtin_amdgcn_s_barrier();
#pragma unroll
    for (int p = 0; p * 64 * W < 32 * kChunks; ++p) {
      const int unit = (p * W + w) * 64 + lane_o, rr = unit / kChunks, ch = unit - rr * kChunks;
      if (unit < 32 * kChunks && row0 + rr <= last_row) {
        const v4i x = *LDS_PTR(const v4i, tile_lds + chunk_at(rr, ch));
        const int q_of = query_of(row0 + rr), head = hk * group + (row0 + rr - q_of * group);
        const unsigned long long at = ((unsigned long long)a.o_bs * b + (unsigned long long)a.o_hs * head + (unsigned long long)a.o_rs * q_of) * 4 * kElem;
        store_row_chunk((uint8_t*)a.o + at + 16 * ch, x);
      }
    }
  };
  if constexpr (kLines8)
    if (fp8_out) return lines(fp8);
  if constexpr (kLines16) lines(fp16);
#endif
}

}  // namespace fa8
#endif  // FA8_SHARED_ROWS_H_
