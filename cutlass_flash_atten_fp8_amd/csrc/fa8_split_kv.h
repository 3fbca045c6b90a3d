// Attention for few query rows over many keys (decode steps, short chunks): the keys of a k/v head are dealt to `splits` workgroups of
// four wavefronts, every wavefront walking its own contiguous range of KV blocks without meeting the others.
//
// The fp8 weights are taken against the running row max over ALL keys before them (that is what the other kernels do, and it decides how a
// weight is rounded), so a range cannot start before the row max of the ranges in front of it is known.  Two passes:
//   logits  reads K, writes S (fp32, masked, live rows only) and the row max of every range
//   values  starts from the max over the ranges before its own, reads S and V, writes O, l and the max of its range; the workgroup
//           that ends last for a row tile adds the ranges up (factors exp2((m_range - m_last) * c) <= 1: the maxima only grow)
// Both are one kernel where the logits of a range fit in LDS (fa8_split_fused_kernel): the workgroups exchange their maxima through the
// workspace while their first tiles of V are on the way, S never goes through memory and one launch, its start and its first accesses
// are saved.  A workgroup waits for those before it in the grid, which start earlier or at the same time; if another stream keeps them off
// the chip it stops waiting after a number of looks and forms the maxima that have not come itself.  Where the logits do not fit, one kernel each.
// Logits, weights and products are those of the other kernels bit for bit; only the order of the fp32 sums over the ranges is another.
//
// Bound: HBM bytes.  K and V are read once; in two kernels S costs 8 bytes per row and key against 2 * head_dim bytes per key for K and V,
// which is why the logits are kept instead of read K again (head dim 128: fewer bytes up to 16 rows a tile, and S comes out of the Infinity
// Cache).  Every wavefront has its own LDS ring, so there is no barrier in either loop.  The rest is latency: a launch and a first memory
// access (kernel arguments and data, 2 us), both twice in two kernels, the exchange of the maxima in one, and the parts' way to the last
// workgroup (stores, a counter, loads: 3 us, with all loads of a step under way together; one by one they took 8).  Measured among other
// calls, inputs rotating, 1 query of 32 heads on 8 k/v heads, head dim 128: 32768 keys 309 us (one wavefront a head) / 151 (shared rows, no
// split) / 20.7 (two kernels, of that 8 logits and 12 values) -> 17.9 us (13 us at the rate of a plain copy).  In a loop of single calls: 4
// sequences of 32768 keys 71.3 (two kernels) -> 55.4, of 4096 keys 23 (shared rows) / 15.9 -> 13.9; 4 queries, 16384 keys 22.7 -> 18.1; 2
// sequences of 60000 keys, 8 k/v heads, head dim 64: 39.8 -> 29.5.
#ifndef FA8_SPLIT_KV_H_
#define FA8_SPLIT_KV_H_
#include <type_traits>

#include "fa8_device.h"

namespace fa8 {

typedef unsigned v4u __attribute__((ext_vector_type(4)));

constexpr int kSplitWaves = 4;  // wavefronts (key ranges) per workgroup
constexpr int kSplitMax = 32;   // most splits of a row tile
// Most looks that a thread takes at the maxima of the workgroups before its own until they have all come, 0.17 us each: 45 us, about what
// forming a few of them from K takes (1 us a block of a wavefront's range; 32768 keys of 8 k/v heads, head dim 128, one late part: 70 us in all, every
// part late: 182; with 2048 looks at each and all K before the workgroup read for a single late one: 470 and 452).
constexpr int kSplitLooks = 256;

// The workspace: arrays one after the other, each of the size of all row tiles together (tile index = (batch * k/v heads + head) * tiles
// + tile).  Offsets in bytes, all multiples of 256.
struct SplitWorkspace {
  long long done;       // [1] unsigned: workgroups that have written their part
  long long range_max;  // [splits * kSplitWaves][32]
  long long split_max;  // [splits][32]
  long long part_m;     // [splits][32]
  long long part_l;     // [splits][32]
  long long part_o;     // [splits][live rows][head_dim]
  long long s;          // [live rows][keys]: masked logits of the keys that some query sees, whole KV blocks
  long long keys;
  long long bytes;
};
// Keys that some query sees: a mask aligned with the first key hides those past the last query.
__host__ __device__ inline int split_visible_keys(int seqlen_q, int seqlen_k, bool causal, bool bottom_right) {
  return causal && !bottom_right && seqlen_q < seqlen_k ? seqlen_q : seqlen_k;
}
__host__ __device__ inline SplitWorkspace split_layout(long long all_tiles, int splits, int live_rows, int head_dim, int visible_keys) {
  auto up = [](long long x) { return (x + 255) / 256 * 256; };
  const long long keys = ((long long)visible_keys + kKvBlock - 1) / kKvBlock * kKvBlock, rows32 = all_tiles * splits * 128;
  SplitWorkspace w;
  w.keys = keys;
  w.done = 0;
  w.range_max = up(all_tiles * 4);
  w.split_max = w.range_max + rows32 * kSplitWaves;
  w.part_m = w.split_max + up(rows32);
  w.part_l = w.part_m + up(rows32);
  w.part_o = w.part_l + up(rows32);
  w.s = w.part_o + up(all_tiles * splits * live_rows * head_dim * 4);
  w.bytes = w.s + all_tiles * live_rows * keys * 4;
  return w;
}

// Two argument blocks of at most 112 bytes (see SharedArgs for the limit, the units of the strides and `mode`).
struct SplitShape {
  uint8_t* workspace;
  float scale_log2;
  int seqlen_q, seqlen_k;
  unsigned mode;
  uint16_t splits, blocks_per_range;  // workgroups per row tile, KV blocks per wavefront
  int heads_k, all_tiles;             // (gridDim would have to be loaded from elsewhere)
};
struct SplitLogitsArgs {
  SplitShape n;
  const uint8_t* q;
  const uint8_t* k;
  unsigned q_bs, q_hs, q_rs;
  unsigned k_bs, k_hs, k_rs;
};
struct SplitValuesArgs {
  SplitShape n;
  const uint8_t* v;
  void* o;
  float* lse;
  unsigned v_bs, v_hs, v_rs;
  unsigned o_bs, o_hs, o_rs;
  unsigned lse_bs, lse_hs;
};
static_assert(sizeof(SplitLogitsArgs) <= 112 && sizeof(SplitValuesArgs) <= 112, "see above");

// What both passes know about a workgroup: grid = k/v heads x batches x (tiles * splits)
struct SplitPlace {
  int hk, b, tile, split, splits;
  long long at;  // row tile index into the workspace
  int wave, lane, qn, h;
  int group, group_shift, shift, live_rows;
  bool causal;
  int row, last_row, qi, hd;  // query row of the lane (clamped), its query and q head
  int first, count;           // KV blocks of this wavefront
  SplitWorkspace ws;
  __device__ __forceinline__ int query_of(int x) const { return group_shift < 31 ? x >> group_shift : x / group; }
};

__device__ __forceinline__ SplitPlace split_place(const SplitShape& n, int head_dim) {
  SplitPlace p;
  p.group = (int)(n.mode >> kSharedGroup);
  p.group_shift = (int)(n.mode >> kSharedShift) & 31;
  p.causal = n.mode & kSharedCausal;
  p.shift = (n.mode & kSharedBottomRight) ? n.seqlen_k - n.seqlen_q : 0;
  p.hk = blockIdx.x;
  p.b = blockIdx.y;
  p.splits = n.splits;
  const int rows = p.group * n.seqlen_q, tiles = (rows + 31) >> 5;
  p.live_rows = min(rows, 32);
  p.last_row = rows - 1;
  p.tile = tiles == 1 ? 0 : (int)blockIdx.z / p.splits;
  p.split = (int)blockIdx.z - p.tile * p.splits;
  p.at = ((long long)p.b * n.heads_k + p.hk) * tiles + p.tile;
  p.ws = split_layout(n.all_tiles, p.splits, p.live_rows, head_dim,
                      split_visible_keys(n.seqlen_q, n.seqlen_k, p.causal, n.mode & kSharedBottomRight));
  p.lane = threadIdx.x & 63;
  p.wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  p.qn = p.lane & 31;
  p.h = p.lane >> 5;
  p.row = p.tile * 32 + p.qn;
  const int rc = min(p.row, p.last_row);
  p.qi = p.query_of(rc);
  p.hd = p.hk * p.group + rc - p.qi * p.group;
  // blocks that some row of the tile sees
  const int q_last = p.query_of(min(p.tile * 32 + 31, p.last_row));
  const int blocks = p.causal ? max(1, (min(n.seqlen_k, q_last + 1 + p.shift) + kKvBlock - 1) / kKvBlock) : (n.seqlen_k + kKvBlock - 1) / kKvBlock;
  p.first = (p.split * kSplitWaves + p.wave) * n.blocks_per_range;
  p.count = max(0, min((int)n.blocks_per_range, blocks - p.first));
  return p;
}

// Waits until at most N vector memory operations of the wavefront are under way (s_waitcnt immediate, gfx9 layout).
template <int N>
__device__ __forceinline__ void wait_loads() {
  static_assert(N < 64, "vmcnt has six bits");
  __builtin_amdgcn_s_waitcnt(0x0F70 | (N & 15) | (N >> 4 << 14));
}

// ---- pass 1: S and the row max of every range ----
template <int D, bool E5M2>
__global__ __launch_bounds__(64 * kSplitWaves) __attribute__((amdgpu_waves_per_eu(2))) void fa8_split_logits_kernel(const SplitLogitsArgs a) {
#if defined(__HIP_DEVICE_COMPILE__)
  constexpr int DP = D <= 32 ? 32 : (D <= 64 ? 64 : (D <= 128 ? 128 : 256));
  constexpr int kTileBytes = kKvBlock * DP, kPasses = kTileBytes / 1024, kKSteps = (D + 63) / 64;
  __shared__ __attribute__((aligned(1024))) uint8_t lds0[kSplitWaves * kTileBytes];
  __shared__ __attribute__((aligned(1024))) uint8_t lds1[kSplitWaves * kTileBytes];
  __shared__ float max_lds[kSplitWaves * 32];
  const SplitPlace p = split_place(a.n, D);
  const int qn = p.qn, h = p.h, lane = p.lane;
  const uint8_t* kp = a.k + ((unsigned long long)a.k_bs * p.b + (unsigned long long)a.k_hs * p.hk) * 16;
  const int k_rs = (int)a.k_rs * 16, seqlen_k = a.n.seqlen_k;
  constexpr unsigned kNoSource = 0x80000000u;
  unsigned src[kPasses];
#pragma unroll
  for (int i = 0; i < kPasses; ++i) {
    int r, ch;
    tile_slot_decode<DP, false>(i * 64 + lane, r, ch);
    src[i] = ch * 16 < D ? (unsigned)(kv_of_lds_row(r) * k_rs + ch * 16) : kNoSource;
  }
  const __amdgpu_buffer_rsrc_t rsrc =
      __builtin_amdgcn_make_buffer_rsrc((void*)kp, 0, (seqlen_k - 1) * k_rs + D, 0x00020000);
  auto issue = [&](int j, uint8_t* dst) __attribute__((always_inline)) {
    const int base = (int)((unsigned)j * kKvBlock * (unsigned)k_rs);
#pragma unroll
    for (int i = 0; i < kPasses; ++i)
      __builtin_amdgcn_raw_ptr_buffer_load_lds(rsrc, LDS_PTR(void, dst + p.wave * kTileBytes + i * 1024), 16, src[i], base, 0, 0);
  };
  v8i qf[kKSteps];
  {
    const uint8_t* q8 = a.q + ((unsigned long long)a.q_bs * p.b + (unsigned long long)a.q_hs * p.hd + (unsigned long long)a.q_rs * p.qi) * 16;
#pragma unroll
    for (int ks = 0; ks < kKSteps; ++ks) {
      const bool upper_exists = 64 * ks + 32 < D;
      const uint8_t* s8 = q8 + 64 * ks + (upper_exists ? 32 * h : 0);
      const v4i lo = *(const v4i*)(s8);
      const v4i hi = *(const v4i*)(s8 + 16);
      qf[ks] = {lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
      if (!upper_exists && h) qf[ks] = v8i{0, 0, 0, 0, 0, 0, 0, 0};
    }
  }
  // (the ranges of a tile are added up by the workgroup that counts itself last: the count starts at 0)
  if (p.split == 0 && threadIdx.x == 0) ((unsigned*)(a.n.workspace + p.ws.done))[p.at] = 0;
  if (p.count > 0) issue(p.first, lds0);
  if (p.count > 1) issue(p.first + 1, lds1);
  int k_off[kKSteps][2];
#pragma unroll
  for (int ks = 0; ks < kKSteps; ++ks)
#pragma unroll
    for (int e = 0; e < 2; ++e) k_off[ks][e] = p.wave * kTileBytes + tile_offset<DP, false>(qn, DP >= 64 ? 4 * ks + 2 * h + e : e);
  const int kv_last = seqlen_k - 1;
  const int kv_limit = p.causal ? min(p.qi + p.shift, kv_last) : kv_last;
  // leading blocks without a masked logit in any row of the tile
  const int q_first = p.query_of(min(p.tile * 32, p.last_row));
  const int n_plain = (p.causal ? max(0, min(q_first + p.shift, seqlen_k)) : seqlen_k) / kKvBlock;
  float* s_out = (float*)(a.n.workspace + p.ws.s) + (p.at * p.live_rows + qn) * p.ws.keys + 32 * h;
  const bool live = qn < p.live_rows && p.row <= p.last_row;  // (lane 0 always is: the stores below are never skipped)
  float m_run = -1.0e30f;
  // Block i of the range: S, then the copy of block i + 2 into the tile just read, then max and stores.  vmcnt counts loads and stores in
  // issue order; what is issued after the copy of block i and may still be under way when its S is formed: the stores of block i - 2
  // (not counted below, they are old by then), the copy of block i + 1 and the stores of block i - 1.  That is what the odd blocks wait
  // for; in front of the even ones' reads the compiler, which does not see that no copy under way writes lds0, waits for everything.
  constexpr int kStores = 8;
  auto block = [&](int i, uint8_t* tile) __attribute__((always_inline)) {
    const int j = p.first + i;
    if (i + 1 < p.count) {
      if (i == 0)
        wait_loads<kPasses>();
      else
        wait_loads<kPasses + kStores>();
    } else {
      if (i == 0)
        wait_loads<0>();
      else
        wait_loads<kStores>();
    }
    v16f s[2];
#pragma unroll
    for (int t = 0; t < 2; ++t) {
#pragma unroll
      for (int e = 0; e < 16; ++e) s[t][e] = 0.f;
#pragma unroll
      for (int ks = 0; ks < kKSteps; ++ks) {
        const v4i lo = *LDS_PTR(const v4i, tile + t * 32 * DP + k_off[ks][0]);
        const v4i hi = *LDS_PTR(const v4i, tile + t * 32 * DP + k_off[ks][1]);
        s[t] = mfma_fp8<E5M2>(v8i{lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]}, qf[ks], s[t]);
      }
    }
    __builtin_amdgcn_sched_barrier(0);
    __builtin_amdgcn_s_waitcnt(0xC07F);  // the tile has been read
    if (i + 2 < p.count) issue(j + 2, tile);
    __builtin_amdgcn_sched_barrier(0);
    if (j >= n_plain) {
#pragma unroll
      for (int t = 0; t < 2; ++t)
#pragma unroll
        for (int e = 0; e < 16; ++e)
          if (j * kKvBlock + 32 * h + 16 * t + e > kv_limit) s[t][e] = -INFINITY;
    }
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
      for (int e = 0; e < 16; e += 2) m_run = max3(s[t][e], s[t][e + 1], m_run);
    if (live) {
#pragma unroll
      for (int t = 0; t < 2; ++t)
#pragma unroll
        for (int e = 0; e < 16; e += 4) *(v4f*)(s_out + (long long)j * kKvBlock + 16 * t + e) = v4f{s[t][e], s[t][e + 1], s[t][e + 2], s[t][e + 3]};
    }
    __builtin_amdgcn_sched_barrier(0);
  };
  for (int i = 0; i < p.count; i += 2) {
    block(i, lds0);
    if (i + 1 < p.count) block(i + 1, lds1);
  }
  m_run = lane32_max(m_run);
  if (h == 0) {
    ((float*)(a.n.workspace + p.ws.range_max))[((p.at * p.splits + p.split) * kSplitWaves + p.wave) * 32 + qn] = m_run;
    max_lds[p.wave * 32 + qn] = m_run;
  }
  __syncthreads();
  if (threadIdx.x < 32) {
    float m = max_lds[threadIdx.x];
#pragma unroll
    for (int x = 1; x < kSplitWaves; ++x) m = __builtin_fmaxf(m, max_lds[x * 32 + threadIdx.x]);
    ((float*)(a.n.workspace + p.ws.split_max))[(p.at * p.splits + p.split) * 32 + threadIdx.x] = m;
  }
#endif
}

// The weights of a KV block (s: its logits) against the running max, and the block's part of O; load_vf(mt) gives a fragment of V^T.
template <bool E5M2, int MTILES, typename LoadVf>
__device__ __forceinline__ void split_weights_and_o(const v4f (&s)[8], float c, float& m_run, float& l_run, v16f (&o_acc)[MTILES], LoadVf&& load_vf) {
  float m = m_run;
#pragma unroll
  for (int i = 0; i < 8; ++i) m = max3(max3(s[i][0], s[i][1], m), s[i][2], s[i][3]);
  const float m_new = lane32_max(m);
  if (__any(m_new != m_run)) {
    const float alpha = __builtin_amdgcn_exp2f((m_run - m_new) * c);
    l_run *= alpha;
#pragma unroll
    for (int mt = 0; mt < MTILES; ++mt)
#pragma unroll
      for (int i = 0; i < 16; ++i) o_acc[mt][i] *= alpha;
    m_run = m_new;
  }
  const float mc = m_new * c;
  float sum0 = 0.f, sum1 = 0.f;
  v8i p8;
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    float x[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) x[e] = __builtin_amdgcn_exp2f(__builtin_fmaf(s[i][e], c, -mc));
    sum0 = sum0 + x[0] + x[2];
    sum1 = sum1 + x[1] + x[3];
    p8[i] = pack4_fp8<E5M2>(x[0], x[1], x[2], x[3]);
  }
  l_run += sum0 + sum1;
#pragma unroll
  for (int mt = 0; mt < MTILES; ++mt) o_acc[mt] = mfma_fp8<E5M2>(load_vf(mt), p8, o_acc[mt]);
}

// ---- end of pass 2: the ranges of a workgroup are added up, then, by the workgroup that ends last, those of all ----
// count_done is called by the first wavefront once its part can be seen by all; lane 0 says whether the others' can be seen too.
// True in the workgroup that wrote the output.
template <int D, bool E5M2, typename Args, typename CountDone>
__device__ __forceinline__ bool split_merge(const Args& a, const SplitPlace& p, const v16f (&o_acc)[D / 32], float m_run, float l_run, uint8_t* lds0,
                                            uint8_t* lds1, float* m_lds, float* l_lds, int* last_lds, CountDone&& count_done) {
  constexpr int kMTiles = D / 32;
  const int qn = p.qn, h = p.h;
  const float c = a.n.scale_log2;
  // ---- the four ranges of the workgroup meet in LDS ----
  if (h == 0) m_lds[p.wave * 32 + qn] = m_run;
  const float l_wave = lane32_sum(l_run);
  __syncthreads();
  const float m_wg = m_lds[(kSplitWaves - 1) * 32 + qn];  // the last range's max is the largest
  const float f = __builtin_amdgcn_exp2f((m_run - m_wg) * c);
  if (h == 0) l_lds[p.wave * 32 + qn] = l_wave * f;
  // [range % 2][row][columns in fours, their number ^ row % 8] in the ring buffer of range / 2: few bank conflicts, no padding
  constexpr int kFours = D / 4;
  auto at4 = [](int row, int four) __attribute__((always_inline)) { return row * kFours + (four ^ (row & 7)); };
  {
    v4f* o_lds = (v4f*)(p.wave < 2 ? lds0 : lds1) + (p.wave & 1) * 32 * kFours;
    if (qn < p.live_rows) {
#pragma unroll
      for (int mt = 0; mt < kMTiles; ++mt)
#pragma unroll
        for (int e = 0; e < 16; e += 4)
          o_lds[at4(qn, 8 * mt + (e >> 1) + h)] = v4f{o_acc[mt][e] * f, o_acc[mt][e + 1] * f, o_acc[mt][e + 2] * f, o_acc[mt][e + 3] * f};
    }
  }
  __syncthreads();
  // ---- this workgroup's part goes out.  The workgroups of a tile sit on different XCDs: stores and loads of the parts carry agent
  // scope (sc1), which passes the XCDs' own L2 caches by ----
  constexpr int kAgent = 16;  // cache policy of the buffer instructions: sc1
  const long long parts = p.at * p.splits;
  const int n = p.live_rows, tid = threadIdx.x, fours = n * kFours;  // of a part
  const int last_bytes = p.splits * 128;
  const __amdgpu_buffer_rsrc_t m_rsrc = __builtin_amdgcn_make_buffer_rsrc(a.n.workspace + p.ws.part_m + parts * 128, 0, last_bytes, 0x00020000);
  const __amdgpu_buffer_rsrc_t l_rsrc = __builtin_amdgcn_make_buffer_rsrc(a.n.workspace + p.ws.part_l + parts * 128, 0, last_bytes, 0x00020000);
  const __amdgpu_buffer_rsrc_t o_rsrc =
      __builtin_amdgcn_make_buffer_rsrc(a.n.workspace + p.ws.part_o + parts * fours * 16, 0, p.splits * fours * 16, 0x00020000);
  for (int x = tid; x < fours; x += 64 * kSplitWaves) {
    const int at = at4(x / kFours, x % kFours);
    const v4f y = (((const v4f*)lds0)[at] + ((const v4f*)lds0)[32 * kFours + at]) + (((const v4f*)lds1)[at] + ((const v4f*)lds1)[32 * kFours + at]);
    __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(v4u, y), o_rsrc, x * 16, p.split * fours * 16, kAgent);
  }
  if (tid < 32) {
    float l = 0.f;
#pragma unroll
    for (int x = 0; x < kSplitWaves; ++x) l += l_lds[x * 32 + tid];
    __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(l), l_rsrc, tid * 4, p.split * 128, kAgent);
    __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(m_lds[(kSplitWaves - 1) * 32 + tid]), m_rsrc, tid * 4, p.split * 128, kAgent);
  }
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // the stores have reached the point where all XCDs see them
  __syncthreads();
  if (tid < 64) {
    const bool last = count_done();
    if (tid == 0) *last_lds = last;
  }
  __syncthreads();
  if (!*last_lds) return false;
  // ---- the last workgroup of the tile adds the parts up ----
  float* factor = (float*)lds0;                 // [split][32]
  float* sums = (float*)lds0 + kSplitMax * 32;  // [split][32]
  {
    constexpr int kEach = kSplitMax * 32 / (64 * kSplitWaves);
    const float m_all = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(m_rsrc, (tid & 31) * 4, (p.splits - 1) * 128, kAgent));  // the largest
    float m[kEach], l[kEach];
#pragma unroll
    for (int e = 0; e < kEach; ++e) {  // (past the last split: 0)
      m[e] = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(m_rsrc, (e * 64 * kSplitWaves + tid) * 4, 0, kAgent));
      l[e] = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(l_rsrc, (e * 64 * kSplitWaves + tid) * 4, 0, kAgent));
    }
#pragma unroll
    for (int e = 0; e < kEach; ++e) {
      const bool exists = e * 64 * kSplitWaves + tid < p.splits * 32;
      factor[e * 64 * kSplitWaves + tid] = exists ? __builtin_amdgcn_exp2f((m[e] - m_all) * c) : 0.f;
      sums[e * 64 * kSplitWaves + tid] = l[e];
    }
  }
  __syncthreads();
  for (int x = tid; x < fours; x += 64 * kSplitWaves) {
    const int row_in = x / kFours, col = (x % kFours) * 4, out_row = p.tile * 32 + row_in;
    v4f y[kSplitMax];  // all parts under way together; past the last split: 0
#pragma unroll
    for (int e = 0; e < kSplitMax; ++e)
      y[e] = __builtin_bit_cast(v4f, __builtin_amdgcn_raw_buffer_load_b128(o_rsrc, x * 16, e * fours * 16, kAgent));
    v4f acc = {0.f, 0.f, 0.f, 0.f};
    float l_all = 0.f;
#pragma unroll
    for (int e = 0; e < kSplitMax; ++e) {
      const float g = factor[e * 32 + row_in];
      l_all = __builtin_fmaf(sums[e * 32 + row_in], g, l_all);
#pragma unroll
      for (int z = 0; z < 4; ++z) acc[z] = __builtin_fmaf(y[e][z], g, acc[z]);
    }
    if (out_row > p.last_row) continue;
    const int q_out = p.query_of(out_row), hd_out = p.hk * p.group + out_row - q_out * p.group;
    const float inv = (l_all == 0.f || l_all != l_all) ? 1.f : 1.f / l_all;
    if (a.lse != nullptr && col == 0) {
      const float m_row = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(m_rsrc, row_in * 4, (p.splits - 1) * 128, kAgent));
      a.lse[(unsigned long long)a.lse_bs * p.b + (unsigned long long)a.lse_hs * hd_out + q_out] =
          l_all > 0.f ? (m_row * c + __builtin_amdgcn_logf(l_all)) * 0.6931471805599453f : (l_all == 0.f ? -INFINITY : l_all);
    }
    const unsigned long long o_at =
        ((unsigned long long)a.o_bs * p.b + (unsigned long long)a.o_hs * hd_out + (unsigned long long)a.o_rs * q_out) * 4 + col;
    if (!(a.n.mode & kSharedFp8Out)) {
      v4h w;
#pragma unroll
      for (int z = 0; z < 4; ++z) w[z] = (_Float16)(acc[z] * inv);
      *(v4h*)((_Float16*)a.o + o_at) = w;
    } else {
      constexpr float kMaxFinite = E5M2 ? 57344.f : 448.f;
      float w[4];
#pragma unroll
      for (int z = 0; z < 4; ++z) {
        const float v = acc[z] * inv;
        w[z] = (v != v) ? v : fminf(fmaxf(v, -kMaxFinite), kMaxFinite);
      }
      *(int*)((uint8_t*)a.o + o_at) = pack4_fp8<E5M2>(w[0], w[1], w[2], w[3]);
    }
  }
  return true;
}

// ---- pass 2: weights and O of every range, and their sum ----
template <int D, bool E5M2, bool VT>
__global__ __launch_bounds__(64 * kSplitWaves) __attribute__((amdgpu_waves_per_eu(D > 128 ? 1 : 2))) void fa8_split_values_kernel(
    const SplitValuesArgs a) {
#if defined(__HIP_DEVICE_COMPILE__)
  constexpr int DP = D <= 32 ? 32 : (D <= 64 ? 64 : (D <= 128 ? 128 : 256));
  constexpr int kTileBytes = kKvBlock * DP, kPasses = kTileBytes / 1024, kMTiles = D / 32;
  // (after the loop each ring buffer holds O of two ranges, later the first one the rescale factors and row sums of all splits)
  constexpr int kRing = kSplitWaves * kTileBytes > kSplitMax * 256 ? kSplitWaves * kTileBytes : kSplitMax * 256;
  static_assert(kSplitWaves * kTileBytes >= 2 * D * 32 * 4, "O of two ranges fits");
  __shared__ __attribute__((aligned(1024))) uint8_t lds0[kRing];
  __shared__ __attribute__((aligned(1024))) uint8_t lds1[kSplitWaves * kTileBytes];
  __shared__ float m_lds[kSplitWaves * 32], l_lds[kSplitWaves * 32];
  __shared__ int last_lds;
  const SplitPlace p = split_place(a.n, D);
  const int qn = p.qn, h = p.h, lane = p.lane;
  const float c = a.n.scale_log2;
  const uint8_t* vp = a.v + ((unsigned long long)a.v_bs * p.b + (unsigned long long)a.v_hs * p.hk) * 16;
  const int v_rs = (int)a.v_rs * 16, seqlen_k = a.n.seqlen_k;
  constexpr unsigned kNoSource = 0x80000000u;
  unsigned src[kPasses];
#pragma unroll
  for (int i = 0; i < kPasses; ++i) {
    int r, ch;
    tile_slot_decode<VT ? 64 : DP, !VT>(i * 64 + lane, r, ch);
    src[i] = VT || ch * 16 < D ? (unsigned)(r * v_rs + ch * 16) : kNoSource;
  }
  const __amdgpu_buffer_rsrc_t rsrc = __builtin_amdgcn_make_buffer_rsrc(
      (void*)vp, 0, VT ? (D - 1) * v_rs + seqlen_k : (seqlen_k - 1) * v_rs + D, 0x00020000);
  auto issue = [&](int j, uint8_t* dst) __attribute__((always_inline)) {
    const int base = VT ? j * kKvBlock : (int)((unsigned)j * kKvBlock * (unsigned)v_rs);
    const bool v_clamp = VT && (j + 1) * kKvBlock > seqlen_k;
#pragma unroll
    for (int i = 0; i < kPasses; ++i) {
      uint8_t* at = dst + p.wave * kTileBytes + i * 1024;
      if (v_clamp) {  // transposed v, ragged last block: see fa8_fwd_kernel
        int r, ch;
        tile_slot_decode<64, false>(i * 64 + lane, r, ch);
        const unsigned off = r < D ? (unsigned)(r * v_rs + min(base + ch * 16, seqlen_k - 16)) : kNoSource;
        __builtin_amdgcn_raw_ptr_buffer_load_lds(rsrc, LDS_PTR(void, at), 16, off, 0, 0, 0);
      } else {
        __builtin_amdgcn_raw_ptr_buffer_load_lds(rsrc, LDS_PTR(void, at), 16, src[i], base, 0, 0);
      }
    }
  };
  const float* s_in = (const float*)(a.n.workspace + p.ws.s) + (p.at * p.live_rows + min(qn, p.live_rows - 1)) * p.ws.keys + 32 * h;
  auto load_s = [&](int j, v4f(&s)[8]) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < 8; ++i) s[i] = *(const v4f*)(s_in + (long long)j * kKvBlock + 4 * i);
  };
  v4f s0[8], s1[8];
  // The running max before this range: over the splits before this one (their loads under way together; the compiler takes their max
  // inside this branch, so a split > 0 waits for them before the loads below start) and the ranges before this one in the split.
  const float* split_max = (const float*)(a.n.workspace + p.ws.split_max) + p.at * p.splits * 32;
  const float* range_max = (const float*)(a.n.workspace + p.ws.range_max) + (p.at * p.splits + p.split) * kSplitWaves * 32;
  float before[kSplitMax / 2 + kSplitWaves - 1];
  if (p.split > 0) {
#pragma unroll
    for (int e = 0; e < kSplitMax / 2; ++e) before[e] = split_max[min(2 * e + h, p.split - 1) * 32 + qn];
  }
#pragma unroll
  for (int x = 0; x < kSplitWaves - 1; ++x) before[kSplitMax / 2 + x] = x < p.wave ? range_max[x * 32 + qn] : -1.0e30f;
  if (p.count > 0) {
    load_s(p.first, s0);
    issue(p.first, lds0);
  }
  float m_run = -1.0e30f;
  if (p.split > 0) {
#pragma unroll
    for (int e = 0; e < kSplitMax / 2; e += 2) m_run = max3(before[e], before[e + 1], m_run);
  }
#pragma unroll
  for (int x = 0; x < kSplitWaves - 1; ++x) m_run = __builtin_fmaxf(m_run, before[kSplitMax / 2 + x]);
  m_run = lane32_max(m_run);

  constexpr int kTrStride = 8 * DP;
  const int tr_j = (lane & 15) >> 1, tr_e = lane & 1, tr_g1 = (lane >> 4) & 1;
  int v_off[kMTiles], vt_off[2];
#pragma unroll
  for (int mt = 0; mt < kMTiles; ++mt) v_off[mt] = p.wave * kTileBytes + tile_offset<DP, true>(32 * h + tr_j, 2 * mt + tr_g1) + 8 * tr_e;
#pragma unroll
  for (int e = 0; e < 2; ++e) vt_off[e] = p.wave * kTileBytes + tile_offset<64, false>(qn, 2 * h + e);
  auto load_vf = [&](const uint8_t* vb, int mt) __attribute__((always_inline)) {
    v8i vf;
    if constexpr (VT) {
      const v4i lo = *LDS_PTR(const v4i, vb + mt * 32 * 64 + vt_off[0]);
      const v4i hi = *LDS_PTR(const v4i, vb + mt * 32 * 64 + vt_off[1]);
      vf = {lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
    } else {
#pragma unroll
      for (int g = 0; g < 4; ++g) {
        const v2i x = __builtin_amdgcn_ds_read_tr8_b64_v2i32(LDS_PTR(v2i, vb + v_off[mt] + g * kTrStride));
        vf[2 * g] = x[0];
        vf[2 * g + 1] = x[1];
      }
    }
    return vf;
  };
  v16f o_acc[kMTiles];
#pragma unroll
  for (int mt = 0; mt < kMTiles; ++mt)
#pragma unroll
    for (int i = 0; i < 16; ++i) o_acc[mt][i] = 0.f;
  float l_run = 0.f;
  auto block = [&](const uint8_t* vb, const v4f(&s)[8]) __attribute__((always_inline)) {
    split_weights_and_o<E5M2, kMTiles>(s, c, m_run, l_run, o_acc, [&](int mt) __attribute__((always_inline)) { return load_vf(vb, mt); });
  };
  // The next block's logits and V are asked for before a block is worked on: the last kPasses + 8 loads may still fly then.  (So they do
  // in front of the blocks in lds0; in front of the V reads from lds1 the compiler waits for everything, as in the logits kernel.)
  constexpr int kNext = kPasses + 8;
  for (int i = 0; i < p.count; i += 2) {
    if (i + 1 < p.count) {
      load_s(p.first + i + 1, s1);
      issue(p.first + i + 1, lds1);
      wait_loads<kNext>();
    } else {
      wait_loads<0>();
    }
    block(lds0, s0);
    if (i + 1 < p.count) {
      if (i + 2 < p.count) {
        load_s(p.first + i + 2, s0);
        issue(p.first + i + 2, lds0);
        wait_loads<kNext>();
      } else {
        wait_loads<0>();
      }
      block(lds1, s1);
    }
  }

  split_merge<D, E5M2>(a, p, o_acc, m_run, l_run, lds0, lds1, m_lds, l_lds, &last_lds, [&]() __attribute__((always_inline)) {
    return threadIdx.x == 0 && __hip_atomic_fetch_add((unsigned*)(a.n.workspace + p.ws.done) + p.at, 1u, __ATOMIC_RELAXED,
                                                      __HIP_MEMORY_SCOPE_AGENT) == (unsigned)p.splits - 1;
  });
#endif
}

// ---- both passes in one kernel, for ranges whose logits fit in LDS ----
struct SplitFusedArgs {
  SplitShape n;
  const uint8_t* q;
  const uint8_t* k;
  const uint8_t* v;
  void* o;
  float* lse;
  unsigned long long tag;  // of this launch: what is in the workspace without it is of no launch or of another one
  unsigned q_bs, q_hs, q_rs;
  unsigned k_bs, k_hs, k_rs;
  unsigned v_bs, v_hs, v_rs;
  unsigned o_bs, o_hs, o_rs;
  unsigned lse_bs, lse_hs;
  unsigned late;  // splits (a bit each) that do not hand on their maximum, for tests
};
// Most LDS bytes for the logits of the four ranges: what the ring of two tiles a wavefront leaves of 160 KB.  (Rings of three and four: 20.3
// and 20.6 us for 32768 keys of 8 k/v heads instead of 18.8 in a loop of single calls, head dim 64 1 - 3 % slower: ranges are rounded up to whole rounds of the ring, and
// the logits have less room.)
constexpr int split_fused_s_bytes(int d) {
  const int dp = d <= 32 ? 32 : (d <= 64 ? 64 : (d <= 128 ? 128 : 256));
  return (160 * 1024 - 2048 - 2 * kSplitWaves * kKvBlock * dp) / 4096 * 4096;
}
// What a launch asks for.  (Held whatever the ranges needed, 161 KB a workgroup, a call had to wait for compute units that another stream's
// kernel left empty: 4 sequences of 8192 keys, 8 k/v heads, head dim 64, beside full attention over 4096 keys of 64 heads, head dim 128: 295 us
// a call, 30 so (the two kernels before: 92); alone 11.7 either way.)
inline long long split_fused_s_used(int live_rows, int blocks_per_range) { return (long long)blocks_per_range * live_rows * kKvBlock * 4 * kSplitWaves; }
inline bool split_fused_fits(int d, int live_rows, int blocks_per_range) {
  return split_fused_s_used(live_rows, blocks_per_range) <= split_fused_s_bytes(d);
}

template <int D, bool E5M2, bool VT>
__global__ __launch_bounds__(64 * kSplitWaves) __attribute__((amdgpu_waves_per_eu(1))) void fa8_split_fused_kernel(const SplitFusedArgs a) {
#if defined(__HIP_DEVICE_COMPILE__)
  constexpr int DP = D <= 32 ? 32 : (D <= 64 ? 64 : (D <= 128 ? 128 : 256));
  constexpr int kTileBytes = kKvBlock * DP, kPasses = kTileBytes / 1024, kKSteps = (D + 63) / 64, kMTiles = D / 32;
  constexpr int R = 2;
  static_assert(kSplitWaves * kTileBytes >= 2 * D * 32 * 4 && kSplitWaves * kTileBytes >= kSplitMax * 256, "see split_merge");
  __shared__ __attribute__((aligned(1024))) uint8_t lds0[kSplitWaves * kTileBytes];
  __shared__ __attribute__((aligned(1024))) uint8_t lds1[kSplitWaves * kTileBytes];
  extern __shared__ __attribute__((aligned(1024))) uint8_t s_lds[];  // split_fused_s_used() bytes
  __shared__ float max_lds[kSplitWaves * 32], m_lds[kSplitWaves * 32], l_lds[kSplitWaves * 32];
  __shared__ int before_lds[32];  // max over the splits before this one, as an integer of the same order
  __shared__ unsigned late_lds;  // splits whose maximum has not come, a bit each
  __shared__ int last_lds;
  const SplitPlace p = split_place(a.n, D);
  const int qn = p.qn, h = p.h, lane = p.lane, tid = threadIdx.x, live = p.live_rows;
  const float c = a.n.scale_log2;
  const int seqlen_k = a.n.seqlen_k, kv_last = seqlen_k - 1;
  const uint8_t* kp = a.k + ((unsigned long long)a.k_bs * p.b + (unsigned long long)a.k_hs * p.hk) * 16;
  const uint8_t* vp = a.v + ((unsigned long long)a.v_bs * p.b + (unsigned long long)a.v_hs * p.hk) * 16;
  const int k_rs = (int)a.k_rs * 16, v_rs = (int)a.v_rs * 16;
  v8i qf[kKSteps];
  {
    const uint8_t* q8 = a.q + ((unsigned long long)a.q_bs * p.b + (unsigned long long)a.q_hs * p.hd + (unsigned long long)a.q_rs * p.qi) * 16;
#pragma unroll
    for (int ks = 0; ks < kKSteps; ++ks) {
      const bool upper_exists = 64 * ks + 32 < D;
      const uint8_t* s8 = q8 + 64 * ks + (upper_exists ? 32 * h : 0);
      const v4i lo = *(const v4i*)(s8);
      const v4i hi = *(const v4i*)(s8 + 16);
      qf[ks] = {lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
      if (!upper_exists && h) qf[ks] = v8i{0, 0, 0, 0, 0, 0, 0, 0};
    }
  }
  // Copies: the K tiles of the range, then its V tiles, go through one ring of R stages.  Every step starts one copy, of a tile that
  // does not exist through a resource of length 0, so that one wait fits every step (see fa8_fwd_kernel).
  constexpr unsigned kNoSource = 0x80000000u;
  unsigned k_src[kPasses], v_src[kPasses];
  int v_chunk = 0;  // transposed v: the lane's first key of a block, the same in every pass
#pragma unroll
  for (int i = 0; i < kPasses; ++i) {
    int r, ch;
    tile_slot_decode<DP, false>(i * 64 + lane, r, ch);
    k_src[i] = ch * 16 < D ? (unsigned)(kv_of_lds_row(r) * k_rs + ch * 16) : kNoSource;
    tile_slot_decode<VT ? 64 : DP, !VT>(i * 64 + lane, r, ch);
    // (transposed v: rows past the head dim lie past the resource's end)
    v_src[i] = VT || ch * 16 < D ? (unsigned)(r * v_rs + ch * 16) : kNoSource;
    if (VT) v_chunk = ch * 16;
  }
  const int k_bytes = kv_last * k_rs + D, v_bytes = VT ? (D - 1) * v_rs + seqlen_k : kv_last * v_rs + D;
  auto issue_k = [&](int i, uint8_t* dst) __attribute__((always_inline)) {
    const bool exists = i < p.count;
    const __amdgpu_buffer_rsrc_t rsrc = __builtin_amdgcn_make_buffer_rsrc((void*)kp, 0, exists ? k_bytes : 0, 0x00020000);
    const int base = exists ? (int)((unsigned)(p.first + i) * kKvBlock * (unsigned)k_rs) : 0;
#pragma unroll
    for (int x = 0; x < kPasses; ++x)
      __builtin_amdgcn_raw_ptr_buffer_load_lds(rsrc, LDS_PTR(void, dst + p.wave * kTileBytes + x * 1024), 16, k_src[x], base, 0, 0);
  };
  auto issue_v = [&](int i, uint8_t* dst) __attribute__((always_inline)) {
    const bool exists = i < p.count;
    const __amdgpu_buffer_rsrc_t rsrc = __builtin_amdgcn_make_buffer_rsrc((void*)vp, 0, exists ? v_bytes : 0, 0x00020000);
    const int key = exists ? (p.first + i) * kKvBlock : 0;
    // transposed v, ragged last block: chunks past the last key are pulled back onto the last chunk (see fa8_fwd_kernel)
    const unsigned shift = VT ? (unsigned)min(key, seqlen_k - 16 - v_chunk) : 0;
    const int base = VT ? 0 : (int)((unsigned)key * (unsigned)v_rs);
#pragma unroll
    for (int x = 0; x < kPasses; ++x)
      __builtin_amdgcn_raw_ptr_buffer_load_lds(rsrc, LDS_PTR(void, dst + p.wave * kTileBytes + x * 1024), 16, v_src[x] + shift, base, 0, 0);
  };
  uint8_t* const ring[R] = {lds0, lds1};
#pragma unroll
  for (int i = 0; i < R; ++i) issue_k(i, ring[i]);
  if (tid < 32) before_lds[tid] = (int)0x80000000;
  if (tid == 0) late_lds = 0;

  // ---- S of the range, into LDS (live rows; a lane reads back what it wrote), and the row max ----
  int k_off[kKSteps][2];
#pragma unroll
  for (int ks = 0; ks < kKSteps; ++ks)
#pragma unroll
    for (int e = 0; e < 2; ++e) k_off[ks][e] = p.wave * kTileBytes + tile_offset<DP, false>(qn, DP >= 64 ? 4 * ks + 2 * h + e : e);
  const int kv_limit = p.causal ? min(p.qi + p.shift, kv_last) : kv_last;
  const int q_first = p.query_of(min(p.tile * 32, p.last_row));
  const int n_plain = (p.causal ? max(0, min(q_first + p.shift, seqlen_k)) : seqlen_k) / kKvBlock;  // blocks without a masked logit
  auto mask = [&](int j, v16f(&s)[2]) __attribute__((always_inline)) {
    if (j >= n_plain) {
#pragma unroll
      for (int t = 0; t < 2; ++t)
#pragma unroll
        for (int e = 0; e < 16; ++e)
          if (j * kKvBlock + 32 * h + 16 * t + e > kv_limit) s[t][e] = -INFINITY;
    }
  };
  uint8_t* const s_at = s_lds + p.wave * a.n.blocks_per_range * live * (kKvBlock * 4) + (h * live + min(qn, live - 1)) * 16;
  float m_run = -1.0e30f;
  const int groups = max(1, (p.count + R - 1) / R);
  // Q has arrived.  (Left to the compiler, which waits in front of the loop, this would be a wait for all copies.)
  wait_loads<R * kPasses>();
#pragma unroll
  for (int ks = 0; ks < kKSteps; ++ks) asm volatile("" : "+v"(qf[ks]));
  const bool stores_s = qn < live;
  auto k_step = [&](auto last_c, int i, int x) __attribute__((always_inline)) {
    wait_loads<(R - 1) * kPasses>();
    __builtin_amdgcn_sched_barrier(0);
    v16f s[2];
    if (i < p.count) {
#pragma unroll
      for (int t = 0; t < 2; ++t) {
#pragma unroll
        for (int e = 0; e < 16; ++e) s[t][e] = 0.f;
#pragma unroll
        for (int ks = 0; ks < kKSteps; ++ks) {
          const v4i lo = *LDS_PTR(const v4i, ring[x] + t * 32 * DP + k_off[ks][0]);
          const v4i hi = *LDS_PTR(const v4i, ring[x] + t * 32 * DP + k_off[ks][1]);
          s[t] = mfma_fp8<E5M2>(v8i{lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]}, qf[ks], s[t]);
        }
      }
    }
    __builtin_amdgcn_sched_barrier(0);
    __builtin_amdgcn_s_waitcnt(0xC07F);  // the tile has been read
    if constexpr (decltype(last_c)::value)
      issue_v(x, ring[x]);
    else
      issue_k(i + R, ring[x]);
    __builtin_amdgcn_sched_barrier(0);
    if (i < p.count) {
      mask(p.first + i, s);
#pragma unroll
      for (int t = 0; t < 2; ++t)
#pragma unroll
        for (int e = 0; e < 16; e += 2) m_run = max3(s[t][e], s[t][e + 1], m_run);
      if (stores_s) {
#pragma unroll
        for (int e = 0; e < 8; ++e)
          *LDS_PTR(v4f, s_at + (i * 8 + e) * live * 32) = v4f{s[e >> 2][4 * (e & 3)], s[e >> 2][4 * (e & 3) + 1], s[e >> 2][4 * (e & 3) + 2], s[e >> 2][4 * (e & 3) + 3]};
      }
    }
    __builtin_amdgcn_sched_barrier(0);
  };
  for (int g = 0; g + 1 < groups; ++g) {
#pragma unroll
    for (int x = 0; x < R; ++x) k_step(std::false_type(), g * R + x, x);
  }
#pragma unroll
  for (int x = 0; x < R; ++x) k_step(std::true_type(), (groups - 1) * R + x, x);

  // ---- the running max before the range ----
  // A bare barrier (the copies of V stay under way), once this wavefront's LDS operations are done.
  auto sync = [&]() __attribute__((always_inline)) {
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
  };
  m_run = lane32_max(m_run);
  if (h == 0) max_lds[p.wave * 32 + qn] = m_run;
  sync();
  // A max travels as two words of half the tag and the value each: no word of an earlier launch passes for one of this launch, so
  // the workspace needs no preparation.  (It is cleared at the end: a captured launch runs again with the same tag.)
  typedef unsigned long long u64;
  const unsigned tag0 = (unsigned)a.tag, tag1 = (unsigned)(a.tag >> 32);
  u64* const maxima = (u64*)(a.n.workspace + p.ws.range_max) + p.at * p.splits * 64;  // [split][row][2]
  u64* const done = (u64*)(a.n.workspace + p.ws.split_max) + p.at * p.splits;         // [split]
  if (tid < live && p.split + 1 < p.splits && !(a.late >> p.split & 1)) {
    float m = max_lds[tid];
#pragma unroll
    for (int x = 1; x < kSplitWaves; ++x) m = __builtin_fmaxf(m, max_lds[x * 32 + tid]);
    const u64 value = (u64)__float_as_uint(m) << 32;
    __hip_atomic_store(maxima + (p.split * 32 + tid) * 2, value | tag0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    __hip_atomic_store(maxima + (p.split * 32 + tid) * 2 + 1, value | tag1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  }
  // (signed integers of the order of the floats; no NaN comes out of the maxima)
  auto ordered = [](float x) __attribute__((always_inline)) { const int i = __float_as_int(x); return i ^ ((i >> 31) & 0x7fffffff); };
  int looks = kSplitLooks;  // of this thread, at all the maxima that it takes
  for (int e = tid; e < p.split * live; e += 64 * kSplitWaves) {
    const int split = e / live, row = e - split * live;
    const u64* const at = maxima + (split * 32 + row) * 2;
    u64 x = 0, y = 0;
    bool there = false;
    do {  // (one look at each, also when the others have used them up)
      x = __hip_atomic_load(at, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      y = __hip_atomic_load(at + 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      there = (unsigned)x == tag0 && (unsigned)y == tag1 && x >> 32 == y >> 32;
    } while (!there && --looks > 0);
    if (there)
      atomicMax(before_lds + row, ordered(__uint_as_float((unsigned)(x >> 32))));
    else
      atomicOr(&late_lds, 1u << split);
  }
  sync();
  const unsigned late = __builtin_amdgcn_readfirstlane(late_lds);
  if (late) {
    // Workgroups before this one have not run yet (the chip is busy with something else): their maxima are formed here, from K in memory.
    float m = -1.0e30f;
    const int blocks = kSplitWaves * a.n.blocks_per_range;  // of a split
    for (unsigned left = late; left != 0; left &= left - 1) {
      const int first = __builtin_ctz(left) * blocks;
      for (int j = first + p.wave; j < first + blocks; j += kSplitWaves) {
        v16f s[2];
#pragma unroll
        for (int t = 0; t < 2; ++t) {
          const uint8_t* row = kp + (long long)min(j * kKvBlock + kv_of_lds_row(32 * t + qn), kv_last) * k_rs;
#pragma unroll
          for (int e = 0; e < 16; ++e) s[t][e] = 0.f;
#pragma unroll
          for (int ks = 0; ks < kKSteps; ++ks) {
            const uint8_t* k8 = row + 64 * ks + (64 * ks + 32 < D ? 32 * h : 0);  // (past the head dim Q is 0)
            const v4i lo = *(const v4i*)(k8);
            const v4i hi = *(const v4i*)(k8 + 16);
            v8i kf = {lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
            if (64 * ks + 32 >= D && h) kf = v8i{0, 0, 0, 0, 0, 0, 0, 0};  // (nor may a NaN meet that 0)
            s[t] = mfma_fp8<E5M2>(kf, qf[ks], s[t]);
          }
        }
        mask(j, s);
#pragma unroll
        for (int t = 0; t < 2; ++t)
#pragma unroll
          for (int e = 0; e < 16; e += 2) m = max3(s[t][e], s[t][e + 1], m);
      }
    }
    m = lane32_max(m);
    if (h == 0) atomicMax(before_lds + qn, ordered(m));
    sync();
  }
  {
    const int i = before_lds[qn];
    m_run = __builtin_fmaxf(-1.0e30f, p.split > 0 ? __int_as_float(i ^ ((i >> 31) & 0x7fffffff)) : -1.0e30f);
#pragma unroll
    for (int x = 0; x < kSplitWaves - 1; ++x)
      if (x < p.wave) m_run = __builtin_fmaxf(m_run, max_lds[x * 32 + qn]);
  }

  // ---- weights and O ----
  constexpr int kTrStride = 8 * DP;
  const int tr_j = (lane & 15) >> 1, tr_e = lane & 1, tr_g1 = (lane >> 4) & 1;
  int v_off[kMTiles], vt_off[2];
#pragma unroll
  for (int mt = 0; mt < kMTiles; ++mt) v_off[mt] = p.wave * kTileBytes + tile_offset<DP, true>(32 * h + tr_j, 2 * mt + tr_g1) + 8 * tr_e;
#pragma unroll
  for (int e = 0; e < 2; ++e) vt_off[e] = p.wave * kTileBytes + tile_offset<64, false>(qn, 2 * h + e);
  auto load_vf = [&](const uint8_t* vb, int mt) __attribute__((always_inline)) {
    v8i vf;
    if constexpr (VT) {
      const v4i lo = *LDS_PTR(const v4i, vb + mt * 32 * 64 + vt_off[0]);
      const v4i hi = *LDS_PTR(const v4i, vb + mt * 32 * 64 + vt_off[1]);
      vf = {lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
    } else {
#pragma unroll
      for (int g = 0; g < 4; ++g) {
        const v2i x = __builtin_amdgcn_ds_read_tr8_b64_v2i32(LDS_PTR(v2i, vb + v_off[mt] + g * kTrStride));
        vf[2 * g] = x[0];
        vf[2 * g + 1] = x[1];
      }
    }
    return vf;
  };
  v16f o_acc[kMTiles];
#pragma unroll
  for (int mt = 0; mt < kMTiles; ++mt)
#pragma unroll
    for (int i = 0; i < 16; ++i) o_acc[mt][i] = 0.f;
  float l_run = 0.f;
  for (int g = 0; g < groups; ++g) {
#pragma unroll
    for (int x = 0; x < R; ++x) {
      const int i = g * R + x;
      wait_loads<(R - 1) * kPasses>();
      __builtin_amdgcn_sched_barrier(0);
      v4f s[8];
      v8i vf[kMTiles];
      if (i < p.count) {
#pragma unroll
        for (int e = 0; e < 8; ++e) s[e] = *LDS_PTR(const v4f, s_at + (i * 8 + e) * live * 32);
#pragma unroll
        for (int mt = 0; mt < kMTiles; ++mt) vf[mt] = load_vf(ring[x], mt);
      }
      __builtin_amdgcn_sched_barrier(0);
      __builtin_amdgcn_s_waitcnt(0xC07F);  // the tile has been read
      issue_v(i + R, ring[x]);
      __builtin_amdgcn_sched_barrier(0);
      if (i < p.count)
        split_weights_and_o<E5M2, kMTiles>(s, c, m_run, l_run, o_acc, [&](int mt) __attribute__((always_inline)) { return vf[mt]; });
      __builtin_amdgcn_sched_barrier(0);
    }
  }
  wait_loads<0>();  // the last copies (of nothing) write the ring no more
  const bool wrote = split_merge<D, E5M2>(a, p, o_acc, m_run, l_run, lds0, lds1, m_lds, l_lds, &last_lds, [&]() __attribute__((always_inline)) {
    // Of the workgroups that end, at least the last one sees the marks of all.  (Several may: they write the same output.)
    if (lane == 0) __hip_atomic_store(done + p.split, a.tag, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    const bool seen = lane >= p.splits || __hip_atomic_load(done + min(lane, p.splits - 1), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == a.tag;
    return (bool)__all(seen);
  });
  if (wrote) {  // every workgroup of the tile has marked its end, so none looks at the maxima any more
    for (int e = tid; e < p.splits * 64; e += 64 * kSplitWaves) __hip_atomic_store(maxima + e, 0ull, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    if (tid < p.splits) __hip_atomic_store(done + tid, 0ull, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  }
#endif
}

}  // namespace fa8
#endif  // FA8_SPLIT_KV_H_
