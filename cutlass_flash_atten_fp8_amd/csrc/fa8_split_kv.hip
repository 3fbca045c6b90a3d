// Launcher of the split-kv kernels (fa8_split_kv.h): the plan, the workspace and the launches.
#include <atomic>

#include "fa8_launch.h"
#include "fa8_split_kv.h"

namespace {

using namespace fa8;

template <int D>
const void* logits_kernel(bool e5m2) {
  return e5m2 ? (const void*)&fa8_split_logits_kernel<D, true> : (const void*)&fa8_split_logits_kernel<D, false>;
}
template <int D>
const void* values_kernel(bool e5m2, bool vt) {
  if (e5m2) return vt ? (const void*)&fa8_split_values_kernel<D, true, true> : (const void*)&fa8_split_values_kernel<D, true, false>;
  return vt ? (const void*)&fa8_split_values_kernel<D, false, true> : (const void*)&fa8_split_values_kernel<D, false, false>;
}

template <int D>
const void* fused_kernel(bool e5m2, bool vt) {
  if (e5m2) return vt ? (const void*)&fa8_split_fused_kernel<D, true, true> : (const void*)&fa8_split_fused_kernel<D, true, false>;
  return vt ? (const void*)&fa8_split_fused_kernel<D, false, true> : (const void*)&fa8_split_fused_kernel<D, false, false>;
}

// A number that no other launch has (SplitFusedArgs::tag): a bijection (splitmix64's) of a count.  Halves of zeros or ones are left out:
// a workspace may be full of them.
unsigned long long next_tag() {
  static std::atomic<unsigned long long> count{0};
  for (;;) {
    unsigned long long x = (count.fetch_add(1, std::memory_order_relaxed) + 1) * 0x9e3779b97f4a7c15ull;
    x = (x ^ x >> 30) * 0xbf58476d1ce4e5b9ull;
    x = (x ^ x >> 27) * 0x94d049bb133111ebull;
    x ^= x >> 31;
    const unsigned lo = (unsigned)x, hi = (unsigned)(x >> 32);
    if (lo != 0 && hi != 0 && ~lo != 0 && ~hi != 0) return x;
  }
}

struct Plan {
  int heads_k, tiles, live_rows, keys, splits, blocks_per_range;
};

Plan plan_of(const Fa8FwdParams* p, int splits) {
  Plan n;
  n.heads_k = p->heads_k > 0 ? p->heads_k : p->heads;
  const long long rows = (long long)(p->heads / n.heads_k) * p->seqlen_q;
  n.tiles = (int)((rows + 31) / 32);
  n.live_rows = rows < 32 ? (int)rows : 32;
  n.keys = split_visible_keys(p->seqlen_q, p->seqlen_k, p->is_causal, p->causal_align == FA8_CAUSAL_BOTTOM_RIGHT);
  const int blocks = (int)(((long long)n.keys + kKvBlock - 1) / kKvBlock);
  n.blocks_per_range = (blocks + splits * kSplitWaves - 1) / (splits * kSplitWaves);
  n.splits = (blocks + n.blocks_per_range * kSplitWaves - 1) / (n.blocks_per_range * kSplitWaves);
  return n;
}

}  // namespace

fa8::SplitForm fa8::split_form(const Fa8FwdParams* p, int splits) {
  const Plan n = plan_of(p, splits);
  return {n.splits, n.blocks_per_range, split_fused_fits(p->head_dim, n.live_rows, n.blocks_per_range)};
}

long long fa8::split_workspace(const Fa8FwdParams* p, int splits) {
  const Plan n = plan_of(p, splits);
  return split_layout((long long)p->batch * n.heads_k * n.tiles, n.splits, n.live_rows, p->head_dim, n.keys).bytes;
}

int fa8::launch_split(const Fa8FwdParams* p, int splits, void* workspace, unsigned late, hipStream_t stream) {
  const Plan n = plan_of(p, splits);
  SplitShape shape;
  shape.workspace = (uint8_t*)workspace;
  shape.scale_log2 = p->softmax_scale * 1.4426950408889634f;
  shape.seqlen_q = p->seqlen_q;
  shape.seqlen_k = p->seqlen_k;
  shape.mode = pack_mode(p);
  shape.splits = (uint16_t)n.splits;
  shape.blocks_per_range = (uint16_t)n.blocks_per_range;
  shape.heads_k = n.heads_k;
  shape.all_tiles = p->batch * n.heads_k * n.tiles;
  const bool e5m2 = p->in_dtype == FA8_DTYPE_E5M2, vt = p->v_layout == FA8_V_TRANSPOSED;
  const dim3 grid((unsigned)n.heads_k, (unsigned)p->batch, (unsigned)(n.tiles * n.splits));
  if (split_fused_fits(p->head_dim, n.live_rows, n.blocks_per_range)) {
    SplitFusedArgs f;
    f.n = shape;
    f.q = (const uint8_t*)p->q;
    f.k = (const uint8_t*)p->k;
    f.v = (const uint8_t*)p->v;
    f.o = p->o;
    f.lse = (float*)p->lse;
    f.tag = next_tag();
    f.late = late;
    f.q_bs = p->q_batch_stride / 16; f.q_hs = p->q_head_stride / 16; f.q_rs = p->q_row_stride / 16;
    f.k_bs = p->k_batch_stride / 16; f.k_hs = p->k_head_stride / 16; f.k_rs = p->k_row_stride / 16;
    f.v_bs = p->v_batch_stride / 16; f.v_hs = p->v_head_stride / 16; f.v_rs = p->v_row_stride / 16;
    f.o_bs = p->o_batch_stride / 4; f.o_hs = p->o_head_stride / 4; f.o_rs = p->o_row_stride / 4;
    f.lse_bs = p->lse_batch_stride; f.lse_hs = p->lse_head_stride;
    const void* fn = nullptr;
    switch (p->head_dim) {
#define FA8_HEAD_DIM_CASE(D_) \
  case D_: fn = fused_kernel<D_>(e5m2, vt); break
      FA8_HEAD_DIM_CASE(32);
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
    void* argv[] = {&f};
    return (int)hipLaunchKernel(fn, grid, dim3(64 * kSplitWaves), argv, (size_t)split_fused_s_used(n.live_rows, n.blocks_per_range), stream);
  }
  SplitLogitsArgs l;
  l.n = shape;
  l.q = (const uint8_t*)p->q;
  l.k = (const uint8_t*)p->k;
  l.q_bs = p->q_batch_stride / 16; l.q_hs = p->q_head_stride / 16; l.q_rs = p->q_row_stride / 16;
  l.k_bs = p->k_batch_stride / 16; l.k_hs = p->k_head_stride / 16; l.k_rs = p->k_row_stride / 16;
  SplitValuesArgs v;
  v.n = shape;
  v.v = (const uint8_t*)p->v;
  v.o = p->o;
  v.lse = (float*)p->lse;
  v.v_bs = p->v_batch_stride / 16; v.v_hs = p->v_head_stride / 16; v.v_rs = p->v_row_stride / 16;
  v.o_bs = p->o_batch_stride / 4; v.o_hs = p->o_head_stride / 4; v.o_rs = p->o_row_stride / 4;
  v.lse_bs = p->lse_batch_stride; v.lse_hs = p->lse_head_stride;
  const void *first = nullptr, *second = nullptr;
  switch (p->head_dim) {
#define FA8_HEAD_DIM_CASE(D_) \
  case D_: first = logits_kernel<D_>(e5m2); second = values_kernel<D_>(e5m2, vt); break
    FA8_HEAD_DIM_CASE(32);
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
  void *argv_l[] = {&l}, *argv_v[] = {&v};
  const hipError_t rc = hipLaunchKernel(first, grid, dim3(64 * kSplitWaves), argv_l, 0, stream);
  if (rc != hipSuccess) return (int)rc;
  return (int)hipLaunchKernel(second, grid, dim3(64 * kSplitWaves), argv_v, 0, stream);
}
