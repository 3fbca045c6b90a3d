// Launcher of fa8_shared_rows_kernel: which (R, W) pairs are built, and the packed argument block.
#include "fa8_launch.h"
#include "fa8_shared_rows.h"
namespace {

using namespace fa8;

template <int D, int R, int W, int STAGES>
const void* pick(bool e5m2, bool vt) {
  if (e5m2)
    return vt ? (const void*)&fa8_shared_rows_kernel<D, true, true, R, W, STAGES, false> : (const void*)&fa8_shared_rows_kernel<D, true, false, R, W, STAGES, false>;
  return vt ? (const void*)&fa8_shared_rows_kernel<D, false, true, R, W, STAGES, false> : (const void*)&fa8_shared_rows_kernel<D, false, false, R, W, STAGES, false>;
}
template <int D>
const void* pick_rw(int r, int w, int stages, bool e5m2, bool vt) {
  // what choose_plan takes; head dim 32 has no use for one stage with (2, 2) (1.0 - 1.2)
  if (r == 1 && w == 4 && stages == 1) return pick<D, 1, 4, 1>(e5m2, vt);
  if constexpr (D <= 128) {
    if (r == 1 && w == 4 && stages == 2) return pick<D, 1, 4, 2>(e5m2, vt);
    if (r == 2 && w == 2 && stages == 2) return pick<D, 2, 2, 2>(e5m2, vt);
  }
  if constexpr (D > 32)
    if (r == 2 && w == 2 && stages == 1) return pick<D, 2, 2, 1>(e5m2, vt);
  if constexpr (D > 64)
    if (r == 2 && w == 4 && stages == (D <= 128 ? 2 : 1)) return pick<D, 2, 4, D <= 128 ? 2 : 1>(e5m2, vt);
  return nullptr;
}

}  // namespace

int fa8::launch_shared(const Fa8FwdParams* p, int r, int w, int stages, bool apart, bool whole_lines, hipStream_t stream) {
  SharedArgs a;
  a.q = (const uint8_t*)p->q;
  a.k = (const uint8_t*)p->k;
  a.v = (const uint8_t*)p->v;
  a.o = p->o;
  a.lse = (float*)p->lse;
  a.scale_log2 = p->softmax_scale * 1.4426950408889634f;
  a.seqlen_q = p->seqlen_q;
  a.seqlen_k = p->seqlen_k;
  const int heads_k = p->heads_k > 0 ? p->heads_k : p->heads, group = p->heads / heads_k;
  a.mode = pack_mode(p) | (whole_lines ? kSharedLines : 0);
  a.q_bs = p->q_batch_stride / 16; a.q_hs = p->q_head_stride / 16; a.q_rs = p->q_row_stride / 16;
  a.k_bs = p->k_batch_stride / 16; a.k_hs = p->k_head_stride / 16; a.k_rs = p->k_row_stride / 16;
  a.v_bs = p->v_batch_stride / 16; a.v_hs = p->v_head_stride / 16; a.v_rs = p->v_row_stride / 16;
  a.o_bs = p->o_batch_stride / 4; a.o_hs = p->o_head_stride / 4; a.o_rs = p->o_row_stride / 4;
  a.lse_bs = p->lse_batch_stride; a.lse_hs = p->lse_head_stride;
  const int tiles = (int)(((long long)group * p->seqlen_q + 32 * r - 1) / (32 * r));
  const bool e5m2 = p->in_dtype == FA8_DTYPE_E5M2, vt = p->v_layout == FA8_V_TRANSPOSED;
  const void* fn = apart ? apart_kernel(p->head_dim, r, w, e5m2, vt) : nullptr;
  if (!apart) switch (p->head_dim) {
#define FA8_HEAD_DIM_CASE(D_) \
  case D_: fn = pick_rw<D_>(r, w, stages, e5m2, vt); break
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
  if (!fn) return FA8_ERR_UNSUPPORTED;
  void* argv[] = {&a.k
#define FA8_FIELD(type, name) , &a.name
                  FA8_SHARED_FIELDS(FA8_FIELD)
#undef FA8_FIELD
  };
  // Head dim 32, two stages: 32 KB that nothing uses keep a compute unit at two workgroups, for which choose_plan takes them; with a third, 1024 tiles
  // take a round of three a compute unit and one of one (1024 heads, 7297 keys: 105 us, 91 so).
  const unsigned unused_lds = p->head_dim == 32 && r == 1 && stages == 2 && !apart ? 32 * 1024 : 0;
  return (int)hipLaunchKernel(fn, dim3((unsigned)heads_k, (unsigned)p->batch, (unsigned)tiles), dim3(64 * r * w), argv, unused_lds, stream);
}
