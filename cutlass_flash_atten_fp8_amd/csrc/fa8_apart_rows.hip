// fa8_shared_rows_kernel with the sums of the wavefronts apart: what is built of it.
#include "fa8_launch.h"
#include "fa8_shared_rows.h"
namespace {

using namespace fa8;

template <int D, int R, int W>
const void* pick(bool e5m2, bool vt) {
  if (e5m2)
    return vt ? (const void*)&fa8_shared_rows_kernel<D, true, true, R, W, 2, true> : (const void*)&fa8_shared_rows_kernel<D, true, false, R, W, 2, true>;
  return vt ? (const void*)&fa8_shared_rows_kernel<D, false, true, R, W, 2, true> : (const void*)&fa8_shared_rows_kernel<D, false, false, R, W, 2, true>;
}
template <int D>
const void* pick_rw(int r, int w, bool e5m2, bool vt) {  // what choose_plan takes
  if (r == 1 && w == 4) return pick<D, 1, 4>(e5m2, vt);
  if (r == 2 && w == 2) return pick<D, 2, 2>(e5m2, vt);
  if constexpr (D > 64)
    if (r == 2 && w == 4) return pick<D, 2, 4>(e5m2, vt);
  return nullptr;
}

}  // namespace

const void* fa8::apart_kernel(int head_dim, int r, int w, bool e5m2, bool vt) {
  switch (head_dim) {
    case 32: return pick_rw<32>(r, w, e5m2, vt);
    case 64: return pick_rw<64>(r, w, e5m2, vt);
    case 96: return pick_rw<96>(r, w, e5m2, vt);
    case 128: return pick_rw<128>(r, w, e5m2, vt);
    default: return nullptr;
  }
}
