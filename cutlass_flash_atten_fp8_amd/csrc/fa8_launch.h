// Launchers of the kernels that live in source files of their own, called by fa8_fwd.
#ifndef FA8_LAUNCH_H_
#define FA8_LAUNCH_H_
#include <hip/hip_runtime.h>

#include "fa8_api.h"

namespace fa8 {

// r row tiles of 32 query rows per workgroup, w wavefronts per row tile, one or two LDS stages where both are built, or the sums of the wavefronts
// apart; two tiles: O as whole lines (fa8_shared_rows.h)
__attribute__((visibility("hidden"))) int launch_shared(const Fa8FwdParams* p, int r, int w, int stages, bool apart, bool whole_lines, hipStream_t stream);

// the kernel with sums apart, nullptr where none is built
__attribute__((visibility("hidden"))) const void* apart_kernel(int head_dim, int r, int w, bool e5m2, bool vt);

// Keys of every row tile dealt to at most `splits` workgroups (fa8_split_kv.h): how (workgroups, KV blocks of a wavefront, whether one kernel does
// it), workspace bytes, launch (late: see fa8_fwd_ws_late).
struct SplitForm {
  int splits, blocks_per_range;
  bool one_kernel;
};
__attribute__((visibility("hidden"))) SplitForm split_form(const Fa8FwdParams* p, int splits);
__attribute__((visibility("hidden"))) long long split_workspace(const Fa8FwdParams* p, int splits);
__attribute__((visibility("hidden"))) int launch_split(const Fa8FwdParams* p, int splits, void* workspace, unsigned late,
                                                            hipStream_t stream);

}  // namespace fa8
#endif  // FA8_LAUNCH_H_
