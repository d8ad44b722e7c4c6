// Runtime-width forward for networks of at most 64 features per layer:
// fwd_kernel.h compiled at width 64.  At width 128 such a network ran four
// times the MFMAs and twice the softplus of its padded features
// (16-64-64-64-4 in fp16 at 262,144 rows, width 128 -> 64: 40 -> 20 us, with
// the stash 65 -> 48 us, 201 MB written).
#include "fwd_kernel.h"

namespace mlpmk {

typedef Gen<Net<64, 64, 64>> G64Net2;
typedef Gen<Net<64, 64, 64, 64>> G64Net3;
typedef Gen<Net<64, 64, 64, 64, 64>> G64Net4;
typedef Gen<Net<64, 64, 64, 64, 64, 64>> G64Net5;

template <bool B>
static int dispatch_t(int L, const FwdParams& p, bool stash, hipStream_t st, LaunchInfo* info) {
  switch (L) {
    case 2: return launch_fwd_any<typename ElemNet<B, G64Net2>::type, 1, 8, 1, 8, 1>(p, stash, st, info);
    case 3: return launch_fwd_any<typename ElemNet<B, G64Net3>::type, 1, 8, 1, 8, 1>(p, stash, st, info);
    case 4: return launch_fwd_any<typename ElemNet<B, G64Net4>::type, 1, 8, 1, 8, 1>(p, stash, st, info);
    default: return launch_fwd_any<typename ElemNet<B, G64Net5>::type, 1, 8, 1, 8, 1>(p, stash, st, info);
  }
}

// dims: a fwd_generic_dims network whose widths are all at most 64.
int fwd_w64_dispatch(int L, const FwdParams& p, bool stash, bool bf, hipStream_t st, LaunchInfo* info) {
  return bf ? dispatch_t<true>(L, p, stash, st, info) : dispatch_t<false>(L, p, stash, st, info);
}

}  // namespace mlpmk
