// The split form of the cross attention (key_split.hpp) at head_dim up to 64.
#include "xattn_kernel.hpp"

namespace svhip {

template <>
void launch_split<2, true>(const XattnParams& p, unsigned g, hipStream_t s, bool vt, bool direct) {
  launch_split_impl<2, true>(p, g, s, vt, direct);
}

template <>
void launch_split<2, false>(const XattnParams& p, unsigned g, hipStream_t s, bool vt, bool direct) {
  launch_split_impl<2, false>(p, g, s, vt, direct);
}

}  // namespace svhip
