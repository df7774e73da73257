// The split form of the cross attention (key_split.hpp) at head_dim 72 to 128.
#include "xattn_kernel.hpp"

namespace svhip {

template <>
void launch_split<3, true>(const XattnParams& p, unsigned g, hipStream_t s, bool vt, bool direct) {
  launch_split_impl<3, true>(p, g, s, vt, direct);
}

template <>
void launch_split<3, false>(const XattnParams& p, unsigned g, hipStream_t s, bool vt, bool direct) {
  launch_split_impl<3, false>(p, g, s, vt, direct);
}

template <>
void launch_split<4, true>(const XattnParams& p, unsigned g, hipStream_t s, bool vt, bool direct) {
  launch_split_impl<4, true>(p, g, s, vt, direct);
}

template <>
void launch_split<4, false>(const XattnParams& p, unsigned g, hipStream_t s, bool vt, bool direct) {
  launch_split_impl<4, false>(p, g, s, vt, direct);
}

}  // namespace svhip
