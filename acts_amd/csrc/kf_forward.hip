// kf_forward.hip -- instantiations of the forward kernel: one precision,
// stepper and navigator per object (KF_MIXED, KF_SYMPY, KF_LAYERS = 0 or 1,
// set by the build).
#include "kf_forward.hpp"

namespace kf {

template <bool Mixed, bool Sympy, bool Layers>
ForwardFn forwardVariant(bool geoInLds, bool rev) {
  if (rev)
    return geoInLds ? fitForwardKernel<Mixed, true, Sympy, true, Layers>
                    : fitForwardKernel<Mixed, false, Sympy, true, Layers>;
  return geoInLds ? fitForwardKernel<Mixed, true, Sympy, false, Layers>
                  : fitForwardKernel<Mixed, false, Sympy, false, Layers>;
}

template ForwardFn forwardVariant<KF_MIXED, KF_SYMPY, KF_LAYERS>(bool, bool);

}  // namespace kf
