// kf_forward.hip -- instantiations of the forward kernel: one precision,
// stepper, navigator and kind of field per object (KF_MIXED, KF_SYMPY,
// KF_LAYERS, KF_MAP = 0 or 1, set by the build).
#include "kf_forward.hpp"

namespace kf {

template <bool Mixed, bool Sympy, bool Layers, bool Map>
ForwardFn forwardVariant(bool geoInLds, bool rev) {
  if (rev)
    return geoInLds ? fitForwardKernel<Mixed, true, Sympy, true, Layers, Map>
                    : fitForwardKernel<Mixed, false, Sympy, true, Layers, Map>;
  return geoInLds ? fitForwardKernel<Mixed, true, Sympy, false, Layers, Map>
                  : fitForwardKernel<Mixed, false, Sympy, false, Layers, Map>;
}

template ForwardFn forwardVariant<KF_MIXED, KF_SYMPY, KF_LAYERS, KF_MAP>(bool, bool);

}  // namespace kf
