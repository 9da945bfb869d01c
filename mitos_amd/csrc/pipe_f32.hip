// The fused pipeline's kernels and launches in float (pipe_impl.h).
#include "pipe_impl.h"

namespace mitos {

template struct Pipe<float>;

}  // namespace mitos
