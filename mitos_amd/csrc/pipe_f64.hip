// The fused pipeline's kernels and launches in double (pipe_impl.h).
#include "pipe_impl.h"

namespace mitos {

template struct Pipe<double>;

}  // namespace mitos
