// Host entry points to the index and weight arithmetic of
// mitos_amd/csrc/particles.h, for tests that need no GPU.
#include <math.h>

#include "../../mitos_amd/csrc/particles.h"

using namespace mitos;

extern "C" {

void check_wrapf(int N, long n, const int* i, int* out) {
    for (long k = 0; k < n; k++) out[k] = wrapf(i[k], N, 1.0f / N);
}

}  // extern "C"
