// Host build of the product's quotient and remainder by a launch constant
// (zillumgl_amd/csrc/zgl_math.h divUniform), for comparison with whole-number division.
#include <cstdint>

#include "../../zillumgl_amd/csrc/zgl_math.h"

extern "C" void probe_div(const int32_t* n, int32_t d, int32_t* q, int32_t* r, int64_t count)
{
    for (int64_t i = 0; i < count; i++) {
        int rem;
        q[i] = zgl::divUniform(n[i], d, 0xffffffffu / (uint32_t)d, rem);
        r[i] = rem;
    }
}
