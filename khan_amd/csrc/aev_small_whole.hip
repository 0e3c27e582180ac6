// The instances of aev_small.hip for float32 with five wavefronts per SIMD,
// a translation unit of its own because it is compiled without the hoisting of constants out of loops (khan_amd/build.py,
// SOURCE_FLAGS).
#define KHAN_UNIT_WHOLE
#include "aev_small.hip"
