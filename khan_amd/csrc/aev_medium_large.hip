// The instances of aev_medium.hip for molecules of more than 256 atoms, those in float64 and the float32 forward kernel,
// a translation unit of its own because it is compiled without the hoisting of constants out of loops (khan_amd/build.py,
// SOURCE_FLAGS).
#define KHAN_UNIT_LARGE
#include "aev_medium.hip"
