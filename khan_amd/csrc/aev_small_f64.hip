// The float64 instances of aev_small.hip,
// a translation unit of its own because it is compiled without the hoisting of constants out of loops (khan_amd/build.py,
// SOURCE_FLAGS).
#define KHAN_UNIT_F64
#include "aev_small.hip"
