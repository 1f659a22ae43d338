// helmholtz3.hpp in FP32 (a file per precision: they compile in parallel).
#include "helmholtz3.hpp"

namespace tpls {
TPLS_INST_HH3(float)
}  // namespace tpls
