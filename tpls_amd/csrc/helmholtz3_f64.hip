// helmholtz3.hpp in FP64 (a file per precision: they compile in parallel).
#include "helmholtz3.hpp"

namespace tpls {
TPLS_INST_HH3(double)
}  // namespace tpls
