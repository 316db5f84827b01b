// Instantiations: K's layers of the preconditioned CG.
#include "pcg_layers.hpp"

namespace qed3 {
QED3_TC_K(QED3_TC_LAUNCH)
}  // namespace qed3
