// Instantiations: the layers of the network applied on its own (horner_apply_solver).
#include "pcg_layers.hpp"

namespace qed3 {
QED3_TC_CHECK(QED3_TC_LAUNCH)
}  // namespace qed3
