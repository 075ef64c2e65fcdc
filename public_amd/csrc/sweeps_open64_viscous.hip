// Kernel instances of one group (instances.hpp).
#include "instances.hpp"

INST_GROUP_OPEN64B()
