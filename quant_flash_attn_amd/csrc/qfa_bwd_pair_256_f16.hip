// The backward's kernel at head_dim 256, Float16 (one instance per file: they are compiled side by side)
#include "qfa_bwd_pair.h"

namespace qfa {
template int launch_bwd_pair<_Float16, 256>(const BwdArgs &, int, int, const BwdArgs &, int, int, int64_t, bool, hipStream_t);
}  // namespace qfa
