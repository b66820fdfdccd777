// The team split kernel (attention_team.h) at head_dim 96, scalar/AVX2 score order:
// XKV and plain BF16 instantiations for every query-row count.
#include "attention_team.h"

namespace kvexp_launch {
KVEXP_TEAM_UNIT(96, 0)
} // namespace kvexp_launch
