// The work descriptor of a base conversion fused with its targets' column pass (conv_cols.h).
#pragma once

#include "arith.h"

namespace ckh {

// One target limb of a conversion. in: the first source limb; out: the converted polynomial (the
// target's limb of it is in the target table). The refs of one conversion are consecutive: ntgt of
// them from index first.
struct ConvColRef {
    const u64* in;
    u64* out;
    u32 first, ntgt;
    u32 src_first, tgt_first;
    u32 nsrc, small;  // small: every source below 2^50
};

}  // namespace ckh
