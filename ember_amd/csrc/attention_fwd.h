// attention_fwd.h -- what the forward's translation units share (not part of
// the public ABI).
#pragma once

#include <stdint.h>

namespace ember {

struct FwdArgs {
    const float *q, *k, *v;
    float *o, *lse;
    int H, S, nqb, nbh;
    float c;  // scale * log2(e)
    int64_t in_sb, in_sh, in_ss, out_sb, out_sh, out_ss;
};

// attention_fwd_tiles.hip: S > 64, one head's query blocks per workgroup.
int launch_fwd_tiles(const FwdArgs &args, int D, bool causal);

}  // namespace ember
