// A sequence of short operations riding in a launch of the small-item GEMV or of learned matrices.
#pragma once

#include "sequence_ops.h"

namespace {

// In `side.n_chains` extra groups behind those of the GEMV a launch can run a sequence of
// short operations that touches nothing the launch touches (sequence_ops.h).
struct RowsSide {
    const NhipSeqOp* ops;
    SeqChains chains;
    int n_chains;
    int n_gemv_groups;
};

// what nhip_gemv_tile_carry armed for this thread, taken over by the launch at hand
__host__ inline bool take_carried(RowsSide& side) {
    side = RowsSide{};
    if (nhip_carried.n_chains <= 0) return false;
    side.ops = static_cast<const NhipSeqOp*>(nhip_carried.ops);
    for (int c = 0; c <= NHIP_SEQ_MAX_CHAINS; ++c) side.chains.first_op[c] = nhip_carried.first_op[c];
    for (int c = 0; c < NHIP_SEQ_MAX_CHAINS; ++c) side.chains.n_staged[c] = nhip_carried.n_staged[c];
    side.n_chains = nhip_carried.n_chains;
    nhip_carried = NhipCarried{};
    return true;
}

// A group behind the GEMV's, or (FIRST) one before them, runs its chain (uniform over the group).
// Launches of long rows take the chains first: their hundreds of groups are short, and a chain that is
// dispatched after them is what the launch waits for (1,024 rows of 1,000 with filters and a chain for
// vectors of 512 elements 7.0 us with the chains behind, 6.3 before; 1,200 rows 6.4 and 5.4).
#define NHIP_ROWS_SIDE_GROUP(side, FIRST)                                                   \
    if ((side).n_chains > 0 && ((FIRST) ? (int)blockIdx.x < (side).n_chains                 \
                                        : (int)blockIdx.x >= (side).n_gemv_groups)) {       \
        __shared__ NhipSeqOp s_ops[SEQ_MAX_OPS];                                             \
        __shared__ __attribute__((aligned(16))) int s_rows[SEQ_MAX_ROWS][SEQ_ROW_WORDS];     \
        const int c = blockIdx.x - ((FIRST) ? 0 : (side).n_gemv_groups);                     \
        sequence_chain((side).ops + (side).chains.first_op[c],                               \
                       (side).chains.first_op[c + 1] - (side).chains.first_op[c],            \
                       (side).chains.n_staged[c], s_ops, s_rows, threadIdx.x);               \
        return;                                                                              \
    }

}  // namespace
