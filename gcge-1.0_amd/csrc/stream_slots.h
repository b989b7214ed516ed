// The block CG's calls that write columns and return sums of them.
#ifndef STREAM_SLOTS_H_
#define STREAM_SLOTS_H_

#include "gcge.h"

namespace gh {

struct StreamSlots {
    decltype(GCGE_OPS::MatDotMultiVecInnerProdDiag) MatDotMultiVecInnerProdDiag;
    decltype(GCGE_OPS::BlockCGResidualUpdate) BlockCGResidualUpdate;
    decltype(GCGE_OPS::BlockPCGResidualUpdate) BlockPCGResidualUpdate;
};

// The slots of `ops` for a caller that goes on with calls of the backend, which
// only queue their work: where a slot is the backend's own, a form that returns
// as soon as the host has the sums, with the columns complete for later calls but
// not yet for other streams.  A slot of the caller's own is returned as it is.
StreamSlots stream_slots(const GCGE_OPS *ops);

}  // namespace gh
#endif
