// Whether a step's captured graph takes the output head along (host code, decoder_step.hip).
#pragma once

#include "common.h"

namespace mynah {

// The head's pointers are part of the captured nodes, so a caller that hands over other rows for the results has the graph captured again: for
// every stream count and every form of the step (decoder_step.hip's Graphs) that steps with them.  One that does so at every step would
// have it captured at every step, and after kMost changes the head runs behind the graph instead.  What counts is the caller's
// change, once, however many forms have to be captured again for it: a batch that goes on through its forms is no further change.
struct HeadRows {
    static constexpr int kMost = 8;
    unsigned long long last[kMaxBatch + 1] = {};   // by stream count: the rows (and head) of its last step, 0 for none
    int changes = 0;
    bool in_graph() const { return changes < kMost; }
    void step(int count, unsigned long long signature) {
        if (last[count] != 0 && last[count] != signature) ++changes;
        last[count] = signature;
    }
};

}  // namespace mynah
