// Which of several timed candidates is taken (host code without dependencies).
#pragma once

namespace nt {

// `measured`: what the GPU takes for a launch of each candidate, in order of preference; `counted`: what the caller is
// charged for it, at least as much where its own pace or a reason against a candidate is counted in.  A later candidate replaces an earlier
// one if it counts for less by more than `margin` (a fraction), or counts for no more and is faster by more than
// `margin` on the GPU -- between candidates that the caller cannot tell apart the GPU's time decides, for callers that can.
// Returns its position, -1 of none.
inline int choose(const float *measured, const float *counted, int candidates, float margin) {
    int best = -1;
    for (int c = 0; c < candidates; ++c)
        if (best < 0 || counted[c] < counted[best] * (1.0f - margin) || (counted[c] <= counted[best] && measured[c] < measured[best] * (1.0f - margin))) best = c;
    return best;
}

}  // namespace nt
