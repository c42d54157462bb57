// How many slices' transmission functions the moving-frame scan builds at a time.  Host code only.
#pragma once
#include <algorithm>

namespace mse_rt {

// ns slices in as few groups of at most `most` as hold them, as even as they come: the slices of
// every group but the last
inline int frame_slices(int ns, int most) {
    most = std::max(1, most);
    const int groups = (ns + most - 1) / most;
    return (ns + groups - 1) / groups;
}

// slices of the group that starts at slice s
inline int frame_group(int ns, int cs, int s) { return std::min(cs, ns - s); }

}  // namespace mse_rt
