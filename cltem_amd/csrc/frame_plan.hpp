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

// frame_slices for memory that may not be there: groups half as deep until try_alloc(slices) has
// room for one; 0 where there is none for a single slice
template <class TryAlloc>
int frame_slices_that_fit(int ns, int most, TryAlloc&& try_alloc) {
    for (int cs = frame_slices(ns, most);; cs = frame_slices(ns, cs / 2)) {
        if (try_alloc(cs)) return cs;
        if (cs == 1) return 0;
    }
}

}  // namespace mse_rt
