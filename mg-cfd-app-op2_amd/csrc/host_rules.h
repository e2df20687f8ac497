// Sizes the host derives for its copies and launches.  Plain C++ (no HIP), so
// that they can be checked without a GPU.
#pragma once

#include <algorithm>
#include <cstddef>

namespace mgcfd {

// Pinned landing buffers of fetches: kFetchSlots of kFetchBytes each.
constexpr int kFetchSlots = 8;
constexpr std::size_t kFetchBytes = 2u << 20;

// How a fetch of cnt elements of rec bytes goes through the buffers: pieces of
// 'rows' whole elements, one to a buffer at a time.  An element that fills
// more than a buffer does not (rows 0).
struct FetchPieces {
    int rows, pieces, slots;
};

inline FetchPieces fetch_pieces(std::size_t rec, int cnt)
{
    if (rec < 1 || rec > kFetchBytes || cnt < 1) return {0, 0, 0};
    const int rows = (int)(kFetchBytes / rec);
    const int pieces = (int)(((long long)cnt + rows - 1) / rows);
    return {rows, pieces, std::min(pieces, kFetchSlots)};
}

// Elements per launch of a loop with a thread for each of an element's five
// doubles: a launch takes fewer than 2^32 threads, so larger sets (from
// 858,993,459 elements) take several launches.
constexpr int kFlatElements = 1 << 29;

// f(first element, elements) for each launch; its first non-zero result ends it.
template <typename F>
int flat_launches(int n, F&& f)
{
    for (long long at = 0; at < n; at += kFlatElements)
        if (int rc = f((std::size_t)at, (int)std::min<long long>(kFlatElements, n - at))) return rc;
    return 0;
}

}  // namespace mgcfd
