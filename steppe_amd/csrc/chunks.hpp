// steppe_amd/csrc/chunks.hpp — many items through workspaces of bounded size.
#pragma once

#include <cstddef>

namespace stp {

// Takes [0, n) in order in chunks of at most max_items items whose size(i) add up to at most
// budget (a chunk holds one item at least): reserve(i0, i1) makes room for a chunk, run(i0, i1)
// works on it.  Where reserve finds no room it returns false, and this and all later chunks
// are cut to at most half of its size; for a chunk of one item it throws instead.
template <class Size, class Reserve, class Run>
void for_chunks(std::size_t n, std::size_t max_items, std::size_t budget, Size&& size, Reserve&& reserve, Run&& run) {
    for (std::size_t i0 = 0; i0 < n;) {
        std::size_t i1 = i0, total = 0;
        while (i1 < n && (i1 == i0 || i1 - i0 < max_items)) {
            const std::size_t s = size(i1);
            if (i1 > i0 && total + s > budget) break;
            total += s;
            ++i1;
        }
        if (!reserve(i0, i1)) {
            budget = total / 2;
            max_items = (i1 - i0) / 2;
            continue;
        }
        run(i0, i1);
        i0 = i1;
    }
}

}  // namespace stp
