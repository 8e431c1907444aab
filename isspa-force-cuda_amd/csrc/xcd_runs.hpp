// The force pass's block table as eight contiguous runs, one an XCD.  Plain C++, with
// neither HIP types nor calls.
#pragma once

#include <algorithm>
#include <cstddef>
#include <utility>
#include <vector>

namespace isspa {

// Workgroup b of a launch goes to XCD b % 8 (round-robin).  The force table's entry of
// workgroup b is the (b / 8)-th of XCD b % 8's run, so the receiver blocks of one group
// of chunks share an L2 instead of being dealt to all eight.  Run x is (nb + 7 - x) / 8
// entries.  A bijection on [0, nb) for any nb.
constexpr int xcd_run_entry(int b, int nb)
{
    const int q = nb >> 3, r = nb & 7, x = b & 7, k = b >> 3;
    return x * q + (x < r ? x : r) + k;
}

// Deals the force blocks of a batch (work, {window .x, receivers .y, chunk group .z}),
// longest first, to the runs by whole chunk groups: the receiver blocks of a group read
// the same records, and an L2 that holds them serves them all.  In one list over all
// XCDs the 4 to 18 receiver blocks of a group went to as many L2s, which fetched its
// records each.  Solvent force of 256 x 1,100 atoms, nMC = 20, 9,042 -> 7,424 us (8,657
// with 5 blocks of 256 receivers), nMC = 5, 2,387 -> 2,017, 32 x 1,100, nMC = 20, 1,118
// -> 1,050, 4 x 1,100 172 -> 162, 80 x 220 232 -> 230; 64 umbrella windows 53 -> 51.
// Every run is longest first and exactly as long as xcd_run_entry has it.  While the
// runs were as long as their groups made them, those after an uneven one were read one
// to 17 entries off, so a longest block (55 points a share among blocks of 16) started
// last on an XCD: the force pass of 10 pairs, 34 chains and 12 lattices of 220 atoms
// took 32.3 us, 26.6 so and 26.2 in one list.
template <class Block>
void groups_to_xcds(std::vector<std::pair<long long, Block>> &blocks)
{
    using Entry = std::pair<long long, Block>;
    const std::size_t nb = blocks.size();
    std::vector<Entry> run[8], over;
    for (auto it = blocks.begin(); it != blocks.end();) {
        const auto end = std::find_if(it, blocks.end(), [it](const Entry &e) {
            return e.second.x != it->second.x || e.second.z != it->second.z;
        });
        auto *shortest = std::min_element(
            run, run + 8, [](const auto &a, const auto &b) { return a.size() < b.size(); });
        shortest->insert(shortest->end(), it, end);
        it = end;
    }
    // what a run has beyond its length, from its short end, fills the others
    auto length = [nb](int x) { return (nb + 7 - x) / 8; };
    for (int x = 0; x < 8; ++x)
        for (; run[x].size() > length(x); run[x].pop_back()) over.push_back(run[x].back());
    blocks.clear();
    for (int x = 0; x < 8; ++x) {
        for (; run[x].size() < length(x); over.pop_back()) run[x].push_back(over.back());
        std::stable_sort(run[x].begin(), run[x].end(),
                         [](const Entry &a, const Entry &b) { return a.first > b.first; });
        blocks.insert(blocks.end(), run[x].begin(), run[x].end());
    }
}

}  // namespace isspa
