// CPU check of a host part of libBaryTree_gpu.so that the C ABI does not show:
// the cover check of the near field's items.
// Test infrastructure only; compiled by tests/test_host_checks.py.
#include <vector>

#include "../barytree_amd/csrc/bt_host.h"
#include "../barytree_amd/csrc/bt_solver.h"

using namespace bt;

// check_items on two keys (targets 0..299 with ranges of 5 and 7 sources,
// targets 300..309 with none) and one more (310..319, 4 sources), whole and
// with one part missing or doubled.  Returns the number of the first case with
// the wrong verdict, 0 if none.
extern "C" int check_cover()
{
    WorkCSR near;
    near.key = {3, 4, 5};
    near.tbeg = {0, 300, 310};
    near.tcnt = {300, 10, 10};
    near.seg_off = {0, 2, 2, 3};
    near.seg_beg = {0, 5, 20};
    near.seg_cnt = {5, 7, 4};
    const std::vector<int> off = {0, 2, 2, 3};
    const std::vector<btk::Tile> tiles = {{0, 0, 256, 0}, {0, 256, 44, 0}, {2, 310, 10, 0}};
    const long long pairs = 300 * 12 + 10 * 4;
    if (!check_items(near, off, tiles, pairs).empty()) return 1;
    if (check_items(near, off, tiles, pairs - 10 * 4).empty()) return 2;               // an item's pairs missing
    if (check_items(near, {0, 1, 1, 2}, tiles, pairs).empty()) return 3;               // a slot missing
    if (check_items(near, off, {tiles[0], tiles[1]}, pairs).empty()) return 4;         // a key not reduced
    if (check_items(near, off, {tiles[0], tiles[2]}, pairs).empty()) return 5;         // targets left out
    if (check_items(near, off, {tiles[0], tiles[1], tiles[1], tiles[2]}, pairs).empty()) return 6;  // twice
    if (check_items(near, off, {tiles[0], tiles[1], {1, 300, 10, 0}, tiles[2]}, pairs).empty()) return 7;
    if (check_items(near, {0, 2, 2}, tiles, pairs).empty()) return 8;
    return 0;
}
