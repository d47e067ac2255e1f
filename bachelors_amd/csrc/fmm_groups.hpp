#pragma once
#include "fmm_gemm.hpp"
#include "fmm_lists.hpp"

namespace fmm {

// Far pairs (t, s) with one target t and sources s that are children of one node: their M2L results
// are summed in the registers of the F16X3 M2L before they are stored.  Groups are sorted by group
// class (level difference and offset of the parent: equal class = equal operator for each child), then
// by the mask of the children that are far pairs of t, then by target.
struct GroupTile {
    int g0, ng;   // groups [g0, g0 + ng) of one class
    int cls;      // group class
    int mask;     // union of the groups' child masks
};
constexpr int GROUP_TILE = 42;   // groups per tile at most (single pairs: always): 126 of 128 columns

struct FarGroups {
    int num = 0, num_classes = 0, num_tiles = 0;
    bool single = false;             // every pair a group of its own, group class = far class
    DevBuf fc, mask;                 // per group: first child of the sources' parent, child mask
    DevBuf cls_ops, cls_mask;        // per group class: far class (operator) of child o at [8 c + o]; children in use
    DevBuf tiles;                    // GroupTile
    // scratch: pairs and groups in (target, parent) order, keys, scans
    DevBuf key, key2, val, perm, perm2, flag, pos, g_t, g_fc, g_mask, g_start, skey, skey2, code, flag2, pos2, cls_begin,
        tcount, toff, counts, tmp;
};

// Groups of the far pairs L (sorted by class; class_flag / class_pos: the class starts and their
// exclusive scan, so pair i has class class_pos[i] + class_flag[i] - 1), up to `tile` groups a tile, and the index of
// the groups by target node for reduce_pairs.  The host waits for the counts.  With fewer than min_pairs far pairs per
// class every pair is a group of its own (no counts, no waits).
void build_far_groups(FarGroups& G, PairIndex& ix, const Lists& L, const uint32_t* class_flag,
                      const uint32_t* class_pos, const TreeDev& S, const TreeDev& T, int min_pairs, int tile, hipStream_t st);

}  // namespace fmm
