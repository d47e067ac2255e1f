// Grouping of the far pairs for the F16X3 M2L (integer work, a few sorts; see fmm_groups.hpp).
//
// The M2L's traffic is its slab: one stored and re-read block per far pair (3 x 304 FP32 at p = 16).
// The traversal descends node by node, so a target usually meets several children of one source node
// as far pairs: 4.2 to 4.5 per (target, parent) on the benchmark's coils and clusters, and the slab
// shrinks by that factor when they are summed in the M2L's accumulators.  A tile runs over the union
// of its groups' children; sorting a class's groups by child mask keeps the union near each mask
// (0.82 to 0.91 of the products are of real pairs there, against 0.76 to 0.79 in target order).
#include "fmm_groups.hpp"
#include "fmm_prims.hpp"

namespace fmm {

static int bits_of(int n) {   // smallest b with 2^b >= n (at least 1)
    int b = 1;
    while (b < 31 && (1 << b) < n) b++;
    return b;
}

// sort key (target, parent of the source; num_nodes stands for "no parent") and value (pair) of a pair
__global__ void k_group_pair_keys(const int* __restrict__ far_t, const int* __restrict__ far_s,
                                  const int* __restrict__ parent, int n, int no_parent, int sbits,
                                  uint64_t* __restrict__ key, int* __restrict__ val) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const int p = parent[far_s[i]];
    key[i] = ((uint64_t)(uint32_t)far_t[i] << sbits) | (uint32_t)(p >= 0 ? p : no_parent);
    val[i] = i;
}
__global__ void k_group_flags(const uint64_t* __restrict__ key, int n, int shift, uint32_t* __restrict__ flag) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) flag[i] = (i == 0 || (key[i] >> shift) != (key[i - 1] >> shift)) ? 1u : 0u;
}
__global__ void k_group_total(const uint32_t* __restrict__ pos, const uint32_t* __restrict__ flag, int n,
                              unsigned* __restrict__ out) {
    *out = pos[n - 1] + flag[n - 1];
}
// pairs in (target, parent) order -> groups: target, first child, child mask, first pair.  A group's
// pairs (at most 8) are consecutive: the thread of its first pair reads them all.
__global__ void k_group_fill(const int* __restrict__ val, const uint32_t* __restrict__ flag,
                             const uint32_t* __restrict__ pos, int n, const int* __restrict__ far_t,
                             const int* __restrict__ far_s, const int* __restrict__ parent,
                             const int* __restrict__ first_child, int* __restrict__ g_t, int* __restrict__ g_fc,
                             int* __restrict__ g_mask, int* __restrict__ g_start) {
    const int k = blockIdx.x * blockDim.x + threadIdx.x;
    if (k >= n || !flag[k]) return;
    const int i = val[k], s = far_s[i], p = parent[s], fc = p >= 0 ? first_child[p] : s, g = (int)pos[k];
    int m = 1 << (s - fc);
    for (int e = k + 1; e < n && !flag[e]; e++) m |= 1 << (far_s[val[e]] - fc);
    g_t[g] = far_t[i];
    g_fc[g] = fc;
    g_mask[g] = m;
    g_start[g] = k;
}

// level difference and offset of the group's parent from its target, per axis in units of the finer
// of the children's and the target's half sizes (whole numbers: the pairs passed the lattice check)
struct HalfSizes {
    double h[MAX_LEVELS][3];
};
struct GroupOffset {
    int d;            // child level - target level
    long long n[3];
    bool root;        // the source is the tree's root (a group of its own, without a parent)
};
__device__ __forceinline__ GroupOffset group_offset(int t, int fc, const double* __restrict__ sc,
                                                    const double* __restrict__ tc, const int* __restrict__ sparent,
                                                    const int* __restrict__ slevel, const int* __restrict__ tlevel,
                                                    const HalfSizes& hs, const HalfSizes& ht) {
    GroupOffset o;
    const int p = sparent[fc], ls = slevel[fc], lt = tlevel[t];
    o.root = p < 0;
    o.d = ls - lt;
    for (int a = 0; a < 3; a++) {
        const double c = sc[3 * (o.root ? fc : p) + a] - tc[3 * t + a];
        o.n[a] = (long long)rint(c / fmin(hs.h[ls][a], ht.h[lt][a]));
    }
    return o;
}

// compact keys: root | level difference (6 bits) | 9 bits per axis | child mask (8 bits).  Pairs with
// offsets of at most 127 give parents of at most 127 + 127 / 2.6 (a child's offset from its parent is
// a half size of the child, and the acceptance keeps pairs at least 2.6 of those apart).
constexpr int COMPACT_AXIS = 9, COMPACT_BITS = 1 + 6 + 3 * COMPACT_AXIS + 8;
__global__ void k_group_keys(const int* __restrict__ g_t, const int* __restrict__ g_fc,
                             const int* __restrict__ g_mask, int ng, const double* __restrict__ sc,
                             const double* __restrict__ tc, const int* __restrict__ sparent,
                             const int* __restrict__ slevel, const int* __restrict__ tlevel, HalfSizes hs, HalfSizes ht,
                             uint64_t* __restrict__ key, int* __restrict__ val, unsigned* __restrict__ err) {
    const int g = blockIdx.x * blockDim.x + threadIdx.x;
    if (g >= ng) return;
    const GroupOffset o = group_offset(g_t[g], g_fc[g], sc, tc, sparent, slevel, tlevel, hs, ht);
    constexpr long long H = 1ll << (COMPACT_AXIS - 1);
    uint64_t code = ((uint64_t)(o.root ? 1 : 0) << 6) | (uint64_t)((o.d + 32) & 63);
    for (int a = 0; a < 3; a++) {
        if (o.n[a] < -H || o.n[a] >= H) atomicOr(err, 1u);
        code = (code << COMPACT_AXIS) | (uint64_t)((o.n[a] + H) & (2 * H - 1));
    }
    key[g] = (code << 8) | (uint64_t)g_mask[g];
    val[g] = g;
}
// wide keys (deep, strongly adaptive trees), two stable sorts: first (root, level difference, child
// mask), then 20 bits per axis
constexpr int WIDE_AXIS = 20;
__global__ void k_group_keys_wide(const int* __restrict__ g_t, const int* __restrict__ g_fc,
                                  const int* __restrict__ g_mask, int ng, const double* __restrict__ sc,
                                  const double* __restrict__ tc, const int* __restrict__ sparent,
                                  const int* __restrict__ slevel, const int* __restrict__ tlevel, HalfSizes hs,
                                  HalfSizes ht, uint32_t* __restrict__ skey, uint64_t* __restrict__ code,
                                  int* __restrict__ val, unsigned* __restrict__ err) {
    const int g = blockIdx.x * blockDim.x + threadIdx.x;
    if (g >= ng) return;
    const GroupOffset o = group_offset(g_t[g], g_fc[g], sc, tc, sparent, slevel, tlevel, hs, ht);
    constexpr long long H = 1ll << (WIDE_AXIS - 1);
    uint64_t c = 0;
    for (int a = 0; a < 3; a++) {
        if (o.n[a] < -H || o.n[a] >= H) atomicOr(err, 1u);
        c = (c << WIDE_AXIS) | (uint64_t)((o.n[a] + H) & (2 * H - 1));
    }
    skey[g] = ((uint32_t)(o.root ? 1 : 0) << 14) | ((uint32_t)((o.d + 32) & 63) << 8) | (uint32_t)g_mask[g];
    code[g] = c;
    val[g] = g;
}
__global__ void k_group_gather_code(const uint64_t* __restrict__ code, const int* __restrict__ perm, int ng,
                                    uint64_t* __restrict__ out) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < ng) out[i] = code[perm[i]];
}
__global__ void k_group_flags_wide(const uint64_t* __restrict__ code, const uint32_t* __restrict__ skey,
                                   const int* __restrict__ perm, int ng, uint32_t* __restrict__ flag) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= ng) return;
    flag[i] = (i == 0 || code[i] != code[i - 1] || (skey[perm[i]] >> 8) != (skey[perm[i - 1]] >> 8)) ? 1u : 0u;
}

// groups into class order; order[g] = the place of group g of the (target, parent) order.  The first
// group of each run of equal class and mask also enters its children into the class: their far class
// (operator), equal for all pairs of the (group class, child).
__global__ void k_group_place(const int* __restrict__ perm, const uint32_t* __restrict__ flag,
                              const uint32_t* __restrict__ pos, int ng, const int* __restrict__ g_fc,
                              const int* __restrict__ g_mask, const int* __restrict__ g_start,
                              const int* __restrict__ val, const int* __restrict__ far_s,
                              const uint32_t* __restrict__ class_flag, const uint32_t* __restrict__ class_pos,
                              int* __restrict__ fc, int* __restrict__ mask, int* __restrict__ order,
                              int* __restrict__ cls_begin, int* __restrict__ cls_mask, int* __restrict__ cls_ops) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= ng) return;
    const int g = perm[i], c = (int)(pos[i] + flag[i]) - 1, m = g_mask[g], f = g_fc[g];
    fc[i] = f;
    mask[i] = m;
    order[g] = i;
    if (flag[i]) cls_begin[c] = i;
    if (i == ng - 1) cls_begin[c + 1] = ng;
    if (!flag[i] && g_mask[perm[i - 1]] == m) return;
    atomicOr(cls_mask + c, m);   // commutative: the result does not depend on the order
    const int k0 = g_start[g];
    for (int e = 0; e < __popc(m); e++) {
        const int q = val[k0 + e];
        cls_ops[8 * (size_t)c + (far_s[q] - f)] = (int)(class_pos[q] + class_flag[q]) - 1;
    }
}
// tiles per class (0 beyond the last class, so the scan's last entry is their number)
__global__ void k_group_tile_counts(const int* __restrict__ cls_begin, const uint32_t* __restrict__ pos,
                                    const uint32_t* __restrict__ flag, int ng, int tile,
                                    uint32_t* __restrict__ count) {
    const int c = blockIdx.x * blockDim.x + threadIdx.x;
    if (c > ng) return;
    const int nc = (int)(pos[ng - 1] + flag[ng - 1]);
    count[c] = c < nc ? (uint32_t)(cls_begin[c + 1] - cls_begin[c] + tile - 1) / tile : 0u;
}
__global__ void k_group_tiles(const int* __restrict__ mask, const uint32_t* __restrict__ pos,
                              const uint32_t* __restrict__ flag, const int* __restrict__ cls_begin,
                              const uint32_t* __restrict__ toff, int ng, int tile, GroupTile* __restrict__ tiles,
                              unsigned* __restrict__ counts) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= ng) return;
    const int c = (int)(pos[i] + flag[i]) - 1, b = cls_begin[c], e = cls_begin[c + 1];
    if (i == 0) {
        counts[1] = pos[ng - 1] + flag[ng - 1];
        counts[2] = toff[ng];
    }
    if ((i - b) % tile) return;
    GroupTile t{i, min(tile, e - i), c, 0};
    for (int j = 0; j < t.ng; j++) t.mask |= mask[i + j];
    tiles[toff[c] + (i - b) / tile] = t;
}

// every pair a group of its own (child 0 of its source), in class order as the pairs are
__global__ void k_single_groups(const int* __restrict__ far_s, const uint32_t* __restrict__ class_flag,
                                const uint32_t* __restrict__ class_pos, int n, int* __restrict__ fc,
                                int* __restrict__ mask, int* __restrict__ cls_begin, int* __restrict__ cls_mask,
                                int* __restrict__ cls_ops) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const int c = (int)(class_pos[i] + class_flag[i]) - 1;
    fc[i] = far_s[i];
    mask[i] = 1;
    if (class_flag[i]) {
        cls_begin[c] = i;
        cls_mask[c] = 1;
        cls_ops[8 * (size_t)c] = c;
    }
    if (i == n - 1) cls_begin[c + 1] = n;
}

static HalfSizes half_sizes(const TreeDev& T) {
    HalfSizes h;
    for (int k = 0; k < MAX_LEVELS; k++)
        for (int a = 0; a < 3; a++) h.h[k][a] = T.half[k][a];
    return h;
}

void build_far_groups(FarGroups& G, PairIndex& ix, const Lists& L, const uint32_t* class_flag,
                      const uint32_t* class_pos, const TreeDev& S, const TreeDev& T, int min_pairs, int tile, hipStream_t st) {
    const int n = L.num_far;
    G.num = G.num_classes = G.num_tiles = 0;
    G.single = false;
    if (!n) {
        build_pair_index(nullptr, 0, T.num_nodes, ix, st);
        return;
    }
    if (n < (long long)min_pairs * L.num_classes) {
        uint32_t *tcount = G.tcount.get<uint32_t>(n + 1), *toff = G.toff.get<uint32_t>(n + 1);
        int *fc = G.fc.get<int>(n), *mask = G.mask.get<int>(n), *cb = G.cls_begin.get<int>(n + 1);
        const int nc = L.num_classes;
        k_single_groups<<<blocks(n), 256, 0, st>>>(L.far_s.as<int>(), class_flag, class_pos, n, fc, mask, cb,
                                                   G.cls_mask.get<int>(nc), G.cls_ops.get<int>(8 * (size_t)nc));
        k_group_tile_counts<<<blocks(n + 1), 256, 0, st>>>(cb, class_pos, class_flag, n, GROUP_TILE, tcount);
        exclusive_scan_u32(tcount, toff, n + 1, G.tmp, st);
        k_group_tiles<<<blocks(n), 256, 0, st>>>(mask, class_pos, class_flag, cb, toff, n, GROUP_TILE, G.tiles.get<GroupTile>(n),
                                                 G.counts.get<unsigned>(4));
        build_pair_index(L.far_t.as<int>(), n, T.num_nodes, ix, st);
        FMM_HIP(hipGetLastError());
        G.num = n;
        G.num_classes = nc;
        G.single = true;
        for (int c = 0; c < nc; c++) G.num_tiles += ceil_div(L.h_class_begin[c + 1] - L.h_class_begin[c], GROUP_TILE);
        return;
    }
    const int sb = bits_of(S.num_nodes + 1), tb = bits_of(T.num_nodes);
    const int *ft = L.far_t.as<int>(), *fs = L.far_s.as<int>(), *par = S.parent.as<int>();
    uint64_t *key = G.key.get<uint64_t>(n), *key2 = G.key2.get<uint64_t>(n);
    int *val0 = G.perm.get<int>(n), *val = G.val.get<int>(n);
    unsigned* counts = G.counts.get<unsigned>(4);   // groups, classes, tiles, range error
    FMM_HIP(hipMemsetAsync(counts, 0, 4 * sizeof(unsigned), st));
    k_group_pair_keys<<<blocks(n), 256, 0, st>>>(ft, fs, par, n, S.num_nodes, sb, key, val0);
    sort_pairs_u64(key, key2, val0, val, n, tb + sb, G.tmp, st);
    uint32_t *flag = G.flag.get<uint32_t>(n), *pos = G.pos.get<uint32_t>(n);
    k_group_flags<<<blocks(n), 256, 0, st>>>(key2, n, 0, flag);
    exclusive_scan_u32(flag, pos, n, G.tmp, st);
    k_group_total<<<1, 1, 0, st>>>(pos, flag, n, counts);
    unsigned hc[4];
    FMM_HIP(hipMemcpyAsync(hc, counts, sizeof(unsigned), hipMemcpyDeviceToHost, st));
    FMM_HIP(hipStreamSynchronize(st));
    const int ng = (int)hc[0];
    int *g_t = G.g_t.get<int>(ng), *g_fc = G.g_fc.get<int>(ng), *g_mask = G.g_mask.get<int>(ng);
    int* g_start = G.g_start.get<int>(ng);
    k_group_fill<<<blocks(n), 256, 0, st>>>(val, flag, pos, n, ft, fs, par, S.first_child.as<int>(), g_t, g_fc, g_mask,
                                             g_start);
    // class order
    int *perm = G.perm.as<int>(), *perm2 = G.perm2.get<int>(ng);   // n >= ng
    uint32_t *flag2 = G.flag2.get<uint32_t>(ng), *pos2 = G.pos2.get<uint32_t>(ng);
    const HalfSizes hs = half_sizes(S), ht = half_sizes(T);
    const double *sc = S.center.as<double>(), *tc = T.center.as<double>();
    const int *sl = S.level.as<int>(), *tl = T.level.as<int>();
    if (!L.wide) {
        k_group_keys<<<blocks(ng), 256, 0, st>>>(g_t, g_fc, g_mask, ng, sc, tc, par, sl, tl, hs, ht, key, perm, counts + 3);
        sort_pairs_u64(key, key2, perm, perm2, ng, COMPACT_BITS, G.tmp, st);
        k_group_flags<<<blocks(ng), 256, 0, st>>>(key2, ng, 8, flag2);
    } else {
        uint32_t *skey = G.skey.get<uint32_t>(ng), *skey2 = G.skey2.get<uint32_t>(ng);
        uint64_t* code = G.code.get<uint64_t>(ng);
        k_group_keys_wide<<<blocks(ng), 256, 0, st>>>(g_t, g_fc, g_mask, ng, sc, tc, par, sl, tl, hs, ht, skey, code, perm2,
                                                      counts + 3);
        sort_pairs_u32(skey, skey2, perm2, perm, ng, 15, G.tmp, st);
        k_group_gather_code<<<blocks(ng), 256, 0, st>>>(code, perm, ng, key);
        sort_pairs_u64(key, key2, perm, perm2, ng, 3 * WIDE_AXIS, G.tmp, st);
        k_group_flags_wide<<<blocks(ng), 256, 0, st>>>(key2, skey, perm2, ng, flag2);
    }
    exclusive_scan_u32(flag2, pos2, ng, G.tmp, st);
    int *fc = G.fc.get<int>(ng), *mask = G.mask.get<int>(ng);
    int *cb = G.cls_begin.get<int>(ng + 1), *cm = G.cls_mask.get<int>(ng), *ops = G.cls_ops.get<int>(8 * (size_t)ng);
    int* order = ix.order.get<int>(ng);
    FMM_HIP(hipMemsetAsync(cm, 0, ng * sizeof(int), st));
    k_group_place<<<blocks(ng), 256, 0, st>>>(perm2, flag2, pos2, ng, g_fc, g_mask, g_start, val, fs, class_flag, class_pos,
                                              fc, mask, order, cb, cm, ops);
    uint32_t *tcount = G.tcount.get<uint32_t>(ng + 1), *toff = G.toff.get<uint32_t>(ng + 1);
    k_group_tile_counts<<<blocks(ng + 1), 256, 0, st>>>(cb, pos2, flag2, ng, tile, tcount);
    exclusive_scan_u32(tcount, toff, ng + 1, G.tmp, st);
    k_group_tiles<<<blocks(ng), 256, 0, st>>>(mask, pos2, flag2, cb, toff, ng, tile, G.tiles.get<GroupTile>(ng), counts);
    // the groups of a target are consecutive in (target, parent) order
    index_sorted_pairs(g_t, ng, T.num_nodes, ix, st);
    FMM_HIP(hipGetLastError());
    FMM_HIP(hipMemcpyAsync(hc, counts, 4 * sizeof(unsigned), hipMemcpyDeviceToHost, st));
    FMM_HIP(hipStreamSynchronize(st));
    if (hc[3]) throw Error(4, "far-pair group offset out of the range of its key");
    G.num = ng;
    G.num_classes = (int)hc[1];
    G.num_tiles = (int)hc[2];
}

}  // namespace fmm
