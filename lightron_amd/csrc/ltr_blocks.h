// Which (batch, kv head) pair, which of its tiles and which of the blocks of that tile a block of the bf16 kernels works on: the grid that the
// host launches (block_grid, pair_group) and the arithmetic that undoes it (block_item_at).  Plain C++, so that it can be checked on a CPU.
#pragma once
#include <algorithm>

#ifdef __HIP__
#define LTR_HOST_DEVICE __host__ __device__ __forceinline__
#else
#define LTR_HOST_DEVICE inline
#endif

struct BlockMap {      // see block_item_at
    int group;         // (batch, kv head) pairs of an XCD whose blocks are handed out together; 0: a linear grid
    int items;         // items (q tile slots, key tiles) per pair
    int groups;
    int inner;         // blocks per item
};

// Block (x, y, z) -> (pair = batch x kv head, item = q tile slot or key tile of the pair, sub = one of the `inner` blocks of an item).
// Consecutive blocks go to the 8 XCDs round-robin.  All blocks of a pair run on one XCD and next to each other in time, so the
// blocks that are resident together stream the same K / V (or Q / dO) through that XCD's L2; the inner blocks of an item follow each
// other.  The items of `group` pairs of an XCD are handed out item by item (the first of every pair, the second of every pair, ...):
// items come longest first, so blocks of unequal length end together (see pair_group).  The grid is (8 XCDs x inner blocks, pairs of a
// group, items of the groups): the hardware counts what would be four divisions (0.3 us of every block, also as multiplications: their
// constants are another trip to the arguments).
struct BlockItem {
    int pair, item, sub;
    int order;   // of the blocks of an XCD
};
LTR_HOST_DEVICE BlockItem block_item_at(const BlockMap &m, int pairs, unsigned x, unsigned y, unsigned z) {
    BlockItem r;
    if (m.group) {
        int g = 0;
        r.item = z;
        if (m.groups > 1) {
            g = r.item / m.items;
            r.item -= g * m.items;
        }
        r.sub = x >> 3;
        r.pair = (g * m.group + y) * 8 + (x & 7);   // past the last pair: a place of the last group that is empty
        r.order = r.sub + m.inner * (y + m.group * z);
    } else {   // pairs that do not divide among the XCDs: one block of every pair, then the next
        const int rest = x / pairs;
        r.pair = x - rest * pairs;
        r.item = rest / m.inner;
        r.sub = rest - r.item * m.inner;
        r.order = x >> 3;
    }
    return r;
}

// How many (batch, kv head) pairs of an XCD hand out their blocks together, longest first across them (block_item_at).  Pair after pair, every
// pair ends with its short blocks and the next one begins with long ones: the launch ends with long blocks running alone.  All
// pairs together, more K / V (or Q / dO) is in use than an L2 holds.  A group is taken as large as two rounds of the blocks that an XCD runs
// at once (`slots`), and equal blocks are left pair after pair.  Kernel us, one pair / 4 pairs / all pairs at a time:
//   dK/dV      B=8  8 kv heads of 32 D=128 causal S=1000   206 / 151 / 154 (8 pairs per XCD)    B=4 16 heads D=128 S=1024   67 / 50 / 51 (8)
//   dK/dV      B=8 32 heads D=128 causal S=2048   685 / 636 / 696 (32)     the same, S=512    94 / 75 / 80 (32)
//   dQ         B=4 12 heads D=64  causal S=2048    69 / 58 / 52 (6)        forward            58 / 48 / 42
//   dK/dV      B=4 32 heads D=128 S=8192 causal  4087 / 4069 / 4453 (16)   no mask          7473 / 7607 / 8515
// A small last group, of less than 1.4 rounds and 0.7 of the others, ends the launch with its own long blocks alone: larger groups are
// taken instead.  Kernel us with the small one / without:
//   dK/dV      B=2 12 heads D=96  causal S=4730   322 / 255 (2+1 pairs, 3)       B=13 8 heads D=96 S=3464   753 / 652 (4+4+4+1, 5+5+3)
//   dK/dV      B=10 8 kv heads of 32 D=64 S=7950  6293 / 5344 (4+4+2, 5+5)        B=8  8 kv heads of 32 D=128, 1306 of 2612 keys  309 / 262 (3+3+2, 4+4)
//   forward    B=5 16 heads D=64  causal S=6284   529 / 465 (4+4+2, 5+5)
inline int pair_group(long long pairs, long long blocks_per_pair, int slots, bool uneven) {
    if (!uneven || pairs % 8) return 1;
    const long long n = pairs / 8, want = std::max(1LL, (2LL * slots + blocks_per_pair - 1) / blocks_per_pair);
    for (long long groups = (n + want / 2) / want; groups > 1; groups--) {
        const long long group = (n + groups - 1) / groups, last = n - (n - 1) / group * group;
        if (last * 10 >= want * 7 || last * 10 >= group * 7) return (int)group;
    }
    return (int)n;
}

// The grid and its map; pairs x items x inner < 2^31 blocks.  The second and third dimension end at 65535: more items of groups than that
// (1024 pairs of 65536 keys in tiles of 128, 131072 pairs of 512) take larger groups, a pair with more items (8 million keys) a linear grid.
// dK/dV without a mask, all pairs block by block as the linear grid has them / groups of two, ms:
//   4096 x 32 heads S=512  D=64 27.0 / 24.2  D=128 52.8 / 48.4      32 x 32 heads D=128, 512 rows against 65600 keys 52.4 / 44.9
constexpr int GRID_YZ_MAX = 65535;
struct BlockGrid {
    BlockMap map;
    unsigned x, y, z;
};
inline BlockGrid block_grid(long long pairs, long long items, long long inner, long long group) {
    const long long per_xcd = pairs / 8;
    if (pairs % 8 == 0 && items > 0 && items <= GRID_YZ_MAX) {
        const long long most = GRID_YZ_MAX / items;   // groups
        group = std::max(group, (per_xcd + most - 1) / most);
        const long long groups = (per_xcd + group - 1) / group;
        if (group <= GRID_YZ_MAX) return {{(int)group, (int)items, (int)groups, (int)inner}, (unsigned)(8 * inner), (unsigned)group, (unsigned)(groups * items)};
    }
    return {{0, (int)items, 1, (int)inner}, (unsigned)(pairs * items * inner), 1, 1};
}

// Blocks of two kinds in one launch (bwd_joint_kernel): all blocks of one kind, each in its own order, then all of the other, on a linear grid.
// The hardware hands blocks out in that order, so the second kind fills the CUs that the first leaves idle, at its end and, where there are
// fewer blocks than CUs, from the start.
struct JointMap {
    unsigned first;    // blocks of the kind that goes first
    int keys_first;    // which that is: dK/dV, or dQ
};
LTR_HOST_DEVICE unsigned map_blocks(const BlockMap &m, int pairs) {   // places of a map, the empty ones of a last group among them
    return m.group ? 8u * m.inner * m.group * m.groups * m.items : (unsigned)pairs * m.items * m.inner;
}
struct JointItem {
    BlockItem item;
    bool keys;         // a dK/dV block
};
LTR_HOST_DEVICE JointItem joint_item_at(const JointMap &j, const BlockMap &q, const BlockMap &kv, int pairs, unsigned id) {
    const bool second = id >= j.first;   // the first kind has a multiple of 8 places where there are groups: the XCD stays id % 8
    if (second) id -= j.first;
    JointItem r;
    r.keys = second != (j.keys_first != 0);
    const BlockMap &m = r.keys ? kv : q;
    if (m.group) {
        const unsigned i = id >> 3, t = i / (unsigned)m.inner, z = t / (unsigned)m.group;
        r.item = block_item_at(m, pairs, (i - t * m.inner) << 3 | (id & 7), t - z * m.group, z);
    } else {
        r.item = block_item_at(m, pairs, id, 0, 0);
    }
    return r;
}

// Time of a launch whose blocks go, in this order, each to the slot (a CU's place for a block) that is free first: what the hardware's in-order
// dispatch comes to.  Blocks come as classes of equal length.  Slots that are free at the same time are counted together; to keep their
// list short, times that differ by less than 3 % of a block are the same.
struct BlockClass {
    double us;
    long long n;
};
struct Dispatch {
    static constexpr int MOST = 48;
    struct Run {
        double at;
        long long n;
    } place[2 * MOST], *run = place;   // slots by the time they are free; the list moves up in its place as runs leave at its front
    int runs = 1, slots;
    double end = 0;                    // of the last block
    explicit Dispatch(int slots_) : slots(slots_) { run[0] = {0, slots_}; }
    Dispatch(const Dispatch &o) : runs(o.runs), slots(o.slots), end(o.end) { std::copy(o.run, o.run + o.runs, place); }
    Dispatch &operator=(const Dispatch &) = delete;
    // more blocks, after those before them; false as soon as one of them ends at `most` or later: `end` is then less than it would have been
    bool add(const BlockClass *classes, int n_classes, double most = 1e300) {
        for (int c = 0; c < n_classes; c++) {
            const double us = classes[c].us, eps = std::max(0.3, 0.03 * us);
            long long left = classes[c].n;
            // whole rounds of equal blocks move all slots alike
            if (left >= 2LL * slots) {
                const long long rounds = left / slots - 1;
                for (int i = 0; i < runs; i++) run[i].at += rounds * us;
                end = std::max(end, run[runs - 1].at);
                left -= rounds * slots;
            }
            while (left > 0) {
                const long long n = std::min(left, run[0].n);
                const double at = run[0].at + us;
                left -= n;
                run[0].n -= n;
                if (run[0].n == 0) {
                    runs--;
                    run++;
                }
                end = std::max(end, at);
                int i = runs;   // the first run that is free at `at` or later: near the end, for the blocks of a launch are much alike
                while (i > 0 && run[i - 1].at >= at - eps) i--;
                if (i < runs && run[i].at <= at + eps) run[i].n += n;
                else if (runs == MOST) run[std::min(i, runs - 1)].n += n;
                else {
                    if (run + runs == place + 2 * MOST) {
                        std::copy(run, run + runs, place);
                        run = place;
                    }
                    for (int k = runs++; k > i; k--) run[k] = run[k - 1];
                    run[i] = {at, n};
                }
            }
            if (end >= most) return false;
        }
        return true;
    }
};
inline double launch_us(const BlockClass *classes, int n_classes, int slots) {
    Dispatch d(slots);
    d.add(classes, n_classes);
    return d.end;
}
