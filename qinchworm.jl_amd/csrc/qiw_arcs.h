// qiw_arcs.h -- open-arc graphs of the diagrams of an integration group, and their device
// programs for models with sector blocks (host only; no HIP).
//
// Summing the diagrams of a group one by one (src/topology_eval.jl:454-556 walks the pair
// assignments of every topology) repeats work: two partial diagrams that have reached the
// same position in the same sector with the same open arcs continue identically, whatever
// arcs they have closed on the way.  The compiler therefore walks the positions once and
// keeps one state per (sector, open arcs); the partial products of all partial diagrams in
// a state are added before they are continued.  What a closed arc leaves behind:
//   * its sign: a perfect matching's parity is (-1)^crossings, and an arc that closes
//     crosses exactly the arcs opened after it that are still open;
//   * connectedness (src/diagrammatics.jl:214-254): every arc has to be linked by crossings
//     to one that straddles the cut.  Before the cut the open arcs carry the partition into
//     linked components (closing an arc links it to all later open ones; a component with
//     no open arc left can no longer be linked: dead).  At the cut every open arc is
//     linked.  After it the linked arcs are a prefix of the open ones.
// At order 4 of the two-orbital model this takes 26 000 states where the assignment trie of
// the same group has more than a million nodes.
#pragma once
#include <algorithm>
#include <array>
#include <cstdint>
#include <cstring>
#include <string>
#include <unordered_map>
#include <vector>

namespace qiwi {

enum { ARC_BOLD = 0, ARC_BARE = 1, ARC_CORR = 2, ARC_SIGMA = 3 };  // = QIW_G_*
constexpr int kArcMax = 6;                                         // largest order

// Sector maps of a model (-1: the operator annihilates the sector).
struct ArcModel {
    int ns = 0, np = 0;
    std::vector<int> dims;
    std::vector<std::vector<int>> head_sf, tail_sf;  // [np][ns]: operators at an arc's earlier / later end
    std::vector<int> table;                          // [np] hybridization table
    std::vector<int> a_sf, b_sf;                     // correlator operators A (at tau_w) and B (at tau_i)
};

struct ArcState {
    uint8_t sector = 0, n = 0, good = 0;     // open arcs; the first `good` of them are linked across the cut
    std::array<uint8_t, kArcMax> comp{};     // components of the arcs after them
    std::array<uint8_t, kArcMax> pos{};      // point at which each arc opened
    std::array<uint16_t, kArcMax> pair{};
    bool operator==(const ArcState &o) const {
        return sector == o.sector && n == o.n && good == o.good && comp == o.comp && pos == o.pos && pair == o.pair;
    }
    bool operator<(const ArcState &o) const {
        if (sector != o.sector) return sector < o.sector;
        if (n != o.n) return n < o.n;
        if (pos != o.pos) return pos < o.pos;
        if (comp != o.comp) return comp < o.comp;
        if (good != o.good) return good < o.good;
        return pair < o.pair;
    }
};
struct ArcStateHash {
    size_t operator()(const ArcState &s) const {
        uint64_t h = 0x9E3779B97F4A7C15ull;
        auto mix = [&](uint64_t v) {
            h ^= v + 0x9E3779B97F4A7C15ull + (h << 6) + (h >> 2);
            h *= 0xBF58476D1CE4E5B9ull;
        };
        mix(s.sector | (s.n << 8) | (s.good << 16));
        for (int i = 0; i < s.n; ++i) mix(s.pos[i] | (s.pair[i] << 8) | ((uint64_t)s.comp[i] << 32));
        return (size_t)h;
    }
};

// What a position applies: nothing, the head or tail operator of a pair, or the operator A.
enum { ARC_ID = 0, ARC_HEAD = 1, ARC_TAIL = 2, ARC_A = 3 };
struct ArcJoin {
    int src, dst;
    uint16_t pair;
    uint8_t op;    // ARC_*
    int8_t sign;
    int8_t head;   // configuration position of the closed arc's head (ARC_TAIL)
};
struct ArcStage {
    int position;  // configuration position (1-based)
    std::vector<ArcJoin> joins;
};
// One initial sector of a group: levels[0] is the root (position 1), levels[i + 1] the
// states after stage i; the last level is the closed state (s0, no arcs).
struct ArcGraph {
    int s0 = 0;
    std::vector<std::vector<ArcState>> levels;
    std::vector<ArcStage> stages;
    double leaves = 0;  // complete diagrams (topology, pair assignment) summed by the graph
};

// fixed: pair of the first fixed.size() arcs opened (the sum over diagrams is cut into one
// graph per choice).  skip_w: leave out the stage of an identity node at tau_w between two
// points (its two propagators are multiplied beforehand).  Returns false when a diagram ends
// outside its initial sector; an empty graph (no stages, no levels) when there is none.
inline bool arc_graph(const ArcModel &m, int kind, int order, int n_after, int s0, const std::vector<int> &fixed,
                      bool skip_w, ArcGraph &out) {
    out = ArcGraph{};
    out.s0 = s0;
    const int np2 = 2 * order;
    const int cut = kind == ARC_BARE ? 0 : kind == ARC_SIGMA ? np2 - 1 : np2 - n_after;  // points before the cut
    const int at_w = kind == ARC_BARE ? -1 : kind == ARC_SIGMA ? np2 : np2 - n_after;    // points before tau_w
    ArcState root;
    root.sector = (uint8_t)s0;
    if (kind == ARC_CORR) {
        if (m.b_sf[s0] < 0) return true;
        root.sector = (uint8_t)m.b_sf[s0];
    }
    std::vector<std::vector<ArcState>> levels{{root}};
    std::vector<std::vector<double>> ways{{1.0}};
    std::vector<ArcStage> stages;
    std::unordered_map<ArcState, int, ArcStateHash> index;
    auto begin = [&](int position) {
        index.clear();
        stages.push_back(ArcStage{position, {}});
        levels.emplace_back();
        ways.emplace_back();
    };
    auto join = [&](int src, const ArcState &d, int op, int pair, int sign, int head) {
        auto it = index.emplace(d, (int)levels.back().size());
        if (it.second) {
            levels.back().push_back(d);
            ways.back().push_back(0.0);
        }
        const int dst = it.first->second;
        ways.back()[dst] += ways[ways.size() - 2][src];
        stages.back().joins.push_back(ArcJoin{src, dst, (uint16_t)pair, (uint8_t)op, (int8_t)sign, (int8_t)head});
    };
    auto linked = [&](ArcState &s) {  // every open arc is linked
        s.good = s.n;
        s.comp.fill(0);
    };
    auto w_node = [&](int position) {
        begin(position);
        const std::vector<ArcState> &src = levels[levels.size() - 2];
        for (int i = 0; i < (int)src.size(); ++i) {
            ArcState d = src[i];
            if (kind == ARC_CORR) {
                if (m.a_sf[d.sector] < 0) continue;
                d.sector = (uint8_t)m.a_sf[d.sector];
            }
            join(i, d, kind == ARC_CORR ? ARC_A : ARC_ID, 0, 1, 0);
        }
    };
    auto position_of = [&](int j) { return 2 + j + (at_w >= 0 && j >= at_w ? 1 : 0); };
    for (int j = 0; j < np2; ++j) {
        if (j == at_w && !skip_w) w_node(2 + at_w);
        begin(position_of(j));
        const std::vector<ArcState> src = levels[levels.size() - 2];
        const int rem = np2 - j;
        const bool all_linked = kind == ARC_BARE || j + 1 == cut;  // the new states stand at the cut
        for (int i = 0; i < (int)src.size(); ++i) {
            const ArcState &s = src[i];
            if (s.n + 1 <= rem - 1) {  // open an arc
                const int nth = (j + s.n) / 2;  // arcs opened so far
                for (int p = 0; p < m.np; ++p) {
                    const int t = m.head_sf[p][s.sector];
                    if (t < 0 || (nth < (int)fixed.size() && fixed[nth] != p)) continue;
                    ArcState d = s;
                    d.sector = (uint8_t)t;
                    d.pos[d.n] = (uint8_t)j;
                    d.pair[d.n] = (uint16_t)p;
                    d.comp[d.n] = d.n > d.good ? (uint8_t)(d.comp[d.n - 1] + 1) : (uint8_t)0;
                    ++d.n;
                    if (all_linked) linked(d);
                    join(i, d, ARC_HEAD, p, 1, 0);
                }
            }
            for (int a = 0; a < s.n; ++a) {  // close an arc
                const int p = s.pair[a], t = m.tail_sf[p][s.sector];
                if (t < 0) continue;
                ArcState d = s;
                d.sector = (uint8_t)t;
                const int own = s.comp[a];
                bool alive = true;
                if (a < s.good) {
                    linked(d);
                } else {  // the later arcs join its component, which must not end here
                    for (int q = a + 1; q < s.n; ++q) d.comp[q] = (uint8_t)own;
                    alive = a + 1 < s.n || (a > s.good && s.comp[a - 1] == own);
                }
                if (!alive) continue;
                for (int q = a; q + 1 < s.n; ++q) {
                    d.comp[q] = d.comp[q + 1];
                    d.pos[q] = d.pos[q + 1];
                    d.pair[q] = d.pair[q + 1];
                }
                --d.n;
                d.comp[d.n] = 0;
                d.pos[d.n] = 0;
                d.pair[d.n] = 0;
                if (a < s.good) {
                    d.good = d.n;
                } else {  // components numbered from 0 without gaps
                    int next = -1, last = -1;
                    for (int q = d.good; q < d.n; ++q) {
                        if (d.comp[q] != last) {
                            last = d.comp[q];
                            ++next;
                        }
                        d.comp[q] = (uint8_t)next;
                    }
                }
                if (all_linked) linked(d);
                join(i, d, ARC_TAIL, p, ((s.n - 1 - a) & 1) ? -1 : 1, position_of(s.pos[a]));
            }
        }
    }
    if (at_w == np2 && !skip_w) w_node(2 + at_w);
    // keep what reaches the closed state
    std::vector<char> alive(levels.back().size(), 0);
    for (size_t i = 0; i < alive.size(); ++i) {
        const ArcState &s = levels.back()[i];
        if (s.n != 0) continue;
        if (s.sector != s0) return false;
        alive[i] = 1;
        out.leaves += ways.back()[i];
    }
    if (out.leaves == 0) return true;
    for (int l = (int)stages.size(); l >= 0; --l) {
        std::vector<int> to(alive.size(), -1);
        std::vector<ArcState> kept;
        for (size_t i = 0; i < alive.size(); ++i)
            if (alive[i]) {
                to[i] = (int)kept.size();
                kept.push_back(levels[l][i]);
            }
        levels[l].swap(kept);
        if (l < (int)stages.size())
            for (ArcJoin &x : stages[l].joins) x.src = to[x.src];
        if (l == 0) break;
        std::vector<char> below(levels[l - 1].size(), 0);
        std::vector<ArcJoin> js;
        for (ArcJoin &x : stages[l - 1].joins)
            if (to[x.dst] >= 0) {
                below[x.src] = 1;
                x.dst = to[x.dst];
                js.push_back(x);
            }
        stages[l - 1].joins.swap(js);
        alive.swap(below);
    }
    out.levels.swap(levels);
    out.stages.swap(stages);
    return true;
}

// ---------------------------------------------------------------------------------------
// Device programs of the arc walk for sector blocks (k_eval_arcs_t)
// ---------------------------------------------------------------------------------------
// A workgroup evaluates one sample at a time: a lane holds one column of one state, the
// states of a level lie in LDS and the levels alternate between the two ends of one region.
// A tile is the work of one wavefront in a stage: up to 64 >> lg states of one sector, times
// 1 << lg columns of the initial sector's block.
//
// The program of a group is a blob of 32-bit words, offsets relative to its start:
//   group    0 segments, 1 arc values, 2 position of the left-out node at tau_w (0: none),
//            3 offset of the arc list, 4-7 byte offsets in LDS of the closed state's columns,
//            the arc values, the propagators and the states, 8.. offsets of the segments
//   arc      head position | tail position << 8 | table << 16
//   segment  0 s0 | m0 << 8 | lg << 16, 1 root sector dimension | stride << 8, 2 root operator
//            block (offset, ARC_NONE: identity), 3 root propagator offset (ARC_NONE: none, the
//            root is the closed state), 4 root state offset, 5 parts of the closed state, 6 offset
//            of their list, 7 where the closed state begins: a float64 array, its element
//            i at offset i of the states (so twice as far behind its beginning in bytes when
//            the states are float32), 8.. of each wavefront the offsets of its records and of its joins
// A wavefront reads two streams without a gap, in packets of ArcLayout::slots slots, so that
// all a packet needs is read while the one before it is at work.  A slot is one or two steps
// of joins, and what its flags say after them; the slots of a tile follow each other.
// Records, 8 words per slot:
//   0 flags, 1 rows | stride << 8 | stride of the source << 16 (a stride is the number of rows
//   that a product computes),
//   2 operator block (offset), 3 state offset, 4 propagator offset (ARC_NONE: none), 5 states,
//   6 (first slot of a packet) set when the packet has a second block of joins
// Joins: blocks of slots x (64 >> lg) words, the slots of a state side by side, one block per
// packet for the first steps and one for the second steps where a slot has one:
//   word     LDS byte address of the source state / 4 | index of the arc value << 20
// Offsets of states and propagators are in elements of the value type.  The arc values are
// 0: 0, 1: 1, then +v, -v of each arc in turn.  A state with fewer joins than its tile is
// filled up with value 0.
constexpr uint32_t ARC_NONE = 0xFFFFFFFFu;
// Flags of a slot: a barrier before it; the end of the segment; no joins; a second step; the
// product of the sum of joins with the block; the tile's end: propagator, store.  Without a
// product the next slot's joins continue the sum (float64; a float32 program has a product in
// every slot).
enum : uint32_t { ARC_BARRIER = 1, ARC_END = 2, ARC_IDLE = 4, ARC_SECOND = 8, ARC_TIMES = 16, ARC_STORE = 32 };
// LDS offsets: 16 times, the grid cells of 16 segments (24 bytes each), the arc values.
constexpr size_t kArcCellsAt = 128, kArcValuesAt = 512;
constexpr int kArcGroupHead = 8, kArcSegHead = 8, kArcSlotWords = 8;
constexpr int kArcTileOps = 28;          // most operators of a tile
constexpr int kArcReadAhead = 6 * 256;   // words a wavefront may read past its streams

// Slots of a packet of the walk whose lanes hold vectors of `rows` values.  The blocks of a packet
// and of the next one stay in registers: with more slots what spills costs more than the longer
// read-ahead saves (two-orbital step of orders 0:4, float32: 22.4, 21.1, 21.1 ms with four, three
// and two slots; three-orbital step of orders 0:3, float32: 31.7 and 31.1 ms with two and one; both
// while the sums over diagrams were float32).
constexpr int arc_slots(int rows) { return rows <= 8 ? 2 : 1; }

struct ArcLayout {
    int elem = 4;             // bytes of the value type
    int mmax = 1;             // largest sector block
    int bt = 0;               // elements of one segment's propagator blocks
    std::vector<int> bt_off;  // [ns]
    int waves = 1;            // wavefronts of the workgroup
    int slots = 4;            // slots of a packet
    size_t cap = 0;           // LDS bytes of the workgroup
};

// Elements a state of m rows takes per column, in a model whose largest block is mmax: fours
// (one 16-byte access) where a block is wider than 8, else pairs up to 6 (6 rows of 4 bytes
// keep the banks of neighbouring lanes apart).
inline int arc_stride(int m, int mmax) {
    return mmax > 8 || m > 6 ? (m + 3) & ~3 : m == 1 ? 1 : (m + 1) & ~1;
}

// LDS of a group in bytes: the times of the positions and cells of the segments, the arc
// values (float64), the closed states of all sectors, the propagators of n - 2 segments and one
// product, then the states (and at the end, in their place, the last propagator).
struct ArcLds {
    size_t fin, arcs, prop, states;
};
inline ArcLds arc_lds(const ArcLayout &l, int n, int n_arcs) {
    auto up = [](size_t b) { return (b + 15) & ~(size_t)15; };
    ArcLds r;
    r.arcs = kArcValuesAt;
    r.fin = r.arcs + up((size_t)(2 + 2 * n_arcs) * 8);
    r.prop = r.fin + up((size_t)l.bt * 8);
    r.states = r.prop + up((size_t)(n - 1) * l.bt * l.elem);
    return r;
}

struct ArcGroupProgram {
    std::vector<uint32_t> blob;
    int n_segments = 0;
    std::vector<double> seg_cost;  // real FLOPs per sample of each segment
    double flops = 0, leaves = 0, joins = 0;
    size_t lds = 0;  // bytes a workgroup needs
    int n_arcs = 0;
};

// Operator blocks as the packer names them: offset of the block of (op, pair, source sector).
struct ArcBlocks {
    std::vector<std::vector<uint32_t>> head, tail;  // [np][ns]
    std::vector<uint32_t> a, b;                     // [ns]
    uint32_t id = 0;                                // the identity
};

struct ArcPacker {
    const ArcModel &m;
    const ArcLayout &l;
    const ArcBlocks &ob;
    int kind, order, n_after, n, w_skipped;
    std::vector<uint32_t> arcs;  // arc list
    std::unordered_map<uint32_t, int> arc_id;

    uint32_t arc_value(int head, int tail, int table, int sign) {
        const uint32_t key = (uint32_t)head | ((uint32_t)tail << 8) | ((uint32_t)table << 16);
        auto it = arc_id.emplace(key, (int)arcs.size());
        if (it.second) arcs.push_back(key);
        return 2u + 2u * (uint32_t)it.first->second + (sign < 0 ? 1u : 0u);
    }
    // slot of the propagators that follow configuration position p: segment p + 1 (slots
    // 0 .. n - 3), or the product over the left-out node at tau_w (slot n - 2)
    int slot_after(int p) const { return w_skipped && p + 1 == w_skipped ? n - 2 : p - 1; }

    struct Tile {
        int sector;
        std::vector<int> states;  // indices in the level (one state `spread` times over)
        int spread = 1;           // the joins of a state are dealt over this many lanes
        std::vector<int> ops;     // keys (op << 16 | pair) this tile sums
        std::vector<int> steps;   // of each operator
    };

    struct Slot {
        std::array<uint32_t, kArcSlotWords> head{};
        std::vector<uint32_t> first, second;  // join words, one per state of the tile
        static Slot idle(uint32_t flags, int per) {
            Slot s;
            s.head[0] = flags;
            s.first.assign(per, 0u);
            return s;
        }
    };

    // States of a level in tiles, with the offsets of every state's parts.
    struct Placed {
        std::vector<Tile> tiles;
        std::vector<int> slots;  // of each tile
        std::vector<size_t> tile_off;
        std::vector<std::vector<size_t>> parts;  // [state] offsets
        size_t size = 0;

        std::vector<int> part_counts() const {
            std::vector<int> n;
            for (const auto &v : parts) n.push_back((int)v.size());
            return n;
        }
        // wavefronts of the tiles, longest first to the least loaded; returns the largest load
        double deal(int waves, std::vector<int> *wave) const {
            std::vector<int> ord(tiles.size());
            for (size_t i = 0; i < ord.size(); ++i) ord[i] = (int)i;
            std::stable_sort(ord.begin(), ord.end(), [&](int x, int y) { return slots[x] > slots[y]; });
            std::vector<double> load(waves, 0.0);
            if (wave) wave->assign(tiles.size(), 0);
            for (int i : ord) {
                const int w = (int)(std::min_element(load.begin(), load.end()) - load.begin());
                load[w] += kTileCost + slots[i];
                if (wave) (*wave)[i] = w;
            }
            return *std::max_element(load.begin(), load.end());
        }
    };
    static constexpr double kTileCost = 0.5, kStageCost = 2.0;  // propagator and store, barrier; in slots

    // The tiles of a stage before their operators are cut: n_src parts of each source state;
    // spread: deal the joins of the closed state over lanes.
    std::vector<Tile> tiles_of(const std::vector<ArcState> &lev, const ArcStage &st, int lg, const std::vector<int> &n_src,
                               bool spread, std::vector<std::vector<int>> &ops_of) const {
        const int per = 64 >> lg;
        ops_of.assign(lev.size(), {});
        for (const ArcJoin &x : st.joins) {
            const int key = (x.op << 16) | x.pair;
            auto &v = ops_of[x.dst];
            if (std::find(v.begin(), v.end(), key) == v.end()) v.push_back(key);
        }
        for (auto &v : ops_of) std::sort(v.begin(), v.end());
        // states opened at this position have one operator: tiles of one operator; the others
        // are tiled by sector
        std::vector<int> ord(lev.size());
        for (size_t i = 0; i < ord.size(); ++i) ord[i] = (int)i;
        auto head_key = [&](int i) {
            return ops_of[i].size() == 1 && (ops_of[i][0] >> 16) == ARC_HEAD ? ops_of[i][0] : -1;
        };
        std::sort(ord.begin(), ord.end(), [&](int x, int y) {
            if (lev[x].sector != lev[y].sector) return lev[x].sector < lev[y].sector;
            const int hx = head_key(x), hy = head_key(y);
            if (hx != hy) return hx < hy;
            return lev[x] < lev[y];
        });
        std::vector<Tile> tiles;
        for (size_t i = 0; i < ord.size();) {
            Tile t;
            t.sector = lev[ord[i]].sector;
            const int hk = head_key(ord[i]);
            while (i < ord.size() && (int)t.states.size() < per && lev[ord[i]].sector == t.sector &&
                   head_key(ord[i]) == hk)
                t.states.push_back(ord[i++]);
            for (int s : t.states)
                for (int key : ops_of[s])
                    if (std::find(t.ops.begin(), t.ops.end(), key) == t.ops.end()) t.ops.push_back(key);
            std::sort(t.ops.begin(), t.ops.end());
            tiles.push_back(t);
        }
        // joins of each state by operator: the steps of a tile's operator are the most of any
        std::vector<std::vector<int>> n_joins(lev.size());
        for (size_t i = 0; i < lev.size(); ++i) n_joins[i].assign(ops_of[i].size(), 0);
        for (const ArcJoin &x : st.joins) {
            const auto &v = ops_of[x.dst];
            const int key = (x.op << 16) | x.pair;
            n_joins[x.dst][std::lower_bound(v.begin(), v.end(), key) - v.begin()] += n_src[x.src];
        }
        for (Tile &t : tiles) {
            t.steps.assign(t.ops.size(), 0);
            for (int s : t.states)
                for (size_t k = 0; k < ops_of[s].size(); ++k) {
                    const size_t q = std::lower_bound(t.ops.begin(), t.ops.end(), ops_of[s][k]) - t.ops.begin();
                    t.steps[q] = std::max(t.steps[q], n_joins[s][k]);
                }
        }
        // the closed state alone leaves most lanes idle: deal its joins over lanes, each a part
        if (spread && lev.size() == 1)
            for (Tile &t : tiles) {
                const int most = *std::max_element(t.steps.begin(), t.steps.end());
                t.spread = std::min(std::min(per, 8), std::max(1, most / 3));
                t.states.assign(t.spread, 0);
                for (int &n : t.steps) n = (n + t.spread - 1) / t.spread;
            }
        return tiles;
    }

    // Cuts the operator sums of tiles longer than `target` slots (0: only those of too many
    // operators) into parts, each a tile of its own with its own copy of the states.
    Placed cut(const std::vector<Tile> &tiles, const std::vector<std::vector<int>> &ops_of, int lg, int target) const {
        Placed p;
        const int cg = 1 << lg;
        for (const Tile &t : tiles) {
            const int no = (int)t.ops.size();
            std::vector<int> upto(no + 1, 0);  // slots before an operator
            for (int i = 0; i < no; ++i) upto[i + 1] = upto[i] + (t.steps[i] + 1) / 2;
            const int k = std::min(no, std::max(target > 0 ? (upto[no] + target - 1) / target : 1,
                                                (no + kArcTileOps - 1) / kArcTileOps));
            for (int q = 0, from = 0; q < k; ++q) {
                int to = from + 1;  // an even share of the slots, an operator at least for each part left
                while (to < no - (k - 1 - q) && to - from < kArcTileOps &&
                       (q == k - 1 || 2 * (long long)upto[to] * k + (upto[to + 1] - upto[to]) * k <= 2LL * upto[no] * (q + 1)))
                    ++to;
                Tile c = t;
                c.ops.assign(t.ops.begin() + from, t.ops.begin() + to);
                c.steps.assign(t.steps.begin() + from, t.steps.begin() + to);
                p.slots.push_back(upto[to] - upto[from]);
                p.tiles.push_back(std::move(c));
                from = to;
                if (q == k - 1 && from < no) --q;  // what the operators' limit left over
            }
        }
        p.parts.assign(ops_of.size(), {});
        for (const Tile &t : p.tiles) {
            const size_t step = (size_t)arc_stride(m.dims[t.sector], l.mmax) * cg;
            p.size = (p.size + 3) & ~(size_t)3;
            p.tile_off.push_back(p.size);
            for (size_t i = 0; i < t.states.size(); ++i)  // a part without any of the state's joins is zero
                for (int key : t.ops)
                    if (std::binary_search(ops_of[t.states[i]].begin(), ops_of[t.states[i]].end(), key)) {
                        p.parts[t.states[i]].push_back(p.size + i * step);
                        break;
                    }
            p.size += t.states.size() * step;
        }
        p.size = (p.size + 3) & ~(size_t)3;
        return p;
    }

    struct Plan {
        std::vector<Placed> placed;  // [stage]
        size_t region = 0;           // elements of the state region, the closed state (float64) at its end
        size_t closed = 0;           // elements of the closed state
        double cost = 0;             // slots on the longest wavefronts, over all column passes
    };

    // Places the states of a graph at 1 << lg columns within `room` elements.  A stage lasts as
    // long as its longest wavefront: tiles are cut towards an even share as far as the parts
    // fit and the steps that they add to the next stage do not cost more.
    bool plan(const ArcGraph &g, int lg, size_t room, Plan &out) const {
        const int cg = 1 << lg, m0 = m.dims[g.s0], per = 64 >> lg;
        const size_t wide = 8 / l.elem;  // elements a value of the closed state takes
        out = Plan{};
        size_t prev = ((size_t)arc_stride(m.dims[g.levels[0][0].sector], l.mmax) * cg + 3) & ~(size_t)3, reg = prev;
        out.closed = prev;
        double c = kStageCost;
        std::vector<int> n_src{1};
        const size_t spare = 8 * (((size_t)arc_stride(m0, l.mmax) * cg + 3) & ~(size_t)3);
        for (size_t s = 0; s < g.stages.size(); ++s) {
            const bool last = s + 1 == g.stages.size();
            std::vector<double> uses(g.levels[s + 1].size(), 0.0);  // lanes' steps that read a state
            if (!last)
                for (const ArcJoin &x : g.stages[s + 1].joins) uses[x.src] += 1.0;
            Placed best;
            double best_cost = -1;
            for (int spread = 1; spread >= (last ? 0 : 1); --spread) {
                std::vector<std::vector<int>> ops_of;
                const std::vector<Tile> tiles = tiles_of(g.levels[s + 1], g.stages[s], lg, n_src, spread != 0, ops_of);
                int longest = 0, sum = 0;
                for (const Tile &t : tiles) {
                    int n = 0;
                    for (int k : t.steps) n += (k + 1) / 2;
                    longest = std::max(longest, n);
                    sum += n;
                }
                for (int target = std::max(1, sum / l.waves);; target += (target + 1) / 2) {
                    const bool uncut = target >= longest;
                    Placed p = cut(tiles, ops_of, lg, uncut ? 0 : target);
                    double cost = p.deal(l.waves, nullptr);
                    if (last)  // the parts are read one by one
                        cost += 0.05 * (double)p.parts[0].size();
                    else
                        for (size_t i = 0; i < uses.size(); ++i)
                            cost += ((double)p.parts[i].size() - 1.0) * uses[i] / (2.0 * per * l.waves);
                    const bool fits = last ? reg + wide * p.size <= room : prev + p.size + spare <= room;
                    if (fits && (best_cost < 0 || cost < best_cost)) {
                        best_cost = cost;
                        best = std::move(p);
                    }
                    if (uncut) break;
                }
                if (best_cost >= 0 && spread) break;
            }
            if (best_cost < 0) return false;
            n_src = best.part_counts();
            if (last)
                out.closed = best.size;
            else
                reg = std::max(reg, prev + best.size);
            prev = best.size;
            c += kStageCost + best.deal(l.waves, nullptr);
            out.placed.push_back(std::move(best));
        }
        out.region = reg + wide * out.closed;
        out.cost = c * ((m0 + cg - 1) / cg);
        return out.region <= room;
    }

    double graph_flops(const ArcGraph &g) const {
        const double m0 = m.dims[g.s0];
        const double mr = m.dims[g.levels[0][0].sector];
        double f = 2.0 * mr * mr * m0 + 2.0 * m0 * m0 * m0;
        for (size_t s = 0; s < g.stages.size(); ++s) {
            std::vector<uint64_t> seen;
            for (const ArcJoin &x : g.stages[s].joins) {
                if (x.op == ARC_TAIL) f += 2.0 * m.dims[g.levels[s][x.src].sector] * m0;
                const uint64_t key = ((uint64_t)x.dst << 20) | ((uint64_t)x.op << 16) | x.pair;
                if (x.op != ARC_ID) seen.push_back(key);
            }
            std::sort(seen.begin(), seen.end());
            seen.erase(std::unique(seen.begin(), seen.end()), seen.end());
            for (uint64_t key : seen) {
                const int op = (int)((key >> 16) & 15), pair = (int)(key & 0xFFFF);
                const int sd = g.levels[s + 1][key >> 20].sector;
                int ss = sd;  // the source sector the operator takes to sd
                for (int q = 0; q < m.ns; ++q) {
                    const int to = op == ARC_HEAD ? m.head_sf[pair][q] : op == ARC_TAIL ? m.tail_sf[pair][q] : m.a_sf[q];
                    if (to == sd) ss = q;
                }
                f += 2.0 * m.dims[ss] * m.dims[sd] * m0;
            }
            if (s + 1 < g.stages.size())
                for (const ArcState &d : g.levels[s + 1]) f += 2.0 * m.dims[d.sector] * m.dims[d.sector] * m0;
        }
        return f;
    }

    void emit(const ArcGraph &g, int lg, const Plan &pn, size_t states_at, ArcGroupProgram &out) {
        std::vector<uint32_t> &b = out.blob;
        while (b.size() % 64) b.push_back(0);
        out.blob[kArcGroupHead + out.n_segments] = (uint32_t)b.size();
        const size_t seg = b.size();
        const int m0 = m.dims[g.s0], s1 = g.levels[0][0].sector, per = 64 >> lg;
        const size_t n_st = g.stages.size();
        b.resize(seg + kArcSegHead + 2 * l.waves, 0u);
        b[seg] = (uint32_t)g.s0 | ((uint32_t)m0 << 8) | ((uint32_t)lg << 16);
        b[seg + 1] = (uint32_t)m.dims[s1] | ((uint32_t)arc_stride(m.dims[s1], l.mmax) << 8);
        b[seg + 2] = kind == ARC_CORR ? ob.b[g.s0] : ARC_NONE;
        // with no stage after it the root is the closed state, and its propagator the last one
        b[seg + 3] = n_st == 0 ? ARC_NONE : (uint32_t)(slot_after(1) * l.bt + l.bt_off[s1]);
        std::vector<std::vector<size_t>> src{{0}};
        std::vector<std::vector<Slot>> stream(l.waves);
        const size_t levels = pn.region - 8 / l.elem * pn.closed;  // elements of the alternating levels
        for (size_t s = 0; s < n_st; ++s) {
            const ArcStage &st = g.stages[s];
            const bool last = s + 1 == n_st;
            const Placed &p = pn.placed[s];
            // the levels alternate between the ends of their region, the closed state follows
            const size_t base = last ? levels : s % 2 == 0 ? levels - p.size : 0;
            std::vector<std::vector<size_t>> dst = p.parts;
            for (auto &v : dst)
                for (size_t &o : v) o += base;
            std::vector<std::vector<int>> by(g.levels[s + 1].size());  // joins by destination
            for (size_t i = 0; i < st.joins.size(); ++i) by[st.joins[i].dst].push_back((int)i);
            // records of the tiles
            std::vector<std::vector<Slot>> recs;
            for (size_t ti = 0; ti < p.tiles.size(); ++ti) {
                const Tile &t = p.tiles[ti];
                const int md = m.dims[t.sector], ns = (int)t.states.size();
                std::vector<Slot> r;
                for (size_t oi = 0; oi < t.ops.size(); ++oi) {
                    const int op = t.ops[oi] >> 16, pair = t.ops[oi] & 0xFFFF;
                    std::vector<std::vector<uint32_t>> words(ns);
                    int ssec = t.sector;
                    size_t most = 0;
                    for (int i = 0; i < ns; ++i) {
                        int dealt = 0;
                        for (int ji : by[t.states[i]]) {
                            const ArcJoin &x = st.joins[ji];
                            if (x.op != op || x.pair != pair) continue;
                            ssec = g.levels[s][x.src].sector;
                            const uint32_t v = op == ARC_TAIL
                                                   ? arc_value(x.head, st.position, m.table[pair], x.sign)
                                                   : 1u;
                            for (size_t off : src[x.src])
                                if (t.spread == 1 || dealt++ % t.spread == i)
                                    words[i].push_back((uint32_t)((states_at + off * l.elem) / 4) | (v << 20));
                        }
                        most = std::max(most, words[i].size());
                    }
                    uint32_t blk = ob.id;
                    if (op == ARC_HEAD) blk = ob.head[pair][ssec];
                    if (op == ARC_TAIL) blk = ob.tail[pair][ssec];
                    if (op == ARC_A) blk = ob.a[ssec];
                    const int ms = m.dims[ssec];
                    uint32_t any = 0;  // a source of the tile, for the fill words
                    for (int i = 0; i < ns; ++i)
                        if (!words[i].empty()) any = words[i][0] & 0xFFFFFu;
                    for (size_t e = 0; e < most; e += 2) {
                        Slot q;
                        q.head[1] = (uint32_t)md | ((uint32_t)arc_stride(md, l.mmax) << 8) |
                                    ((uint32_t)arc_stride(ms, l.mmax) << 16);
                        for (int i = 0; i < per; ++i)
                            q.first.push_back(i < ns && e < words[i].size() ? words[i][e] : any);
                        if (e + 1 < most) {
                            q.head[0] |= ARC_SECOND;
                            for (int i = 0; i < per; ++i)
                                q.second.push_back(i < ns && e + 1 < words[i].size() ? words[i][e + 1] : any);
                        }
                        if (e + 2 >= most || l.elem == 4) {
                            q.head[0] |= ARC_TIMES;
                            q.head[2] = blk;
                        }
                        r.push_back(std::move(q));
                    }
                    out.joins += (double)most * ns;
                }
                r.back().head[0] |= ARC_STORE;
                r.back().head[3] = (uint32_t)(base + p.tile_off[ti]);
                r.back().head[4] = last ? ARC_NONE : (uint32_t)(slot_after(st.position) * l.bt + l.bt_off[t.sector]);
                r.back().head[5] = (uint32_t)ns;
                recs.push_back(std::move(r));
            }
            // each wavefront's first slot of a stage waits for the barrier
            std::vector<int> wave;
            p.deal(l.waves, &wave);
            std::vector<char> begun(l.waves, 0);
            auto append = [&](int w, std::vector<Slot> r) {
                if (!begun[w]) r[0].head[0] |= ARC_BARRIER;
                begun[w] = 1;
                stream[w].insert(stream[w].end(), r.begin(), r.end());
            };
            for (size_t i = 0; i < recs.size(); ++i) append(wave[i], recs[i]);
            for (int w = 0; w < l.waves; ++w)
                if (!begun[w]) append(w, {Slot::idle(ARC_IDLE, per)});  // nothing to do in this stage
            src.swap(dst);
        }
        for (int w = 0; w < l.waves; ++w) {
            std::vector<Slot> &q = stream[w];
            const size_t at_end = q.size() / l.slots * l.slots;  // first slot of the last packet
            q.push_back(Slot::idle(ARC_BARRIER | ARC_END | ARC_IDLE, per));
            // a wavefront fetches the operator blocks of one packet more
            do q.push_back(Slot::idle(ARC_IDLE, per));
            while (q.size() % l.slots || (int)(q.size() - at_end) <= l.slots);
            std::vector<uint32_t> joins;
            while (b.size() % 64) b.push_back(0);
            b[seg + kArcSegHead + 2 * w] = (uint32_t)b.size();
            for (size_t i = 0; i < q.size(); i += l.slots) {
                bool second = false;
                for (int o = 0; o < l.slots; ++o) second = second || (q[i + o].head[0] & ARC_SECOND);
                q[i].head[6] = second;
                for (int o = 0; o < l.slots; ++o) b.insert(b.end(), q[i + o].head.begin(), q[i + o].head.end());
                for (int sl = 0; sl < per; ++sl)
                    for (int o = 0; o < l.slots; ++o) joins.push_back(q[i + o].first[sl]);
                for (int sl = 0; second && sl < per; ++sl)
                    for (int o = 0; o < l.slots; ++o)
                        joins.push_back(q[i + o].second.empty() ? 0u : q[i + o].second[sl]);
            }
            while (b.size() % 64) b.push_back(0);
            b[seg + kArcSegHead + 2 * w + 1] = (uint32_t)b.size();
            b.insert(b.end(), joins.begin(), joins.end());
        }
        if (n_st == 0) src[0][0] = levels;
        b[seg + 4] = n_st == 0 ? (uint32_t)levels : 0u;
        b[seg + 5] = (uint32_t)src[0].size();  // the parts of the closed state
        b[seg + 6] = (uint32_t)b.size();
        b[seg + 7] = (uint32_t)levels;
        for (size_t off : src[0]) b.push_back((uint32_t)off);
        out.n_segments++;
        const double f = graph_flops(g);
        out.seg_cost.push_back(f);
        out.flops += f;
        out.leaves += g.leaves;
    }
};

// Compiles a group: all initial sectors, cut by the pairs of the first n_fixed arcs.
// Returns 0, 1 when a diagram ends outside its initial sector, or 2 when the states do not
// fit the layout's LDS (or the word formats).
inline int arc_compile(const ArcModel &m, const ArcLayout &l, const ArcBlocks &ob, int kind, int order, int n_after,
                       int n_fixed, ArcGroupProgram &out) {
    out = ArcGroupProgram{};
    const int n = kind == ARC_BARE ? 2 * order + 2 : 2 * order + 3;
    const bool skip_w = kind == ARC_BOLD && order > 0;
    const int pos_w = kind == ARC_BARE ? 0 : 2 * order - n_after + 2;
    ArcPacker pk{m, l, ob, kind, order, n_after, n, skip_w ? pos_w : 0, {}, {}};
    std::vector<ArcGraph> graphs;
    std::vector<int> fix(std::min(n_fixed, order), 0);
    double total = 1;
    for (size_t i = 0; i < fix.size(); ++i) total *= m.np;
    for (int s0 = 0; s0 < m.ns; ++s0)
        for (double c = 0; c < total; ++c) {
            double r = c;
            for (size_t i = 0; i < fix.size(); ++i) {
                fix[i] = (int)((long long)r % m.np);
                r = (double)((long long)r / m.np);
            }
            ArcGraph g;
            if (!arc_graph(m, kind, order, n_after, s0, fix, skip_w, g)) return 1;
            if (!g.levels.empty()) graphs.push_back(std::move(g));
        }
    int n_tables = 0;  // (none in a model without pairs)
    for (int t : m.table) n_tables = std::max(n_tables, t + 1);
    const int most_arcs = order * (2 * order - 1) * n_tables;
    const ArcLds at = arc_lds(l, n, order > 0 ? most_arcs : 0);
    if (at.states + (size_t)l.bt * 8 > l.cap || 2 + 2 * most_arcs >= 4096) return 2;
    const size_t room = (l.cap - at.states) / l.elem;
    out.blob.assign(kArcGroupHead + graphs.size(), 0u);
    out.lds = at.states + (size_t)l.bt * 8;
    for (const ArcGraph &g : graphs) {
        int best = -1;
        ArcPacker::Plan plan, best_plan;
        for (int lg = 0; lg <= 5; ++lg) {
            if (lg > 0 && (1 << (lg - 1)) >= m.dims[g.s0]) break;
            if (!pk.plan(g, lg, room, plan)) break;
            if (best < 0 || plan.cost < best_plan.cost) {
                best = lg;
                best_plan = std::move(plan);
            }
        }
        if (best < 0) return 2;
        pk.emit(g, best, best_plan, at.states, out);
        out.lds = std::max(out.lds, at.states + best_plan.region * l.elem);
    }
    while (out.blob.size() % 4) out.blob.push_back(0);
    out.blob[0] = (uint32_t)out.n_segments;
    out.blob[1] = (uint32_t)pk.arcs.size();
    out.blob[2] = (uint32_t)pk.w_skipped;
    out.blob[3] = (uint32_t)out.blob.size();
    out.blob[4] = (uint32_t)at.fin;
    out.blob[5] = (uint32_t)at.arcs;
    out.blob[6] = (uint32_t)at.prop;
    out.blob[7] = (uint32_t)at.states;
    out.n_arcs = (int)pk.arcs.size();
    out.blob.insert(out.blob.end(), pk.arcs.begin(), pk.arcs.end());
    out.blob.resize(out.blob.size() + kArcReadAhead, 0u);
    return 0;
}

// ---------------------------------------------------------------------------------------
// Device programs of the scalar arc walk (all sectors 1x1; k_eval_sarcs_t)
// ---------------------------------------------------------------------------------------
// A lane holds one sample; a workgroup of kScalarWaves wavefronts shares 64 samples.  Per
// sample every factor of the diagrams is one row of a table in LDS: constants, arc values,
// and propagators per segment and sector.  Each wavefront runs its own program: a state is
// the sum over its joins (TERM words: accumulate source slot times a row), then its product
// with the propagator that follows (STORE: destination slot = accumulator times a row).  The
// states live in 64 registers slots, given out in the order a greedy schedule computes them
// (the state that frees most sources first), so order 4 of the single-orbital model needs
// 47 slots where its two widest neighbouring levels hold 120 states.
//   word     bits 0-7 twice the slot, 9-17 row, 31 set for all but a positive TERM, 30 set
//            for a negative TERM (clear: STORE)
// Slots 0-7 are the results (of initial sectors 0-7), slot 8 holds 1, slot 9 takes the padding.
// The program of a group is a blob of 32-bit words, offsets relative to its start:
//   0 constants, 1 their offset (float64 pairs; rows 0 ..), 2 arcs, 3 their offset,
//   4 propagators, 5 their offset, 6 scaled rows, 7 their offset, 8-11 program offsets of the
//   wavefronts, 12-15 their lengths in blocks of 16 words
//   arc      head | tail << 8, then the rows of tables 0, 1 and 2, 3 (16 bits each, 0xFFFF none)
//   prop     a pair of sectors s, s + 1 (s even; those with no state in either are left out):
//            row of s | s << 16 | 1 << 24 if s + 1 is a sector (the next row), segment | second
//            segment of a product << 8 (0: none)
//   scaled   row, source row, constant row
// A wavefront reads eight words past its program (zeros).
constexpr int kScalarWaves = 4, kScalarSlots = 64, kScalarFree = 10, kScalarRows = 300;
// Results that a wavefront stores, for n_out in use; rows of LDS before the times (the
// results take the place of the first rows), and with the times of the positions 0 .. n.
constexpr int scalar_out_rows(int n_out) { return n_out <= 2 ? 2 : n_out <= 4 ? 4 : 8; }
inline int scalar_table_rows(int rows, int n_out) { return std::max(rows, kScalarWaves * scalar_out_rows(n_out)); }
inline int scalar_lds_rows(int rows, int n_out, int n) { return scalar_table_rows(rows, n_out) + std::max(n + 1, n_out); }
constexpr uint32_t SARC_SPECIAL = 1u << 31, SARC_MINUS = 1u << 30;

// Operator matrix elements of a scalar model.
struct ArcValues {
    std::vector<std::vector<double>> head, tail;  // [np][ns]
    std::vector<double> a, b;                     // [ns]
};

struct ScalarProgram {
    std::vector<uint32_t> blob;
    double leaves = 0, words = 0;
    int rows = 0, slots = 0;  // LDS rows and register slots it needs
};

struct ScalarPacker {
    int kind, n, w_skipped;
    std::vector<double> consts{1.0};
    struct Arc {
        uint32_t ends;
        int row[4];
    };
    std::vector<Arc> arcs;
    struct Scaled {
        int row, src, c;
    };
    std::vector<Scaled> scaled;
    // rows are numbered by kind first and placed when all are known
    enum { R_CONST = 0, R_ARC = 1, R_PROP = 2, R_SCALED = 3 };
    struct Row {
        int kind, a, b;  // constant index | arc, table | slot, sector | scaled index
    };
    std::vector<Row> rows;
    std::unordered_map<uint64_t, int> row_id;
    int row(int k, int a, int b) {
        const uint64_t key = ((uint64_t)k << 48) | ((uint64_t)(uint32_t)a << 16) | (uint32_t)b;
        auto it = row_id.emplace(key, (int)rows.size());
        if (it.second) rows.push_back(Row{k, a, b});
        return it.first->second;
    }
    int const_row(double v) {
        size_t i = std::find(consts.begin(), consts.end(), v) - consts.begin();
        if (i == consts.size()) consts.push_back(v);
        return row(R_CONST, (int)i, 0);
    }
    int arc_row(int head, int tail, int table) {
        const uint32_t ends = (uint32_t)head | ((uint32_t)tail << 8);
        size_t i = 0;
        while (i < arcs.size() && arcs[i].ends != ends) ++i;
        if (i == arcs.size()) arcs.push_back(Arc{ends, {-1, -1, -1, -1}});
        return row(R_ARC, (int)i, table);
    }
    // segment index after position p as in ArcPacker (n - 2: the product), n - 1: the last
    int slot_after(int p) const { return w_skipped && p + 1 == w_skipped ? n - 2 : p + 1 == n ? n - 1 : p - 1; }

    struct Node {
        std::vector<int> src;
        std::vector<double> c;   // operator element and crossing sign
        std::vector<int> base;   // row the coefficient multiplies (-1: none)
        int prop, level;
    };
    struct Segment {
        std::vector<uint32_t> words;  // rows by id in bits 9..
        int result;                   // slot it adds to
    };

    // One initial sector: states in the greedy order, slots from the free list.  Returns
    // false when the states need more slots than there are.
    bool segment(const ArcModel &m, const ArcValues &val, const ArcGraph &g, int result, Segment &out) {
        std::vector<Node> node;
        std::vector<std::vector<int>> id(g.levels.size());
        for (size_t l = 0; l < g.levels.size(); ++l)
            for (size_t i = 0; i < g.levels[l].size(); ++i) {
                id[l].push_back((int)node.size());
                const int p = l == 0 ? 1 : g.stages[l - 1].position;
                const bool last = l + 1 == g.levels.size();
                Node x;
                x.level = (int)l;
                x.prop = row(R_PROP, last ? n - 1 : slot_after(p), g.levels[l][i].sector);
                node.push_back(x);
            }
        for (size_t s = 0; s < g.stages.size(); ++s)
            for (const ArcJoin &j : g.stages[s].joins) {
                const int ss = g.levels[s][j.src].sector;
                double c = j.sign;
                if (j.op == ARC_HEAD) c *= val.head[j.pair][ss];
                if (j.op == ARC_TAIL) c *= val.tail[j.pair][ss];
                if (j.op == ARC_A) c *= val.a[ss];
                Node &d = node[id[s + 1][j.dst]];
                d.src.push_back(id[s][j.src]);
                d.c.push_back(c);
                d.base.push_back(j.op == ARC_TAIL ? arc_row(j.head, g.stages[s].position, m.table[j.pair]) : -1);
            }
        const int N = (int)node.size();
        // sign of each state as it is kept: the majority of its joins become positive
        std::vector<double> sg(N, 1.0);
        for (int i = 1; i + 1 < N; ++i) {
            int plus = 0;
            for (size_t q = 0; q < node[i].src.size(); ++q) plus += node[i].c[q] * sg[node[i].src[q]] > 0 ? 1 : -1;
            if (plus < 0) sg[i] = -1.0;
        }
        std::vector<std::vector<int>> succ(N);
        std::vector<int> pending(N, 0), uses(N, 0), slot(N, -1);
        for (int i = 0; i < N; ++i) {
            std::vector<int> u(node[i].src);
            std::sort(u.begin(), u.end());
            u.erase(std::unique(u.begin(), u.end()), u.end());
            for (int p : u) {
                succ[p].push_back(i);
                ++uses[p];
            }
            pending[i] = (int)u.size();
        }
        std::vector<int> pool;
        for (int i = kScalarSlots - 1; i >= kScalarFree; --i) pool.push_back(i);
        auto put = [&](uint32_t flags, int sl, int r) {
            out.words.push_back(flags | ((uint32_t)r << 9) | (uint32_t)(2 * sl));
        };
        auto coef = [&](double c, int base) {  // row of |c| times a row (a constant row without one)
            c = c < 0 ? -c : c;
            if (base < 0) return const_row(c);
            if (c == 1.0) return base;
            const int cr = const_row(c);
            for (size_t i = 0; i < scaled.size(); ++i)
                if (scaled[i].src == base && scaled[i].c == cr) return scaled[i].row;
            const int r = row(R_SCALED, (int)scaled.size(), 0);
            scaled.push_back(Scaled{r, base, cr});
            return r;
        };
        auto store = [&](int i) {
            if (i + 1 == N) {  // the closed state
                slot[i] = result;
            } else {
                if (pool.empty()) return false;
                slot[i] = pool.back();
                pool.pop_back();
            }
            put(SARC_SPECIAL, slot[i], node[i].prop);
            return true;
        };
        const double b0 = kind == ARC_CORR ? val.b[g.s0] : 1.0;
        put(b0 < 0 ? SARC_SPECIAL | SARC_MINUS : 0u, 8, coef(b0, -1));
        if (!store(0)) return false;
        std::vector<int> ready;
        auto done = [&](int i) {
            for (int q : succ[i])
                if (--pending[q] == 0) ready.push_back(q);
        };
        done(0);
        while (!ready.empty()) {
            size_t best = 0;
            int bf = -1, bl = -1;
            for (size_t r = 0; r < ready.size(); ++r) {
                const Node &x = node[ready[r]];
                int f = 0;
                for (size_t q = 0; q < x.src.size(); ++q)
                    if (uses[x.src[q]] == 1 && std::find(x.src.begin(), x.src.begin() + q, x.src[q]) == x.src.begin() + q) ++f;
                if (f > bf || (f == bf && x.level > bl)) {
                    best = r;
                    bf = f;
                    bl = x.level;
                }
            }
            const int i = ready[best];
            ready.erase(ready.begin() + best);
            const Node &x = node[i];
            for (int neg = 0; neg < 2; ++neg)
                for (size_t q = 0; q < x.src.size(); ++q) {
                    const double c = x.c[q] * sg[x.src[q]] * sg[i];
                    if ((c < 0) != (neg == 1)) continue;
                    put(neg ? SARC_SPECIAL | SARC_MINUS : 0u, slot[x.src[q]], coef(c, x.base[q]));
                }
            for (size_t q = 0; q < x.src.size(); ++q)
                if (std::find(x.src.begin(), x.src.begin() + q, x.src[q]) == x.src.begin() + q && --uses[x.src[q]] == 0)
                    pool.push_back(slot[x.src[q]]);
            if (!store(i)) return false;
            done(i);
        }
        out.result = result;
        return true;
    }
};

// Compiles a scalar group.  models: one, whose results are its initial sectors, or several
// that differ in A and B alone (and their values), with one result each, the sum over the
// initial sectors (the trace): what they share is computed once.  max_words: cut the graphs by the
// pairs of their first arcs until a segment holds at most this many words (0: as few segments as
// fit).  Returns 0, 1 when a diagram ends outside its initial sector, or 2 when the program does
// not fit the slots, the rows or the tables of the walk.
inline int arc_compile_scalar(const std::vector<ArcModel> &models, const std::vector<ArcValues> &values, int kind, int order,
                              int n_after, int max_words, ScalarProgram &out) {
    out = ScalarProgram{};
    const ArcModel &m = models[0];
    const int n_models = (int)models.size();
    if (n_models > 8) return 2;
    const int n = kind == ARC_BARE ? 2 * order + 2 : 2 * order + 3;
    const bool skip_w = kind == ARC_BOLD && order > 0;
    const int pos_w = kind == ARC_BARE ? 0 : 2 * order - n_after + 2;
    if (m.ns > 8) return 2;
    for (int t : m.table)
        if (t > 3) return 2;
    for (int n_fixed = 0; n_fixed <= order; ++n_fixed) {
        ScalarPacker pk{kind, n, skip_w ? pos_w : 0};
        pk.const_row(1.0);
        std::vector<ScalarPacker::Segment> segs;
        double leaves = 0, total = 1;
        std::vector<int> fix(n_fixed, 0);
        for (int i = 0; i < n_fixed; ++i) total *= m.np;
        bool fits = total <= 4096;
        for (int ms = 0; ms < n_models * m.ns && fits; ++ms)
            for (double c = 0; c < total && fits; ++c) {
                const int im = ms / m.ns, s0 = ms % m.ns;
                long long r = (long long)c;
                for (int i = 0; i < n_fixed; ++i) {
                    fix[i] = (int)(r % m.np);
                    r /= m.np;
                }
                ArcGraph g;
                if (!arc_graph(models[im], kind, order, n_after, s0, fix, skip_w, g)) return 1;
                if (g.levels.empty()) continue;
                leaves += g.leaves;
                size_t states = 0;
                for (const auto &l : g.levels) states += l.size();
                ScalarPacker::Segment sg;
                if (states > 20000 || !pk.segment(models[im], values[im], g, n_models > 1 ? im : s0, sg))
                    fits = false;
                else
                    segs.push_back(std::move(sg));
            }
        if (!fits) continue;
        if (max_words > 0 && n_fixed < std::min(order, 2)) {
            size_t longest = 0;
            for (const auto &sg : segs) longest = std::max(longest, sg.words.size());
            if (longest > (size_t)max_words) continue;
        }
        if (pk.rows.size() + m.ns > (size_t)kScalarRows) return 2;
        // rows: constants, arcs, scaled rows, then the propagators by pairs of sectors
        std::vector<int> at(pk.rows.size(), -1);
        std::vector<std::array<int, 4>> prop_row(n + 1, std::array<int, 4>{-1, -1, -1, -1});
        int next = (int)pk.consts.size();
        for (size_t i = 0; i < pk.rows.size(); ++i) {
            const auto &r = pk.rows[i];
            if (r.kind == ScalarPacker::R_CONST) at[i] = r.a;
            if (r.kind == ScalarPacker::R_ARC) pk.arcs[r.a].row[r.b] = at[i] = next++;
            if (r.kind == ScalarPacker::R_SCALED) at[i] = next++;
        }
        for (size_t i = 0; i < pk.rows.size(); ++i) {
            const auto &r = pk.rows[i];
            if (r.kind != ScalarPacker::R_PROP) continue;
            int &pair = prop_row[r.a][r.b / 2];
            if (pair < 0) {
                pair = next;
                next += std::min(2, m.ns - r.b / 2 * 2);
            }
            at[i] = pair + r.b % 2;
        }
        if (next > kScalarRows) return 2;
        std::vector<uint32_t> &b = out.blob;
        b.assign(16, 0u);
        b[0] = (uint32_t)pk.consts.size();
        b[1] = (uint32_t)b.size();
        for (double v : pk.consts) {
            uint32_t w[2];
            std::memcpy(w, &v, 8);
            b.push_back(w[0]);
            b.push_back(w[1]);
        }
        b[2] = (uint32_t)pk.arcs.size();
        b[3] = (uint32_t)b.size();
        auto half = [](int r) { return r < 0 ? 0xFFFFu : (uint32_t)r; };
        for (const auto &a : pk.arcs) {
            b.push_back(a.ends);
            b.push_back(half(a.row[0]) | (half(a.row[1]) << 16));
            b.push_back(half(a.row[2]) | (half(a.row[3]) << 16));
        }
        b[5] = (uint32_t)b.size();
        for (int q = 0; q < n; ++q)
            for (int pair = 0; pair < 4; ++pair)
                if (prop_row[q][pair] >= 0) {
                    b[4]++;
                    b.push_back((uint32_t)prop_row[q][pair] | (uint32_t)(2 * pair) << 16 |
                                (2 * pair + 1 < m.ns ? 1u << 24 : 0u));
                    b.push_back((uint32_t)(q == n - 2 ? pos_w | (pos_w + 1) << 8 : q == n - 1 ? n : q + 2));
                }
        if (b[4] > 64) return 2;  // one record per lane
        b[6] = (uint32_t)pk.scaled.size();
        b[7] = (uint32_t)b.size();
        for (const auto &sc : pk.scaled) {
            b.push_back((uint32_t)at[sc.row]);
            b.push_back((uint32_t)at[sc.src]);
            b.push_back((uint32_t)at[sc.c]);
        }
        // segments to wavefronts, longest first to the least loaded
        std::vector<size_t> ord(segs.size());
        for (size_t i = 0; i < ord.size(); ++i) ord[i] = i;
        std::stable_sort(ord.begin(), ord.end(), [&](size_t x, size_t y) { return segs[x].words.size() > segs[y].words.size(); });
        std::vector<std::vector<uint32_t>> prog(kScalarWaves);
        std::vector<std::vector<char>> seen(kScalarWaves, std::vector<char>(8, 0));
        for (size_t i : ord) {
            int w = 0;
            for (int q = 1; q < kScalarWaves; ++q)
                if (prog[q].size() < prog[w].size()) w = q;
            std::vector<uint32_t> ws = segs[i].words;
            for (uint32_t &x : ws) x = (x & ~(0x1FFu << 9)) | ((uint32_t)at[(x >> 9) & 0x1FFu] << 9);
            const int s0 = segs[i].result;
            if (seen[w][s0]) {  // add to the result of this wavefront
                ws.back() = (ws.back() & ~0xFFu) | (2u * 9u);
                ws.push_back(2u * 9u);
                ws.push_back(2u * (uint32_t)s0);
                ws.push_back(SARC_SPECIAL | 2u * (uint32_t)s0);
            }
            seen[w][s0] = 1;
            prog[w].insert(prog[w].end(), ws.begin(), ws.end());
        }
        for (int w = 0; w < kScalarWaves; ++w) {
            out.words += (double)prog[w].size();
            while (b.size() % 16) b.push_back(0);
            while (prog[w].size() % 16) prog[w].push_back(SARC_SPECIAL | 2u * 9u);
            b[8 + w] = (uint32_t)b.size();
            b[12 + w] = (uint32_t)(prog[w].size() / 16);
            b.insert(b.end(), prog[w].begin(), prog[w].end());
            for (uint32_t x : prog[w]) out.slots = std::max(out.slots, (int)(x & 255u) / 2 + 1);
        }
        b.resize(b.size() + 16, 0u);  // zeros behind the last program; the others run into words or zeros
        out.leaves = leaves;
        out.rows = next;
        return 0;
    }
    return 2;
}

inline int arc_compile_scalar(const ArcModel &m, const ArcValues &val, int kind, int order, int n_after, int max_words,
                              ScalarProgram &out) {
    return arc_compile_scalar(std::vector<ArcModel>{m}, std::vector<ArcValues>{val}, kind, order, n_after, max_words, out);
}

}  // namespace qiwi
