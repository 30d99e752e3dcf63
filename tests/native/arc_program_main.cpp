// Runs the block-sector programs of qiw_arcs.h on the CPU, word for word as the arc walk
// reads them, with every access checked, against the plain sum over topologies and pair
// assignments.  Arguments: kind order n_after n_fixed waves cap_bytes elem modes seed [largest block, 5].
// The model: `modes` fermionic modes, one sector per particle number with random dimensions,
// random operator blocks, propagators and arc values.  elem 0: the scalar program (blocks 1x1;
// n_fixed > 0: cut into as many segments as it can be).  Prints the largest deviation relative
// to the largest element, and the count of diagrams of the program and of the plain sum.
#include <cmath>
#include <cstdio>
#include <cstdlib>
#include <functional>
#include <map>
#include <random>

#include "qiw_arcs.h"

using namespace qiwi;

static std::mt19937_64 rng;
static double rnd() { return std::uniform_real_distribution<double>(-1.0, 1.0)(rng); }
static void die(const char *what) {
    std::printf("FAIL %s\n", what);
    std::exit(1);
}

typedef std::vector<std::pair<int, int>> Pairs;
struct Topo {
    Pairs p;
    int parity;
};
static void gen(Pairs &part, int parity, std::vector<int> open, std::vector<Topo> &out) {
    if (open.empty()) {
        out.push_back({part, parity});
        return;
    }
    for (size_t i = 1; i < open.size(); ++i) {
        std::vector<int> rest;
        for (size_t q = 1; q < open.size(); ++q)
            if (q != i) rest.push_back(open[q]);
        part.push_back({open[0], open[i]});
        gen(part, i % 2 ? parity : -parity, rest, out);
        part.pop_back();
    }
}
static bool connected(const Pairs &t, int k) {
    Pairs stack, rest;
    for (auto &p : t) ((p.first <= k && p.second > k) ? stack : rest).push_back(p);
    while (!stack.empty()) {
        auto c = stack.back();
        stack.pop_back();
        for (size_t i = rest.size(); i-- > 0;) {
            auto a = c, b = rest[i];
            if (a.first > b.first) std::swap(a, b);
            if (a.second > b.first && a.second < b.second) {
                stack.push_back(rest[i]);
                rest.erase(rest.begin() + i);
            }
        }
    }
    return rest.empty();
}

int main(int argc, char **argv) {
    if (argc < 10) return 2;
    const int kind = std::atoi(argv[1]), order = std::atoi(argv[2]), n_after = std::atoi(argv[3]);
    const int n_fixed = std::atoi(argv[4]), waves = std::atoi(argv[5]), cap = std::atoi(argv[6]);
    const int elem = std::atoi(argv[7]), modes = std::atoi(argv[8]);
    rng.seed(std::atoi(argv[9]));
    const int most = argc > 10 ? std::atoi(argv[10]) : 5;
    ArcModel m;
    m.ns = modes + 1;
    m.np = 2 * modes;
    for (int s = 0; s < m.ns; ++s) m.dims.push_back(1 + (int)(rng() % most));
    if (modes > 1) m.dims[1] = 1;
    std::vector<int> off(m.ns + 1, 0);
    for (int s = 0; s < m.ns; ++s) off[s + 1] = off[s] + m.dims[s] * m.dims[s];
    ArcLayout l;
    l.elem = elem;
    l.mmax = *std::max_element(m.dims.begin(), m.dims.end());
    l.bt = off[m.ns];
    l.bt_off.assign(off.begin(), off.end() - 1);
    l.waves = waves;
    l.slots = arc_slots(l.mmax <= 8 ? 8 : l.mmax <= 20 ? 20 : 32);
    l.cap = cap;
    std::vector<std::vector<double>> blocks;  // operator blocks, named by index
    std::vector<std::pair<int, int>> shape;
    ArcBlocks ob;
    auto block = [&](int from, int to) -> uint32_t {
        if (to < 0) return ARC_NONE;
        std::vector<double> v(m.dims[to] * m.dims[from]);
        for (double &x : v) x = rnd();
        blocks.push_back(v);
        shape.push_back({m.dims[to], m.dims[from]});
        return (uint32_t)blocks.size() - 1;
    };
    ob.id = 1u << 30;
    for (int p = 0; p < m.np; ++p) {
        std::vector<int> h, t;
        std::vector<uint32_t> hb, tb;
        for (int s = 0; s < m.ns; ++s) {
            const int up = s + 1 < m.ns ? s + 1 : -1, dn = s - 1;
            h.push_back(p % 2 ? up : dn);
            t.push_back(p % 2 ? dn : up);
            hb.push_back(block(s, h.back()));
            tb.push_back(block(s, t.back()));
        }
        m.head_sf.push_back(h);
        m.tail_sf.push_back(t);
        ob.head.push_back(hb);
        ob.tail.push_back(tb);
        m.table.push_back(p % 2);
    }
    for (int s = 0; s < m.ns; ++s) {
        m.a_sf.push_back(s - 1);
        m.b_sf.push_back(s + 1 < m.ns ? s + 1 : -1);
        ob.a.push_back(block(s, m.a_sf[s]));
        ob.b.push_back(block(s, m.b_sf[s]));
    }
    const int n = kind == ARC_BARE ? 2 * order + 2 : 2 * order + 3;
    std::vector<std::vector<double>> prop(n + 1, std::vector<double>(l.bt));  // segment L
    for (auto &v : prop)
        for (double &x : v) x = rnd();
    std::map<uint32_t, double> arcs;
    auto arc = [&](int head, int tail, int tab) {
        const uint32_t k = (uint32_t)head | ((uint32_t)tail << 8) | ((uint32_t)tab << 16);
        auto it = arcs.find(k);
        if (it == arcs.end()) it = arcs.emplace(k, rnd()).first;
        return it->second;
    };

    std::vector<double> res(l.bt, 0.0), ref(l.bt, 0.0);
    ArcGroupProgram pg;
    if (elem == 0) {  // the scalar program (all blocks 1x1), read as the scalar walk reads it
        ArcValues val;
        auto pick = [&](const std::vector<uint32_t> &v) {
            std::vector<double> x;
            for (uint32_t b : v) x.push_back(b == ARC_NONE ? 0.0 : blocks[b][0]);
            return x;
        };
        for (int p = 0; p < m.np; ++p) {
            val.head.push_back(pick(ob.head[p]));
            val.tail.push_back(pick(ob.tail[p]));
        }
        val.a = pick(ob.a);
        val.b = pick(ob.b);
        ScalarProgram sp;
        const int rc = arc_compile_scalar(m, val, kind, order, n_after, n_fixed ? 1 : 0, sp);
        if (rc) {
            std::printf("rc %d\n", rc);
            return 0;
        }
        auto run = [&](const ScalarProgram &sp) {  // the results of its slots 0 .. 7
        std::array<double, 8> out{};
        const std::vector<uint32_t> &b = sp.blob;
        auto at = [&](size_t i) -> uint32_t {
            if (i >= b.size()) die("word out of the program");
            return b[i];
        };
        if (sp.rows > 300) die("rows");
        std::vector<double> tab(sp.rows, NAN);
        auto set = [&](uint32_t r, double v) {
            if (r >= tab.size() || !std::isnan(tab[r])) die("row");
            tab[r] = v;
        };
        for (uint32_t i = 0; i < at(0); ++i) {
            const uint32_t w[2] = {at(at(1) + 2 * i), at(at(1) + 2 * i + 1)};
            double v;
            std::memcpy(&v, w, 8);
            set(i, v);
        }
        for (uint32_t i = 0; i < at(2); ++i)
            for (int q = 0; q < 4; ++q) {
                const uint32_t r = (at(at(3) + 3 * i + 1 + q / 2) >> (16 * (q & 1))) & 0xFFFF;
                const uint32_t e = at(at(3) + 3 * i);
                if (r != 0xFFFF) set(r, arc(e & 255, e >> 8, q));
            }
        for (uint32_t i = 0; i < at(4); ++i) {
            const uint32_t r = at(at(5) + 2 * i), seg = at(at(5) + 2 * i + 1), L = seg & 255, L2 = seg >> 8;
            const int s = (int)((r >> 16) & 255);
            if (L < 2 || L > (uint32_t)n || L2 > (uint32_t)n || s % 2 || s + (int)(r >> 24) >= m.ns || i >= 64) die("segment");
            for (int q = 0; q <= (int)(r >> 24); ++q) set((r & 0xFFFF) + q, prop[L][s + q] * (L2 ? prop[L2][s + q] : 1.0));
        }
        for (uint32_t i = 0; i < at(6); ++i)
            set(at(at(7) + 3 * i), tab.at(at(at(7) + 3 * i + 1)) * tab.at(at(at(7) + 3 * i + 2)));
        for (int w = 0; w < kScalarWaves; ++w) {
            if (at(8 + w) % 16 && at(12 + w)) die("program alignment");
            std::vector<double> slot(kScalarSlots, NAN);
            for (int s = 0; s < 8; ++s) slot[s] = 0.0;
            slot[8] = 1.0;
            slot[9] = 0.0;
            double acc = 0.0;
            for (uint32_t i = 0; i < 16 * at(12 + w); ++i) {
                const uint32_t x = at(at(8 + w) + i), sl = (x & 255) / 2, r = (x >> 9) & 511;
                if ((x & 1) || (x & 256) || sl >= (uint32_t)sp.slots || sp.slots > kScalarSlots || r >= tab.size() || std::isnan(tab[r])) die("word");
                if ((x & SARC_SPECIAL) && !(x & SARC_MINUS)) {
                    if (sl == 8) die("the constant slot is written");
                    slot[sl] = acc * tab[r];
                    acc = 0.0;
                } else {
                    if (std::isnan(slot[sl])) die("slot read before it is written");
                    acc += (x & SARC_SPECIAL ? -1.0 : 1.0) * slot[sl] * tab[r];
                }
            }
            for (int s = 0; s < 8; ++s) out[s] += slot[s];
            for (uint32_t i = 0; i < 8; ++i)  // words read ahead, the rows of the first four too
                if (((at(at(8 + w) + 16 * at(12 + w) + i) >> 9) & 511) >= tab.size()) die("row read ahead");
        }
        return out;
        };
        const std::array<double, 8> single = run(sp);
        for (int s = 0; s < m.ns; ++s) res[s] += single[s];
        if (kind == ARC_CORR) {  // with the operators' roles exchanged too: both traces in one program
            std::vector<ArcModel> models{m, m};
            std::vector<ArcValues> values{val, val};
            std::swap(models[1].a_sf, models[1].b_sf);
            std::swap(values[1].a, values[1].b);
            ScalarProgram both, other;
            if (arc_compile_scalar(models, values, kind, order, n_after, n_fixed ? 1 : 0, both) ||
                arc_compile_scalar(models[1], values[1], kind, order, n_after, n_fixed ? 1 : 0, other))
                die("programs of two pairs");
            const std::array<double, 8> o = run(other), t = run(both);
            double t0 = 0, t1 = 0, size = 1e-300;
            for (int s = 0; s < m.ns; ++s) {
                t0 += single[s];
                t1 += o[s];
                size += std::fabs(single[s]) + std::fabs(o[s]);
            }
            if (!(std::fabs(t0 - t[0]) < 1e-9 * size && std::fabs(t1 - t[1]) < 1e-9 * size)) die("traces of two pairs");
        }
        pg.leaves = sp.leaves;
        pg.n_segments = (int)sp.words;
        pg.lds = (size_t)sp.rows * 512;
    } else {
    // ---- the program ----
    const int rc = arc_compile(m, l, ob, kind, order, n_after, n_fixed, pg);
    if (rc) {
        std::printf("rc %d\n", rc);
        return 0;
    }
    const std::vector<uint32_t> &b = pg.blob;
    auto at = [&](size_t i) -> uint32_t {
        if (i >= b.size()) die("word out of the program");
        return b[i];
    };
    const size_t region = (pg.lds - at(7)) / elem;
    if (pg.lds > l.cap) die("more LDS than the cap");
    if (at(5) != kArcValuesAt || at(4) % 16 || at(6) % 16 || at(7) % 16) die("alignment");
    const size_t dv_size = (at(4) - at(5)) / elem, prop_size = (at(7) - at(6)) / elem;
    std::vector<double> dv(2 + 2 * at(1));
    if (dv.size() > dv_size) die("arc values");
    dv[1] = 1.0;
    for (uint32_t i = 0; i < at(1); ++i) {
        const uint32_t a = at(at(3) + i);
        dv[2 + 2 * i] = arc(a & 255, (a >> 8) & 255, a >> 16);
        dv[3 + 2 * i] = -dv[2 + 2 * i];
    }
    std::vector<double> pl((size_t)(n - 1) * l.bt, NAN);
    if (pl.size() > prop_size) die("propagators");
    for (int L = 2; L < n; ++L) std::copy(prop[L].begin(), prop[L].end(), pl.begin() + (size_t)(L - 2) * l.bt);
    if (at(2))
        for (int s = 0; s < m.ns; ++s)
            for (int i = 0; i < m.dims[s]; ++i)
                for (int j = 0; j < m.dims[s]; ++j) {
                    double v = 0;
                    for (int q = 0; q < m.dims[s]; ++q)
                        v += prop[at(2) + 1][off[s] + i + q * m.dims[s]] * prop[at(2)][off[s] + q + j * m.dims[s]];
                    pl[(size_t)(n - 2) * l.bt + off[s] + i + j * m.dims[s]] = v;
                }
    for (uint32_t sg = 0; sg < at(0); ++sg) {
        const size_t h = at(kArcGroupHead + sg);
        const int s0 = at(h) & 255, m0 = (at(h) >> 8) & 255, lg = at(h) >> 16, cg = 1 << lg;
        if (m0 != m.dims[s0]) die("m0");
        for (int c0 = 0; c0 < m0; c0 += cg) {
            std::vector<double> st(region, NAN);
            auto get = [&](size_t i) -> double {
                if (i >= st.size()) die("state read out of the region");
                return st[i];
            };
            auto put = [&](size_t i, double v) {
                if (i >= st.size()) die("state write out of the region");
                st[i] = v;
            };
            auto times = [&](size_t po, int mm, const std::vector<double> &x) {
                std::vector<double> y(mm, 0.0);
                for (int i = 0; i < mm; ++i)
                    for (int q = 0; q < mm; ++q) {
                        if (po + i + q * mm >= pl.size()) die("propagator read");
                        y[i] += pl[po + i + q * mm] * x[q];
                    }
                return y;
            };
            const int m1 = at(h + 1) & 255, str1 = at(h + 1) >> 8, per = 64 >> lg;
            for (int col = 0; col < cg; ++col) {
                std::vector<double> x(m1, 0.0);
                for (int k = 0; k < m1; ++k)
                    if (c0 + col < m0)
                        x[k] = at(h + 2) == ARC_NONE ? (k == c0 + col) : blocks.at(at(h + 2)).at((c0 + col) * m1 + k);
                if (at(h + 3) != ARC_NONE) x = times(at(h + 3), m1, x);
                for (int k = 0; k < str1; ++k) put(at(h + 4) + col * str1 + k, k < m1 ? x[k] : 0.0);
            }
            int stf = str1;
            // of each wavefront: slot and block of joins it has come to
            std::vector<size_t> pos(waves, 0), joins(waves), packet(waves, ~(size_t)0), second(waves, 0);
            std::vector<std::vector<std::vector<double>>> acc(waves), y(waves);  // per lane
            for (int w = 0; w < waves; ++w) {
                joins[w] = at(h + kArcSegHead + 2 * w + 1);
                if (at(h + kArcSegHead + 2 * w) % 64 || joins[w] % 64) die("stream alignment");
                acc[w].assign(64, {});
                y[w].assign(64, {});
            }
            const size_t block = (size_t)l.slots * per;  // words of a block of joins
            for (bool more = true; more;) {  // a stage: every wavefront's slots up to its next barrier
                std::vector<std::pair<size_t, double>> writes;
                std::vector<std::pair<size_t, int>> reads;
                for (int w = 0; w < waves; ++w) {
                    for (bool first = true;; first = false) {
                        const size_t rec = at(h + kArcSegHead + 2 * w), pk = pos[w] / l.slots, o = pos[w] % l.slots;
                        const size_t r = rec + kArcSlotWords * pos[w];
                        if (packet[w] != pk) {
                            if (packet[w] != ~(size_t)0) joins[w] += (1 + second[w]) * block;
                            packet[w] = pk;
                            second[w] = at(rec + kArcSlotWords * l.slots * pk + 6);
                            if (second[w] > 1) die("packet");
                        }
                        const uint32_t fl = at(r);
                        if (first != ((fl & ARC_BARRIER) != 0)) {
                            if (first) die("no barrier at a stage");
                            break;
                        }
                        if (fl & ARC_END) {
                            if (w > 0 && more) die("wavefronts end apart");
                            more = false;
                            // what the wavefront reads ahead: two packets of records, one of joins
                            (void)at(rec + kArcSlotWords * l.slots * (pk + 2) + 63);
                            for (int i = 0; i < l.slots; ++i)  // blocks are fetched one packet ahead
                                if (at(rec + kArcSlotWords * (l.slots * (pk + 1) + i)) & ARC_TIMES) die("block past the end");
                            (void)at(joins[w] + 4 * block - 1);
                            break;
                        }
                        if (!more) die("wavefronts end apart");
                        pos[w]++;
                        if (fl & ARC_IDLE) continue;
                        const int rows = at(r + 1) & 255, str = (at(r + 1) >> 8) & 255, ss = at(r + 1) >> 16;
                        const int ns = at(r + 5);
                        if (str != arc_stride(rows, l.mmax)) die("stride");
                        if ((fl & ARC_SECOND) && !second[w]) die("no second steps");
                        if ((fl & ARC_STORE) && !(fl & ARC_TIMES)) die("sum left over");
                        for (int lane = 0; lane < 64; ++lane) {
                            const int col = lane & (cg - 1), sl = lane >> lg;
                            std::vector<double> &v = y[w][lane], &x = acc[w][lane];
                            if (v.empty()) v.assign(ss, 0.0);
                            if ((int)v.size() != ss) die("continued sum");
                            for (int e = 0; e < (fl & ARC_SECOND ? 2 : 1); ++e) {
                                const uint32_t q = at(joins[w] + e * block + sl * l.slots + o);
                                for (int k = 0; k < ss; ++k) {  // the walk reads whole strides
                                    const size_t byte = (q & 0xFFFF) * 4;
                                    if ((q & 0xF0000) || byte < at(7) || (byte - at(7)) % elem) die("state address");
                                    const size_t i = (byte - at(7)) / elem + col * ss + k;
                                    const double sv = get(i);
                                    if (std::isnan(sv)) die("state read before it is written");
                                    reads.push_back({i, 0});
                                    v[k] += dv.at(q >> 20) * sv;
                                }
                            }
                            if (x.empty()) x.assign(rows, 0.0);
                            if ((int)x.size() != rows) die("rows of a tile");
                            if (fl & ARC_TIMES) {
                                const uint32_t blk = at(r + 2);
                                if (blk == ob.id) {
                                    if (ss != str) die("identity");
                                    for (int k = 0; k < ss; ++k)
                                        if (k < rows) x[k] += v[k];
                                } else {
                                    const int ms = shape.at(blk).second;
                                    if (shape[blk].first != rows || arc_stride(ms, l.mmax) != ss) die("operator shape");
                                    for (int k = 0; k < ms; ++k)
                                        for (int i = 0; i < rows; ++i) x[i] += blocks[blk][i + k * rows] * v[k];
                                }
                                v.clear();
                            }
                            if (!(fl & ARC_STORE)) continue;
                            if (ns < 1 || ns > per) die("tile");
                            if (lane < (ns << lg)) {
                                std::vector<double> d = at(r + 4) != ARC_NONE ? times(at(r + 4), rows, x) : x;
                                for (int k = 0; k < str; ++k)
                                    writes.push_back({at(r + 3) + lane * str + k, k < rows ? d[k] : 0.0});
                            }
                            x.clear();
                            stf = str;
                        }
                    }
                }
                // a stage may not write what it reads: the new states are stored after all reads
                std::vector<char> hit(region, 0);
                for (auto &w : writes) {
                    if (w.first >= region || hit[w.first]) die("two states in one place");
                    hit[w.first] = 1;
                }
                for (auto &q : reads)
                    if (hit[q.first]) die("a stage overwrites its source");
                for (auto &w : writes) put(w.first, w.second);
            }
            for (int col = 0; col < cg && c0 + col < m0; ++col) {
                std::vector<double> x(m0, 0.0);
                for (uint32_t p = 0; p < at(h + 5); ++p)
                    for (int k = 0; k < m0; ++k) x[k] += get(at(at(h + 6) + p) + col * stf + k);
                for (int i = 0; i < m0; ++i)
                    for (int q = 0; q < m0; ++q)
                        res[off[s0] + i + (c0 + col) * m0] += prop[n][off[s0] + i + q * m0] * x[q];
            }
        }
    }

    }

    // ---- the plain sum ----
    const int pos_w = kind == ARC_BARE ? -1 : kind == ARC_SIGMA ? 2 * order + 2 : 2 * order - n_after + 2;
    std::vector<Topo> all;
    Pairs part;
    std::vector<int> pts;
    for (int i = 1; i <= 2 * order; ++i) pts.push_back(i);
    gen(part, 1, pts, all);
    double leaves = 0;
    auto point_pos = [&](int pt) {  // point 1 is the latest
        int pos = n - pt;
        if (kind == ARC_SIGMA) return pos - 1;
        if (pos_w > 0 && pos <= pos_w) --pos;
        return pos;
    };
    const int cut = kind == ARC_SIGMA ? 1 : n_after;
    for (const Topo &t : all) {
        if (kind != ARC_BARE && !connected(t.p, cut)) continue;
        std::vector<int> arc_at(n + 1, -1), is_head(n + 1, 0);
        for (size_t a = 0; a < t.p.size(); ++a) {
            const int head = point_pos(t.p[a].second), tail = point_pos(t.p[a].first);
            arc_at[head] = arc_at[tail] = (int)a;
            is_head[head] = 1;
        }
        for (int s0 = 0; s0 < m.ns; ++s0) {
            std::vector<int> sel(order + 1, 0);
            // X: dims[s] x dims[s0]
            struct Rec {
                static void go(int pos, int s, std::vector<double> X, double wgt, int n, int pos_w, int kind, int s0,
                               const ArcModel &m, const std::vector<int> &off, const std::vector<std::vector<double>> &prop,
                               const std::vector<int> &arc_at, const std::vector<int> &is_head, const Topo &t,
                               std::vector<int> &sel, const ArcBlocks &ob, const std::vector<std::vector<double>> &blocks,
                               const std::function<double(int, int, int)> &arc, const std::function<int(int)> &pp,
                               std::vector<double> &ref, double &leaves) {
                    const int ms = m.dims[s], m0 = m.dims[s0];
                    std::vector<double> Y(ms * m0, 0.0);
                    for (int c = 0; c < m0; ++c)
                        for (int i = 0; i < ms; ++i)
                            for (int q = 0; q < ms; ++q) Y[i + c * ms] += prop[pos][off[s] + i + q * ms] * X[q + c * ms];
                    if (pos == n) {
                        if (s != s0) die("the test's model leaves its sector");
                        leaves += 1;
                        for (int i = 0; i < ms * m0; ++i) ref[off[s0] + i] += wgt * Y[i];
                        return;
                    }
                    auto next = [&](int to, uint32_t blk, double w2) {
                        std::vector<double> Z(m.dims[to] * m0, 0.0);
                        for (int c = 0; c < m0; ++c)
                            for (int i = 0; i < m.dims[to]; ++i)
                                for (int q = 0; q < ms; ++q) Z[i + c * m.dims[to]] += blocks[blk][i + q * m.dims[to]] * Y[q + c * ms];
                        go(pos + 1, to, Z, w2, n, pos_w, kind, s0, m, off, prop, arc_at, is_head, t, sel, ob, blocks, arc, pp, ref, leaves);
                    };
                    if (pos == pos_w) {
                        if (kind == ARC_CORR) {
                            if (m.a_sf[s] >= 0) next(m.a_sf[s], ob.a[s], wgt);
                        } else {
                            go(pos + 1, s, Y, wgt, n, pos_w, kind, s0, m, off, prop, arc_at, is_head, t, sel, ob, blocks, arc, pp, ref, leaves);
                        }
                        return;
                    }
                    const int a = arc_at[pos];
                    if (is_head[pos]) {
                        for (int p = 0; p < m.np; ++p)
                            if (m.head_sf[p][s] >= 0) {
                                sel[a] = p;
                                next(m.head_sf[p][s], ob.head[p][s], wgt);
                            }
                    } else {
                        const int p = sel[a];
                        if (m.tail_sf[p][s] >= 0) next(m.tail_sf[p][s], ob.tail[p][s], wgt * arc(pp(t.p[a].second), pos, m.table[p]));
                    }
                }
            };
            int s1 = s0;
            std::vector<double> X;
            if (kind == ARC_CORR) {
                if (m.b_sf[s0] < 0) continue;
                s1 = m.b_sf[s0];
                X = blocks[ob.b[s0]];
            } else {
                X.assign(m.dims[s0] * m.dims[s0], 0.0);
                for (int i = 0; i < m.dims[s0]; ++i) X[i + i * m.dims[s0]] = 1.0;
            }
            Rec::go(2, s1, X, t.parity, n, pos_w, kind, s0, m, off, prop, arc_at, is_head, t, sel, ob, blocks,
                    [&](int x, int y, int z) { return arc(x, y, z); }, [&](int x) { return point_pos(x); }, ref, leaves);
        }
    }
    double dev = 0, mx = 0;
    for (int i = 0; i < l.bt; ++i) {
        dev = std::max(dev, std::fabs(res[i] - ref[i]));
        mx = std::max(mx, std::fabs(ref[i]));
    }
    std::printf("dev %.3e leaves %.0f %.0f lds %zu segments %d\n", mx > 0 ? dev / mx : dev, pg.leaves, leaves, pg.lds, pg.n_segments);
    return 0;
}
