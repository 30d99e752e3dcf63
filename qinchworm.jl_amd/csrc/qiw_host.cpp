// qiw_host.cpp -- the C ABI of libqiw (include/qiw.h): context, model staging, compilation
// of configuration tries into device programs, and the inchworm!/correlator_2p drivers.
//
// The drivers keep all per-step state on the device: every inchworm step is one launch of
// the evaluator over all (order, n_pts_after, topology, sample) work of the step followed by
// one launch of the bookkeeping kernel (set_ppgf! + normalize!), so the n_tau-2 serial steps
// run without a host round trip.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <chrono>
#include <cmath>
#include <complex>
#include <cstdio>
#include <cstring>
#include <map>
#include <mutex>
#include <string>
#include <vector>

#include "../../include/qiw.h"
#include "qiw_arcs.h"
#include "qiw_chunks.h"
#include "qiw_ctx.h"
#include "qiw_device.h"

using namespace qiwi;

// ---------------------------------------------------------------------------------------
// Topologies (src/diagrammatics.jl:288-337)
// ---------------------------------------------------------------------------------------
namespace {

struct Topology {
    std::vector<std::pair<int, int>> pairs;
    int parity;
};

void gen_topologies(std::vector<std::pair<int, int>> &partial, int parity, std::vector<int> unpaired,
                    std::vector<Topology> &out) {
    if (unpaired.empty()) {
        out.push_back({partial, parity});
        return;
    }
    for (size_t i = 2; i <= unpaired.size(); ++i) {
        // pairing the first open point with the i-th adds a transposition per skipped point
        std::vector<int> rest;
        for (size_t q = 1; q < unpaired.size(); ++q)
            if (q != i - 1) rest.push_back(unpaired[q]);
        partial.push_back({unpaired[0], unpaired[i - 1]});
        gen_topologies(partial, (i % 2 == 0) ? parity : -parity, rest, out);
        partial.pop_back();
    }
}

bool arcs_cross(std::pair<int, int> a, std::pair<int, int> b) {
    if (a.first > a.second) std::swap(a.first, a.second);
    if (b.first > b.second) std::swap(b.first, b.second);
    return (a.first < b.first && b.first < a.second && a.second < b.second) ||
           (b.first < a.first && a.first < b.second && b.second < a.second);
}

bool doubly_k_connected(const Topology &t, int k) {
    auto straddles = [k](std::pair<int, int> p) {
        return (p.first <= k && p.second > k) || (p.second <= k && p.first > k);
    };
    std::vector<std::pair<int, int>> stack, rest;
    for (auto &p : t.pairs) (straddles(p) ? stack : rest).push_back(p);
    while (!stack.empty()) {
        auto c = stack.back();
        stack.pop_back();
        for (int i = (int)rest.size() - 1; i >= 0; --i)
            if (arcs_cross(c, rest[i])) {
                stack.push_back(rest[i]);
                rest.erase(rest.begin() + i);
            }
    }
    return rest.empty();
}

std::vector<Topology> topologies_at_order(int order, int k, bool external_arc) {
    std::vector<Topology> all;
    std::vector<std::pair<int, int>> partial;
    std::vector<int> pts;
    for (int i = 1; i <= 2 * order; ++i) pts.push_back(i);
    gen_topologies(partial, 1, pts, all);
    if (k < 0) return all;
    std::vector<Topology> out;
    for (auto &t : all)
        if (doubly_k_connected(t, k)) out.push_back(t);
    if (external_arc)
        for (auto &t : out) t.parity *= (k % 2 == 0) ? 1 : -1;
    return out;
}

}  // namespace

namespace qiwi {

int fail(qiw_ctx *c, int code, const std::string &msg) {
    if (c) c->err = msg;
    return code;
}

// Buffers that one step call fills and reads back (per-task partial sums, the i*P table
// and its order slots, the bookkeeping's sums and counter): a no-alloc call takes them from
// the device's static scratch array.
static bool per_call_buffer(const std::string &name) {
    static const char *const names[] = {"partial", "ptab",     "porders",  "lambda",      "fin.scratch",
                                        "fin.gsum", "diag",     "fin.done", "porders_std", "sobol.m"};
    for (const char *n : names)
        if (name == n) return true;
    return false;
}

void *dev(qiw_ctx *c, const std::string &name, size_t bytes, int *rc) {
    if (c->no_alloc) {
        if (per_call_buffer(name)) {
            const size_t off = (c->scratch_used + 255) & ~(size_t)255;
            if (off + bytes > kNoAllocScratchBytes) {
                *rc = fail(c, QIW_E_LIMIT, "the step needs more than the " + std::to_string(kNoAllocScratchBytes >> 20) +
                                               " MiB scratch array of qiw_inchworm_step_noalloc (" + name + ")");
                return nullptr;
            }
            c->scratch_used = off + bytes;
            return (char *)c->scratch + off;
        }
        DevBuf &b = c->bufs[name];
        if (b.n < bytes) {
            *rc = fail(c, QIW_E_STATE, "device buffer " + name +
                                           " is not resident: call qiw_inchworm_step once with the same run first");
            return nullptr;
        }
        return b.p;
    }
    DevBuf &b = c->bufs[name];
    if (b.n < bytes) {
        if (b.p) (void)hipFree(b.p);
        b.p = nullptr;
        b.n = 0;
        if (hipMalloc(&b.p, std::max<size_t>(bytes, 256)) != hipSuccess) {
            *rc = fail(c, QIW_E_DEVICE, "hipMalloc failed for " + name);
            return nullptr;
        }
        b.n = std::max<size_t>(bytes, 256);
    }
    return b.p;
}

}  // namespace qiwi

namespace {

// natural cubic spline of uniformly spaced real values -> per-interval local cubic
// coefficients (src/spline_gf.jl:194-202: BSpline(Cubic(Line(OnGrid()))) on the grid)
void natural_spline_coef(const std::vector<double> &y, double h, double *c) {
    int n = (int)y.size();
    std::vector<double> M(n, 0.0);
    if (n >= 3) {
        int m = n - 2;
        std::vector<double> cp(m), dp(m);
        for (int i = 0; i < m; ++i) {
            double rhs = 6.0 * (y[i + 2] - 2.0 * y[i + 1] + y[i]) / (h * h);
            double den = 4.0 - (i > 0 ? cp[i - 1] : 0.0);
            cp[i] = (i < m - 1 ? 1.0 : 0.0) / den;
            dp[i] = (rhs - (i > 0 ? dp[i - 1] : 0.0)) / den;
        }
        for (int i = m - 1; i >= 0; --i) M[i + 1] = dp[i] - (i < m - 1 ? cp[i] * M[i + 2] : 0.0);
    }
    const double h26 = h * h / 6.0;
    for (int j = 0; j < n - 1; ++j) {
        c[4 * j + 0] = y[j];
        c[4 * j + 1] = (y[j + 1] - y[j]) - h26 * (2.0 * M[j] + M[j + 1]);
        c[4 * j + 2] = 3.0 * h26 * M[j];
        c[4 * j + 3] = h26 * (M[j + 1] - M[j]);
    }
}

int load_scalar_op(qiw_ctx *c, const qiw_sbm &in, const std::vector<int> &dims, ScalarOp &out, bool *scalar,
                   std::vector<double> &op_data, std::vector<int32_t> &op_desc) {
    int ns = (int)dims.size();
    out.sf.assign(ns, -1);
    out.val.assign(ns, 0.0);
    out.blk.assign(ns, -1);
    size_t off = 0;
    for (int b = 0; b < in.n_blocks; ++b) {
        int si = in.s_i[b], sf = in.s_f[b];
        if (si < 0 || si >= ns || sf < 0 || sf >= ns)
            return fail(c, QIW_E_ARG, "operator block sector index out of range");
        if (out.sf[si] != -1)
            return fail(c, QIW_E_NOT_SBM,
                        "Operator is not representable by a SectorBlockMatrix (more than one non-zero blocks per column)");
        size_t sz = (size_t)dims[sf] * dims[si];
        if (sz != 1) *scalar = false;
        for (size_t e = 0; e < sz; ++e)
            if (std::fabs(in.data[2 * (off + e) + 1]) > 1e-13 * (1.0 + std::fabs(in.data[2 * (off + e)])))
                return fail(c, QIW_E_ARG, "complex operator matrix elements are not supported by the GPU kernels");
        out.sf[si] = sf;
        out.val[si] = in.data[2 * off];
        out.blk[si] = (int)op_desc.size() / 3;
        op_desc.push_back((int32_t)op_data.size());
        op_desc.push_back(dims[sf]);
        op_desc.push_back(dims[si]);
        for (size_t e = 0; e < sz; ++e) op_data.push_back(in.data[2 * (off + e)]);
        off += sz;
    }
    return QIW_OK;
}

// ---------------------------------------------------------------------------------------
// Group compilation: the depth-first traversal of src/topology_eval.jl:454-556 for every
// (topology, initial sector), recorded as a trie and emitted in preorder.
// ---------------------------------------------------------------------------------------
enum NodeKind { N_PAIR_HEAD, N_PAIR_TAIL, N_IDENTITY, N_OPERATOR };

// Program formats: the walks of the assignment tries (scalar, LDS block, vector), and the arc
// walks (sector blocks, scalar).
enum ProgFormat { FMT_SCALAR = 0, FMT_BLOCK = 1, FMT_VEC = 2, FMT_ARC = 3, FMT_SARC = 4 };

// Format of the assignment tries.  Vector programs also drive the matrix-core walk of wide
// blocks (float32 chain products).
int program_format(const HostModel &m, int max_order, int precision) {
    if (m.scalar_kernel) return FMT_SCALAR;
    if (m.vec_ok && max_order <= 4) return FMT_VEC;
    if (m.mfma_ok && max_order <= 4 && precision == QIW_PREC_FP32) return FMT_VEC;
    return FMT_BLOCK;
}

// Chains are in float32 where a walk of the tries has them so; what runs on the LDS block walk
// (orders beyond 4, wide blocks of more than two tables) is float64 in the arc walk too.
int chain_precision(const HostModel &m, int max_order, int precision) {
    return program_format(m, max_order, precision) == FMT_BLOCK ? QIW_PREC_FP64 : precision;
}

// Models run the arc walks wherever the states of their groups fit (a CU's LDS; the slots
// and rows of the scalar walk; compile_group), and the assignment tries otherwise.
int eval_format(const HostModel &m, int max_order, int precision) {
    const int fmt = program_format(m, max_order, precision);
    return fmt == FMT_SCALAR ? FMT_SARC : m.ns > 255 ? fmt : FMT_ARC;
}

// Stride of the W slots: the table count of the register walk instantiation that runs the
// program, or the model's table count for the LDS block walk.
int w_stride(const HostModel &m, int fmt, int max_order) {
    if (fmt == FMT_BLOCK) return m.ntab;
    if (fmt == FMT_SCALAR) return qiw_scalar_tm(max_order, m.ns, m.ntab);
    return qiw_vec_tm(m.ntab);
}

struct Compiled {
    QiwGroup g{};
    std::vector<uint64_t> prog;
    std::vector<uint32_t> topo;   // per topology: head/tail nibbles of arcs 0-3, of arcs 4-5
    std::vector<double> coefs;    // scalar programs: leaf coefficients other than +-1
    std::vector<int32_t> chunks{0};  // program offsets (64-bit words) of the topology chunks
    std::vector<double> chunk_share;  // vector programs: each chunk's share of the group's cost
    int64_t leaves_per_sample = 0;
    int64_t edges_per_sample = 0;
    // block programs: real FLOPs of the chain products one sample costs (per column of the
    // initial sector: i*P times the partial product once per node with children, the
    // operator block per edge, the leaf accumulation)
    double flops_per_sample = 0;
    int n_top = 0;
    // arc programs: initial-sector segments, shape (wavefronts of a workgroup; scalar: register
    // slots) and LDS bytes of a workgroup
    int n_segments = 0, shape = 1;
    size_t lds_bytes = 0;
    int replica_of = -1;  // randomized qMC: another sequence of group `replica_of` (no program of its own)
};

struct TrieNode {
    int level, pslot, wslot, parent;
    bool tail, leaf;
    double coef;
    std::vector<int> children;
    int s_in = 0, s_out = 0, blk = 0xFFFF;  // block programs: sectors and operator block
};

constexpr char kOffDiagonal[] =
    "A block off-diagonal contribution to a pseudo-particle propagator detected, try passing more "
    "'symmetry_breakers' when constructing the local exact diagonalization object";

struct Compiler {
    const HostModel &m;
    int kind, order, n_after, corr, fmt;
    int wstride;  // W slot of arc a, table t: a * wstride + t
    int pstride;  // scalar programs: inner P entry of level L, sector s: (nm - 1 - L) * pstride + s
    int nm;       // scalar programs: positions of the largest order of the instantiation
    std::vector<uint32_t> p32;  // scalar program words
    int chunk_words = 0;        // scalar programs: start a new chunk at a topology once the
                                // current one holds this many words (0: one chunk)
    int64_t chunk_cost = 0;     // vector programs: the same, in words x columns replayed

    // appends a scalar program word; the last word of every 64-word block is NEXT
    void put32(uint32_t w) {
        if (p32.size() % QIW_WAVE == QIW_WAVE - 1) p32.push_back((uint32_t)QIW_FL_OP_NEXT << 28);
        p32.push_back(w);
    }
    int n = 0, pos_w = 0;
    std::vector<int> conf_kind, conf_arc;
    std::vector<int> selected;
    std::vector<TrieNode> trie;
    int s0 = 0, parity = 1;
    std::string err;

    Compiler(const HostModel &m_, int kind_, int order_, int n_after_, int corr_, int fmt_, int max_order)
        : m(m_), kind(kind_), order(order_), n_after(n_after_), corr(corr_), fmt(fmt_),
          wstride(w_stride(m_, fmt_, max_order)), pstride(qiw_scalar_sm(max_order, m_.ns, m_.ntab)),
          nm(2 * qiw_scalar_km(max_order, m_.ns, m_.ntab) + 3) {}

    int add(int parent, int level, int s_in, int wslot, bool tail, int s_out = 0, int blk = 0xFFFF) {
        TrieNode t{level, (level - 2) * m.ns + s_in, wslot, parent, tail, false, 0.0, {}, s_in, s_out, blk};
        trie.push_back(t);
        int id = (int)trie.size() - 1;
        if (parent >= 0) trie[parent].children.push_back(id);
        return id;
    }

    // Child `id` was just added under `node`: keep it if its subtree reaches a leaf, else
    // drop it (a pair whose tail operator annihilates the sector reached by then).  Returns
    // -1 on error, 0 for a dead subtree, 1 for a live one.
    int keep_child(int node, int id, int r) {
        if (r <= 0) {
            trie.erase(trie.begin() + id, trie.end());
            trie[node].children.pop_back();
        }
        return r;
    }

    int dfs(int node, int pos, int s, double c) {
        if (pos > n) {
            if (s != s0) {
                err = kOffDiagonal;
                return -1;
            }
            trie[node].leaf = true;
            trie[node].coef = c * parity * ((order % 2 == 0) ? 1.0 : -1.0);
            return 1;
        }
        int k = conf_kind[pos];
        // block programs keep the operator blocks as matrices: no constant folding
        const bool fold = (fmt == FMT_SCALAR);
        int live = 0;
        if (k == N_PAIR_HEAD) {
            int a = conf_arc[pos];
            for (int p : m.attachable[s]) {
                selected[a] = p;
                int id = add(node, pos, s, 0, false, m.op_i[p].sf[s], m.op_i[p].blk[s]);
                int r = keep_child(node, id, dfs(id, pos + 1, m.op_i[p].sf[s], fold ? c * m.op_i[p].val[s] : c));
                if (r < 0) return -1;
                live |= r;
            }
        } else if (k == N_PAIR_TAIL) {
            int a = conf_arc[pos];
            int p = selected[a];
            if (m.op_f[p].sf[s] >= 0) {
                int id = add(node, pos, s, a * wstride + m.pair_table[p], true, m.op_f[p].sf[s], m.op_f[p].blk[s]);
                live = keep_child(node, id, dfs(id, pos + 1, m.op_f[p].sf[s], fold ? c * m.op_f[p].val[s] : c));
            }
        } else if (k == N_OPERATOR) {
            const ScalarOp &A = m.corr_A[corr];
            if (A.sf[s] >= 0) {
                int id = add(node, pos, s, 0, false, A.sf[s], A.blk[s]);
                live = keep_child(node, id, dfs(id, pos + 1, A.sf[s], fold ? c * A.val[s] : c));
            }
        } else {
            int id = add(node, pos, s, 0, false, s, 0xFFFF);
            live = keep_child(node, id, dfs(id, pos + 1, s, c));
        }
        return live;
    }

    void emit(int id, Compiled &out) {
        const TrieNode &t = trie[id];
        uint64_t w;
        if (fmt == FMT_VEC) {
            w = (uint64_t)m.dims[t.s_out] | ((uint64_t)t.wslot << 16) |
                ((uint64_t)t.children.size() << 24) | (op_offset(t.blk) << 32) | (blk_off(t.s_out) << 52);
        } else {
            w = (uint64_t)t.level | ((uint64_t)t.s_in << 8) | ((uint64_t)t.wslot << 16) |
                ((uint64_t)(t.blk & 0xFFFF) << 24) | ((uint64_t)t.s_out << 40);
        }
        if (t.tail) w |= QIW_F_TAIL;
        if (t.leaf) w |= QIW_F_LEAF;
        {
            const double m0 = m.dims[s0], mi = m.dims[t.s_in], mo = m.dims[t.s_out];
            if (t.blk != 0xFFFF) out.flops_per_sample += 2.0 * mo * mi * m0;
            if (t.leaf) out.flops_per_sample += 2.0 * mo * m0;
            if (!t.children.empty() && t.level + 1 < n) out.flops_per_sample += 2.0 * mo * mo * m0;
        }
        const bool unit = t.leaf && fmt != FMT_BLOCK && std::fabs(t.coef) == 1.0;
        if (unit) w |= QIW_FV_UNIT | (t.coef < 0 ? QIW_FV_NEG : 0);
        out.edges_per_sample++;
        out.prog.push_back(w);
        if (unit) out.leaves_per_sample++;
        if (t.leaf && !unit) {  // the leaf coefficient follows as a raw float64 word
            uint64_t cw;
            std::memcpy(&cw, &t.coef, 8);
            out.prog.push_back(cw);
            out.leaves_per_sample++;
        }
        for (size_t i = 0; i < t.children.size(); ++i) emit(t.children[i], out);
    }

    // Leaf coefficient bits of a scalar program word: UNIT/NEG, or the index into the
    // group's table of other coefficients.
    bool coef_bits(double coef, uint32_t &w, Compiled &out) {
        if (std::fabs(coef) == 1.0) {
            w |= QIW_FL_UNIT | (coef < 0 ? QIW_FL_NEG : 0u);
            return true;
        }
        size_t ci = std::find(out.coefs.begin(), out.coefs.end(), coef) - out.coefs.begin();
        if (ci == out.coefs.size()) out.coefs.push_back(coef);
        if (ci > 255) {
            err = "more than 256 distinct leaf coefficients in one group";
            return false;
        }
        w |= (uint32_t)ci;
        return true;
    }

    // Scalar program words of node `id` at level L and its subtree (format in qiw_device.h).
    // `pop`: the node is not its parent's first child, so it restores the parent's product.
    bool emit_flat(int id, int L, bool pop, Compiled &out) {
        const TrieNode &t = trie[id];
        const bool leaf = (L + 1 == n);  // the only child is the leaf at the last position
        uint32_t w;
        if (id == 0) {  // root, position 1
            w = (uint32_t)QIW_FL_OP_ROOT << 28;
            if (!leaf) w |= (uint32_t)t.s_out;
        } else {
            w = (uint32_t)L << 16;
            if (pop) w |= QIW_FL_POP;
            if (t.tail) w |= QIW_FL_TAIL | ((uint32_t)t.wslot << 8);
            out.edges_per_sample++;
        }
        if (leaf) {
            w |= QIW_FL_LEAF;
            out.edges_per_sample++;
            out.leaves_per_sample++;
            if (!coef_bits(trie[t.children.at(0)].coef, w, out)) return false;
            put32(w);
            return true;
        }
        if (id != 0) w |= (uint32_t)(2 * ((nm - 1 - (L + 1)) * pstride + t.s_out));
        if (t.children.size() > 1) w |= QIW_FL_PUSH;
        put32(w);
        for (size_t i = 0; i < t.children.size(); ++i)
            if (!emit_flat(t.children[i], L + 1, i > 0, out)) return false;
        return true;
    }

    // offset of operator block blk in the operator data (0xFFFF: identity)
    uint64_t op_offset(int blk) const {
        if (blk == 0xFFFF) return 0xFFFF;
        return wide() ? (uint64_t)m.op_rm_off[blk] : (uint64_t)m.op_desc[3 * blk];
    }
    // vector programs of models with blocks wider than 6 run on the matrix-core walk, which
    // reads the row-major operator blocks and its own LDS layout of the i*P blocks
    bool wide() const { return fmt == FMT_VEC && m.mmax > 6; }
    uint64_t blk_off(int s) const { return wide() ? (uint64_t)m.lds_off[s] : (uint64_t)m.bt_off[s]; }

    bool compile(Compiled &out) {
        n = (kind == QIW_G_BARE) ? 2 * order + 2 : 2 * order + 3;
        // self-energy groups: all 2k pair positions before tau_w (= tau_f_prev = tau_f)
        int d_after = (kind == QIW_G_BARE) ? 2 * order : (kind == QIW_G_SIGMA) ? 0 : n_after;
        int d_before = 2 * order - d_after;
        pos_w = (kind == QIW_G_BARE) ? 0 : d_before + 2;
        conf_kind.assign(n + 2, N_IDENTITY);
        conf_arc.assign(n + 2, -1);
        if (kind == QIW_G_CORR) {
            conf_kind[1] = N_OPERATOR;  // B at tau = 0; handled at the root
            conf_kind[pos_w] = N_OPERATOR;
        }
        std::vector<int> top_to_conf;  // topology point -> configuration position
        for (int pos = n; pos >= 1; --pos) {
            bool fixed = (pos == 1 || pos == n || pos == pos_w);
            if (!fixed) top_to_conf.push_back(pos);
        }
        // self-energy: get_topologies_at_order(order, 1) (src/inchworm.jl:715)
        std::vector<Topology> tops = (kind == QIW_G_BARE)    ? topologies_at_order(order, -1, false)
                                     : (kind == QIW_G_SIGMA) ? topologies_at_order(order, 1, false)
                                                             : topologies_at_order(order, n_after, kind == QIW_G_CORR);
        selected.assign(std::max(order, 1), -1);
        out.n_top = (int)tops.size();
        // vector format: segments per initial sector, collected first
        // vector format: words of every (topology, initial sector), regrouped into chunks
        const bool vec_like = (fmt == FMT_VEC);
        std::vector<std::vector<std::vector<uint64_t>>> vtop(vec_like ? tops.size() : 0,
                                                             std::vector<std::vector<uint64_t>>(m.ns));
        for (int ti = 0; ti < (int)tops.size(); ++ti) {
            const Topology &top = tops[ti];
            parity = top.parity;
            uint64_t topo_word = (uint64_t)QIW_OP_TOPO << 48;
            uint32_t tw[2] = {0, 0};
            for (int a = 0; a < order; ++a) {
                int head = top_to_conf[top.pairs[a].second - 1];
                int tail = top_to_conf[top.pairs[a].first - 1];
                conf_kind[head] = N_PAIR_HEAD;
                conf_kind[tail] = N_PAIR_TAIL;
                conf_arc[head] = conf_arc[tail] = a;
                topo_word |= ((uint64_t)head << (8 * a)) | ((uint64_t)tail << (8 * a + 4));
                // flat scalar programs name arc ends by simplex coordinate: j = n - 1 - p
                // after tau_w, d_after + pos_w - 1 - p before it
                auto coord = [&](int p) { return p > pos_w ? n - 1 - p : d_after + pos_w - 1 - p; };
                tw[a / 4] |= (uint32_t)(coord(head) | (coord(tail) << 4)) << (8 * (a % 4));
            }
            out.topo.push_back(tw[0]);
            out.topo.push_back(tw[1]);
            if (fmt == FMT_SCALAR && chunk_words > 0 && ti > 0 &&
                (int)p32.size() - 2 * out.chunks.back() >= chunk_words) {
                // close the chunk: END, then END up to the next 64-word block
                put32((uint32_t)QIW_FL_OP_END << 28);
                while (p32.size() % QIW_WAVE) p32.push_back((uint32_t)QIW_FL_OP_END << 28);
                out.chunks.push_back((int32_t)(p32.size() / 2));
            }
            if (order > 0 && fmt == FMT_SCALAR) put32(((uint32_t)QIW_FL_OP_TOPO << 28) | (uint32_t)ti);
            if (order > 0 && fmt == FMT_BLOCK) out.prog.push_back(topo_word);
            for (s0 = 0; s0 < m.ns; ++s0) {
                trie.clear();
                // root: configuration position 1 (identity, or the B operator)
                double c = 1.0;
                int s = s0, root_blk = 0xFFFF;
                if (kind == QIW_G_CORR) {
                    const ScalarOp &B = m.corr_B[corr];
                    if (B.sf[s0] < 0) continue;
                    c = (fmt == FMT_SCALAR) ? B.val[s0] : 1.0;  // other formats apply the B block at the root
                    s = B.sf[s0];
                    root_blk = B.blk[s0];
                }
                TrieNode root{1, 0, 0, -1, false, false, 0.0, {}};
                trie.push_back(root);
                if (dfs(0, 2, s, c) < 0) return false;
                if (trie[0].children.empty()) continue;
                if (fmt == FMT_SCALAR) {  // position 1 is the root, level 1
                    trie[0].s_out = s;
                    if (!emit_flat(0, 1, true, out)) return false;
                    put32(((uint32_t)QIW_FL_OP_FLUSH << 28) | (uint32_t)s0);
                    continue;
                }
                if (trie[0].children.size() > 255) {
                    err = "too many pair interactions attachable to one sector";
                    return false;
                }
                if (fmt == FMT_VEC) {
                    std::vector<uint64_t> saved;
                    saved.swap(out.prog);
                    if (order > 0) out.prog.push_back(topo_word);
                    out.prog.push_back(((uint64_t)QIW_OP_ROOT << 48) | (uint64_t)m.dims[s] |
                                       ((uint64_t)trie[0].children.size() << 24) | (op_offset(root_blk) << 32) |
                                       (blk_off(s) << 52));
                    // the root's i*P (level 2) for its children
                    if (n > 2) out.flops_per_sample += 2.0 * m.dims[s] * m.dims[s] * m.dims[s0];
                    for (size_t i = 0; i < trie[0].children.size(); ++i) emit(trie[0].children[i], out);
                    vtop[ti][s0] = out.prog;
                    saved.swap(out.prog);
                    continue;
                }
                out.prog.push_back(((uint64_t)QIW_OP_ROOT << 48) | ((uint64_t)s0 << 8) |
                                   ((uint64_t)(root_blk & 0xFFFF) << 24) | ((uint64_t)s << 40));
                for (size_t i = 0; i < trie[0].children.size(); ++i) emit(trie[0].children[i], out);
                out.prog.push_back(((uint64_t)QIW_OP_FLUSH << 48) | ((uint64_t)s0 << 8));
            }
        }
        if (vec_like) {
            // Chunks of topologies, each a program of its own: every initial sector gets a
            // segment in every chunk, so every output element of a task row is written.
            // Where the chunks start: qiw_chunk_starts, on the topologies' words weighted by
            // the columns each segment is replayed for.
            auto put_chunk = [&](size_t t0, size_t t1) {
                for (int s = 0; s < m.ns; ++s) {
                    out.prog.push_back(((uint64_t)QIW_OP_SEG << 48) | (uint64_t)m.dims[s] | ((uint64_t)s << 8) |
                                       (blk_off(s) << 52));
                    for (size_t t = t0; t < t1; ++t) out.prog.insert(out.prog.end(), vtop[t][s].begin(), vtop[t][s].end());
                    out.prog.push_back((uint64_t)QIW_OP_FLUSH << 48);
                }
            };
            std::vector<int64_t> tcost(vtop.size(), 0);
            int64_t total = 0;
            for (size_t t = 0; t < vtop.size(); ++t) {
                for (int s = 0; s < m.ns; ++s) tcost[t] += (int64_t)m.dims[s] * (int64_t)vtop[t][s].size();
                total += tcost[t];
            }
            const std::vector<size_t> chunk_first = qiw_chunk_starts(tcost, chunk_cost, wide() ? QIW_MFMA_WAVES : 1);
            size_t t0 = 0;
            for (size_t ci = 1; ci < chunk_first.size(); ++ci) {
                const size_t t = chunk_first[ci];
                put_chunk(t0, t);
                out.prog.push_back((uint64_t)QIW_OP_END << 48);
                while (out.prog.size() % QIW_WAVE) out.prog.push_back((uint64_t)QIW_OP_END << 48);
                out.chunks.push_back((int32_t)out.prog.size());
                t0 = t;
            }
            put_chunk(t0, vtop.size());
            out.chunk_share.assign(out.chunks.size(), 0.0);  // the chunks' shares of the cost
            for (size_t t = 0, ci = 0; t < vtop.size(); ++t) {
                while (ci + 1 < chunk_first.size() && t == chunk_first[ci + 1]) ++ci;
                out.chunk_share[ci] += total > 0 ? (double)tcost[t] / (double)total : 1.0 / (double)vtop.size();
            }
        }
        if (fmt == FMT_SCALAR) {  // 32-bit words, two to a 64-bit program element
            put32((uint32_t)QIW_FL_OP_END << 28);
            if (p32.size() % 2) p32.push_back((uint32_t)QIW_FL_OP_END << 28);
            for (size_t i = 0; i < p32.size(); i += 2) out.prog.push_back(p32[i] | ((uint64_t)p32[i + 1] << 32));
        } else {
            out.prog.push_back((uint64_t)QIW_OP_END << 48);
        }
        QiwGroup &g = out.g;
        g.kind = kind;
        g.order = order;
        g.n_after = d_after;
        g.n_nodes = n;
        g.d_before = d_before;
        g.d_after = d_after;
        g.pos_w = pos_w;
        g.n_pslots = (n - 1) * m.ns;
        g.n_wslots = order * wstride;
        return true;
    }
};

// ---- arc programs (qiw_arcs.h) ----
ArcModel arc_model(const HostModel &m, int corr) {
    ArcModel a;
    a.ns = m.ns;
    a.np = m.np;
    a.dims = m.dims;
    a.table = m.pair_table;
    for (int p = 0; p < m.np; ++p) {
        a.head_sf.push_back(m.op_i[p].sf);
        a.tail_sf.push_back(m.op_f[p].sf);
    }
    if (corr >= 0) {
        a.a_sf = m.corr_A[corr].sf;
        a.b_sf = m.corr_B[corr].sf;
    }
    return a;
}

// Elements of a stored operator block in the instantiation for the model's blocks: float32
// slice registers (64 floats each), or float64 blocks padded to its size.
uint32_t arc_block_size(const HostModel &m, bool fp32) {
    const int mb = qiw_arc_rows(m.mmax);
    return fp32 ? 64u * (uint32_t)((mb / 4 * mb + 15) / 16) : (uint32_t)(mb * mb);
}

ArcBlocks arc_blocks(const HostModel &m, int corr, int precision) {
    ArcBlocks o;
    const uint32_t per = arc_block_size(m, precision == QIW_PREC_FP32);
    auto offsets = [&](const ScalarOp &op, bool column_major) {
        std::vector<uint32_t> v(m.ns, ARC_NONE);
        for (int s = 0; s < m.ns; ++s)
            if (op.blk[s] >= 0)
                v[s] = column_major ? (uint32_t)m.op_desc[3 * op.blk[s]] : per * (uint32_t)op.blk[s];
        return v;
    };
    for (int p = 0; p < m.np; ++p) {
        o.head.push_back(offsets(m.op_i[p], false));
        o.tail.push_back(offsets(m.op_f[p], false));
    }
    if (corr >= 0) {
        o.a = offsets(m.corr_A[corr], false);
        o.b = offsets(m.corr_B[corr], true);  // the root reads columns of B
    }
    o.id = per * (uint32_t)(m.op_desc.size() / 3);  // past the operators' blocks
    return o;
}

// Workgroup shapes of the arc walk, narrowest first: wavefronts, the LDS they may take, and
// the widest level, in 64-state tiles, that the shape is for.  Small levels take two
// wavefronts: one (20 KB) leaves the set-up of a sample to 64 lanes, four meet at more barriers
// than their tiles are worth (two-orbital solve of orders 0:2, N = 2^10: 21.9, 16.6, 20.5 ms
// with one, two, four).  Order 3 of the same model takes four in 53 KB (8.9 ms a step at N =
// 2^12; 11.1 in 40 KB, 11.2 with eight in 80 KB, 13.7 with two).  Wide blocks take all of a
// CU's LDS: the more columns fit beside each other, the fewer lanes idle in the tiles of one
// operator (three-orbital step of orders 0:2, N = 2^8, float64: 8.6 ms with two workgroups of
// 80 KB per CU, which left seven in a hundred lanes at work, 3.1 with one of 160 KB).  So do the
// programs that are cut by their first pairs, whose states did not fit otherwise: two-orbital steps
// in float64, orders 0:4, 5.1 -> 3.5, 41.8 -> 26.9 and 331 -> 213 ms at N = 2^5, 2^9 and 2^12, orders
// 0:5 at N = 2^4 118 -> 73 ms, against the first shape that the cut states fit (80 KB).
struct ArcShape {
    int waves;
    size_t cap;
    int tiles;
};
constexpr ArcShape kArcShapes[] = {{2, 40 << 10, 2}, {4, 53 << 10, 12}, {8, 80 << 10, 32}, {16, 160 << 10, 1 << 30}};
constexpr ArcShape kArcShapesWide[] = {{8, 160 << 10, 1 << 30}};  // mmax > 8; at most qiw_arc_waves

// Algorithmic real FLOPs of one sample of a compiled group: the scalar walk's multiply per
// trie edge and leaf, or the block programs' chain products.
double sample_flops(const Compiled &cg) {
    if (cg.flops_per_sample > 0) return cg.flops_per_sample;
    return 2.0 * cg.edges_per_sample + 2.0 * cg.leaves_per_sample;
}

// The group record and program of an arc-compiled group.
void set_arc_group(const HostModel &m, int kind, int order, int n_after, std::vector<uint32_t> &blob, Compiled &out) {
    const int d_after = (kind == QIW_G_BARE) ? 2 * order : (kind == QIW_G_SIGMA) ? 0 : n_after;
    out.n_top = (int)((kind == QIW_G_BARE)    ? topologies_at_order(order, -1, false)
                      : (kind == QIW_G_SIGMA) ? topologies_at_order(order, 1, false)
                                              : topologies_at_order(order, n_after, false))
                    .size();
    if (blob.size() % 2) blob.push_back(0);
    out.prog.resize(blob.size() / 2);
    std::memcpy(out.prog.data(), blob.data(), blob.size() * 4);
    QiwGroup &g = out.g;
    g.kind = kind;
    g.order = order;
    g.n_after = d_after;
    g.n_nodes = kind == QIW_G_BARE ? 2 * order + 2 : 2 * order + 3;
    g.d_before = 2 * order - d_after;
    g.d_after = d_after;
    g.pos_w = kind == QIW_G_BARE ? 0 : g.d_before + 2;
    g.n_pslots = (g.n_nodes - 1) * m.ns;
    g.n_wslots = order * qiw_vec_tm(m.ntab);
}

// Compiles a group as an arc program.  Returns 0, 1 when a diagram ends outside its initial
// sector, 2 when the states do not fit.
int compile_arcs(const HostModel &m, int kind, int order, int n_after, int corr, int precision, Compiled &out) {
    const ArcModel am = arc_model(m, corr);
    if (m.np > 127) return 2;
    const ArcBlocks ob = arc_blocks(m, corr, precision);
    const bool fp32 = precision == QIW_PREC_FP32;
    const int max_waves = qiw_arc_waves(m.mmax, fp32 ? 1 : 0);
    ArcLayout l;
    l.elem = fp32 ? 4 : 8;
    l.slots = arc_slots(qiw_arc_rows(m.mmax));
    l.mmax = m.mmax;
    l.bt = m.bt;
    l.bt_off.assign(m.bt_off.begin(), m.bt_off.end());
    // the widest level decides the shape to start from
    size_t widest = 0;
    for (int s0 = 0; s0 < m.ns; ++s0) {
        ArcGraph g;
        if (!arc_graph(am, kind, order, n_after, s0, {}, kind == QIW_G_BOLD && order > 0, g)) return 1;
        for (const auto &lev : g.levels) widest = std::max(widest, lev.size());
    }
    const bool wide = m.mmax > 8;
    const ArcShape *shapes = wide ? kArcShapesWide : kArcShapes;
    const int n_shapes = wide ? 1 : 4;
    ArcGroupProgram pg;
    int rc = 2;
    for (int n_fixed = 0; n_fixed <= order && rc == 2; ++n_fixed)
        for (int i = 0; i < n_shapes; ++i) {
            const ArcShape &sh = shapes[i];
            if (n_fixed == 0 ? (widest + 63) / 64 > (size_t)sh.tiles : i + 1 < n_shapes) continue;
            l.waves = std::min(sh.waves, max_waves);
            l.cap = sh.cap;
            rc = arc_compile(am, l, ob, kind, order, n_after, n_fixed, pg);
            if (rc != 2) break;
        }
    if (rc) return rc;
    set_arc_group(m, kind, order, n_after, pg.blob, out);
    out.n_segments = pg.n_segments;
    out.shape = l.waves;
    out.lds_bytes = pg.lds;
    out.leaves_per_sample = (int64_t)pg.leaves;
    out.edges_per_sample = (int64_t)pg.joins;
    out.flops_per_sample = pg.flops;
    return 0;
}

// Compiles a group of a scalar model as an arc program.  Returns as compile_arcs.
// corrs: the operator pair (-1: none), or several pairs for the traces of all.
int compile_scalar_arcs(const HostModel &m, int kind, int order, int n_after, const std::vector<int> &corrs, int max_words,
                        Compiled &out) {
    std::vector<ArcModel> models;
    std::vector<ArcValues> values;
    for (int corr : corrs) {
        ArcValues v;
        for (int p = 0; p < m.np; ++p) {
            v.head.push_back(m.op_i[p].val);
            v.tail.push_back(m.op_f[p].val);
        }
        if (corr >= 0) {
            v.a = m.corr_A[corr].val;
            v.b = m.corr_B[corr].val;
        }
        models.push_back(arc_model(m, corr));
        values.push_back(std::move(v));
    }
    const int n_out = corrs.size() > 1 ? (int)corrs.size() : m.ns;
    ScalarProgram sp;
    const int rc = arc_compile_scalar(models, values, kind, order, n_after, max_words, sp);
    if (rc) return rc;
    set_arc_group(m, kind, order, n_after, sp.blob, out);
    out.g.n_pslots = scalar_table_rows(sp.rows, n_out);
    out.shape = qiw_sarc_slots(sp.slots);
    out.lds_bytes = (size_t)scalar_lds_rows(sp.rows, n_out, out.g.n_nodes) * QIW_WAVE * 8;
    out.leaves_per_sample = (int64_t)sp.leaves;
    out.edges_per_sample = (int64_t)sp.words;
    out.flops_per_sample = 2.0 * sp.words;
    return 0;
}

// LDS doubles of one evaluator wavefront.  Scalar trie programs keep their state in registers;
// block programs hold per-sample state shared by the lanes (iP slots, W slots, stack, X,
// acc, out).
int lds_slots(const Compiled &cg, const HostModel &m, int fmt) {
    const QiwGroup &g = cg.g;
    if (fmt != FMT_BLOCK) return 0;  // register-resident walks, and the arc walks (Compiled::lds_bytes)
    int mm = m.mmax * m.mmax;
    return (g.n_nodes - 1) * m.bt + g.n_wslots + 1 + (g.n_nodes + 1) * mm + 2 * mm + m.bt;
}

// ---------------------------------------------------------------------------------------
// A batch of compiled groups resident on the device
// ---------------------------------------------------------------------------------------
struct Batch {
    std::vector<Compiled> groups;   // one entry per evaluated sequence of each group
    std::vector<QiwTask> tasks;
    std::vector<int32_t> g_first, g_count, g_slot;  // per group: task rows, order slot
    std::vector<int32_t> r_first, r_count;  // per (order, n_pts_after) group: its sequences' entries
    int n_eval = 1;        // sequences evaluated per sampled group
    bool scrambled = false;  // coordinates are drawn per step (randomized qMC)
    bool given = false;      // ... from the caller's sequences
    int64_t ut_total = 0;    // doubles of simplex coordinates of one launch (one tau row)
    int lds = 0;
    int fmt = FMT_SCALAR;  // program format of every group of the batch
    int spt = QIW_WAVE;    // samples per task
    int precision = QIW_PREC_FP64;
    int max_order = 0;  // largest order of the batch: selects the kernel instantiation
    double flops_per_launch = 0;  // algorithmic FLOPs of one launch
    int64_t leaves_per_launch = 0, diagram_evals_per_launch = 0;
    bool overflow = false;  // the launch would exceed kMaxTasks workgroups
    int n_out = 0;          // scalar arc walk: outputs per task (0: the sectors)
    struct Launch {         // arc walks: one launch per workgroup shape
        int first, count, shape;
        size_t lds;
    };
    std::vector<Launch> launches;
    int wg_waves = 1;       // wavefronts per workgroup: consecutive tasks of a workgroup share
                            // its sample block (matrix-core walk: kMfmaWaves)
};

// Wavefronts per workgroup of the matrix-core walk: they walk different topology chunks of
// the same samples and share the samples' i*P blocks in LDS (four: two workgroups of 65 KB
// per CU, two wavefronts per SIMD at the walk's 256 registers, on the three-orbital model).
constexpr int kMfmaWaves = QIW_MFMA_WAVES;

// Workgroups of one launch: task rows and grid sizes are 32-bit and every task is a
// 24-byte record on the host and the device, so a launch holds at most 2^28 tasks
// (e.g. N = 2^30 samples of 16 groups in 64-sample tasks is already 2^28).
constexpr int64_t kMaxTasks = (int64_t)1 << 28;
// Per-row coordinates of a correlator run on caller-drawn sequences stay below this.
constexpr double kMaxGivenCoordBytes = 64.0 * (1ull << 30);
inline bool tasks_fit(Batch &b, int64_t more) {
    if ((int64_t)b.tasks.size() + more > kMaxTasks) b.overflow = true;
    return !b.overflow;
}

// Evaluator launches of a batch: one per workgroup shape for the arc walks.
int eval_launches(const Batch &b) { return std::max<int>(1, (int)b.launches.size()); }

// Most task rows of a group (the reduction's block is sized by it).
int most_rows(const Batch &b) { return b.g_count.empty() ? 0 : *std::max_element(b.g_count.begin(), b.g_count.end()); }

struct DevBatch {
    QiwGroup *groups = nullptr;
    QiwTask *tasks = nullptr;
    uint64_t *prog = nullptr;
    uint32_t *topo = nullptr;
    double *coefs = nullptr;
    double *ut = nullptr;
    int32_t *g_first = nullptr, *g_count = nullptr, *g_slot = nullptr;
    int32_t *r_first = nullptr, *r_count = nullptr;
};

// Warp group index of a bold group (order k <= 4, n_after points after tau_w), else -1.
int warp_gid(const QiwGroup &g) {
    if (g.kind != QIW_G_BOLD || g.order < 1 || g.order > 4) return -1;
    return (g.order - 1) * (g.order - 1) + g.n_after - 1;
}

// weighted: the sampled bold groups carry a per-sample weight row (learned warp);
// per_sample: offsets of the groups' samples in a per-sample output are assigned.
int upload(qiw_ctx *c, const std::string &tag, Batch &b, int64_t N, DevBatch &d, bool weighted = false) {
    int rc = 0;
    std::vector<uint64_t> prog;
    std::vector<uint32_t> topo;
    std::vector<double> coefs;
    std::vector<QiwGroup> gs;
    // END words between and after the programs (never executed: prefetch and alignment)
    const uint64_t end_fl = (uint64_t)QIW_FL_OP_END << 28;
    const uint64_t pad = b.fmt >= FMT_ARC      ? 0ull
                         : b.fmt == FMT_SCALAR ? (end_fl | (end_fl << 32))
                                               : (uint64_t)QIW_OP_END << 48;
    int64_t ut_total = 0, ps_total = 0;
    for (auto &cg : b.groups) {
        QiwGroup g = cg.g;
        if (cg.replica_of >= 0) {  // another sequence of an earlier group: same program
            g.prog_off = gs[cg.replica_of].prog_off;
            g.topo_off = gs[cg.replica_of].topo_off;
            g.coef_off = gs[cg.replica_of].coef_off;
        } else {
            // programs start on a 64-word block boundary (the NOP placement assumes it)
            while (prog.size() % QIW_WAVE) prog.push_back(pad);
            g.prog_off = (int32_t)prog.size();
            g.topo_off = (int32_t)topo.size();
            g.coef_off = (int32_t)coefs.size();
        }
        g.sampled = g.order > 0;
        g.n_samples = (g.sampled && !qiw_group_exact(g)) ? (int32_t)N : 1;
        g.weighted = (weighted && g.sampled && warp_gid(g) >= 0) ? 1 : 0;
        g.ps_off = ps_total;
        ps_total += g.n_samples;
        g.ut_off = ut_total;
        if (g.sampled) ut_total += (int64_t)(g.d_before + g.d_after + g.weighted) * g.n_samples;
        prog.insert(prog.end(), cg.prog.begin(), cg.prog.end());
        topo.insert(topo.end(), cg.topo.begin(), cg.topo.end());
        coefs.insert(coefs.end(), cg.coefs.begin(), cg.coefs.end());
        cg.g = g;
        gs.push_back(g);
    }
    // two blocks of END words after the last program: the evaluator prefetches one block ahead
    prog.insert(prog.end(), 2 * QIW_WAVE, pad);
    b.ut_total = ut_total;
    if (topo.empty()) topo.push_back(0);
    if (coefs.empty()) coefs.push_back(0.0);
    d.groups = (QiwGroup *)dev(c, tag + ".groups", gs.size() * sizeof(QiwGroup), &rc);
    d.prog = (uint64_t *)dev(c, tag + ".prog", prog.size() * 8, &rc);
    d.topo = (uint32_t *)dev(c, tag + ".topo", topo.size() * 4, &rc);
    d.coefs = (double *)dev(c, tag + ".coefs", coefs.size() * 8, &rc);
    d.ut = (double *)dev(c, tag + ".ut", std::max<int64_t>(ut_total, 1) * 8, &rc);
    d.tasks = (QiwTask *)dev(c, tag + ".tasks", b.tasks.size() * sizeof(QiwTask), &rc);
    d.g_first = (int32_t *)dev(c, tag + ".gfirst", b.g_first.size() * 4 + 4, &rc);
    d.g_count = (int32_t *)dev(c, tag + ".gcount", b.g_count.size() * 4 + 4, &rc);
    d.g_slot = (int32_t *)dev(c, tag + ".gslot", b.g_slot.size() * 4 + 4, &rc);
    d.r_first = (int32_t *)dev(c, tag + ".rfirst", b.r_first.size() * 4 + 4, &rc);
    d.r_count = (int32_t *)dev(c, tag + ".rcount", b.r_count.size() * 4 + 4, &rc);
    if (rc) return rc;
    HIPCHK(c, hipMemcpy(d.groups, gs.data(), gs.size() * sizeof(QiwGroup), hipMemcpyHostToDevice));
    HIPCHK(c, hipMemcpy(d.prog, prog.data(), prog.size() * 8, hipMemcpyHostToDevice));
    HIPCHK(c, hipMemcpy(d.topo, topo.data(), topo.size() * 4, hipMemcpyHostToDevice));
    HIPCHK(c, hipMemcpy(d.coefs, coefs.data(), coefs.size() * 8, hipMemcpyHostToDevice));
    HIPCHK(c, hipMemcpy(d.tasks, b.tasks.data(), b.tasks.size() * sizeof(QiwTask), hipMemcpyHostToDevice));
    if (!b.g_first.empty()) {
        HIPCHK(c, hipMemcpy(d.g_first, b.g_first.data(), b.g_first.size() * 4, hipMemcpyHostToDevice));
        HIPCHK(c, hipMemcpy(d.g_count, b.g_count.data(), b.g_count.size() * 4, hipMemcpyHostToDevice));
        HIPCHK(c, hipMemcpy(d.g_slot, b.g_slot.data(), b.g_slot.size() * 4, hipMemcpyHostToDevice));
    }
    if (!b.r_first.empty()) {
        HIPCHK(c, hipMemcpy(d.r_first, b.r_first.data(), b.r_first.size() * 4, hipMemcpyHostToDevice));
        HIPCHK(c, hipMemcpy(d.r_count, b.r_count.data(), b.r_count.size() * 4, hipMemcpyHostToDevice));
    }
    // simplex coordinates of every sampled group (step independent unless scrambled per step)
    uint32_t *sm = (uint32_t *)dev(c, "sobol.m", c->sob_m.size() * 4, &rc);
    uint32_t *sx = (uint32_t *)dev(c, "sobol.x", c->sob_x.size() * 4, &rc);
    if (rc) return rc;
    HIPCHK(c, hipMemcpy(sm, c->sob_m.data(), c->sob_m.size() * 4, hipMemcpyHostToDevice));
    HIPCHK(c, hipMemcpy(sx, c->sob_x.data(), c->sob_x.size() * 4, hipMemcpyHostToDevice));
    for (auto &cg : b.groups) {
        if (!cg.g.sampled) continue;
        int dim = cg.g.d_before + cg.g.d_after;
        if (dim > c->sob_dim) return fail(c, QIW_E_DIM, "Sobol dimension beyond the staged direction numbers");
        if (b.scrambled) continue;
        if (cg.g.kind == QIW_G_SIGMA)
            HIPCHK(c, qiw_launch_sigma_coords(c->stream, sm, sx, cg.g.order, cg.g.n_samples, d.ut + cg.g.ut_off));
        else
            HIPCHK(c, qiw_launch_simplex_coords(c->stream, sm, sx, cg.g.d_before, cg.g.d_after, N, d.ut + cg.g.ut_off));
    }
    return 0;
}

// Randomized qMC parameters of a run (RandomizationParams, src/randomization.jl:46-57).
struct RandPlan {
    int n_seqs = 1;
    bool scrambled = false;
    bool given = false;   // the sequences are the caller's (qiw_set_scrambles or qiw_set_points)
    bool points = false;  // ... given as points (qiw_set_points)
    uint64_t seed = 0;
    double target_std = 0.0;
    int n_eval() const { return scrambled ? n_seqs : 1; }  // sequences evaluated per group
};
RandPlan rand_plan(const qiw_run *run) {
    RandPlan r;
    if (run && run->rand_params) {
        r.n_seqs = run->rand_params->N_seqs;
        r.scrambled = run->rand_params->scramble != 0;
        r.given = run->rand_params->scramble == 2 || run->rand_params->scramble == 3;
        r.points = run->rand_params->scramble == 3;
        r.seed = run->rand_params->seed;
        r.target_std = run->rand_params->target_std;
    }
    return r;
}

// Caller-drawn sequences of one launch row (a step, a correlator tau row): the sequences
// the reference constructs for the batch's groups, in group order (src/randomization.jl:
// 93-99): N_seqs per sampled group, except that a group whose integral vanishes
// identically -- no leaves in its programs, or a simplex of zero volume (`flat`) -- takes
// min(2, N_seqs), since with target_std = 0 the reference stops after the second sequence,
// whose deviation is exactly 0.  idx[g] is the sequence of entry g (-1: exact group; unused
// replicas repeat their group's first), used[r] the sequences real group r takes (1 for an
// exact one, as the bookkeeping counts it).  Returns the row's total.
// (With idx and used null, only the dimensions 2k of the row's sequences are appended to
// dims.)
template <class Flat>
int64_t given_row(const Batch &b, int n_seqs, int64_t base, Flat flat, int64_t *idx, int32_t *used,
                  std::vector<int32_t> *dims = nullptr) {
    int64_t n = 0;
    for (size_t r = 0; r < b.r_first.size(); ++r) {
        const int first = b.r_first[r], cnt = b.r_count[r];
        const Compiled &cg = b.groups[first];
        if (cg.g.order == 0 || (cg.g.kind == QIW_G_SIGMA && cg.g.order == 1)) {  // exact
            for (int q = 0; q < cnt && idx; ++q) idx[first + q] = -1;
            if (used) used[r] = 1;
            continue;
        }
        const int u = (cg.leaves_per_sample == 0 || flat(cg.g)) ? std::min(2, n_seqs) : n_seqs;
        for (int q = 0; q < cnt && idx; ++q) idx[first + q] = base + n + (q < u ? q : 0);
        if (used) used[r] = u;
        if (dims) dims->insert(dims->end(), u, 2 * cg.g.order);
        n += u;
    }
    return n;
}

// The reference's stopping rule ended real groups where given_row assumed it would: a
// group that given_row takes to vary (or to vanish) but whose sequences gave identical (or
// different) values would have made the reference consume other sequences from then on.
int check_given_use(qiw_ctx *c, const Batch &b, const std::vector<int32_t> &expect, const int32_t *dev_nuse,
                    const std::vector<int> &rows) {
    const size_t nr = b.r_first.size();
    if (!dev_nuse || nr == 0 || rows.empty()) return 0;
    const int max_row = *std::max_element(rows.begin(), rows.end());
    std::vector<int32_t> got((size_t)(max_row + 1) * nr);
    HIPCHK(c, hipMemcpy(got.data(), dev_nuse, got.size() * 4, hipMemcpyDeviceToHost));
    for (size_t i = 0; i < rows.size(); ++i)
        for (size_t r = 0; r < nr; ++r)
            if (got[(size_t)rows[i] * nr + r] != expect[i * nr + r]) {
                const QiwGroup &g = b.groups[b.r_first[r]].g;
                return fail(c, QIW_E_ARG,
                            "caller-drawn sequences: the group of order " + std::to_string(g.order) + ", n_pts_after " +
                                std::to_string(g.n_after) + " stopped after " + std::to_string(got[(size_t)rows[i] * nr + r]) +
                                " sequences, not " + std::to_string(expect[i * nr + r]) +
                                ": its values are identical across sequences without a structural zero, so the "
                                "reference would consume the caller's sequences differently");
            }
    return 0;
}

// The caller's sequences for a call that consumes `need` of them, for groups up to order
// max_order and N_samples n: checks the staged ones and returns their device copies
// (scrambled Sobol states, or points with `points`).
int given_buffers(qiw_ctx *c, bool points, int max_order, int64_t need, int64_t n, GivenSrc *src) {
    const int64_t have = points ? c->points_n : c->given_n;
    const int stride = points ? c->points_stride : c->given_stride;
    const char *what = points ? " caller-supplied point sequences, " : " caller-drawn sequences, ";
    const char *how = points ? " are staged (qiw_set_points)" : " are staged (qiw_set_scrambles)";
    if (need > have) return fail(c, QIW_E_ARG, "the call consumes " + std::to_string(need) + what + std::to_string(have) + how);
    if (need > 0 && stride < 2 * max_order)
        return fail(c, QIW_E_ARG, "the caller's sequences have fewer dimensions than 2 * order");
    if (need > 0 && points && c->points_npts < n)
        return fail(c, QIW_E_ARG, "the caller's point sequences hold fewer points than N_samples");
    int rc = 0;
    *src = GivenSrc{};
    src->stride = stride;
    if (points) {
        src->npts = c->points_npts;
        src->pts = (const double *)dev(c, "given.pts", (size_t)std::max<int64_t>(have, 1) * std::max<int64_t>(c->points_npts, 1) * std::max(stride, 1) * 8, &rc);
    } else {
        const size_t rows = (size_t)std::max<int64_t>(have, 1) * std::max(stride, 1);
        src->gm = (const uint32_t *)dev(c, "given.m", rows * 32 * 4, &rc);
        src->gx = (const uint32_t *)dev(c, "given.x", rows * 4, &rc);
    }
    return rc;
}

// Appends group cg (compiled) and, for a sampled group of a randomized run, its further
// sequences as replicas; `add_tasks(gi)` appends the tasks of entry gi.
template <class AddTasks>
void push_sequences(Batch &b, Compiled &&cg, int n_eval, AddTasks add_tasks) {
    const bool exact = cg.g.order == 0 || (cg.g.kind == QIW_G_SIGMA && cg.g.order == 1);
    const int n = exact ? 1 : n_eval;
    const int first = (int)b.groups.size();
    b.r_first.push_back(first);
    b.r_count.push_back(n);
    Compiled rep;
    if (n > 1) {  // the replicas carry no program
        rep.g = cg.g;
        rep.chunks = cg.chunks;
        rep.leaves_per_sample = cg.leaves_per_sample;
        rep.edges_per_sample = cg.edges_per_sample;
        rep.flops_per_sample = cg.flops_per_sample;
        rep.n_top = cg.n_top;
        rep.n_segments = cg.n_segments;
        rep.shape = cg.shape;
        rep.lds_bytes = cg.lds_bytes;
        rep.replica_of = first;
    }
    b.groups.push_back(std::move(cg));
    add_tasks(first);
    for (int q = 1; q < n; ++q) {
        b.groups.push_back(rep);
        b.groups.back().g.seq = q;
        add_tasks(first + q);
    }
}

int check_run(qiw_ctx *c, const qiw_run *run) {
    if (!c->has_model) return fail(c, QIW_E_STATE, "no model staged (qiw_set_model)");
    if (!run) return fail(c, QIW_E_ARG, "null run");
    if (!(run->N_samples == 0 || (run->N_samples > 0 && (run->N_samples & (run->N_samples - 1)) == 0)))
        return fail(c, QIW_E_NOT_POW2, "N_samples must be 0 or a power of 2");
    if (run->N_samples > (int64_t)1 << 30) return fail(c, QIW_E_LIMIT, "N_samples beyond 2^30");
    for (int i = 0; i < run->n_orders; ++i)
        if (run->orders[i] < 0 || run->orders[i] > QIW_KMAX) return fail(c, QIW_E_LIMIT, "order beyond QIW_KMAX");
    for (int i = 0; i < run->n_orders_bare; ++i)
        if (run->orders_bare[i] < 0 || run->orders_bare[i] > QIW_KMAX)
            return fail(c, QIW_E_LIMIT, "order beyond QIW_KMAX");
    if (c->sob_dim == 0) return fail(c, QIW_E_STATE, "no Sobol direction numbers staged (qiw_set_sobol)");
    if (run->rand_params) {
        const qiw_rand &r = *run->rand_params;
        if (r.N_seqs < 1) return fail(c, QIW_E_ARG, "rand_params.N_seqs must be > 0");
        if (r.N_seqs > QIW_MAX_SEQS) return fail(c, QIW_E_LIMIT, "rand_params.N_seqs beyond 64");
        if (r.scramble < 0 || r.scramble > 3) return fail(c, QIW_E_ARG, "rand_params.scramble must be 0, 1, 2 or 3");
        // the reference draws sequence s + 1 of a group only if it does not stop after s
        if (r.scramble >= 2 && r.target_std != 0.0)
            return fail(c, QIW_E_ARG, "the caller's sequences (scramble = 2, 3) need target_std = 0");
        if (!(r.target_std >= 0.0)) return fail(c, QIW_E_ARG, "rand_params.target_std must be >= 0");
    }
    return 0;
}

// Workgroup i of a launch runs on XCD i % 8 (round-robin dispatch over the 8 XCDs, each
// with its own L2).  The chunk tasks of one (group, sample block, tau) read the same
// coordinates and propagator rows, so they are kept on one XCD: bundles of such tasks go
// round-robin to the XCDs, and each XCD's list is laid out at positions x, x + 8, ...
constexpr int kXcds = 8;
void xcd_interleave(std::vector<QiwTask> &tasks) {
    std::vector<std::vector<QiwTask>> lists(kXcds);
    int xcd = -1;
    for (size_t i = 0; i < tasks.size(); ++i) {
        const QiwTask &t = tasks[i];
        const bool same = i > 0 && t.group == tasks[i - 1].group && t.first_sample == tasks[i - 1].first_sample &&
                          t.tau_index == tasks[i - 1].tau_index;
        if (!same) xcd = (xcd + 1) % kXcds;
        lists[xcd].push_back(t);
    }
    std::vector<QiwTask> out;
    out.reserve(tasks.size());
    std::vector<size_t> pos(kXcds, 0);
    for (bool more = true; more;) {  // one task of each XCD list per round; short lists drop out
        more = false;
        for (int x = 0; x < kXcds; ++x)
            if (pos[x] < lists[x].size()) {
                out.push_back(lists[x][pos[x]++]);
                more = true;
            }
    }
    tasks.swap(out);
}

// Vector programs are large (a group's trie runs to megabytes) and every sample block
// streams its chunk's program once per column pass, so the chunk, not the sample block, is
// what an XCD's L2 should keep: all tasks of one program chunk (its sample blocks, tau
// rows and sequences) go to one XCD back to back.  Chunks are assigned heaviest first to
// the least-loaded XCD, each XCD's list is laid out at positions x, x + 8, ...  (On the
// two-orbital step at N = 2^14 this takes the L2 fetches of a launch from 41 GiB to
// 0.17 GiB at the same run time.)
// A one-wavefront task is priced at its chunk's share of its group's cost (the compiler's
// words x columns), so that a group's short last chunk does not count as a full one
// (two-orbital step at N = 2^14: 5.08 s -> 4.90 s against equal shares).  With units of w
// tasks (the tasks of one workgroup, consecutive), a unit is placed as one, by the chunk of
// its first task, at w equal shares: pricing units by their chunks' shares (summed, or the
// longest) made the three-orbital step 0.4-0.6 % slower.
void xcd_by_chunk(Batch &b, int w) {
    std::map<std::pair<int, int>, size_t> key_of;  // (program, chunk) -> bucket
    std::vector<std::vector<QiwTask>> buckets;
    std::vector<double> cost;
    for (size_t u = 0; u < b.tasks.size(); u += w) {
        const QiwTask &t = b.tasks[u];
        const Compiled &cg = b.groups[t.group];
        const int prog = cg.replica_of >= 0 ? cg.replica_of : t.group;
        auto it = key_of.emplace(std::make_pair(prog, t.chunk), buckets.size()).first;
        if (it->second == buckets.size()) {
            buckets.emplace_back();
            cost.push_back(0.0);
        }
        buckets[it->second].insert(buckets[it->second].end(), b.tasks.begin() + u, b.tasks.begin() + u + w);
        const Compiled &pc = b.groups[prog];
        const double work = (double)(cg.edges_per_sample + cg.leaves_per_sample);
        const double even = 1.0 / (double)std::max<size_t>(pc.chunks.size(), 1);
        if (w == 1) {
            const size_t ci = std::lower_bound(pc.chunks.begin(), pc.chunks.end(), t.chunk) - pc.chunks.begin();
            cost[it->second] += work * (ci < pc.chunk_share.size() ? pc.chunk_share[ci] : even);
        } else {
            cost[it->second] += (double)w * work * even;
        }
    }
    std::vector<size_t> order(buckets.size());
    for (size_t i = 0; i < order.size(); ++i) order[i] = i;
    std::stable_sort(order.begin(), order.end(), [&](size_t x, size_t y) { return cost[x] > cost[y]; });
    std::vector<std::vector<QiwTask>> lists(kXcds);
    std::vector<double> load(kXcds, 0.0);
    for (size_t bi : order) {
        const int x = (int)(std::min_element(load.begin(), load.end()) - load.begin());
        lists[x].insert(lists[x].end(), buckets[bi].begin(), buckets[bi].end());
        load[x] += cost[bi];
    }
    std::vector<QiwTask> out;
    out.reserve(b.tasks.size());
    std::vector<size_t> pos(kXcds, 0);
    for (bool more = true; more;) {
        more = false;
        for (int x = 0; x < kXcds; ++x)
            if (pos[x] < lists[x].size()) {
                out.insert(out.end(), lists[x].begin() + pos[x], lists[x].begin() + pos[x] + w);
                pos[x] += w;
                more = true;
            }
    }
    b.tasks.swap(out);
}

// Workgroups of b.wg_waves tasks: the tasks of one sample block of a group (its topology
// chunks, consecutive after order_tasks' bucketing) are cut into units of wg_waves, the
// last one filled up with empty tasks (chunk -1, no output row).
void unit_tasks(Batch &b) {
    const int w = b.wg_waves;
    std::vector<QiwTask> out;
    out.reserve(b.tasks.size() + b.tasks.size() / 2 + w);
    size_t i = 0;
    while (i < b.tasks.size()) {
        size_t j = i + 1;
        const QiwTask &t0 = b.tasks[i];
        while (j < b.tasks.size() && b.tasks[j].group == t0.group && b.tasks[j].first_sample == t0.first_sample &&
               b.tasks[j].tau_index == t0.tau_index)
            ++j;
        out.insert(out.end(), b.tasks.begin() + i, b.tasks.begin() + j);
        for (size_t k = j - i; k % w; ++k) out.push_back(QiwTask{t0.group, t0.first_sample, t0.tau_index, -1, -1, 0});
        i = j;
    }
    b.tasks.swap(out);
}

// Heaviest groups first: workgroups are dispatched in task order, so the long tasks do
// not form the tail of the launch.  Each task keeps its output row, so the summation
// order of the results does not change.  Tasks are bucketed by group (linear time).
void order_tasks(Batch &b) {
    const size_t ng = b.groups.size();
    std::vector<int> go(ng);
    for (size_t i = 0; i < ng; ++i) go[i] = (int)i;
    if (b.fmt == FMT_SARC) {  // one launch for all: the small groups fill the large ones' tail
        int shape = 0;
        for (const Compiled &cg : b.groups) shape = std::max(shape, cg.shape);
        for (Compiled &cg : b.groups) cg.shape = shape;
    }
    if (b.fmt >= FMT_ARC) {  // one launch per workgroup shape, heaviest groups first in each
        std::stable_sort(go.begin(), go.end(), [&](int x, int y) {
            const Compiled &p = b.groups[x], &q = b.groups[y];
            return p.shape != q.shape ? p.shape > q.shape : p.flops_per_sample > q.flops_per_sample;
        });
        std::vector<std::vector<QiwTask>> of(ng);
        for (const QiwTask &t : b.tasks) of[t.group].push_back(t);
        b.tasks.clear();
        for (int gi : go) {
            const Compiled &cg = b.groups[gi];
            if (of[gi].empty()) continue;
            if (b.launches.empty() || b.launches.back().shape != cg.shape)
                b.launches.push_back({(int)b.tasks.size(), 0, cg.shape, 0});
            Batch::Launch &ln = b.launches.back();
            ln.count += (int)of[gi].size();
            ln.lds = std::max(ln.lds, cg.lds_bytes);
            b.tasks.insert(b.tasks.end(), of[gi].begin(), of[gi].end());
        }
        return;
    }
    auto weight = [&](int gi) { return b.groups[gi].edges_per_sample + b.groups[gi].leaves_per_sample; };
    std::stable_sort(go.begin(), go.end(), [&](int x, int y) { return weight(x) > weight(y); });
    std::vector<size_t> count(ng, 0), start(ng, 0);
    for (const QiwTask &t : b.tasks) count[t.group]++;
    size_t pos = 0;
    for (int gi : go) {
        start[gi] = pos;
        pos += count[gi];
    }
    std::vector<QiwTask> out(b.tasks.size());
    for (const QiwTask &t : b.tasks) out[start[t.group]++] = t;
    b.tasks.swap(out);
    if (b.wg_waves > 1) {
        unit_tasks(b);
        xcd_by_chunk(b, b.wg_waves);
    } else if (b.fmt == FMT_VEC) {
        xcd_by_chunk(b, 1);
    } else {
        xcd_interleave(b.tasks);
    }
}

// The matrix-core walk's layout of the operator blocks and of the i*P blocks of a segment:
// row-major, rows padded to a multiple of 4 floats, every block 16-byte aligned, so a lane
// reads four consecutive elements of a row with one load.
static void wide_layout(HostModel &m) {
    const size_t nb = m.op_desc.size() / 3;
    m.op_rm_off.assign(nb, 0);
    m.ops_rm.clear();
    for (size_t b = 0; b < nb; ++b) {
        const int off = m.op_desc[3 * b], mf = m.op_desc[3 * b + 1], mi = m.op_desc[3 * b + 2];
        const int ldr = (mi + 3) & ~3;
        m.op_rm_off[b] = (int32_t)m.ops_rm.size();
        m.ops_rm.resize(m.ops_rm.size() + (size_t)mf * ldr, 0.f);
        for (int i = 0; i < mf; ++i)
            for (int j = 0; j < mi; ++j) m.ops_rm[m.op_rm_off[b] + (size_t)i * ldr + j] = (float)m.op_data[off + i + j * mf];
    }
    m.ops_rm.resize(m.ops_rm.size() + 4, 0.f);  // the four zeros read by lanes outside a block
    m.lds_off.assign(m.ns, 0);
    m.btp = 0;
    for (int s = 0; s < m.ns; ++s) {
        m.lds_off[s] = m.btp;
        m.btp += m.dims[s] * ((m.dims[s] + 3) & ~3);
    }
    m.pinv.assign(m.btp, -1);
    for (int s = 0; s < m.ns; ++s) {
        const int d = m.dims[s], ldr = (d + 3) & ~3;
        for (int i = 0; i < d; ++i)
            for (int j = 0; j < d; ++j) m.pinv[m.lds_off[s] + i * ldr + j] = m.bt_off[s] + i + j * d;
    }
}

// Rows the Y stack of the matrix-core walk can hold at once: the largest sum of block sizes
// over `levels` consecutive levels of a path.  Consecutive levels are joined by an operator
// (of a pair, or of a correlator) or, at most once per path, by the identity node at tau_w.
static int ystack_rows(const HostModel &m, int levels) {
    if (levels <= 0) return 0;
    std::vector<std::vector<int>> nb(m.ns);  // nb[s]: sectors an operator takes to s
    for (const std::vector<ScalarOp> *ops : {&m.op_i, &m.op_f, &m.corr_A, &m.corr_B})
        for (const ScalarOp &o : *ops)
            for (int s = 0; s < m.ns && s < (int)o.sf.size(); ++s)
                if (o.sf[s] >= 0) nb[o.sf[s]].push_back(s);
    // best[u][s]: largest sum over paths ending in sector s, u = identity node used
    std::vector<int> b0(m.dims.begin(), m.dims.end()), b1(m.ns, -1), n0(m.ns), n1(m.ns);
    for (int l = 1; l < levels; ++l) {
        for (int s = 0; s < m.ns; ++s) {
            int x0 = -1, x1 = b0[s];
            for (int p : nb[s]) {
                x0 = std::max(x0, b0[p]);
                x1 = std::max(x1, b1[p]);
            }
            n0[s] = x0 < 0 ? -1 : m.dims[s] + x0;
            n1[s] = x1 < 0 ? -1 : m.dims[s] + x1;
        }
        b0.swap(n0);
        b1.swap(n1);
    }
    int r = 0;
    for (int s = 0; s < m.ns; ++s) r = std::max(r, std::max(b0[s], b1[s]));
    return r;
}

// Samples per task.  The scalar and vector walks map one sample to a lane (64 per task);
// the block and matrix-core walks evaluate one sample at a time per wavefront, so their
// tasks are cut smaller until a launch holds at least 4 tasks per SIMD of the device.
// The arc walk takes a workgroup per sample: its tasks are cut until a launch holds 4096, or as
// many as there may be rows (rows: for its sample blocks; step_rows).
int samples_per_task(const qiw_ctx *c, const HostModel &m, int fmt, int64_t total_samples, int64_t rows = INT64_MAX) {
    if (fmt == FMT_SCALAR || fmt == FMT_SARC || (fmt == FMT_VEC && m.mmax <= 6)) return QIW_WAVE;
    if (c->tune.samples_per_task > 0) {
        int spt = c->tune.samples_per_task;  // blocks up to 6, whose vector walk takes 64: within the rows
        while (fmt == FMT_ARC && m.mmax <= 6 && spt < QIW_WAVE && total_samples / spt > rows) spt *= 2;
        return spt;
    }
    int spt = QIW_WAVE;
    while (spt > 1 && total_samples / spt < 4096 && (fmt != FMT_ARC || 2 * total_samples / spt <= rows)) spt /= 2;
    return spt;
}

// Task rows of a step that fit the scratch array of qiw_inchworm_step_noalloc beside its other
// per-call buffers (per_call_buffer): n_slots order slots, n_groups groups of n_eval sequences.
int64_t step_rows(const qiw_ctx *c, const RandPlan &rq, int64_t n_slots, int64_t n_groups) {
    const HostModel &m = c->m;
    const bool rqmc = rq.n_seqs > 1;
    const int64_t row = 8 * (int64_t)m.bt, up = 10 * 256;  // (each buffer starts at 256 bytes)
    const int64_t others = row * (m.ntau * (1 + n_slots * (rqmc ? 2 : 1)) + n_groups * (rq.n_eval() + (rqmc ? 2 : 0))) +
                           8 * (int64_t)m.ntau + 4 * (int64_t)m.bt + (rq.scrambled ? 4 * (int64_t)c->sob_m.size() : 0) + up;
    return std::max<int64_t>(0, (int64_t)kNoAllocScratchBytes - others) / row;
}

std::vector<int> orders_all(const qiw_run *run) {
    std::vector<int> v(run->orders, run->orders + run->n_orders);
    v.insert(v.end(), run->orders_bare, run->orders_bare + run->n_orders_bare);
    std::sort(v.begin(), v.end());
    v.erase(std::unique(v.begin(), v.end()), v.end());
    return v;
}

// Build the groups of a bold step (src/inchworm.jl:422-452) or the bare step (:373-392).
// Words per topology chunk of flat scalar programs: long groups are cut into several tasks
// per sample block so that no single task sets the length of a launch.
constexpr int kChunkWords = 896;
// The same for the self-energy batches of the differential steps: their launches are small
// (one τ_f row, orders 1..), and shorter chunks keep more workgroups in flight (C1,
// 199 steps: 24.1 ms at 640 words against 26.7 ms at 896).
constexpr int kChunkWordsDiff = 640;
// Column-words (program words x columns each segment is replayed for) per topology chunk of
// vector programs, for the vector and matrix-core walks.
constexpr int64_t kChunkCost = 1 << 18;
// With few sample blocks a launch holds few tasks and its length is that of one chunk, so
// the chunks shrink in proportion below 256 sample blocks (x tau rows), down to 2^14
// column-words (the two-orbital inchworm! at N = 2^8 has 4 blocks per group).
int64_t vec_chunk_cost(const qiw_ctx *c, int64_t N, int64_t rows) {
    if (c->tune.chunk_cost > 0) return c->tune.chunk_cost;
    const int64_t blocks = std::max<int64_t>(1, (N + QIW_WAVE - 1) / QIW_WAVE) * std::max<int64_t>(rows, 1);
    if (blocks >= 256) return kChunkCost;
    return std::max<int64_t>((int64_t)1 << 14, kChunkCost * blocks / 256);
}

// A group that does not fit the arc walk: the batch is built again from assignment tries.
constexpr int kArcNoFit = 1;

// Compiles one group in the batch's format.  chunk_words, chunk_cost: as in Compiler.
int compile_group(qiw_ctx *c, const Batch &b, int kind, int order, int n_after, int corr, int chunk_words,
                  int64_t chunk_cost, Compiled &cg) {
    if (b.fmt == FMT_ARC) {
        const int rc = compile_arcs(c->m, kind, order, n_after, corr, b.precision, cg);
        return rc == 1 ? fail(c, QIW_E_OFFDIAG, kOffDiagonal) : rc == 2 ? kArcNoFit : 0;
    }
    if (b.fmt == FMT_SARC) {
        const int rc = compile_scalar_arcs(c->m, kind, order, n_after, {corr}, c->tune.chunk_words, cg);
        return rc == 1 ? fail(c, QIW_E_OFFDIAG, kOffDiagonal) : rc == 2 ? kArcNoFit : 0;
    }
    Compiler comp(c->m, kind, order, n_after, corr, b.fmt, b.max_order);
    comp.chunk_words = chunk_words;
    comp.chunk_cost = chunk_cost;
    return comp.compile(cg) ? 0 : fail(c, QIW_E_OFFDIAG, comp.err);
}

// Format and workgroup width of a batch (max_order and precision set).
void set_format(const HostModel &m, Batch &b, bool arcs) {
    b.fmt = arcs ? eval_format(m, b.max_order, b.precision) : program_format(m, b.max_order, b.precision);
    b.wg_waves = (b.fmt == FMT_VEC && m.mmax > 6) ? kMfmaWaves : 1;
}

// The program parts of a group that get tasks of their own per sample block (QiwTask::chunk
// and pad_): topology chunks, or for the arc walk its segments in up to `most` parts.
std::vector<std::pair<int32_t, int32_t>> task_parts(const Batch &b, const Compiled &cg, int64_t most) {
    std::vector<std::pair<int32_t, int32_t>> v;
    if (b.fmt != FMT_ARC) {
        for (int32_t ch : cg.chunks) v.push_back({ch, 0});
    } else if (most > 1 && cg.n_segments > 1) {
        const int64_t n = std::min<int64_t>(most, cg.n_segments);
        for (int64_t i = 0; i < n; ++i) {
            const int32_t first = (int32_t)(i * cg.n_segments / n);
            v.push_back({first, (int32_t)((i + 1) * cg.n_segments / n) - first});
        }
    } else {
        v.push_back({-1, 0});
    }
    return v;
}

// Estimated seconds of a batch's evaluator at N samples per sampled group and `rows` tau rows, for
// the choice between the arc walk and the walks of the assignment tries.  The arc walk takes a
// workgroup per sample, whose set-up (times, arc values, every sector's propagators) and barriers
// it pays for however little there is to sum; the vector walk takes a sample per lane and only
// the blocks of its chains.  So at order 1, and for blocks of two or three at order 2, the vector
// walk is faster once its launch, as long as one wavefront's walk of the longest program, is
// full; likewise the LDS block walk for wide blocks in float64.  Measured (arc walk, trie walk; ms):
//   two orbitals, order 1, N = 2^12 .283 .681, 2^15 1.52 .765, 2^18 11.4 2.68; orders 0:2, N = 2^18
//   63.8 131 (float32 43.2 47.7); orders 0:3, N = 2^12 8.2 126;
//   blocks up to 3, order 1, N = 2^18 5.53 .540; orders 0:2, N = 2^12 .582 .896, 2^18 27.7 10.1; orders
//   0:3, N = 2^12 1.75 9.6;
//   128 blocks of 4, order 1, N = 2^9 1.58 5.25, 2^12 10.4 5.15, 2^15 76.8 6.34;
//   blocks up to 10 in float64, order 1, N = 2^15 7.37 2.80; orders 0:2, N = 2^12 6.14 12.4.
// The rates are fits to these and to 110 further sizes: the walk chosen is the faster one or within a
// fifth of it, but for launches below 0.5 ms.
int64_t group_samples(const QiwGroup &g, int64_t N) {
    return g.order == 0 || (g.kind == QIW_G_SIGMA && g.order == 1) ? 1 : std::max<int64_t>(N, 1);
}
double arc_seconds(const HostModel &m, const Batch &b, int64_t N, int64_t rows) {
    double t = 8e-5;
    for (const Compiled &cg : b.groups) {
        // workgroups at a time; a barrier per stage and segment; a lookup per propagator element
        const double wgs = 256.0 * std::max<size_t>(1, std::min<size_t>(12 / cg.shape, (160 << 10) / std::max<size_t>(cg.lds_bytes, 1)));
        const double sample = (cg.n_segments * (2.0 * cg.g.order + 1) + 4) * 1.6e-6 / wgs + m.bt * (cg.g.n_nodes - 1.0) * 5e-11;
        t += (double)rows * group_samples(cg.g, N) * sample * (b.precision == QIW_PREC_FP32 ? 0.7 : 1.0);
    }
    return t;
}
// least: of an arc batch, what the tries would take at least (4.5 words per diagram, the FLOPs of
// the merged diagrams).
double trie_seconds(const HostModel &m, const Batch &b, bool least, int64_t N, int64_t rows) {
    double longest = 0, t = 0;
    const bool vec = m.mmax <= 6;
    for (const Compiled &cg : b.groups) {
        const Compiled &own = cg.replica_of >= 0 ? b.groups[cg.replica_of] : cg;  // (sequences share a program)
        const double words = least ? 4.5 * cg.leaves_per_sample : (double)own.prog.size();
        longest = std::max(longest, words);
        t += (double)rows * group_samples(cg.g, N) * (vec ? words * m.mmax * 2e-11 : sample_flops(cg) / 1.3e12);
    }
    const bool fp32 = b.precision == QIW_PREC_FP32;
    return vec ? 1e-4 + std::max(longest * (m.mmax * 8e-7 + m.bt * 1e-9) * (fp32 ? 0.6 : 1.0), t * (fp32 ? 0.5 : 1.0))
               : 5e-5 + std::max(longest * m.mmax * 1e-7, t);
}
// Whether the batch `arcs` would be faster on the walks of the tries (tries: builds the batch there).
template <class Build>
int prefer_tries(const HostModel &m, Batch &arcs, int64_t N, int64_t rows, Build build) {
    if (arcs.fmt != FMT_ARC || (m.mmax > 6 && arcs.precision == QIW_PREC_FP32)) return 0;
    if (program_format(m, arcs.max_order, arcs.precision) == FMT_BLOCK && m.mmax <= 6) return 0;
    const double t = arc_seconds(m, arcs, N, rows);
    if (trie_seconds(m, arcs, true, N, rows) >= t) return 0;
    Batch tries;
    const int rc = build(tries);
    if (rc) return rc;
    const bool fits = arcs.groups.empty() || tries.fmt != FMT_BLOCK || (size_t)tries.lds * 8 <= 160 * 1024;
    if (fits && trie_seconds(m, tries, false, N, rows) < t) arcs = std::move(tries);
    return 0;
}

// Parts the segments of an arc program may be cut into: as many as there are when the sample
// blocks alone are fewer than 2048 workgroups, within `rows` task rows for `blocks` blocks.  A
// program cut by its first pairs has hundreds of segments (three orbitals, order 3, float64: 84),
// whose rows would take more than the scratch array of a no-alloc step.
int64_t most_parts(int64_t total_blocks, int64_t blocks, int64_t rows) {
    return total_blocks < 2048 ? std::max<int64_t>(1, rows / std::max<int64_t>(1, blocks)) : 1;
}
// Rows of a call that allocates what it needs: as many as the scratch array would hold.
int64_t call_rows(const HostModel &m) { return (int64_t)kNoAllocScratchBytes / (8 * (int64_t)m.bt); }

int build_step_batch_as(qiw_ctx *c, const qiw_run *run, bool bare, const std::vector<int> &oall, Batch &b, bool split,
                        bool arcs) {
    const HostModel &m = c->m;
    int n_o = bare ? run->n_orders_bare : run->n_orders;
    const int32_t *ord = bare ? run->orders_bare : run->orders;
    int max_order = 0;
    int64_t n_groups = 0;
    for (int oi = 0; oi < n_o; ++oi) {
        max_order = std::max(max_order, (int)ord[oi]);
        if (ord[oi] > 0) n_groups += bare ? 1 : 2 * ord[oi] - 1;
    }
    const RandPlan rq = rand_plan(run);
    b.n_eval = rq.n_eval();
    b.scrambled = rq.scrambled;
    b.given = rq.given;
    b.max_order = max_order;
    b.precision = chain_precision(m, max_order, run->precision);
    set_format(m, b, arcs);
    const int64_t total = n_groups * b.n_eval * std::max<int64_t>(run->N_samples, 1);
    const int64_t rows = step_rows(c, rq, (int64_t)oall.size(), n_groups + 1);
    b.spt = samples_per_task(c, m, b.fmt, total, rows - n_groups * b.n_eval - 1);
    const int64_t blocks = n_groups * b.n_eval * ((run->N_samples + b.spt - 1) / b.spt) + 1;
    for (int oi = 0; oi < n_o; ++oi) {
        int order = ord[oi];
        if (order > 0 && run->N_samples <= 0) continue;
        std::vector<int> nas;
        if (bare)
            nas.push_back(2 * order);
        else if (order == 0)
            nas.push_back(0);
        else
            for (int na = 1; na <= 2 * order - 1; ++na)
                if (run->n_pts_after_max <= 0 || na <= run->n_pts_after_max) nas.push_back(na);
        for (int na : nas) {
            Compiled cg;
            const int words = c->tune.chunk_words > 0 ? c->tune.chunk_words : kChunkWords;
            const int rc = compile_group(c, b, bare ? QIW_G_BARE : QIW_G_BOLD, order, na, -1, split ? words : 0,
                                         split ? vec_chunk_cost(c, run->N_samples, 1) : 0, cg);
            if (rc) return rc;
            if (cg.n_top == 0) continue;
            if (cg.g.n_wslots > 255 || m.ns > 255)
                return fail(c, QIW_E_LIMIT, "too many slots");
            b.lds = std::max(b.lds, lds_slots(cg, m, b.fmt));
            int slot = (int)(std::find(oall.begin(), oall.end(), order) - oall.begin());
            int64_t N = order > 0 ? run->N_samples : 1;
            const auto parts = task_parts(b, cg, split ? most_parts(total / b.spt, blocks, rows) : 1);
            const double flops = (double)N * sample_flops(cg);
            const int64_t leaves = N * cg.leaves_per_sample, evals = N * cg.n_top;
            push_sequences(b, std::move(cg), b.n_eval, [&](int gi) {
                b.g_first.push_back((int32_t)b.tasks.size());
                const int64_t nt64 = (N + b.spt - 1) / b.spt;
                const int nt = tasks_fit(b, nt64 * (int64_t)parts.size()) ? (int)nt64 : 0;
                for (int t = 0; t < nt; ++t)
                    for (auto &p : parts)
                        b.tasks.push_back({gi, t * b.spt, 0, (int32_t)b.tasks.size(), p.first, p.second});
                b.g_count.push_back(nt * (int)parts.size());
                b.g_slot.push_back(slot);
                b.flops_per_launch += flops;
                b.leaves_per_launch += leaves;
                b.diagram_evals_per_launch += evals;
            });
        }
    }
    if (b.r_first.size() > 64) return fail(c, QIW_E_LIMIT, "more than 64 (order, n_pts_after) groups in one step");
    if (b.overflow) return fail(c, QIW_E_LIMIT, "more than 2^28 workgroups in one launch (lower N_samples)");
    order_tasks(b);
    return 0;
}

int build_step_batch(qiw_ctx *c, const qiw_run *run, bool bare, const std::vector<int> &oall, Batch &b,
                     bool split = true) {
    b = Batch{};
    const int rc = build_step_batch_as(c, run, bare, oall, b, split, true);
    if (rc == 0)
        return prefer_tries(c->m, b, run->N_samples, 1,
                            [&](Batch &t) { return build_step_batch_as(c, run, bare, oall, t, split, false); });
    if (rc != kArcNoFit) return rc;
    b = Batch{};
    return build_step_batch_as(c, run, bare, oall, b, split, false);
}

}  // namespace

// ---------------------------------------------------------------------------------------
// Plans: a compiled batch and its device copy (programs, tasks, simplex coordinates) kept
// under its buffer tag, and reused while the model content, the Sobol tables and the run
// parameters it was built from stay the same.  Warped coordinates are rewritten on every
// step, so a plan of warped groups is never reused.
// ---------------------------------------------------------------------------------------
namespace qiwi {
struct Plan {
    std::string key;
    Batch b;
    DevBatch d;
    bool first_is_order0 = false;  // correlator plans: the leading group is order 0
    bool fits = false;             // plan of all pairs: its groups fit the scalar arc walk
    int32_t *rf = nullptr, *rcnt = nullptr;  // correlator plans: per (tau row, group) task ranges
};
struct PlanStore {
    std::map<std::string, Plan> by_tag;
    std::map<std::string, uint64_t> last_use;  // step plans: use counter of each buffer tag
    uint64_t clock = 0;
};
void plans_destroy(PlanStore *p) { delete p; }

// The bold-step loop of an inchworm run (per step: coordinates when scrambled, the
// evaluator's launches, the bookkeeping kernel) captured once and replayed while every launch is
// the same: `key` holds the bytes of their arguments, and of the evaluators' workgroup counts,
// shapes and LDS (launch_eval), which two programs of one order and sample count need not share.
struct StepGraph {
    std::string key;
    hipGraph_t graph = nullptr;
    hipGraphExec_t exec = nullptr;
    std::vector<hipEvent_t> ev;  // two around each replay
    void clear() {
        if (exec) (void)hipGraphExecDestroy(exec);
        if (graph) (void)hipGraphDestroy(graph);
        for (auto e : ev) (void)hipEventDestroy(e);
        exec = nullptr;
        graph = nullptr;
        ev.clear();
        key.clear();
    }
};
void step_graph_destroy(StepGraph *g) {
    if (g) g->clear();
    delete g;
}
}  // namespace qiwi

namespace {

Plan &plan_slot(qiw_ctx *c, const std::string &tag) {
    if (!c->plans) c->plans = new PlanStore;
    return c->plans->by_tag[tag];
}

std::string plan_key(const qiw_ctx *c, const qiw_run *run, const std::vector<int> &oall, const std::string &kind) {
    std::string k = kind;
    auto put = [&](const void *p, size_t n) { k.append((const char *)p, n); };
    put(&run->N_samples, 8);
    put(&run->n_pts_after_max, 4);
    put(&run->precision, 4);
    put(&run->n_orders, 4);
    put(run->orders, 4 * (size_t)run->n_orders);
    put(&run->n_orders_bare, 4);
    put(run->orders_bare, 4 * (size_t)run->n_orders_bare);
    const int no = (int)oall.size();
    put(&no, 4);
    put(oall.data(), 4 * (size_t)no);
    put(&c->sob_dim, 4);
    put(c->sob_m.data(), 4 * c->sob_m.size());
    put(c->sob_x.data(), 4 * c->sob_x.size());
    put(&c->tune.chunk_words, 4);
    put(&c->tune.samples_per_task, 4);
    put(&c->tune.chunk_cost, 8);
    const RandPlan rq = rand_plan(run);
    const int rk[2] = {rq.n_eval(), rq.given ? 2 : rq.scrambled ? 1 : 0};
    put(rk, 8);
    return k + c->model_fp;
}

// Step plans kept per kind (bare / bold), so that runs alternating between settings (two
// sample counts, the tuner's candidates) reuse them; the least recently used is replaced.
constexpr int kStepPlanSlots = 2;

// The plan of a bare or bold step batch (buffer tags "bare", "bare.1", "bold", "bold.1"),
// built and uploaded unless a resident one matches.
int step_plan(qiw_ctx *c, const qiw_run *run, const std::vector<int> &oall, bool bare, bool warp, Plan *&out) {
    const std::string kind = bare ? "bare" : "bold";
    const std::string key = plan_key(c, run, oall, kind);
    if (!c->plans) c->plans = new PlanStore;
    PlanStore &ps = *c->plans;
    std::string tag = kind;
    uint64_t oldest = UINT64_MAX;
    for (int i = 0; i < kStepPlanSlots; ++i) {
        const std::string t = i == 0 ? kind : kind + "." + std::to_string(i);
        auto it = ps.by_tag.find(t);
        if (!warp && it != ps.by_tag.end() && it->second.key == key) {
            tag = t;
            oldest = 0;
            break;
        }
        const uint64_t u = it == ps.by_tag.end() ? 0 : ps.last_use[t];
        if (u < oldest) {
            oldest = u;
            tag = t;
        }
    }
    Plan &p = plan_slot(c, tag);
    out = &p;
    ps.last_use[tag] = ++ps.clock;
    if (!warp && p.key == key) return 0;
    if (c->no_alloc)
        return fail(c, QIW_E_STATE, "no resident plan for this run: call qiw_inchworm_step once with the same run first");
    p = Plan{};
    int rc = build_step_batch(c, run, bare, oall, p.b);
    if (rc) return rc;
    const bool weighted = warp && !p.b.groups.empty();
    if (weighted && program_format(c->m, p.b.max_order, p.b.precision) == FMT_BLOCK)
        return fail(c, QIW_E_LIMIT, "the learned warp needs sector blocks <= 6 and orders <= 4");
    if (!p.b.groups.empty() && (rc = upload(c, tag, p.b, run->N_samples, p.d, weighted))) return rc;
    if (!weighted) p.key = key;
    return 0;
}

// Transfers of a call through the context's pinned buffer: what a call hands over (tables,
// zeros) goes to the device in one kernel that reads the buffer, and its results come back in
// one that writes it.  Nine synchronous copies and three fills took 130 us of a small step.
// Pieces of more than kStageDirect bytes are copied on the stream, where a copy engine is
// faster than loads over the bus.  Without a buffer (no-alloc calls that need more than there
// is) every piece is copied by itself.
constexpr size_t kStageDirect = 64 << 10;
struct Stage {
    qiw_ctx *c;
    struct Piece {
        void *to;
        const void *from;  // null: zeros
        size_t bytes;
    };
    std::vector<Piece> pieces;
    explicit Stage(qiw_ctx *c_) : c(c_) {}
    void add(void *to, const void *from, size_t bytes) {
        if (bytes) pieces.push_back({to, from, bytes});
    }
    template <class T>
    void add(void *to, const std::vector<T> &v) {
        add(to, v.data(), v.size() * sizeof(T));
    }
    static size_t up(size_t b) { return (b + 15) & ~(size_t)15; }
    char *pinned(size_t bytes) {
        if (c->pin_busy) {  // a call that failed may have left work that reads it
            if (hipStreamSynchronize(c->stream) != hipSuccess) return nullptr;
            c->pin_busy = false;
        }
        if (c->pin_bytes >= bytes) return (char *)c->pin;
        if (c->no_alloc) return nullptr;
        if (c->pin) (void)hipHostFree(c->pin);
        c->pin = nullptr;
        c->pin_bytes = 0;
        const size_t n = std::max<size_t>(bytes, 256 << 10);
        if (hipHostMalloc(&c->pin, n, hipHostMallocDefault) != hipSuccess) {
            (void)hipGetLastError();
            c->pin = nullptr;
            return nullptr;
        }
        c->pin_bytes = n;
        return (char *)c->pin;
    }
    hipError_t launch(const std::vector<StageOp> &ops) {
        hipError_t e = hipSuccess;
        for (size_t i = 0; i < ops.size() && e == hipSuccess; i += kStageOps) {
            StageArgs a{};
            a.n = (int)std::min<size_t>(kStageOps, ops.size() - i);
            std::copy(ops.begin() + i, ops.begin() + i + a.n, a.op);
            e = qiw_launch_stage(c->stream, a);
        }
        return e;
    }
    // To the device, in stream order.
    int upload() {
        size_t total = 0;
        for (const Piece &p : pieces)
            if (p.from) total += up(p.bytes);
        char *pin = pinned(total);
        std::vector<StageOp> ops;
        size_t at = 0;
        if (pin) c->pin_busy = true;
        for (const Piece &p : pieces) {
            if (p.from && !pin) {
                HIPCHK(c, hipMemcpy(p.to, p.from, p.bytes, hipMemcpyHostToDevice));
                continue;
            }
            if (p.from) {
                std::memcpy(pin + at, p.from, p.bytes);
                if (p.bytes > kStageDirect) {
                    HIPCHK(c, hipMemcpyAsync(p.to, pin + at, p.bytes, hipMemcpyHostToDevice, c->stream));
                    at += up(p.bytes);
                    continue;
                }
            }
            ops.push_back(StageOp{(uint32_t *)p.to, p.from ? (const uint32_t *)(pin + at) : nullptr, (int64_t)(p.bytes / 4)});
            if (p.from) at += up(p.bytes);
        }
        HIPCHK(c, launch(ops));
        pieces.clear();
        return 0;
    }
    // Back to the host; the stream is idle afterwards.
    int download() {
        size_t total = 0;
        for (const Piece &p : pieces) total += up(p.bytes);
        if (c->pin_busy && c->pin_bytes < total) {
            HIPCHK(c, hipStreamSynchronize(c->stream));
            c->pin_busy = false;
        }
        // what the upload left in the buffer has been read when the kernels below run
        char *pin = c->pin_bytes >= total ? (char *)c->pin : pinned(total);
        std::vector<StageOp> ops;
        size_t at = 0;
        for (const Piece &p : pieces) {
            if (!pin) break;
            if (p.bytes > kStageDirect)
                HIPCHK(c, hipMemcpyAsync(pin + at, p.from, p.bytes, hipMemcpyDeviceToHost, c->stream));
            else
                ops.push_back(StageOp{(uint32_t *)(pin + at), (const uint32_t *)p.from, (int64_t)(p.bytes / 4)});
            at += up(p.bytes);
        }
        HIPCHK(c, launch(ops));
        HIPCHK(c, hipStreamSynchronize(c->stream));
        c->pin_busy = false;
        at = 0;
        for (const Piece &p : pieces) {
            if (pin)
                std::memcpy(p.to, pin + at, p.bytes);
            else
                HIPCHK(c, hipMemcpy(p.to, p.from, p.bytes, hipMemcpyDeviceToHost));
            at += up(p.bytes);
        }
        pieces.clear();
        return 0;
    }
};

int ensure_model_buffers(qiw_ctx *c, double **dcoef, int32_t **dkind, double **eshift, Stage *stage = nullptr) {
    int rc = 0;
    const HostModel &m = c->m;
    *dcoef = (double *)dev(c, "delta.coef", std::max<size_t>(m.dcoef.size(), 1) * 8, &rc);
    *dkind = (int32_t *)dev(c, "delta.kind", std::max<size_t>(m.dkind.size(), 1) * 4, &rc);
    double *ddlr = (double *)dev(c, "delta.dlr", std::max<size_t>(m.dlr.size(), 1) * 8, &rc);
    size_t n_eig = 0;
    for (int s = 0; s < m.ns; ++s) n_eig += m.dims[s];
    *eshift = (double *)dev(c, "eshift", n_eig * 8, &rc);
    if (rc) return rc;
    c->es.clear();  // E + lambda per eigenvalue, sector-major
    for (int s = 0; s < m.ns; ++s)
        for (double e : m.E[s]) c->es.push_back(e + m.lambda0);
    Stage own(c), &st = stage ? *stage : own;
    st.add(ddlr, m.dlr);
    st.add(*dcoef, m.dcoef);
    st.add(*dkind, m.dkind);
    st.add(*eshift, c->es);
    return stage ? 0 : own.upload();
}

// Device tables of the arc walk: the operator blocks (as the products read them, and
// column-major), E + lambda and the layout of the blocks.  Staged once per model and
// precision (synchronous copies).
int stage_arcs(qiw_ctx *c, int precision, ArcArgs *aa) {
    const HostModel &m = c->m;
    const bool fp32 = precision == QIW_PREC_FP32;
    const size_t pad = 64, nb = m.op_desc.size() / 3, per = arc_block_size(m, fp32), el = fp32 ? 4 : 8;
    int rc = 0;
    void *blocks = dev(c, fp32 ? "arc.slices" : "arc.blocks", (nb + 1) * per * el, &rc);
    void *cm = dev(c, fp32 ? "arc.ops32" : "arc.ops", (m.op_data.size() + pad) * el, &rc);
    double *ediag = (double *)dev(c, "arc.ediag", (size_t)m.bt * 8, &rc);
    uint8_t *emask = (uint8_t *)dev(c, "arc.emask", (size_t)m.bt, &rc);
    int32_t *lay = (int32_t *)dev(c, "arc.layout", ((size_t)m.bt + 2 * m.ns) * 4, &rc);
    if (rc) return rc;
    if (!(c->arc_staged & (fp32 ? 2 : 1))) {
        HIPCHK(c, hipStreamSynchronize(c->stream));
        const int mb = qiw_arc_rows(m.mmax);
        std::vector<double> o(m.op_data), s((nb + 1) * per, 0.0);
        o.resize(m.op_data.size() + pad, 0.0);
        auto at = [&](size_t b, int i, int k) -> double & {  // element (i, k) of a block
            const int slice = (i / 4) * mb + k;              // float32: slice registers
            return s[b * per + (fp32 ? (size_t)(slice / 16) * 64 + 4 * (slice % 16) + i % 4 : (size_t)k * mb + i)];
        };
        for (size_t b = 0; b < nb; ++b) {
            const int off = m.op_desc[3 * b], mf = m.op_desc[3 * b + 1], mi = m.op_desc[3 * b + 2];
            for (int i = 0; i < mf; ++i)
                for (int k = 0; k < mi; ++k) at(b, i, k) = m.op_data[off + i + k * mf];
        }
        for (int i = 0; i < mb; ++i) at(nb, i, i) = 1.0;
        if (fp32) {
            const std::vector<float> s32(s.begin(), s.end()), o32(o.begin(), o.end());
            HIPCHK(c, hipMemcpy(blocks, s32.data(), s32.size() * 4, hipMemcpyHostToDevice));
            HIPCHK(c, hipMemcpy(cm, o32.data(), o32.size() * 4, hipMemcpyHostToDevice));
        } else {
            HIPCHK(c, hipMemcpy(blocks, s.data(), s.size() * 8, hipMemcpyHostToDevice));
            HIPCHK(c, hipMemcpy(cm, o.data(), o.size() * 8, hipMemcpyHostToDevice));
        }
        std::vector<double> ed((size_t)m.bt, 0.0);
        std::vector<uint8_t> mk((size_t)m.bt, 0);
        std::vector<int32_t> l((size_t)m.bt + 2 * m.ns);
        for (int q = 0; q < m.ns; ++q) {
            const int d = m.dims[q];
            for (int e = 0; e < d * d; ++e)  // bt < 2^16 where the propagators fit in LDS
                l[m.bt_off[q] + e] = (int32_t)((uint32_t)m.bt_off[q] | (uint32_t)(e % d) << 16 | (uint32_t)(e / d) << 21 |
                                               (uint32_t)(d - 1) << 26);
            for (int i = 0; i < d; ++i) {
                ed[m.bt_off[q] + i + i * d] = m.E[q][i] + m.lambda0;
                mk[m.bt_off[q] + i + i * d] = 1;
            }
            l[m.bt + q] = m.bt_off[q];
            l[m.bt + m.ns + q] = arc_stride(d, m.mmax);
        }
        HIPCHK(c, hipMemcpy(ediag, ed.data(), ed.size() * 8, hipMemcpyHostToDevice));
        HIPCHK(c, hipMemcpy(emask, mk.data(), mk.size(), hipMemcpyHostToDevice));
        HIPCHK(c, hipMemcpy(lay, l.data(), l.size() * 4, hipMemcpyHostToDevice));
        c->arc_staged |= fp32 ? 2 : 1;
    }
    aa->ops = blocks;
    aa->ops_cm = cm;
    aa->ediag = ediag;
    aa->emask = emask;
    aa->element = (const uint32_t *)lay;
    aa->bt_off = lay + m.bt;
    aa->stride = lay + m.bt + m.ns;
    aa->bt = m.bt;
    return 0;
}

// Launches the evaluator matching the model's sector structure.  The arc walk of sector blocks and
// the vector and matrix-core walks stage their tables on the first call after qiw_set_model
// (synchronous copies), so a call with `record` comes before a capture.  record: append the bytes of
// every launch (arguments, workgroups, shape, LDS) instead of launching; two calls of one format
// and precision with the same bytes launch the same.
int launch_eval(qiw_ctx *c, const EvalArgs &a, const Batch &batch, std::string *record = nullptr) {
    const HostModel &m = c->m;
    auto put = [&](const auto &args, int count, int shape, size_t lds) {
        record->append((const char *)&args, sizeof(args));
        const int64_t v[4] = {m.mmax, count, shape, (int64_t)lds};
        record->append((const char *)v, sizeof(v));
    };
    const int n_tasks = (int)batch.tasks.size(), fmt = batch.fmt, precision = batch.precision;
    if (fmt == FMT_ARC) {
        ArcArgs aa{};
        int rc = stage_arcs(c, precision, &aa);
        if (rc) return rc;
        aa.e = a;
        for (const Batch::Launch &ln : batch.launches) {
            aa.e.tasks = a.tasks + ln.first;
            if (record) {
                put(aa, ln.count, ln.shape, ln.lds);
                continue;
            }
            HIPCHK(c, qiw_launch_eval_arcs(c->stream, aa, ln.count, m.mmax, precision == QIW_PREC_FP32 ? 1 : 0, ln.shape,
                                           ln.lds));
        }
        return 0;
    }
    const size_t lds_bytes = (size_t)a.lds_slots * sizeof(double);
    if (lds_bytes > 160 * 1024) return fail(c, QIW_E_LIMIT, "evaluator state exceeds the 160 KiB of LDS of a CU");
    if (fmt == FMT_SARC) {
        EvalArgs e = a;
        for (const Batch::Launch &ln : batch.launches) {
            e.tasks = a.tasks + ln.first;
            if (record) {
                put(e, ln.count, ln.shape, ln.lds);
                continue;
            }
            HIPCHK(c, qiw_launch_eval_sarcs(c->stream, e, ln.count, ln.shape, batch.groups[0].g.kind == QIW_G_BARE, ln.lds));
        }
        return 0;
    }
    if (fmt == FMT_SCALAR) {
        if (record) {
            put(a, n_tasks, 0, 0);
            return 0;
        }
        HIPCHK(c, qiw_launch_eval_flat(c->stream, a, n_tasks, a.max_order, m.ns, m.ntab));
        return 0;
    }
    if (fmt == FMT_VEC && m.mmax > 6) {  // wide blocks: the matrix-core walk
        int rc = 0;
        const size_t pad = 64;
        float *ops32 = (float *)dev(c, "mfma.ops32", (m.ops_rm.size() + pad) * 4, &rc);
        double *ediag = (double *)dev(c, "mfma.ediag", ((size_t)m.bt + pad) * 8, &rc);
        uint8_t *emask = (uint8_t *)dev(c, "mfma.emask", (size_t)m.bt + pad, &rc);
        int32_t *pinv = (int32_t *)dev(c, "mfma.pinv", ((size_t)m.btp + pad) * 4, &rc);
        int32_t *bto = (int32_t *)dev(c, "mfma.bto", ((size_t)m.ns + pad) * 4, &rc);
        if (rc) return rc;
        if (!c->mfma_staged) {  // once per model
            std::vector<float> o32(m.ops_rm.begin(), m.ops_rm.end());
            o32.resize(m.ops_rm.size() + pad, 0.0f);
            std::vector<double> ed((size_t)m.bt + pad, 0.0);
            std::vector<uint8_t> mk((size_t)m.bt + pad, 0);
            for (int s = 0; s < m.ns; ++s)
                for (int i = 0; i < m.dims[s]; ++i) {
                    ed[m.bt_off[s] + i + i * m.dims[s]] = m.E[s][i] + m.lambda0;
                    mk[m.bt_off[s] + i + i * m.dims[s]] = 1;
                }
            HIPCHK(c, hipStreamSynchronize(c->stream));
            HIPCHK(c, hipMemcpy(ops32, o32.data(), o32.size() * 4, hipMemcpyHostToDevice));
            HIPCHK(c, hipMemcpy(ediag, ed.data(), ed.size() * 8, hipMemcpyHostToDevice));
            HIPCHK(c, hipMemcpy(emask, mk.data(), mk.size(), hipMemcpyHostToDevice));
            HIPCHK(c, hipMemcpy(pinv, m.pinv.data(), m.pinv.size() * 4, hipMemcpyHostToDevice));
            HIPCHK(c, hipMemcpy(bto, m.bt_off.data(), m.bt_off.size() * 4, hipMemcpyHostToDevice));
            c->mfma_staged = true;
        }
        const int KM = a.max_order <= 3 ? 3 : 4, NM = 2 * KM + 3;
        // i*P blocks and four 0.0 read by lanes outside a block, shared by the workgroup; per
        // wavefront 64 floats for the writes of absent rows and the stack of its walk (a
        // 4-float header and the rows of each frame)
        const size_t wave_lds = 64 + (size_t)(NM - 2) * 4 + (size_t)ystack_rows(m, NM - 2) * 16;
        const size_t lds = ((((size_t)(NM - 1) * m.btp + 3) & ~(size_t)3) + 4 + QIW_MFMA_WAVES * wave_lds) * 4;
        if (lds > 160 * 1024) return fail(c, QIW_E_LIMIT, "propagator blocks exceed the 160 KiB of LDS of a CU");
        MfmaArgs mf{};
        mf.e = a;
        mf.ops = ops32;
        mf.ediag = ediag;
        mf.emask = emask;
        mf.pinv = pinv;
        mf.bto = bto;
        mf.bt = m.bt;
        mf.btp = m.btp;
        mf.ops_zero = (int)m.ops_rm.size() - 4;
        mf.wave_lds = (int)wave_lds;
        if (record) {
            put(mf, n_tasks, 0, lds);
            return 0;
        }
        HIPCHK(c, qiw_launch_eval_mfma(c->stream, mf, n_tasks, a.max_order, m.ntab, lds));
        return 0;
    }
    if (fmt == FMT_VEC) {
        // operator blocks and E + lambda on the BT diagonal, both padded so that the
        // fixed-length vector loops stay inside the allocations
        int rc = 0;
        const size_t pad = 64;
        double *ops = (double *)dev(c, "vec.ops", (m.op_data.size() + pad) * 8, &rc);
        double *ediag = (double *)dev(c, "vec.ediag", ((size_t)m.bt + 2 * pad) * 8, &rc);
        double2 *pt = (double2 *)dev(c, "vec.pt", ((size_t)(m.ntau - 1) * m.bt + pad) * 16, &rc);
        double *ptm = (double *)dev(c, "vec.ptm", ((size_t)(m.ntau - 1) * m.bt + pad) * 8, &rc);
        float *ops32 = (float *)dev(c, "vec.ops32", (m.op_data.size() + pad) * 4, &rc);
        QiwCell32 *pt32 = (QiwCell32 *)dev(c, "vec.pt32", ((size_t)(m.ntau - 1) * m.bt + pad) * sizeof(QiwCell32), &rc);
        if (rc) return rc;
        if (!c->vec_staged) {  // once per model
            std::vector<double> o(m.op_data), ed((size_t)m.bt + 2 * pad, 0.0);
            o.resize(m.op_data.size() + pad, 0.0);
            std::vector<float> o32(o.begin(), o.end());
            HIPCHK(c, hipMemcpy(ops32, o32.data(), o32.size() * 4, hipMemcpyHostToDevice));
            HIPCHK(c, hipMemset(pt32, 0, ((size_t)(m.ntau - 1) * m.bt + pad) * sizeof(QiwCell32)));
            HIPCHK(c, hipMemset(ptm, 0, ((size_t)(m.ntau - 1) * m.bt + pad) * 8));
            for (int s = 0; s < m.ns; ++s)
                for (int i = 0; i < m.dims[s]; ++i) ed[m.bt_off[s] + i + i * m.dims[s]] = m.E[s][i] + m.lambda0;
            HIPCHK(c, hipStreamSynchronize(c->stream));
            HIPCHK(c, hipMemcpy(ops, o.data(), o.size() * 8, hipMemcpyHostToDevice));
            HIPCHK(c, hipMemcpy(ediag, ed.data(), ed.size() * 8, hipMemcpyHostToDevice));
            HIPCHK(c, hipMemset(pt, 0, ((size_t)(m.ntau - 1) * m.bt + pad) * 16));
            c->vec_staged = true;
        }
        VecArgs v{};
        v.e = a;
        v.pt = pt;
        v.ptm = ptm;
        v.pt32 = pt32;
        v.ediag = ediag;
        v.ops = ops;
        v.ops32 = ops32;
        v.bt = m.bt;
        if (record) {
            put(v, n_tasks, 0, 0);
            return 0;
        }
        HIPCHK(c, qiw_launch_ptab_cells(c->stream, a.ptab, m.ntau, m.bt, pt, ptm, pt32));
        HIPCHK(c, qiw_launch_eval_vec(c->stream, v, n_tasks, m.mmax, a.max_order, m.ntab,
                                      precision == QIW_PREC_FP32 ? 1 : 0));
        return 0;
    }
    int rc = 0;
    double *opd = (double *)dev(c, "op.data", m.op_data.size() * 8, &rc);
    int32_t *opdesc = (int32_t *)dev(c, "op.desc", std::max<size_t>(m.op_desc.size(), 1) * 4, &rc);
    int32_t *dims = (int32_t *)dev(c, "dims", m.ns * 4, &rc);
    int32_t *btoff = (int32_t *)dev(c, "btoff", m.ns * 4, &rc);
    if (rc) return rc;
    std::vector<int32_t> d32(m.dims.begin(), m.dims.end()), o32(m.bt_off.begin(), m.bt_off.end());
    HIPCHK(c, hipMemcpyAsync(opd, m.op_data.data(), m.op_data.size() * 8, hipMemcpyHostToDevice, c->stream));
    if (!m.op_desc.empty())
        HIPCHK(c, hipMemcpyAsync(opdesc, m.op_desc.data(), m.op_desc.size() * 4, hipMemcpyHostToDevice, c->stream));
    HIPCHK(c, hipMemcpyAsync(dims, d32.data(), m.ns * 4, hipMemcpyHostToDevice, c->stream));
    HIPCHK(c, hipMemcpyAsync(btoff, o32.data(), m.ns * 4, hipMemcpyHostToDevice, c->stream));
    BlockArgs b{};
    b.e = a;
    b.op_data = opd;
    b.op_desc = opdesc;
    b.dims = dims;
    b.bt_off = btoff;
    b.bt = m.bt;
    b.mmax = m.mmax;
    HIPCHK(c, qiw_launch_eval_block(c->stream, b, n_tasks, lds_bytes));
    return 0;
}

EvalArgs make_eval_args(qiw_ctx *c, const Batch &bt, const DevBatch &d, double *ptab, double *eshift, double *dcoef,
                        int32_t *dkind, double *partial) {
    const HostModel &m = c->m;
    EvalArgs a{};
    int lds = bt.lds;
    a.max_order = bt.max_order;
    a.groups = d.groups;
    a.tasks = d.tasks;
    a.prog = d.prog;
    a.topo = d.topo;
    a.coefs = d.coefs;
    a.ut = d.ut;
    a.ptab = ptab;
    a.e_shift = eshift;
    a.dtab.n_tables = m.ntab;
    a.dtab.n_tau = m.ntau;
    a.dtab.h = m.h;
    a.dtab.beta = m.beta;
    a.dtab.kind = dkind;
    a.dtab.grid_mask = 0;
    a.dtab.dlr_mask = 0;
    a.dtab.dlr_rank = m.dlr_rank;
    {
        int rc = 0;
        a.dtab.dlr = (const double *)dev(c, "delta.dlr", std::max<size_t>(m.dlr.size(), 1) * 8, &rc);
    }
    for (int t = 0; t < m.ntab; ++t)
        if (m.dkind[t] == QIW_GF_DLR) a.dtab.dlr_mask |= 1 << t;
    for (int t = 0; t < m.ntab && t < 31; ++t)
        if (m.dkind[t] == QIW_GF_GRID_LINEAR) a.dtab.grid_mask |= 1 << t;
    a.dtab.coef = dcoef;
    a.ns = m.ns;
    a.n_tau = m.ntau;
    a.h = m.h;
    a.beta = m.beta;
    a.lds_slots = lds;
    a.n_out = bt.n_out ? bt.n_out : m.ns;
    a.step_w = 0;
    a.partial = partial;
    a.spt = bt.spt;
    return a;
}

void atomic_ip(const HostModel &m, std::vector<double> &ip) {  // src/ppgf.jl:144-207
    ip.assign((size_t)m.ntau * m.bt, 0.0);
    for (int j = 0; j < m.ntau; ++j)
        for (int s = 0; s < m.ns; ++s)
            for (int i = 0; i < m.dims[s]; ++i)
                ip[(size_t)j * m.bt + m.bt_off[s] + i + i * m.dims[s]] = std::exp(-(j * m.h) * (m.E[s][i] + m.lambda0));
}

void store_complex_from_ip(double ipv, double *out) {  // P = -i * (i P)
    out[0] = 0.0;
    out[1] = -ipv;
}

}  // namespace

// =======================================================================================
// Scratch of qiw_inchworm_step_noalloc: one static array per GPU, held until the process
// ends.  Host code never uses the array's name as an address: at qiw_create, once per
// device and with that device current, hipGetSymbolAddress gives the device address, which
// every later call on that device uses.
// =======================================================================================
static __device__ __align__(256) unsigned char scratch[kNoAllocScratchBytes];

namespace {
constexpr int kMaxDevices = 64;
std::mutex g_scratch_mu;
void *g_scratch_ptr[kMaxDevices] = {};

// The device address of `device`'s scratch array (that device is current).
int scratch_address(int device, void **out) {
    if (device < 0 || device >= kMaxDevices) return QIW_E_LIMIT;
    std::lock_guard<std::mutex> lock(g_scratch_mu);
    if (!g_scratch_ptr[device]) {
        void *p = nullptr;
        if (hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)) != hipSuccess || !p) return QIW_E_DEVICE;
        g_scratch_ptr[device] = p;
    }
    *out = g_scratch_ptr[device];
    return QIW_OK;
}
}  // namespace

// =======================================================================================
// C ABI
// =======================================================================================
extern "C" int qiw_abi_version(void) { return QIW_ABI_VERSION; }

static int qiw_create_impl(qiw_ctx **out, int device) {
    if (!out) return QIW_E_ARG;
    *out = nullptr;
    int n = 0;
    if (hipGetDeviceCount(&n) != hipSuccess || n <= device || device < 0) return QIW_E_NO_GPU;
    qiw_ctx *c = new qiw_ctx();
    c->device = device;
    if (hipSetDevice(device) != hipSuccess || hipStreamCreate(&c->stream) != hipSuccess) {
        delete c;
        return QIW_E_DEVICE;
    }
    const int rc = scratch_address(device, &c->scratch);
    if (rc != QIW_OK) {
        (void)hipStreamDestroy(c->stream);
        delete c;
        return rc;
    }
    *out = c;
    return QIW_OK;
}

namespace {
// Bytes of everything the compiled programs and task lists depend on: sector structure,
// operator elements and blocks, pair tables, correlator operators, grid size.
std::string model_fingerprint(const HostModel &m) {
    std::string k;
    auto put = [&](const void *p, size_t n) { k.append((const char *)p, n); };
    auto vec = [&](const auto &v) {
        const size_t n = v.size();
        put(&n, sizeof n);
        if (n) put(v.data(), n * sizeof(v[0]));
    };
    put(&m.ntau, sizeof m.ntau);
    put(&m.ns, sizeof m.ns);
    put(&m.ntab, sizeof m.ntab);
    vec(m.dims);
    vec(m.pair_table);
    vec(m.op_data);
    vec(m.op_desc);
    for (const auto *ops : {&m.op_i, &m.op_f, &m.corr_A, &m.corr_B}) {
        const size_t n = ops->size();
        put(&n, sizeof n);
        for (const ScalarOp &o : *ops) {
            vec(o.sf);
            vec(o.val);
            vec(o.blk);
        }
    }
    return k;
}
}  // namespace

static void qiw_destroy_impl(qiw_ctx *c) {
    if (!c) return;
    (void)hipSetDevice(c->device);
    if (c->stream) (void)hipStreamSynchronize(c->stream);
    warp_destroy(c->warp);
    plans_destroy(c->plans);
    step_graph_destroy(c->graph);
    if (c->pin) (void)hipHostFree(c->pin);
    for (auto e : c->evpool) (void)hipEventDestroy(e);
    for (auto &kv : c->bufs)
        if (kv.second.p) (void)hipFree(kv.second.p);
    if (c->stream) (void)hipStreamDestroy(c->stream);
    delete c;
}

extern "C" const char *qiw_last_error(const qiw_ctx *c) { return c ? c->err.c_str() : "null context"; }

static int qiw_set_model_impl(qiw_ctx *c, const qiw_model *mi) {
    if (!c || !mi) return QIW_E_ARG;
    if (mi->n_tau < 3 || mi->n_sectors < 1 || !(mi->beta > 0)) return fail(c, QIW_E_ARG, "bad grid or sectors");
    HostModel m;
    m.beta = mi->beta;
    m.ntau = mi->n_tau;
    m.h = m.beta / (m.ntau - 1);
    m.ns = mi->n_sectors;
    m.dims.assign(mi->sector_dim, mi->sector_dim + m.ns);
    size_t off = 0;
    double emin = 1e300;
    for (int s = 0; s < m.ns; ++s) {
        if (m.dims[s] < 1) return fail(c, QIW_E_ARG, "empty sector");
        m.E.emplace_back(mi->energies + off, mi->energies + off + m.dims[s]);
        off += m.dims[s];
        for (double e : m.E.back()) emin = std::min(emin, e);
        if (m.dims[s] != 1) m.scalar = false;
    }
    double zs = 0;
    for (auto &v : m.E)
        for (double e : v) zs += std::exp(-m.beta * (e - emin));
    m.lambda0 = (std::log(zs) - m.beta * emin) / m.beta;  // log(Z)/beta, src/exact_atomic_ppgf.jl:130-135
    m.ppgf_kind = mi->ppgf_kind;
    if (m.ppgf_kind != QIW_GF_GRID_LINEAR && m.ppgf_kind != QIW_GF_INC_SPLINE)
        return fail(c, QIW_E_ARG, "ppgf_kind must be QIW_GF_GRID_LINEAR or QIW_GF_INC_SPLINE");
    m.np = mi->n_pairs;
    m.op_i.resize(m.np);
    m.op_f.resize(m.np);
    m.pair_table.resize(m.np);
    std::vector<std::vector<double>> tabs;
    std::vector<int> tab_kind;
    m.dlr_rank = 0;
    for (int p = 0; p < m.np; ++p)
        if (mi->pair_prop_kind[p] == QIW_GF_DLR) {
            if (mi->dlr_rank < 1 || !mi->pair_dlr_omega || !mi->pair_dlr_coef)
                return fail(c, QIW_E_ARG, "a QIW_GF_DLR pair needs dlr_rank > 0, pair_dlr_omega and pair_dlr_coef");
            if (mi->dlr_rank > 512) return fail(c, QIW_E_LIMIT, "dlr_rank beyond 512");
            m.dlr_rank = mi->dlr_rank;
        }
    for (int p = 0; p < m.np; ++p) {
        int rc = load_scalar_op(c, mi->pair_op_i[p], m.dims, m.op_i[p], &m.scalar, m.op_data, m.op_desc);
        if (rc) return rc;
        if ((rc = load_scalar_op(c, mi->pair_op_f[p], m.dims, m.op_f[p], &m.scalar, m.op_data, m.op_desc))) return rc;
        int kind = mi->pair_prop_kind[p];
        if (kind != QIW_GF_GRID_LINEAR && kind != QIW_GF_CUBIC_SPLINE && kind != QIW_GF_DLR)
            return fail(c, QIW_E_ARG, "pair propagator kind must be GRID_LINEAR, CUBIC_SPLINE or DLR");
        // i * Delta_p must be real: grid values, or (frequency, coefficient) pairs of a DLR
        std::vector<double> y;
        if (kind == QIW_GF_DLR) {
            for (int k = 0; k < m.dlr_rank; ++k) {
                const size_t i = (size_t)p * m.dlr_rank + k;
                const double re = mi->pair_dlr_coef[2 * i], im = mi->pair_dlr_coef[2 * i + 1];
                if (std::fabs(re) > 1e-13 * (1.0 + std::fabs(im)))
                    return fail(c, QIW_E_ARG, "i*Delta must be real for the GPU kernels (DLR coefficients)");
                y.push_back(mi->pair_dlr_omega[i]);
                y.push_back(-im);
            }
        } else {
            y.resize(m.ntau);
            for (int j = 0; j < m.ntau; ++j) {
                double re = mi->pair_prop[2 * ((size_t)p * m.ntau + j)], im = mi->pair_prop[2 * ((size_t)p * m.ntau + j) + 1];
                if (std::fabs(re) > 1e-13 * (1.0 + std::fabs(im)))
                    return fail(c, QIW_E_ARG, "i*Delta must be real for the GPU kernels");
                y[j] = -im;
            }
        }
        int found = -1;
        for (size_t t = 0; t < tabs.size(); ++t)
            if (tab_kind[t] == kind && tabs[t] == y) found = (int)t;
        if (found < 0) {
            tabs.push_back(y);
            tab_kind.push_back(kind);
            found = (int)tabs.size() - 1;
        }
        m.pair_table[p] = found;
    }
    m.ntab = (int)tabs.size();
    if (m.ntab > 31) return fail(c, QIW_E_LIMIT, "more than 31 distinct hybridization tables");
    m.dcoef.assign((size_t)std::max(m.ntab, 1) * (m.ntau - 1) * 4, 0.0);
    m.dlr.assign((size_t)std::max(m.ntab, 1) * std::max(m.dlr_rank, 1) * 2, 0.0);
    m.dkind = tab_kind;
    for (int t = 0; t < m.ntab; ++t) {
        double *cc = m.dcoef.data() + (size_t)t * (m.ntau - 1) * 4;
        if (tab_kind[t] == QIW_GF_DLR) {
            std::copy(tabs[t].begin(), tabs[t].end(), m.dlr.begin() + (size_t)t * m.dlr_rank * 2);
        } else if (tab_kind[t] == QIW_GF_CUBIC_SPLINE) {
            natural_spline_coef(tabs[t], m.h, cc);
        } else {  // grid container: value, forward and backward difference per index
            for (int j = 0; j < m.ntau - 1; ++j) {
                cc[4 * j] = tabs[t][j];
                cc[4 * j + 1] = tabs[t][j + 1] - tabs[t][j];
                cc[4 * j + 2] = j > 0 ? tabs[t][j] - tabs[t][j - 1] : cc[4 * j + 1];
            }
        }
    }
    m.ncorr = mi->n_corr;
    m.corr_A.resize(m.ncorr);
    m.corr_B.resize(m.ncorr);
    for (int i = 0; i < m.ncorr; ++i) {
        int rc = load_scalar_op(c, mi->corr_A[i], m.dims, m.corr_A[i], &m.scalar, m.op_data, m.op_desc);
        if (rc) return rc;
        if ((rc = load_scalar_op(c, mi->corr_B[i], m.dims, m.corr_B[i], &m.scalar, m.op_data, m.op_desc))) return rc;
    }
    m.attachable.assign(m.ns, {});  // src/expansion.jl:180-183
    for (int s = 0; s < m.ns; ++s)
        for (int p = 0; p < m.np; ++p)
            if (m.op_i[p].sf[s] >= 0) m.attachable[s].push_back(p);
    m.bt_off.resize(m.ns);
    m.bt = 0;
    for (int s = 0; s < m.ns; ++s) {
        m.bt_off[s] = m.bt;
        m.bt += m.dims[s] * m.dims[s];
        m.mmax = std::max(m.mmax, m.dims[s]);
    }
    if (m.mmax > 32) return fail(c, QIW_E_LIMIT, "sector blocks larger than 32 are not supported");
    m.scalar_kernel = m.scalar && m.ns <= 8 && m.ntab <= 4;
    if (m.op_data.empty()) m.op_data.push_back(0.0);
    m.vec_ok = !m.scalar_kernel && m.mmax <= 6 && m.ntab <= 4 && m.ns <= 255 && m.bt < 4096 &&
               m.op_data.size() < 0xFFFF - 64;
    if (m.mmax > 6) wide_layout(m);
    m.mfma_ok = !m.scalar_kernel && m.mmax <= 32 && m.ntab <= 2 && m.ns <= 255 && m.bt < 4096 &&
                m.op_data.size() < 0xFFFF - 64 && m.ops_rm.size() < 0xFFFF && m.btp < 4096;
    c->m = std::move(m);
    c->has_model = true;
    std::string fp = model_fingerprint(c->m);
    if (fp != c->model_fp) c->tune = qiw_tuning{};  // the work mapping was chosen for another model
    c->model_fp = fp;
    c->vec_staged = false;
    c->mfma_staged = false;
    c->arc_staged = 0;
    atomic_ip(c->m, c->ip);
    c->n_known = (c->m.ppgf_kind == QIW_GF_INC_SPLINE) ? 1 : c->m.ntau;
    c->der0.assign(c->m.bt, cd(0.0));  // initial_ppgf_derivative: -i diag(-E - lambda), src/ppgf.jl:710-720
    for (int s = 0; s < c->m.ns; ++s)
        for (int i = 0; i < c->m.dims[s]; ++i) c->der0[c->m.bt_off[s] + i + i * c->m.dims[s]] = cd(0.0, c->m.E[s][i] + c->m.lambda0);
    c->lambdas.assign(c->m.ntau, 0.0);
    return QIW_OK;
}

static int qiw_set_sobol_impl(qiw_ctx *c, int32_t dim, const uint32_t *m, const uint32_t *shift) {
    if (!c || !m || dim < 1 || dim > 2 * QIW_KMAX) return c ? fail(c, QIW_E_DIM, "Sobol dimension out of range") : QIW_E_ARG;
    c->sob_dim = dim;
    c->sob_m.assign(m, m + (size_t)dim * 32);
    c->sob_x.assign(dim, 0u);
    if (shift) c->sob_x.assign(shift, shift + dim);
    return QIW_OK;
}

static int qiw_set_scrambles_impl(qiw_ctx *c, int64_t n, int32_t stride, const uint32_t *m, const uint32_t *shift) {
    if (!c) return QIW_E_ARG;
    if (n < 0 || (n > 0 && (!m || stride < 1 || stride > 2 * QIW_KMAX)))
        return fail(c, QIW_E_ARG, "qiw_set_scrambles: n >= 0 sequences of 1 .. 12 dimensions");
    if (n > ((int64_t)1 << 40) / (32 * std::max(stride, 1)))
        return fail(c, QIW_E_LIMIT, "qiw_set_scrambles: too many sequences");
    (void)hipSetDevice(c->device);
    c->given_n = 0;
    c->given_stride = 0;
    if (n == 0) return QIW_OK;
    const size_t rows = (size_t)n * stride;
    int rc = 0;
    uint32_t *gm = (uint32_t *)dev(c, "given.m", rows * 32 * 4, &rc);
    uint32_t *gx = (uint32_t *)dev(c, "given.x", rows * 4, &rc);
    if (rc) return rc;
    HIPCHK(c, hipStreamSynchronize(c->stream));  // earlier calls may still read the buffers
    HIPCHK(c, hipMemcpy(gm, m, rows * 32 * 4, hipMemcpyHostToDevice));
    if (shift) {
        HIPCHK(c, hipMemcpy(gx, shift, rows * 4, hipMemcpyHostToDevice));
    } else {
        const std::vector<uint32_t> zero(rows, 0u);
        HIPCHK(c, hipMemcpy(gx, zero.data(), rows * 4, hipMemcpyHostToDevice));
    }
    c->given_n = n;
    c->given_stride = stride;
    return QIW_OK;
}

static int qiw_set_points_impl(qiw_ctx *c, int64_t n, int64_t n_points, int32_t stride, const double *x) {
    if (!c) return QIW_E_ARG;
    if (n < 0 || (n > 0 && (!x || n_points < 1 || stride < 1 || stride > 2 * QIW_KMAX)))
        return fail(c, QIW_E_ARG, "qiw_set_points: n >= 0 sequences of n_points >= 1 points of 1 .. 12 dimensions");
    if ((double)n * (double)n_points * stride * 8 > kMaxGivenCoordBytes)
        return fail(c, QIW_E_LIMIT, "qiw_set_points: the points exceed 64 GiB");
    (void)hipSetDevice(c->device);
    c->points_n = 0;
    c->points_npts = 0;
    c->points_stride = 0;
    if (n == 0) return QIW_OK;
    const size_t count = (size_t)n * n_points * stride;
    for (size_t i = 0; i < count; ++i)
        if (!(x[i] >= 0.0 && x[i] <= 1.0)) return fail(c, QIW_E_ARG, "qiw_set_points: points must lie in [0, 1]");
    int rc = 0;
    double *p = (double *)dev(c, "given.pts", count * 8, &rc);
    if (rc) return rc;
    HIPCHK(c, hipStreamSynchronize(c->stream));  // earlier calls may still read the buffer
    HIPCHK(c, hipMemcpy(p, x, count * 8, hipMemcpyHostToDevice));
    c->points_n = n;
    c->points_npts = n_points;
    c->points_stride = stride;
    return QIW_OK;
}

static int qiw_set_ppgf_impl(qiw_ctx *c, int32_t n_known, const double *P, const double *der0) {
    if (!c || !P) return QIW_E_ARG;
    if (!c->has_model) return fail(c, QIW_E_STATE, "no model staged");
    const HostModel &m = c->m;
    if (n_known < 1 || n_known > m.ntau) return fail(c, QIW_E_ARG, "n_known out of range");
    for (size_t i = 0; i < (size_t)m.ntau * m.bt; ++i) {
        double re = P[2 * i], im = P[2 * i + 1];
        if (std::fabs(re) > 1e-12 * (1.0 + std::fabs(im))) return fail(c, QIW_E_ARG, "i*P must be real for the GPU kernels");
        c->ip[i] = -im;
    }
    c->n_known = (m.ppgf_kind == QIW_GF_INC_SPLINE) ? n_known : m.ntau;
    if (der0)
        for (int e = 0; e < m.bt; ++e) c->der0[e] = cd(der0[2 * e], der0[2 * e + 1]);
    return QIW_OK;
}

static int qiw_get_ppgf_impl(qiw_ctx *c, int32_t *n_known_out, double *P, double *der0) {
    if (!c) return QIW_E_ARG;
    if (!c->has_model) return fail(c, QIW_E_STATE, "no model staged");
    const HostModel &m = c->m;
    if (n_known_out) *n_known_out = c->n_known;
    if (P)
        for (size_t i = 0; i < (size_t)m.ntau * m.bt; ++i) store_complex_from_ip(c->ip[i], P + 2 * i);
    if (der0)
        for (int e = 0; e < m.bt; ++e) {
            der0[2 * e] = c->der0[e].real();
            der0[2 * e + 1] = c->der0[e].imag();
        }
    return QIW_OK;
}

namespace {

// Runs the initial step and then bold steps jw = first_w .. last_w on the device; the
// device tables are initialized from the host mirror and copied back at the end.
constexpr int kGraphSteps = 4;
int run_inchworm(qiw_ctx *c, const qiw_run *run, bool do_bare, int first_w, int last_w, bool normalize,
                 bool store_host_P, double *P_orders_out, double *P_orders_std_out, std::vector<double> *step_value,
                 std::vector<double> *step_orders) {
    const HostModel &m = c->m;
    auto t0 = std::chrono::steady_clock::now();
    std::vector<int> oall = orders_all(run);
    if (step_orders) {  // single step: order slots follow run->orders
        oall.assign(run->orders, run->orders + run->n_orders);
    }
    int n_slots = std::max<int>((int)oall.size(), 1);
    int rc = 0;
    Plan none, *bp = &none, *sp = &none;
    const bool want_warp = warp_enabled(c->warp);
    const RandPlan rq = rand_plan(run);
    const bool rqmc = rq.n_seqs > 1;  // mean and deviation over several sequences
    if (want_warp && (rqmc || rq.scrambled))
        return fail(c, QIW_E_ARG, "the learned warp takes one unscrambled sequence (rand_params)");
    if (do_bare && (rc = step_plan(c, run, oall, true, false, bp))) return rc;
    if (last_w >= first_w && (rc = step_plan(c, run, oall, false, want_warp, sp))) return rc;
    Batch &bare_b = bp->b, &bold_b = sp->b;
    DevBatch &bare_d = bp->d, &bold_d = sp->d;
    // caller-drawn sequences: the initial step's, then every bold step's in step order
    GivenSrc gsrc;
    const int64_t *gidx_bare = nullptr, *gidx_bold = nullptr;
    int32_t *nuse_bare = nullptr, *nuse_bold = nullptr;  // sequences the bookkeeping used (N_seqs >= 3)
    std::vector<int32_t> use_bare, use_bold;
    std::vector<int> rows_bare, rows_bold;
    if (rq.given) {
        if (c->no_alloc) return fail(c, QIW_E_ARG, "caller-drawn sequences need qiw_inchworm_step");
        const auto none = [](const QiwGroup &) { return false; };  // bare and bold simplices have volume
        std::vector<int64_t> idx;
        int64_t n = 0;
        const size_t ngb = bare_b.groups.size(), ngo = bold_b.groups.size();
        if (do_bare && ngb) {
            idx.resize(ngb);
            use_bare.resize(bare_b.r_first.size());
            n += given_row(bare_b, rq.n_seqs, n, none, idx.data(), use_bare.data());
            rows_bare.push_back(1);
        }
        for (int jw = first_w; jw <= last_w && ngo; ++jw) {
            const size_t o = idx.size(), ou = use_bold.size();
            idx.resize(o + ngo);
            use_bold.resize(ou + bold_b.r_first.size());
            n += given_row(bold_b, rq.n_seqs, n, none, idx.data() + o, use_bold.data() + ou);
            rows_bold.push_back(jw + 1);
        }
        if ((rc = given_buffers(c, rq.points, std::max(bare_b.max_order, bold_b.max_order), n, run->N_samples, &gsrc)))
            return rc;
        int64_t *didx = (int64_t *)dev(c, "given.idx", std::max<size_t>(idx.size(), 1) * 8, &rc);
        if (rq.n_seqs >= 3) {
            nuse_bare = (int32_t *)dev(c, "given.nuse_bare", (size_t)m.ntau * std::max<size_t>(bare_b.r_first.size(), 1) * 4, &rc);
            nuse_bold = (int32_t *)dev(c, "given.nuse_bold", (size_t)m.ntau * std::max<size_t>(bold_b.r_first.size(), 1) * 4, &rc);
        }
        if (rc) return rc;
        if (!idx.empty()) HIPCHK(c, hipMemcpy(didx, idx.data(), idx.size() * 8, hipMemcpyHostToDevice));
        gidx_bare = didx;
        gidx_bold = didx + (rows_bare.empty() ? 0 : ngb);
    }
    const bool warped = want_warp && !bold_b.groups.empty();
    if (warped) {
        std::vector<WarpGroup> wg;
        for (auto &cg : bold_b.groups)
            if (cg.g.weighted)
                wg.push_back({cg.g.order, cg.g.n_after, cg.g.d_before, cg.g.d_after, warp_gid(cg.g), cg.g.ut_off});
        if ((rc = warp_prepare(c, wg, run->N_samples))) return rc;
    }
    double *dcoef, *eshift;
    int32_t *dkind;
    Stage stage(c);
    if ((rc = ensure_model_buffers(c, &dcoef, &dkind, &eshift, &stage))) return rc;
    size_t rows = std::max(bare_b.tasks.size(), bold_b.tasks.size());
    double *partial = (double *)dev(c, "partial", std::max<size_t>(rows, 1) * m.bt * 8, &rc);
    double *ptab = (double *)dev(c, "ptab", (size_t)m.ntau * m.bt * 8, &rc);
    double *porders = (double *)dev(c, "porders", (size_t)n_slots * m.ntau * m.bt * 8, &rc);
    double *lam = (double *)dev(c, "lambda", (size_t)m.ntau * 8, &rc);
    double *scratch = (double *)dev(
        c, "fin.scratch", (rqmc ? std::max(bare_b.r_first.size(), bold_b.r_first.size()) * 2 * m.bt : 0) * 8 + 8, &rc);
    double *gsum = (double *)dev(c, "fin.gsum",
                                 (size_t)std::max(bare_b.groups.size(), bold_b.groups.size()) * m.bt * 8 + 8, &rc);
    int32_t *diag = (int32_t *)dev(c, "diag", (size_t)m.bt * 4, &rc);
    unsigned *done = (unsigned *)dev(c, "fin.done", 4, &rc);
    double *pstd = rqmc ? (double *)dev(c, "porders_std", (size_t)n_slots * m.ntau * m.bt * 8, &rc) : nullptr;
    uint32_t *sobm = rq.scrambled ? (uint32_t *)dev(c, "sobol.m", c->sob_m.size() * 4, &rc) : nullptr;
    if (rc) return rc;
    std::vector<int32_t> dg;
    for (int s = 0; s < m.ns; ++s)
        for (int i = 0; i < m.dims[s]; ++i) dg.push_back(m.bt_off[s] + i + i * m.dims[s]);
    if (sobm) stage.add(sobm, c->sob_m);
    stage.add(diag, dg);
    stage.add(ptab, c->ip);
    stage.add(done, nullptr, 4);
    stage.add(porders, nullptr, (size_t)n_slots * m.ntau * m.bt * 8);
    stage.add(lam, nullptr, (size_t)m.ntau * 8);
    if (pstd) stage.add(pstd, nullptr, (size_t)n_slots * m.ntau * m.bt * 8);
    if ((rc = stage.upload())) return rc;

    FinalizeArgs fa{};
    fa.partial = partial;
    fa.bt = m.bt;
    fa.diag_idx = diag;
    fa.n_diag = (int)dg.size();
    fa.ptab = ptab;
    fa.porders = porders;
    fa.lambda_out = lam;
    fa.n_tau = m.ntau;
    fa.h = m.h;
    fa.n_order_slots = n_slots;
    fa.scratch = scratch;
    fa.gsum = gsum;
    fa.done = done;
    fa.n_seqs = rq.n_seqs;
    fa.target_std = rq.target_std;
    fa.porders_std = pstd;
    auto rqmc_args = [&](const Batch &b, const DevBatch &d, int domain, int key) {
        return RqmcCoords{d.groups, sobm, (int)b.groups.size(), run->N_samples, rq.seed, (uint64_t)domain, (uint64_t)key, d.ut};
    };
    // next_w: the bold step whose coordinates are drawn beside the bookkeeping (-1: none)
    auto finalize = [&](const Batch &b, const DevBatch &d, int next_w) -> hipError_t {
        fa.n_real = (int)b.r_first.size();
        fa.real_first = d.r_first;
        fa.real_count = d.r_count;
        if (!rqmc) return qiw_launch_finalize_step(c->stream, fa);
        const RqmcCoords next = rqmc_args(b, d, QIW_RQ_BOLD, next_w);
        return qiw_launch_finalize_step_rqmc(c->stream, fa, next_w >= 0 ? &next : nullptr);
    };
    // per-step scrambled sequences: coordinates of every group's sequences for this step
    auto coords = [&](const Batch &b, const DevBatch &d, int domain, int key, const int64_t *gidx) -> hipError_t {
        if (!b.scrambled || run->N_samples <= 0) return hipSuccess;  // N = 0: order 0 only
        if (b.given)
            return qiw_launch_given_coords(c->stream, d.groups, (int)b.groups.size(), run->N_samples, gsrc, gidx, 1, 0, 0,
                                           d.ut);
        return qiw_launch_rqmc_coords(c->stream, rqmc_args(b, d, domain, key), 2 * b.max_order);
    };
    // the bookkeeping of a randomized step draws the next step's coordinates (2^24 samples at most)
    const bool draws_next = rqmc && bold_b.scrambled && !bold_b.given && run->N_samples > 0 && run->N_samples <= (1 << 24);
    auto next_of = [&](int jw) { return draws_next && jw < last_w ? jw + 1 : -1; };

    // every evaluator launch is bracketed by an event pair on the launch stream
    // timing events from the context's pool (created once, reused by every call)
    size_t n_ev = 0;
    auto mark = [&](void) -> hipError_t {
        if (c->no_alloc) return hipSuccess;  // creates no events: no timing of a no-alloc call
        if (n_ev == c->evpool.size()) {
            hipEvent_t e;
            hipError_t r = hipEventCreate(&e);
            if (r != hipSuccess) return r;
            c->evpool.push_back(e);
        }
        return hipEventRecord(c->evpool[n_ev++], c->stream);
    };
    int64_t launches = 0;
    int n_known = c->n_known;
    if (!bare_b.groups.empty()) {
        EvalArgs a = make_eval_args(c, bare_b, bare_d, ptab, eshift, dcoef, dkind, partial);
        HIPCHK(c, coords(bare_b, bare_d, QIW_RQ_BARE, 0, gidx_bare));
        HIPCHK(c, mark());
        if ((rc = launch_eval(c, a, bare_b))) return rc;
        HIPCHK(c, mark());
        fa.groups = bare_d.groups;
        fa.group_task_first = bare_d.g_first;
        fa.group_task_count = bare_d.g_count;
        fa.most_rows = most_rows(bare_b);
        fa.group_order_slot = bare_d.g_slot;
        fa.n_groups = (int)bare_b.groups.size();
        fa.jf = fa.jt = 1;
        fa.tau_w = 0.0;
        fa.tau_f = m.h;
        fa.bare = 1;
        fa.normalize = 0;
        fa.n_known = 0;
        fa.nuse_out = nuse_bare;
        HIPCHK(c, finalize(bare_b, bare_d, -1));
        launches += eval_launches(bare_b);
        if (m.ppgf_kind == QIW_GF_INC_SPLINE) n_known = 2;
        c->stats.flops += bare_b.flops_per_launch;
        c->stats.leaves += bare_b.leaves_per_launch;
        c->stats.diagram_evals += bare_b.diagram_evals_per_launch;
    }
    std::vector<std::pair<hipEvent_t, hipEvent_t>> graph_ev;  // timing events of a replayed loop
    if (!bold_b.groups.empty()) {
        EvalArgs a = make_eval_args(c, bold_b, bold_d, ptab, eshift, dcoef, dkind, partial);
        fa.groups = bold_d.groups;
        fa.group_task_first = bold_d.g_first;
        fa.group_task_count = bold_d.g_count;
        fa.most_rows = most_rows(bold_b);
        fa.group_order_slot = bold_d.g_slot;
        fa.n_groups = (int)bold_b.groups.size();
        fa.bare = 0;
        fa.nuse_out = nuse_bold;
        // arguments of every step, as the eager loop below would launch them
        auto step_args = [&](int jw) {
            a.step_w = jw;
            fa.jf = fa.jt = jw + 1;
            fa.tau_w = jw * m.h;
            fa.tau_f = (jw + 1) * m.h;
            if (m.ppgf_kind == QIW_GF_INC_SPLINE && normalize) n_known = std::max(n_known, jw + 2);
            fa.n_known = (m.ppgf_kind == QIW_GF_INC_SPLINE) ? n_known : m.ntau;
            fa.normalize = normalize ? 1 : 0;
        };
        // without the warp the whole loop is one hipGraph, replayed while its launches are the same;
        // the walks with tables on the device stage them before the capture (launch_eval, for the
        // key), but the LDS block walk copies host data per launch and stays eager
        // a few steps launch faster one by one than a graph is replayed, or captured for new times
        bool graph = c->graphs && bold_b.fmt != FMT_BLOCK && !warped && !c->no_alloc && !rq.given &&
                     last_w - first_w >= kGraphSteps;
        const int n_known_start = n_known;
        if (graph) {
            if (!c->graph) c->graph = new StepGraph;
            StepGraph &G = *c->graph;
            const int n_known0 = n_known;
            std::string key;
            auto put = [&](const void *p, size_t n) { key.append((const char *)p, n); };
            if ((rc = launch_eval(c, a, bold_b, &key))) return rc;
            put(&bold_b.max_order, 4);
            put(&rq.seed, 8);
            const uint32_t *sm = sobm;
            put(&sm, sizeof(sm));
            const int scr = bold_b.scrambled ? 1 : 0;
            put(&scr, 4);
            put(&run->N_samples, 8);
            put(&m.ns, 4);
            put(&m.ntab, 4);
            put(&bold_b.fmt, 4);
            put(&bold_b.precision, 4);
            fa.n_real = (int)bold_b.r_first.size();  // as finalize() sets them for this batch
            fa.real_first = bold_d.r_first;
            fa.real_count = bold_d.r_count;
            for (int jw = first_w; jw <= last_w; ++jw) {
                step_args(jw);
                put(&a, sizeof(a));
                put(&fa, sizeof(fa));
            }
            if (G.key != key || !G.exec) {
                G.clear();
                n_known = n_known0;
                for (int i = 0; i < 2; ++i) {
                    hipEvent_t e;
                    HIPCHK(c, hipEventCreate(&e));
                    G.ev.push_back(e);
                }
                HIPCHK(c, hipStreamBeginCapture(c->stream, hipStreamCaptureModeThreadLocal));
                hipError_t err = hipSuccess;
                for (int jw = first_w; jw <= last_w && err == hipSuccess; ++jw) {
                    step_args(jw);
                    if ((jw == first_w || !draws_next) &&
                        (err = coords(bold_b, bold_d, QIW_RQ_BOLD, jw, nullptr)) != hipSuccess)
                        break;  // never given
                    if (launch_eval(c, a, bold_b) != 0) {
                        err = hipErrorUnknown;
                        break;
                    }
                    err = finalize(bold_b, bold_d, next_of(jw));
                }
                hipGraph_t gr = nullptr;
                const hipError_t e2 = hipStreamEndCapture(c->stream, &gr);
                G.graph = gr;
                if (err == hipSuccess) err = e2;
                if (err == hipSuccess) err = hipGraphInstantiate(&G.exec, G.graph, nullptr, nullptr, 0);
                if (err != hipSuccess) {  // capture not available: the eager loop from now on
                    G.clear();
                    (void)hipGetLastError();
                    c->graphs = false;
                    graph = false;
                    n_known = n_known0;
                } else {
                    G.key = key;
                }
            }
        }
        if (graph) {
            // events recorded inside a captured graph carry no timing here: the replay is timed
            // as a whole (evaluators, bookkeeping and the gaps between them)
            StepGraph &G = *c->graph;
            HIPCHK(c, hipEventRecord(G.ev[0], c->stream));
            HIPCHK(c, hipGraphLaunch(G.exec, c->stream));
            c->stats.graph_replays += 1;
            HIPCHK(c, hipEventRecord(G.ev[1], c->stream));
            graph_ev.push_back({G.ev[0], G.ev[1]});
            n_known = n_known_start;
            for (int jw = first_w; jw <= last_w; ++jw) {  // host-side state of the loop
                step_args(jw);
                launches += eval_launches(bold_b);
                c->stats.flops += bold_b.flops_per_launch;
                c->stats.leaves += bold_b.leaves_per_launch;
                c->stats.diagram_evals += bold_b.diagram_evals_per_launch;
            }
        }
        for (int jw = first_w; jw <= last_w && !graph; ++jw) {
            a.step_w = jw;
            if (warped && (rc = warp_points(c, jw * m.h / m.beta, bold_d.ut))) return rc;
            if (jw == first_w || !draws_next)
                HIPCHK(c, coords(bold_b, bold_d, QIW_RQ_BOLD, jw,
                                 gidx_bold ? gidx_bold + (size_t)(jw - first_w) * bold_b.groups.size() : nullptr));
            HIPCHK(c, mark());
            if ((rc = launch_eval(c, a, bold_b))) return rc;
            HIPCHK(c, mark());
            fa.jf = fa.jt = jw + 1;
            fa.tau_w = jw * m.h;
            fa.tau_f = (jw + 1) * m.h;
            if (m.ppgf_kind == QIW_GF_INC_SPLINE && normalize) n_known = std::max(n_known, jw + 2);
            fa.n_known = (m.ppgf_kind == QIW_GF_INC_SPLINE) ? n_known : m.ntau;
            fa.normalize = normalize ? 1 : 0;
            HIPCHK(c, finalize(bold_b, bold_d, next_of(jw)));
            launches += eval_launches(bold_b);
            c->stats.flops += bold_b.flops_per_launch;
            c->stats.leaves += bold_b.leaves_per_launch;
            c->stats.diagram_evals += bold_b.diagram_evals_per_launch;
        }
    }
    // a step returns its own row, the other calls all rows
    const bool one_row = step_value && !store_host_P && !P_orders_out && !P_orders_std_out;
    const int row0 = one_row ? (do_bare ? 1 : first_w + 1) : 0, n_rows = one_row ? 1 : m.ntau;
    std::vector<double> ptab_h((size_t)n_rows * m.bt), por((size_t)n_slots * n_rows * m.bt), lam_h(one_row ? 0 : m.ntau);
    std::vector<double> pstd_h(pstd && !one_row ? por.size() : 0);
    stage.add(ptab_h.data(), ptab + (size_t)row0 * m.bt, ptab_h.size() * 8);
    if (one_row)
        for (int o = 0; o < n_slots; ++o)
            stage.add(por.data() + (size_t)o * m.bt, porders + ((size_t)o * m.ntau + row0) * m.bt, (size_t)m.bt * 8);
    else
        stage.add(por.data(), porders, por.size() * 8);
    stage.add(lam_h.data(), lam, lam_h.size() * 8);
    stage.add(pstd_h.data(), pstd, pstd_h.size() * 8);
    if ((rc = stage.download())) return rc;
    for (size_t i = 0; i + 1 < n_ev; i += 2) {
        float ms = 0;
        HIPCHK(c, hipEventElapsedTime(&ms, c->evpool[i], c->evpool[i + 1]));
        c->stats.kernel_ms += ms;
    }
    for (auto &pr : graph_ev) {
        float ms = 0;
        HIPCHK(c, hipEventElapsedTime(&ms, pr.first, pr.second));
        c->stats.kernel_ms += ms;
    }
    c->stats.n_kernel_launches += launches;
    if ((rc = check_given_use(c, bare_b, use_bare, nuse_bare, rows_bare))) return rc;
    if ((rc = check_given_use(c, bold_b, use_bold, nuse_bold, rows_bold))) return rc;

    if (store_host_P) {
        c->ip = ptab_h;
        c->n_known = (m.ppgf_kind == QIW_GF_INC_SPLINE) ? n_known : m.ntau;
        c->lambdas = lam_h;
    }
    if (P_orders_out || P_orders_std_out) {
        const double nan = std::nan("");
        for (size_t o = 0; o < oall.size(); ++o) {
            bool in_bare = std::find(run->orders_bare, run->orders_bare + run->n_orders_bare, oall[o]) !=
                           run->orders_bare + run->n_orders_bare;
            bool in_bold = std::find(run->orders, run->orders + run->n_orders, oall[o]) != run->orders + run->n_orders;
            for (int j = 0; j < m.ntau; ++j)
                for (int e = 0; e < m.bt; ++e) {
                    size_t i = ((size_t)o * m.ntau + j) * m.bt + e;
                    if (P_orders_out) store_complex_from_ip(por[i], P_orders_out + 2 * i);
                    if (P_orders_std_out && pstd) {  // real: sqrt of the variance of complex values
                        P_orders_std_out[2 * i] = pstd_h[i];
                        P_orders_std_out[2 * i + 1] = 0.0;
                    } else if (P_orders_std_out) {
                        bool sampled_here = oall[o] > 0 && run->N_samples > 0 &&
                                            ((j == 1 && in_bare && do_bare) || (j >= first_w + 1 && j <= last_w + 1 && in_bold));
                        P_orders_std_out[2 * i] = sampled_here ? nan : 0.0;
                        P_orders_std_out[2 * i + 1] = sampled_here ? nan : 0.0;
                    }
                }
        }
    }
    if (step_value) {
        const int jf = (do_bare ? 1 : first_w + 1) - row0;
        step_value->assign(ptab_h.begin() + (size_t)jf * m.bt, ptab_h.begin() + (size_t)(jf + 1) * m.bt);
        step_orders->clear();
        for (int o = 0; o < n_slots; ++o)
            step_orders->insert(step_orders->end(), por.begin() + ((size_t)o * n_rows + jf) * m.bt,
                                por.begin() + ((size_t)o * n_rows + jf + 1) * m.bt);
    }
    c->stats.wall_s += std::chrono::duration<double>(std::chrono::steady_clock::now() - t0).count();
    return 0;
}

}  // namespace

static int qiw_inchworm_impl(qiw_ctx *c, const qiw_run *run, double *P_out, double *P_orders_out,
                            double *P_orders_std_out) {
    if (!c) return QIW_E_ARG;
    int rc = check_run(c, run);
    if (rc) return rc;
    (void)hipSetDevice(c->device);
    c->stats = qiw_stats{};
    atomic_ip(c->m, c->ip);  // inchworm! starts from the staged atomic propagator
    c->n_known = (c->m.ppgf_kind == QIW_GF_INC_SPLINE) ? 1 : c->m.ntau;
    for (int s = 0; s < c->m.ns; ++s)
        for (int i = 0; i < c->m.dims[s]; ++i)
            c->der0[c->m.bt_off[s] + i + i * c->m.dims[s]] = cd(0.0, c->m.E[s][i] + c->m.lambda0);
    rc = run_inchworm(c, run, true, 1, c->m.ntau - 2, true, true, P_orders_out, P_orders_std_out, nullptr, nullptr);
    if (rc) return rc;
    if (c->m.ppgf_kind == QIW_GF_INC_SPLINE) {
        // derivative at 0 of the incremental splines after every normalize!
        // (src/ppgf.jl:687-688: der - i*lambda*P(0) with P(0) = -i on the diagonal)
        for (int j = 2; j < c->m.ntau; ++j)
            for (int s = 0; s < c->m.ns; ++s)
                for (int i = 0; i < c->m.dims[s]; ++i) c->der0[c->m.bt_off[s] + i + i * c->m.dims[s]] -= c->lambdas[j];
    }
    if (P_out) qiw_get_ppgf(c, nullptr, P_out, nullptr);
    return QIW_OK;
}

// ---------------------------------------------------------------------------------------
// Differential inchworm (src/inchworm.jl:528-778)
// ---------------------------------------------------------------------------------------
namespace {

// Self-energy groups of run->orders (order 0 has none; order 1 is exact), slot = index in
// run->orders.
int build_diff_batch_as(qiw_ctx *c, const qiw_run *run, Batch &b, bool arcs) {
    const HostModel &m = c->m;
    int max_order = 0;
    int64_t n_groups = 0;
    for (int oi = 0; oi < run->n_orders; ++oi) {
        max_order = std::max(max_order, (int)run->orders[oi]);
        n_groups += run->orders[oi] > 0;
    }
    const RandPlan rq = rand_plan(run);
    b.n_eval = rq.n_eval();
    b.scrambled = rq.scrambled;
    b.given = rq.given;
    b.max_order = max_order;
    b.precision = chain_precision(m, max_order, run->precision);
    set_format(m, b, arcs);
    const int64_t total = n_groups * b.n_eval * std::max<int64_t>(run->N_samples, 1);
    b.spt = samples_per_task(c, m, b.fmt, total);
    for (int oi = 0; oi < run->n_orders; ++oi) {
        const int order = run->orders[oi];
        if (order == 0 || (order > 1 && run->N_samples <= 0)) continue;  // :557, :567
        Compiled cg;
        const int rc = compile_group(c, b, QIW_G_SIGMA, order, 1, -1,
                                     c->tune.chunk_words > 0 ? c->tune.chunk_words : kChunkWordsDiff,
                                     vec_chunk_cost(c, run->N_samples, 1), cg);
        if (rc) return rc;
        if (cg.n_top == 0) continue;
        if (cg.g.n_wslots > 255 || m.ns > 255) return fail(c, QIW_E_LIMIT, "too many slots");
        b.lds = std::max(b.lds, lds_slots(cg, m, b.fmt));
        const int64_t N = order == 1 ? 1 : run->N_samples;
        const auto parts = task_parts(b, cg, most_parts(total / b.spt, total / b.spt + n_groups * b.n_eval, call_rows(m)));
        const double flops = (double)N * sample_flops(cg);
        const int64_t leaves = N * cg.leaves_per_sample, evals = N * cg.n_top;
        push_sequences(b, std::move(cg), b.n_eval, [&](int gi) {
            b.g_first.push_back((int32_t)b.tasks.size());
            const int64_t nt64 = (N + b.spt - 1) / b.spt;
            const int nt = tasks_fit(b, nt64 * (int64_t)parts.size()) ? (int)nt64 : 0;
            for (int t = 0; t < nt; ++t)
                for (auto &p : parts) b.tasks.push_back({gi, t * b.spt, 0, (int32_t)b.tasks.size(), p.first, p.second});
            b.g_count.push_back(nt * (int)parts.size());
            b.g_slot.push_back(oi);
            b.flops_per_launch += flops;
            b.leaves_per_launch += leaves;
            b.diagram_evals_per_launch += evals;
        });
    }
    if (b.r_first.size() > 64) return fail(c, QIW_E_LIMIT, "more than 64 self-energy groups");
    if (b.overflow) return fail(c, QIW_E_LIMIT, "more than 2^28 workgroups in one launch (lower N_samples)");
    order_tasks(b);
    return 0;
}

int build_diff_batch(qiw_ctx *c, const qiw_run *run, Batch &b) {
    b = Batch{};
    const int rc = build_diff_batch_as(c, run, b, true);
    if (rc == 0)
        return prefer_tries(c->m, b, run->N_samples, 1, [&](Batch &t) { return build_diff_batch_as(c, run, t, false); });
    if (rc != kArcNoFit) return rc;
    b = Batch{};
    return build_diff_batch_as(c, run, b, false);
}

// diff_inchworm!: n_tau - 1 steps from the atomic propagator, each one evaluator launch
// over the self-energy groups at tau_f_prev = grid[a] and one k_diff_reduce_finalize
// (self-energy row, Σ * P convolution, Euler step into row a + 1).
int run_diff(qiw_ctx *c, const qiw_run *run, double *S_out, double *S_std_out) {
    const HostModel &m = c->m;
    auto t0 = std::chrono::steady_clock::now();
    const RandPlan rq = rand_plan(run);
    const bool rqmc = rq.n_seqs > 1;
    const std::vector<int> oslots(run->orders, run->orders + run->n_orders);
    const int n_slots = std::max(run->n_orders, 1);
    int rc = 0;
    Plan &p = plan_slot(c, "diff");
    const std::string key = plan_key(c, run, oslots, "diff");
    if (p.key != key) {
        p = Plan{};
        if ((rc = build_diff_batch(c, run, p.b))) return rc;
        if (!p.b.groups.empty() && (rc = upload(c, "diff", p.b, run->N_samples, p.d))) return rc;
        p.key = key;
    }
    const Batch &b = p.b;
    const DevBatch &d = p.d;
    // the reference sums the orders' self-energies (src/inchworm.jl:606), which needs one
    if (b.groups.empty()) return fail(c, QIW_E_ARG, "diff_inchworm needs a self-energy order >= 1");
    // caller-drawn sequences: every step's in step order; at tau_f_prev = tau_i (step 0) the
    // sampled self-energy simplices have zero volume
    GivenSrc gsrc;
    const int64_t *gidx = nullptr;
    int32_t *nuse = nullptr;
    std::vector<int32_t> use;
    std::vector<int> rows;
    if (rq.given && run->N_samples > 0) {
        const size_t ng = b.groups.size(), nr = b.r_first.size();
        std::vector<int64_t> idx((size_t)(m.ntau - 1) * ng);
        use.resize((size_t)(m.ntau - 1) * nr);
        int64_t n = 0;
        for (int st = 0; st + 1 < m.ntau; ++st) {
            n += given_row(b, rq.n_seqs, n, [&](const QiwGroup &) { return st == 0; }, idx.data() + st * ng,
                           use.data() + st * nr);
            rows.push_back(st + 1);
        }
        if ((rc = given_buffers(c, rq.points, b.max_order, n, run->N_samples, &gsrc))) return rc;
        int64_t *didx = (int64_t *)dev(c, "given.idx", std::max<size_t>(idx.size(), 1) * 8, &rc);
        if (rq.n_seqs >= 3) nuse = (int32_t *)dev(c, "given.nuse_diff", (size_t)m.ntau * std::max<size_t>(nr, 1) * 4, &rc);
        if (rc) return rc;
        HIPCHK(c, hipMemcpy(didx, idx.data(), idx.size() * 8, hipMemcpyHostToDevice));
        gidx = didx;
    }
    double *dcoef, *eshift;
    int32_t *dkind;
    if ((rc = ensure_model_buffers(c, &dcoef, &dkind, &eshift))) return rc;
    const size_t tab = (size_t)m.ntau * m.bt;
    double *partial = (double *)dev(c, "partial", std::max<size_t>(b.tasks.size(), 1) * m.bt * 8, &rc);
    double *ptab = (double *)dev(c, "ptab", tab * 8, &rc);
    double *sig = (double *)dev(c, "diff.sigma", tab * 8, &rc);
    double *porders = (double *)dev(c, "porders", (size_t)n_slots * tab * 8, &rc);
    double *pstd = rqmc ? (double *)dev(c, "porders_std", (size_t)n_slots * tab * 8, &rc) : nullptr;
    double *scratch = (double *)dev(c, "fin.scratch", b.r_first.size() * 2 * m.bt * 8 + 8, &rc);
    double *gsum = (double *)dev(c, "fin.gsum", std::max<size_t>(b.groups.size(), 1) * m.bt * 8, &rc);
    double *hdiag = (double *)dev(c, "diff.hdiag", (size_t)m.bt * 8, &rc);
    int32_t *ddims = (int32_t *)dev(c, "diff.dims", (size_t)m.ns * 4, &rc);
    int32_t *dbtoff = (int32_t *)dev(c, "diff.btoff", (size_t)m.ns * 4, &rc);
    unsigned *done = (unsigned *)dev(c, "fin.done", 4, &rc);
    uint32_t *sobm = rq.scrambled ? (uint32_t *)dev(c, "sobol.m", c->sob_m.size() * 4, &rc) : nullptr;
    if (rc) return rc;
    std::vector<double> hd((size_t)m.bt, 0.0);
    for (int s = 0; s < m.ns; ++s)
        for (int i = 0; i < m.dims[s]; ++i) hd[m.bt_off[s] + i + i * m.dims[s]] = m.E[s][i] + m.lambda0;
    std::vector<int32_t> d32(m.dims.begin(), m.dims.end()), o32(m.bt_off.begin(), m.bt_off.end());
    HIPCHK(c, hipMemcpy(hdiag, hd.data(), hd.size() * 8, hipMemcpyHostToDevice));
    HIPCHK(c, hipMemcpy(ddims, d32.data(), (size_t)m.ns * 4, hipMemcpyHostToDevice));
    HIPCHK(c, hipMemcpy(dbtoff, o32.data(), (size_t)m.ns * 4, hipMemcpyHostToDevice));
    HIPCHK(c, hipMemcpy(ptab, c->ip.data(), c->ip.size() * 8, hipMemcpyHostToDevice));
    HIPCHK(c, hipMemsetAsync(done, 0, 4, c->stream));
    HIPCHK(c, hipMemsetAsync(sig, 0, tab * 8, c->stream));
    HIPCHK(c, hipMemsetAsync(porders, 0, (size_t)n_slots * tab * 8, c->stream));
    if (pstd) HIPCHK(c, hipMemsetAsync(pstd, 0, (size_t)n_slots * tab * 8, c->stream));
    if (sobm) HIPCHK(c, hipMemcpy(sobm, c->sob_m.data(), c->sob_m.size() * 4, hipMemcpyHostToDevice));

    FinalizeArgs fa{};
    fa.groups = d.groups;
    fa.group_task_first = d.g_first;
    fa.group_task_count = d.g_count;
    fa.most_rows = most_rows(b);
    fa.group_order_slot = d.g_slot;
    fa.n_groups = (int)b.groups.size();
    fa.n_order_slots = n_slots;
    fa.partial = partial;
    fa.bt = m.bt;
    fa.ptab = sig;  // the self-energy table
    fa.porders = porders;
    fa.n_tau = m.ntau;
    fa.h = m.h;
    fa.bare = 0;
    fa.normalize = 0;
    fa.scratch = scratch;
    fa.gsum = gsum;
    fa.done = done;
    fa.n_real = (int)b.r_first.size();
    fa.real_first = d.r_first;
    fa.real_count = d.r_count;
    fa.n_seqs = rq.n_seqs;
    fa.target_std = rq.target_std;
    fa.porders_std = pstd;
    fa.nuse_out = nuse;
    fa.P = ptab;
    fa.hdiag = hdiag;
    fa.dims = ddims;
    fa.bt_off = dbtoff;
    fa.ns = m.ns;
    // set_ppgf! on Σ: an incremental container appends (row a + 1 at step a), a grid one
    // writes the row of tau_f_prev (row a)
    const int sig_shift = (m.ppgf_kind == QIW_GF_INC_SPLINE) ? 1 : 0;

    // timing events from the context's pool (created once, reused by every call)
    size_t n_ev = 0;
    auto mark = [&](void) -> hipError_t {
        if (c->no_alloc) return hipSuccess;  // creates no events: no timing of a no-alloc call
        if (n_ev == c->evpool.size()) {
            hipEvent_t e;
            hipError_t r = hipEventCreate(&e);
            if (r != hipSuccess) return r;
            c->evpool.push_back(e);
        }
        return hipEventRecord(c->evpool[n_ev++], c->stream);
    };
    EvalArgs a = make_eval_args(c, b, d, ptab, eshift, dcoef, dkind, partial);
    int64_t launches = 0;
    // the loop is timed as a whole: an event before and after every evaluator kept the GPU waiting
    // for a third of each step
    HIPCHK(c, mark());
    for (int st = 0; st + 1 < m.ntau; ++st) {
        fa.a = st;
        fa.jf = st + 1;  // Σ_orders at tau_f (src/inchworm.jl:770-773)
        fa.jt = st + sig_shift;
        fa.tau_w = fa.tau_f = st * m.h;
        a.step_w = st;
        if (gidx)
            HIPCHK(c, qiw_launch_given_coords(c->stream, d.groups, (int)b.groups.size(), run->N_samples, gsrc,
                                              gidx + (size_t)st * b.groups.size(), 1, 0, 0, d.ut));
        else if (b.scrambled && !b.given)
            HIPCHK(c, qiw_launch_rqmc_coords(c->stream,
                                             RqmcCoords{d.groups, sobm, (int)b.groups.size(),
                                                        run->N_samples > 0 ? run->N_samples : 1, rq.seed, QIW_RQ_DIFF,
                                                        (uint64_t)st, d.ut},
                                             2 * b.max_order));
        if ((rc = launch_eval(c, a, b))) return rc;
        HIPCHK(c, qiw_launch_finalize_diff(c->stream, fa, rqmc ? 1 : 0));
        launches += eval_launches(b);
        c->stats.flops += b.flops_per_launch;
        c->stats.leaves += b.leaves_per_launch;
        c->stats.diagram_evals += b.diagram_evals_per_launch;
    }
    HIPCHK(c, mark());
    HIPCHK(c, hipStreamSynchronize(c->stream));
    for (size_t i = 0; i + 1 < n_ev; i += 2) {
        float ms = 0;
        HIPCHK(c, hipEventElapsedTime(&ms, c->evpool[i], c->evpool[i + 1]));
        c->stats.kernel_ms += ms;
    }
    c->stats.n_kernel_launches += launches;
    if ((rc = check_given_use(c, b, use, nuse, rows))) return rc;
    std::vector<double> P_h(tab), por((size_t)n_slots * tab), pstd_h(pstd ? por.size() : 0);
    HIPCHK(c, hipMemcpy(P_h.data(), ptab, tab * 8, hipMemcpyDeviceToHost));
    HIPCHK(c, hipMemcpy(por.data(), porders, por.size() * 8, hipMemcpyDeviceToHost));
    if (pstd) HIPCHK(c, hipMemcpy(pstd_h.data(), pstd, pstd_h.size() * 8, hipMemcpyDeviceToHost));
    c->ip = P_h;
    c->n_known = m.ntau;
    std::vector<char> sampled(n_slots, 0);  // orders with a qMC group (std NaN for one sequence)
    for (size_t gi = 0; gi < b.groups.size(); ++gi)
        if (!qiw_group_exact(b.groups[gi].g)) sampled[b.g_slot[gi]] = 1;
    const double nan = std::nan("");
    for (int o = 0; o < run->n_orders; ++o)
        for (int j = 0; j < m.ntau; ++j)
            for (int e = 0; e < m.bt; ++e) {
                const size_t i = ((size_t)o * m.ntau + j) * m.bt + e;
                if (S_out) {  // Σ = i sigma
                    S_out[2 * i] = 0.0;
                    S_out[2 * i + 1] = por[i];
                }
                if (S_std_out) {
                    const double v = pstd ? pstd_h[i] : (sampled[o] && j >= 1 ? nan : 0.0);
                    S_std_out[2 * i] = v;
                    S_std_out[2 * i + 1] = pstd ? 0.0 : v;
                }
            }
    c->stats.wall_s += std::chrono::duration<double>(std::chrono::steady_clock::now() - t0).count();
    return 0;
}
}  // namespace

static int qiw_diff_inchworm_impl(qiw_ctx *c, const qiw_run *run, double *P_out, double *Sigma_orders_out,
                                 double *Sigma_orders_std_out) {
    if (!c) return QIW_E_ARG;
    int rc = check_run(c, run);
    if (rc) return rc;
    (void)hipSetDevice(c->device);
    c->stats = qiw_stats{};
    atomic_ip(c->m, c->ip);  // diff_inchworm! starts from the staged atomic propagator
    for (int s = 0; s < c->m.ns; ++s)
        for (int i = 0; i < c->m.dims[s]; ++i)
            c->der0[c->m.bt_off[s] + i + i * c->m.dims[s]] = cd(0.0, c->m.E[s][i] + c->m.lambda0);
    if ((rc = run_diff(c, run, Sigma_orders_out, Sigma_orders_std_out))) return rc;
    if (P_out) qiw_get_ppgf(c, nullptr, P_out, nullptr);
    return QIW_OK;
}

static int qiw_inchworm_step_impl(qiw_ctx *c, const qiw_run *run, int32_t n_w, double *value_out, double *orders_out) {
    if (!c) return QIW_E_ARG;
    int rc = check_run(c, run);
    if (rc) return rc;
    if (n_w < 1 || n_w > c->m.ntau - 2) return fail(c, QIW_E_ARG, "n_w out of range");
    (void)hipSetDevice(c->device);
    c->stats = qiw_stats{};
    std::vector<double> val, per;
    rc = run_inchworm(c, run, false, n_w, n_w, false, false, nullptr, nullptr, &val, &per);
    if (rc) return rc;
    for (int e = 0; e < c->m.bt; ++e)
        if (value_out) store_complex_from_ip(val[e], value_out + 2 * e);
    if (orders_out)
        for (size_t i = 0; i < per.size() && i < (size_t)run->n_orders * c->m.bt; ++i)
            store_complex_from_ip(per[i], orders_out + 2 * i);
    return QIW_OK;
}

// The same step with nothing allocated: the plan, model tables and walk buffers of a
// previous qiw_inchworm_step with the same run stay in use, the per-call buffers come from
// the device's static scratch array, and no timing events or graphs are made.
static int qiw_inchworm_step_noalloc_impl(qiw_ctx *c, const qiw_run *run, int32_t n_w, double *value_out,
                                          double *orders_out) {
    if (!c) return QIW_E_ARG;
    if (!c->scratch) return fail(c, QIW_E_STATE, "no scratch array on this device");
    if (warp_enabled(c->warp)) return fail(c, QIW_E_ARG, "the learned warp is not available without allocation");
    struct Mode {
        qiw_ctx *c;
        ~Mode() { c->no_alloc = false; }
    } mode{c};
    c->no_alloc = true;
    c->scratch_used = 0;
    return qiw_inchworm_step_impl(c, run, n_w, value_out, orders_out);
}

static int qiw_inchworm_step_bare_impl(qiw_ctx *c, const qiw_run *run, double *value_out, double *orders_out) {
    if (!c) return QIW_E_ARG;
    int rc = check_run(c, run);
    if (rc) return rc;
    (void)hipSetDevice(c->device);
    c->stats = qiw_stats{};
    qiw_run r2 = *run;
    r2.orders = run->orders_bare;  // order slots follow orders_bare
    r2.n_orders = run->n_orders_bare;
    std::vector<double> val, per;
    rc = run_inchworm(c, &r2, true, 1, 0, false, false, nullptr, nullptr, &val, &per);
    if (rc) return rc;
    for (int e = 0; e < c->m.bt; ++e)
        if (value_out) store_complex_from_ip(val[e], value_out + 2 * e);
    if (orders_out)
        for (size_t i = 0; i < per.size() && i < (size_t)run->n_orders_bare * c->m.bt; ++i)
            store_complex_from_ip(per[i], orders_out + 2 * i);
    return QIW_OK;
}

namespace {
// The groups of operator pair ci (src/inchworm.jl:957-981): every n_pts_after of every
// order with topologies, compiled.
int build_corr_groups_as(qiw_ctx *c, const qiw_run *run, int ci, Batch &b, bool *first_is_order0, bool arcs) {
    const HostModel &m = c->m;
    const RandPlan rq = rand_plan(run);
    int max_order = 0;
    for (int oi = 0; oi < run->n_orders; ++oi) max_order = std::max(max_order, (int)run->orders[oi]);
    b.max_order = max_order;
    b.precision = chain_precision(m, max_order, run->precision);
    set_format(m, b, arcs);
    b.n_eval = rq.n_eval();
    b.scrambled = rq.scrambled;
    b.given = rq.given;
    *first_is_order0 = false;
    for (int oi = 0; oi < run->n_orders; ++oi) {
        int order = run->orders[oi];
        if (order > 0 && run->N_samples <= 0) continue;
        int lo = order == 0 ? 0 : 1, hi = order == 0 ? 0 : 2 * order - 1;
        for (int na = lo; na <= hi; ++na) {
            Compiled cg;
            const int rc = compile_group(c, b, QIW_G_CORR, order, na, ci,
                                         c->tune.chunk_words > 0 ? c->tune.chunk_words : kChunkWords,
                                         vec_chunk_cost(c, run->N_samples, m.ntau), cg);
            if (rc) return rc;
            if (cg.n_top == 0) continue;
            if (b.groups.empty() && order == 0) *first_is_order0 = true;
            b.lds = std::max(b.lds, lds_slots(cg, m, b.fmt));
            push_sequences(b, std::move(cg), b.n_eval, [](int) {});
        }
    }
    if (b.r_first.size() > 64) return fail(c, QIW_E_LIMIT, "more than 64 (order, n_pts_after) groups");
    return 0;
}

int build_corr_groups(qiw_ctx *c, const qiw_run *run, int ci, Batch &b, bool *first_is_order0) {
    b = Batch{};
    const int rc = build_corr_groups_as(c, run, ci, b, first_is_order0, true);
    if (rc == 0)
        return prefer_tries(c->m, b, run->N_samples, c->m.ntau,
                            [&](Batch &t) { return build_corr_groups_as(c, run, ci, t, first_is_order0, false); });
    if (rc != kArcNoFit) return rc;
    b = Batch{};
    return build_corr_groups_as(c, run, ci, b, first_is_order0, false);
}

// The groups of all operator pairs in one batch, one output per pair: a scalar model's pairs
// on the same points share times, arc values and propagators, which is what a correlator of
// low order spends its time on (three pairs of orders 0:3 on 200 points, N = 2^14: 6.9 ms one
// after the other, 3.5 ms together).  Returns kArcNoFit when a group does not fit the walk.
bool corr_together(const HostModel &m, const RandPlan &rq) {
    return m.scalar_kernel && m.ncorr > 1 && m.ncorr <= 8 && !rq.scrambled && !rq.given && rq.n_seqs == 1;
}
int build_corr_all(qiw_ctx *c, const qiw_run *run, Batch &b, bool *first_is_order0) {
    const HostModel &m = c->m;
    std::vector<int> all;
    for (int ci = 0; ci < m.ncorr; ++ci) all.push_back(ci);
    for (int oi = 0; oi < run->n_orders; ++oi) b.max_order = std::max(b.max_order, (int)run->orders[oi]);
    b.precision = run->precision;
    set_format(m, b, true);
    if (b.fmt != FMT_SARC) return kArcNoFit;
    b.n_out = m.ncorr;
    *first_is_order0 = false;
    for (int oi = 0; oi < run->n_orders; ++oi) {
        const int order = run->orders[oi];
        if (order > 0 && run->N_samples <= 0) continue;
        for (int na = order == 0 ? 0 : 1; na <= (order == 0 ? 0 : 2 * order - 1); ++na) {
            Compiled cg;
            const int rc = compile_scalar_arcs(m, QIW_G_CORR, order, na, all, c->tune.chunk_words, cg);
            if (rc) return rc == 1 ? fail(c, QIW_E_OFFDIAG, kOffDiagonal) : kArcNoFit;
            if (cg.n_top == 0) continue;
            if (b.groups.empty() && order == 0) *first_is_order0 = true;
            push_sequences(b, std::move(cg), 1, [](int) {});
        }
    }
    if (b.r_first.size() > 64) return fail(c, QIW_E_LIMIT, "more than 64 (order, n_pts_after) groups");
    return 0;
}

// correlator_2p(expansion, grid, orders, N_samples, RequestStdDev(); rand_params)
// (src/inchworm.jl:918-1052); corr_std_out may be NULL.
int run_correlator(qiw_ctx *c, const qiw_run *run, double *corr_out, double *corr_std_out) {
    if (!c || !corr_out) return QIW_E_ARG;
    int rc = check_run(c, run);
    if (rc) return rc;
    (void)hipSetDevice(c->device);
    c->stats = qiw_stats{};
    auto t0 = std::chrono::steady_clock::now();
    const HostModel &m = c->m;
    const RandPlan rq = rand_plan(run);
    const bool rqmc = rq.n_seqs > 1;
    std::memset(corr_out, 0, sizeof(double) * 2 * (size_t)m.ncorr * m.ntau);
    if (corr_std_out) std::memset(corr_std_out, 0, sizeof(double) * 2 * (size_t)m.ncorr * m.ntau);
    if (m.ncorr == 0 || run->n_orders == 0) return QIW_OK;
    double Z = 0;  // partition_function(P) = sum_s tr iP_s(beta), src/ppgf.jl:611-617
    for (int s = 0; s < m.ns; ++s)
        for (int i = 0; i < m.dims[s]; ++i) Z += c->ip[(size_t)(m.ntau - 1) * m.bt + m.bt_off[s] + i + i * m.dims[s]];
    double *dcoef, *eshift;
    int32_t *dkind;
    if ((rc = ensure_model_buffers(c, &dcoef, &dkind, &eshift))) return rc;
    double *ptab = (double *)dev(c, "ptab", (size_t)m.ntau * m.bt * 8, &rc);
    if (rc) return rc;
    HIPCHK(c, hipMemcpy(ptab, c->ip.data(), c->ip.size() * 8, hipMemcpyHostToDevice));
    std::vector<int> oall(run->orders, run->orders + run->n_orders);
    std::vector<int32_t> dg;  // BT indices of the diagonal elements (the trace)
    for (int s = 0; s < m.ns; ++s)
        for (int i = 0; i < m.dims[s]; ++i) dg.push_back(m.bt_off[s] + i + i * m.dims[s]);
    // all pairs in one batch where they can be
    bool together = corr_together(m, rq);
    if (together) {
        Plan &p = plan_slot(c, "corr.all");
        const std::string key = plan_key(c, run, oall, "corr.all");
        if (p.key != key) {
            p = Plan{};
            rc = build_corr_all(c, run, p.b, &p.first_is_order0);
            if (rc && rc != kArcNoFit) return rc;
            p.fits = rc == 0;
            rc = 0;
        }
        together = p.fits;
        if (!together) p.key = key;
    }
    if (together)
        for (int ci = 0; ci < m.ncorr; ++ci) dg.push_back(ci);  // behind the trace: each pair's output
    const int dg_trace = (int)dg.size() - (together ? m.ncorr : 0);
    int32_t *diag = (int32_t *)dev(c, "corr.diag", dg.size() * 4, &rc);
    uint32_t *sobm = rq.scrambled ? (uint32_t *)dev(c, "sobol.m", c->sob_m.size() * 4, &rc) : nullptr;
    if (rc) return rc;
    HIPCHK(c, hipMemcpy(diag, dg.data(), dg.size() * 4, hipMemcpyHostToDevice));
    if (sobm) HIPCHK(c, hipMemcpy(sobm, c->sob_m.data(), c->sob_m.size() * 4, hipMemcpyHostToDevice));
    // the pairs are queued on the stream back to back; their results are read after one
    // synchronisation
    struct PairOut {
        int ci, n;  // pairs ci .. ci + n - 1
        std::vector<double> out, out_std;
        hipEvent_t e0, e1;
        bool any_sampled;
    };
    std::vector<PairOut> pending;
    pending.reserve(m.ncorr);
    int64_t given_next = 0;  // caller-drawn sequences taken by the pairs so far
    const int n_pairs = together ? m.ncorr : 1;  // of a launch
    for (int ci = 0; ci < m.ncorr; ci += n_pairs) {
        // groups (src/inchworm.jl:957-981): every n_pts_after of every order
        const std::string tag = together ? "corr.all" : "corr" + std::to_string(ci);
        Plan &p = plan_slot(c, tag);
        const std::string key = plan_key(c, run, oall, tag);
        if (p.key != key) {
            Batch &b = p.b;
            if (!together) {
                p = Plan{};
                if ((rc = build_corr_groups(c, run, ci, b, &p.first_is_order0))) return rc;
            }
            if (!b.groups.empty()) {
                int ng = (int)b.groups.size();
                const int64_t total = (int64_t)m.ntau * ng * std::max<int64_t>(run->N_samples, 1);
                b.spt = samples_per_task(c, m, b.fmt, total);
                std::vector<int32_t> rf((size_t)m.ntau * ng, 0), rcnt((size_t)m.ntau * ng, 0);
                for (int j = 0; j < m.ntau; ++j)
                    for (int gi = 0; gi < ng; ++gi) {
                        // tau_A = tau_B: only the leading order-0 group (src/inchworm.jl:1014-1024)
                        if (j == 0 && !(gi == 0 && p.first_is_order0)) continue;
                        int64_t N = b.groups[gi].g.order > 0 ? run->N_samples : 1;
                        const auto parts = task_parts(
                            b, b.groups[gi], most_parts(total / b.spt, total / b.spt + (int64_t)m.ntau * ng, call_rows(m)));
                        const int64_t nt64 = (N + b.spt - 1) / b.spt;
                        if (!tasks_fit(b, nt64 * (int64_t)parts.size()))
                            return fail(c, QIW_E_LIMIT, "more than 2^28 workgroups in one launch (lower N_samples)");
                        const int nt = (int)nt64;
                        rf[(size_t)j * ng + gi] = (int32_t)b.tasks.size();
                        rcnt[(size_t)j * ng + gi] = nt * (int)parts.size();
                        for (int t = 0; t < nt; ++t)
                            for (auto &q : parts)
                                b.tasks.push_back({gi, t * b.spt, j, (int32_t)b.tasks.size(), q.first, q.second});
                        b.flops_per_launch += (double)N * sample_flops(b.groups[gi]);
                        b.leaves_per_launch += N * b.groups[gi].leaves_per_sample;
                        b.diagram_evals_per_launch += N * b.groups[gi].n_top * n_pairs;
                    }
                order_tasks(b);
                if ((rc = upload(c, tag, b, run->N_samples, p.d))) return rc;
                p.rf = (int32_t *)dev(c, tag + ".rf", rf.size() * 4, &rc);
                p.rcnt = (int32_t *)dev(c, tag + ".rc", rcnt.size() * 4, &rc);
                if (rc) return rc;
                HIPCHK(c, hipMemcpy(p.rf, rf.data(), rf.size() * 4, hipMemcpyHostToDevice));
                HIPCHK(c, hipMemcpy(p.rcnt, rcnt.data(), rcnt.size() * 4, hipMemcpyHostToDevice));
            }
            p.key = key;
        }
        Batch &b = p.b;
        DevBatch &d = p.d;
        if (b.groups.empty()) continue;
        int ng = (int)b.groups.size();
        // the device buffers are reused by the next pair in stream order (its evaluator runs
        // after this pair's bookkeeping and copies); the host results stay per pair
        const int n_out = together ? m.ncorr : m.bt;
        const size_t partial_bytes = b.tasks.size() * n_out * 8;
        if (c->bufs["corr.partial"].n < partial_bytes)  // the buffer grows: let queued pairs finish with it
            HIPCHK(c, hipStreamSynchronize(c->stream));
        double *partial = (double *)dev(c, "corr.partial", partial_bytes, &rc);
        int32_t *drf = p.rf, *drc = p.rcnt;
        double *dout = (double *)dev(c, "corr.out", (size_t)n_pairs * m.ntau * 8, &rc);
        double *dout_std = rqmc ? (double *)dev(c, "corr.out_std", (size_t)m.ntau * 8, &rc) : nullptr;
        if (rc) return rc;
        // caller-drawn sequences: tau rows 1 .. n_tau-1 of every pair in turn, each with its own
        // coordinates (row j at ut + j * ut_total); at tau_A = beta the simplices after tau_A
        // have zero volume
        double *ut_rows = nullptr;
        int32_t *nuse = nullptr;
        std::vector<int32_t> use;
        std::vector<int> rows;
        if (b.given && run->N_samples > 0) {
            const size_t nr = b.r_first.size();
            std::vector<int64_t> idx((size_t)(m.ntau - 1) * ng);
            use.resize((size_t)(m.ntau - 1) * nr);
            int64_t n = 0;
            for (int j = 1; j < m.ntau; ++j) {
                n += given_row(b, rq.n_seqs, given_next + n,
                               [&](const QiwGroup &g) { return g.d_after > 0 && j == m.ntau - 1; },
                               idx.data() + (size_t)(j - 1) * ng, use.data() + (size_t)(j - 1) * nr);
                rows.push_back(j);
            }
            GivenSrc gsrc;
            if ((rc = given_buffers(c, rq.points, b.max_order, given_next + n, run->N_samples, &gsrc))) return rc;
            given_next += n;
            if ((double)m.ntau * b.ut_total * 8 > kMaxGivenCoordBytes)
                return fail(c, QIW_E_LIMIT, "coordinates of every tau row exceed 64 GiB (lower N_samples or N_seqs)");
            // the buffers are reused by the next pair: queued pairs finish with them first
            HIPCHK(c, hipStreamSynchronize(c->stream));
            ut_rows = (double *)dev(c, "corr.ut_rows", (size_t)m.ntau * b.ut_total * 8, &rc);
            int64_t *didx = (int64_t *)dev(c, "given.idx", idx.size() * 8, &rc);
            if (rq.n_seqs >= 3) nuse = (int32_t *)dev(c, "given.nuse_corr", (size_t)m.ntau * nr * 4, &rc);
            if (rc) return rc;
            HIPCHK(c, hipMemcpy(didx, idx.data(), idx.size() * 8, hipMemcpyHostToDevice));
            HIPCHK(c, qiw_launch_given_coords(c->stream, d.groups, ng, run->N_samples, gsrc, didx, m.ntau - 1, 1,
                                              b.ut_total, ut_rows));
        } else if (sobm && !b.given && run->N_samples > 0) {  // one set of scrambled sequences for all tau rows
            HIPCHK(c, qiw_launch_rqmc_coords(c->stream,
                                             RqmcCoords{d.groups, sobm, ng, run->N_samples, rq.seed, QIW_RQ_CORR,
                                                        (uint64_t)ci, d.ut},
                                             2 * b.max_order));
        }
        pending.push_back(PairOut{ci, n_pairs, std::vector<double>((size_t)n_pairs * m.ntau),
                                  std::vector<double>(m.ntau, 0.0), nullptr, nullptr, false});
        PairOut &po = pending.back();
        for (auto &cg : b.groups) po.any_sampled = po.any_sampled || cg.g.sampled;
        hipEvent_t &e0 = po.e0, &e1 = po.e1;
        HIPCHK(c, hipEventCreate(&e0));
        HIPCHK(c, hipEventCreate(&e1));
        HIPCHK(c, hipEventRecord(e0, c->stream));
        EvalArgs a = make_eval_args(c, b, d, ptab, eshift, dcoef, dkind, partial);
        if (ut_rows) {
            a.ut = ut_rows;
            a.ut_row_stride = b.ut_total;
        }
        if ((rc = launch_eval(c, a, b))) return rc;
        HIPCHK(c, hipEventRecord(e1, c->stream));
        CorrFinalizeArgs fa{};
        fa.groups = d.groups;
        fa.row_task_first = drf;
        fa.row_task_count = drc;
        fa.n_groups = ng;
        fa.n_rows = m.ntau;
        fa.n_tau = m.ntau;
        fa.partial = partial;
        fa.bt = n_out;
        fa.diag_idx = together ? diag + dg_trace : diag;
        fa.n_diag = together ? 1 : dg_trace;
        fa.n_pairs = n_pairs;
        fa.h = m.h;
        fa.beta = m.beta;
        fa.out = dout;
        fa.n_real = (int)b.r_first.size();
        fa.real_first = d.r_first;
        fa.real_count = d.r_count;
        fa.n_seqs = rq.n_seqs;
        fa.target_std = rq.target_std;
        fa.out_std = dout_std;
        fa.nuse_out = nuse;
        HIPCHK(c, rqmc ? qiw_launch_finalize_corr_rqmc(c->stream, fa) : qiw_launch_finalize_corr(c->stream, fa));
        if ((rc = check_given_use(c, b, use, nuse, rows))) return rc;
        HIPCHK(c, hipMemcpyAsync(po.out.data(), dout, po.out.size() * 8, hipMemcpyDeviceToHost, c->stream));
        if (dout_std)
            HIPCHK(c, hipMemcpyAsync(po.out_std.data(), dout_std, m.ntau * 8, hipMemcpyDeviceToHost, c->stream));
        c->stats.n_kernel_launches += eval_launches(b);
        c->stats.flops += b.flops_per_launch;
        c->stats.leaves += b.leaves_per_launch;
        c->stats.diagram_evals += b.diagram_evals_per_launch;
    }
    HIPCHK(c, hipStreamSynchronize(c->stream));
    for (PairOut &po : pending) {
        float ms = 0;
        HIPCHK(c, hipEventElapsedTime(&ms, po.e0, po.e1));
        (void)hipEventDestroy(po.e0);
        (void)hipEventDestroy(po.e1);
        c->stats.kernel_ms += ms;
        const std::vector<double> &out = po.out, &out_std = po.out_std;
        const bool any_sampled = po.any_sampled;
        for (int k = 0; k < po.n * m.ntau; ++k) {  // value = -i * out / Z
            const int j = k % m.ntau;
            const size_t i = (size_t)po.ci * m.ntau + k;
            corr_out[2 * i] = 0.0;
            corr_out[2 * i + 1] = -out[k] / Z;
            if (!corr_std_out) continue;
            if (rqmc) {  // sum of the groups' deviations / Z (real)
                corr_std_out[2 * i] = out_std[j] / Z;
                corr_std_out[2 * i + 1] = 0.0;
            } else {  // one sequence: the deviation of one sample is NaN; tau = 0 is exact
                const double v = (j > 0 && any_sampled) ? std::nan("") : 0.0;
                corr_std_out[2 * i] = v;
                corr_std_out[2 * i + 1] = v;
            }
        }
    }
    c->stats.wall_s = std::chrono::duration<double>(std::chrono::steady_clock::now() - t0).count();
    return QIW_OK;
}
}  // namespace

static int qiw_correlator_2p_impl(qiw_ctx *c, const qiw_run *run, double *corr_out) {
    return run_correlator(c, run, corr_out, nullptr);
}

static int qiw_correlator_2p_std_impl(qiw_ctx *c, const qiw_run *run, double *corr_out, double *corr_std_out) {
    if (!corr_std_out) return c ? fail(c, QIW_E_ARG, "null corr_std_out") : QIW_E_ARG;
    return run_correlator(c, run, corr_out, corr_std_out);
}

static int qiw_partition_function_impl(qiw_ctx *c, double *Z_out) {
    if (!c || !Z_out) return QIW_E_ARG;
    if (!c->has_model) return fail(c, QIW_E_STATE, "no model staged");
    const HostModel &m = c->m;
    double Z = 0;
    for (int s = 0; s < m.ns; ++s)
        for (int i = 0; i < m.dims[s]; ++i) Z += c->ip[(size_t)(m.ntau - 1) * m.bt + m.bt_off[s] + i + i * m.dims[s]];
    Z_out[0] = Z;
    Z_out[1] = 0.0;
    return QIW_OK;
}

static int qiw_density_matrix_impl(qiw_ctx *c, double *rho_out) {
    if (!c || !rho_out) return QIW_E_ARG;
    double Z[2];
    int rc = qiw_partition_function(c, Z);
    if (rc) return rc;
    const HostModel &m = c->m;
    // normalize!(P, beta) then rho = i P(beta)  (src/ppgf.jl:629-636, :729-733)
    double lam = std::log(Z[0]) / m.beta;
    double f = std::exp(-m.beta * lam);
    for (int e = 0; e < m.bt; ++e) {
        rho_out[2 * e] = c->ip[(size_t)(m.ntau - 1) * m.bt + e] * f;
        rho_out[2 * e + 1] = 0.0;
    }
    return QIW_OK;
}

static int qiw_sobol_points_impl(qiw_ctx *c, int32_t dim, int64_t first, int64_t n, double *out) {
    if (!c || !out || n < 0 || first < 0) return QIW_E_ARG;
    if (dim < 1 || dim > c->sob_dim) return fail(c, QIW_E_DIM, "Sobol dimension beyond the staged direction numbers");
    (void)hipSetDevice(c->device);
    int rc = 0;
    uint32_t *sm = (uint32_t *)dev(c, "sobol.m", c->sob_m.size() * 4, &rc);
    uint32_t *sx = (uint32_t *)dev(c, "sobol.x", c->sob_x.size() * 4, &rc);
    double *o = (double *)dev(c, "sobol.out", (size_t)std::max<int64_t>(n, 1) * dim * 8, &rc);
    if (rc) return rc;
    HIPCHK(c, hipMemcpy(sm, c->sob_m.data(), c->sob_m.size() * 4, hipMemcpyHostToDevice));
    HIPCHK(c, hipMemcpy(sx, c->sob_x.data(), c->sob_x.size() * 4, hipMemcpyHostToDevice));
    if (n == 0) return QIW_OK;
    HIPCHK(c, qiw_launch_sobol_points(c->stream, sm, sx, dim, first, n, o));
    HIPCHK(c, hipMemcpyAsync(out, o, (size_t)n * dim * 8, hipMemcpyDeviceToHost, c->stream));
    HIPCHK(c, hipStreamSynchronize(c->stream));
    return QIW_OK;
}

static int qiw_simplex_points_impl(qiw_ctx *c, int32_t d_before, int32_t d_after, double t_i, double t_w, double t_f,
                                  int64_t n, double *out) {
    if (!c || !out || n < 0 || d_before < 0 || d_after < 0) return QIW_E_ARG;
    int d = d_before + d_after;
    if (d < 1 || d > c->sob_dim) return fail(c, QIW_E_DIM, "Sobol dimension beyond the staged direction numbers");
    (void)hipSetDevice(c->device);
    int rc = 0;
    uint32_t *sm = (uint32_t *)dev(c, "sobol.m", c->sob_m.size() * 4, &rc);
    uint32_t *sx = (uint32_t *)dev(c, "sobol.x", c->sob_x.size() * 4, &rc);
    double *o = (double *)dev(c, "simplex.out", (size_t)std::max<int64_t>(n, 1) * d * 8, &rc);
    if (rc) return rc;
    HIPCHK(c, hipMemcpy(sm, c->sob_m.data(), c->sob_m.size() * 4, hipMemcpyHostToDevice));
    HIPCHK(c, hipMemcpy(sx, c->sob_x.data(), c->sob_x.size() * 4, hipMemcpyHostToDevice));
    if (n == 0) return QIW_OK;
    HIPCHK(c, qiw_launch_simplex_points(c->stream, sm, sx, d_before, d_after, t_i, t_w, t_f, n, o));
    HIPCHK(c, hipMemcpyAsync(out, o, (size_t)n * d * 8, hipMemcpyDeviceToHost, c->stream));
    HIPCHK(c, hipStreamSynchronize(c->stream));
    return QIW_OK;
}

static int qiw_get_stats_impl(qiw_ctx *c, qiw_stats *out) {
    if (!c || !out) return QIW_E_ARG;
    *out = c->stats;
    return QIW_OK;
}

// ---------------------------------------------------------------------------------------
// Training data of the learned warp
// ---------------------------------------------------------------------------------------
namespace qiwi {

int warp_collect(qiw_ctx *c, const qiw_run *run, const std::vector<int> &steps, int64_t n,
                 std::vector<WarpGroup> &gs, std::vector<double> &mag) {
    const HostModel &m = c->m;
    int rc = 0;
    qiw_run r = *run;
    r.N_samples = n;
    r.n_orders_bare = 0;
    r.rand_params = nullptr;  // training points: the staged sequence
    std::vector<int> oall = orders_all(&r);
    Batch b;
    DevBatch d;
    if ((rc = build_step_batch(c, &r, false, oall, b, false))) return rc;  // per-sample sums: one chunk
    if (program_format(m, b.max_order, b.precision) == FMT_BLOCK)
        return fail(c, QIW_E_LIMIT, "the learned warp needs sector blocks <= 6 and orders <= 4");
    if (b.groups.empty()) return fail(c, QIW_E_ARG, "no sampled bold groups to train on");
    if ((rc = upload(c, "wtrain", b, n, d))) return rc;
    double *dcoef, *eshift;
    int32_t *dkind;
    if ((rc = ensure_model_buffers(c, &dcoef, &dkind, &eshift))) return rc;
    int64_t ps_total = 0;
    for (auto &cg : b.groups) ps_total += cg.g.n_samples;
    double *partial = (double *)dev(c, "partial", std::max<size_t>(b.tasks.size(), 1) * m.bt * 8, &rc);
    double *ptab = (double *)dev(c, "ptab", (size_t)m.ntau * m.bt * 8, &rc);
    double *ps = (double *)dev(c, "wtrain.ps", (size_t)ps_total * 8, &rc);
    if (rc) return rc;
    HIPCHK(c, hipMemcpy(ptab, c->ip.data(), c->ip.size() * 8, hipMemcpyHostToDevice));
    gs.clear();
    for (auto &cg : b.groups)
        if (cg.g.sampled && warp_gid(cg.g) >= 0)
            gs.push_back({cg.g.order, cg.g.n_after, cg.g.d_before, cg.g.d_after, warp_gid(cg.g), cg.g.ps_off});
    mag.assign(steps.size() * gs.size() * (size_t)n, 0.0);
    std::vector<double> host((size_t)ps_total);
    EvalArgs a = make_eval_args(c, b, d, ptab, eshift, dcoef, dkind, partial);
    a.per_sample = ps;
    for (size_t si = 0; si < steps.size(); ++si) {
        a.step_w = steps[si];
        if ((rc = launch_eval(c, a, b))) return rc;
        HIPCHK(c, hipMemcpyAsync(host.data(), ps, (size_t)ps_total * 8, hipMemcpyDeviceToHost, c->stream));
        HIPCHK(c, hipStreamSynchronize(c->stream));
        for (size_t gi = 0; gi < gs.size(); ++gi)
            std::copy(host.begin() + gs[gi].off, host.begin() + gs[gi].off + n,
                      mag.begin() + (si * gs.size() + gi) * (size_t)n);
    }
    return QIW_OK;
}

}  // namespace qiwi

// ---------------------------------------------------------------------------------------
// Work mapping: fixed settings and the tuner
// ---------------------------------------------------------------------------------------
namespace {
int check_tuning(qiw_ctx *c, const qiw_tuning &t) {
    if (t.chunk_words < 0 || (t.chunk_words > 0 && t.chunk_words < 64))
        return fail(c, QIW_E_ARG, "chunk_words must be 0 or >= 64");
    if (t.chunk_cost < 0) return fail(c, QIW_E_ARG, "chunk_cost must be >= 0");
    const int s = t.samples_per_task;
    if (s < 0 || s > QIW_WAVE || (s & (s - 1))) return fail(c, QIW_E_ARG, "samples_per_task must be 0 or a power of 2 <= 64");
    return 0;
}

// Evaluator time (ms, best of 2 after a warm-up launch) of one bold step of `run` at
// tau_w = grid[n_tau/2] under the context's current work mapping.
int time_bold_step(qiw_ctx *c, const qiw_run *run, double *ms_out) {
    const HostModel &m = c->m;
    int rc = 0;
    qiw_run r = *run;
    r.n_orders_bare = 0;
    r.rand_params = nullptr;  // the work mapping is timed on one sequence
    std::vector<int> oall(r.orders, r.orders + r.n_orders);
    Batch b;
    DevBatch d;
    if ((rc = build_step_batch(c, &r, false, oall, b))) return rc;
    if (b.groups.empty()) return fail(c, QIW_E_ARG, "no bold groups to time");
    if ((rc = upload(c, "tune", b, r.N_samples, d))) return rc;
    double *dcoef, *eshift;
    int32_t *dkind;
    if ((rc = ensure_model_buffers(c, &dcoef, &dkind, &eshift))) return rc;
    double *partial = (double *)dev(c, "tune.partial", std::max<size_t>(b.tasks.size(), 1) * m.bt * 8, &rc);
    double *ptab = (double *)dev(c, "ptab", (size_t)m.ntau * m.bt * 8, &rc);
    if (rc) return rc;
    HIPCHK(c, hipMemcpy(ptab, c->ip.data(), c->ip.size() * 8, hipMemcpyHostToDevice));
    EvalArgs a = make_eval_args(c, b, d, ptab, eshift, dcoef, dkind, partial);
    a.step_w = std::max(1, m.ntau / 2 - 1);
    hipEvent_t e0, e1;
    HIPCHK(c, hipEventCreate(&e0));
    HIPCHK(c, hipEventCreate(&e1));
    double best = 1e300;
    for (int rep = 0; rep < 3; ++rep) {
        HIPCHK(c, hipEventRecord(e0, c->stream));
        if ((rc = launch_eval(c, a, b))) return rc;
        HIPCHK(c, hipEventRecord(e1, c->stream));
        HIPCHK(c, hipEventSynchronize(e1));
        float ms = 0;
        HIPCHK(c, hipEventElapsedTime(&ms, e0, e1));
        if (rep > 0) best = std::min(best, (double)ms);
    }
    (void)hipEventDestroy(e0);
    (void)hipEventDestroy(e1);
    *ms_out = best;
    return 0;
}

void free_tag(qiw_ctx *c, const std::string &prefix) {
    for (auto it = c->bufs.begin(); it != c->bufs.end();) {
        if (it->first.compare(0, prefix.size(), prefix) == 0) {
            if (it->second.p) (void)hipFree(it->second.p);
            it = c->bufs.erase(it);
        } else {
            ++it;
        }
    }
}
}  // namespace

static int qiw_set_graphs_impl(qiw_ctx *c, int32_t on) {
    if (!c) return QIW_E_ARG;
    c->graphs = on != 0;
    return QIW_OK;
}

static int qiw_set_tuning_impl(qiw_ctx *c, const qiw_tuning *t) {
    if (!c || !t) return QIW_E_ARG;
    int rc = check_tuning(c, *t);
    if (rc) return rc;
    c->tune = *t;
    c->tune.n_tried = 0;
    c->tune.best_ms = 0.0;
    return QIW_OK;
}

static int qiw_get_tuning_impl(qiw_ctx *c, qiw_tuning *out) {
    if (!c || !out) return QIW_E_ARG;
    *out = c->tune;
    return QIW_OK;
}

static int qiw_autotune_impl(qiw_ctx *c, const qiw_run *run, qiw_tuning *out) {
    if (!c) return QIW_E_ARG;
    int rc = check_run(c, run);
    if (rc) return rc;
    if (run->N_samples <= 0 || run->n_orders == 0) return fail(c, QIW_E_ARG, "autotune needs sampled orders");
    (void)hipSetDevice(c->device);
    const HostModel &m = c->m;
    int fmt;  // of the walk that the step runs on, which need not be the one tried first
    {
        qiw_run r = *run;
        r.n_orders_bare = 0;
        r.rand_params = nullptr;
        Batch b;
        if ((rc = build_step_batch(c, &r, false, std::vector<int>(r.orders, r.orders + r.n_orders), b))) return rc;
        fmt = b.fmt;
    }
    std::vector<qiw_tuning> cand;
    if (fmt == FMT_SCALAR || fmt == FMT_SARC) {
        for (int w : {256, 384, 512, 640, 896, 1024, 2048}) cand.push_back(qiw_tuning{w, 0, 0, 0, 0, 0.0});
    } else if (fmt == FMT_VEC && m.mmax <= 6) {
        for (int e = 16; e <= 20; ++e) cand.push_back(qiw_tuning{0, 0, (int64_t)1 << e, 0, 0, 0.0});
    } else if (fmt == FMT_VEC) {
        for (int e = 17; e <= 19; ++e)
            for (int spt : {1, 2, 4, 8, 16}) cand.push_back(qiw_tuning{0, spt, (int64_t)1 << e, 0, 0, 0.0});
    } else {
        for (int spt : {1, 2, 4, 8, 16, 32, 64}) cand.push_back(qiw_tuning{0, spt, 0, 0, 0, 0.0});
    }
    const qiw_tuning keep = c->tune;
    qiw_tuning best = keep;
    double best_ms = 1e300;
    for (const qiw_tuning &t : cand) {
        c->tune = t;
        double ms = 0;
        if ((rc = time_bold_step(c, run, &ms))) {
            c->tune = keep;
            free_tag(c, "tune");
            return rc;
        }
        if (ms < best_ms) {
            best_ms = ms;
            best = t;
        }
    }
    free_tag(c, "tune");
    best.n_tried = (int32_t)cand.size();
    best.best_ms = best_ms;
    c->tune = best;
    if (out) *out = best;
    return QIW_OK;
}

// ---- C ABI: every entry point runs its body through guarded() ----
extern "C" int qiw_create(qiw_ctx **out, int device) {
    return guarded(nullptr, [&] { return qiw_create_impl(out, device); });
}

extern "C" void qiw_destroy(qiw_ctx *c) {
    guarded(nullptr, [&] {
        qiw_destroy_impl(c);
        return 0;
    });
}

extern "C" int qiw_set_model(qiw_ctx *c, const qiw_model *mi) {
    return guarded(c, [&] { return qiw_set_model_impl(c, mi); });
}

// The dimensions of the caller-drawn sequences a call consumes, in order (as the runs
// above assign them).
static int64_t qiw_scramble_dims_impl(qiw_ctx *c, const qiw_run *run, int32_t call, int64_t cap, int32_t *dims) {
    if (!c) return QIW_E_ARG;
    if (cap > 0 && !dims) return fail(c, QIW_E_ARG, "null dims");
    int rc = check_run(c, run);
    if (rc) return rc;
    const HostModel &m = c->m;
    const RandPlan rq = rand_plan(run);
    std::vector<int32_t> out;
    const auto none = [](const QiwGroup &) { return false; };
    if (run->N_samples > 0) {
        if (call == QIW_CALL_INCHWORM || call == QIW_CALL_STEP_BARE) {
            Batch b;
            if ((rc = build_step_batch(c, run, true, orders_all(run), b))) return rc;
            given_row(b, rq.n_seqs, 0, none, nullptr, nullptr, &out);
        }
        if (call == QIW_CALL_INCHWORM || call == QIW_CALL_STEP) {
            Batch b;
            if ((rc = build_step_batch(c, run, false, orders_all(run), b))) return rc;
            const int steps = call == QIW_CALL_STEP ? 1 : m.ntau - 2;
            for (int i = 0; i < steps; ++i) given_row(b, rq.n_seqs, 0, none, nullptr, nullptr, &out);
        } else if (call == QIW_CALL_CORRELATOR) {
            for (int ci = 0; ci < m.ncorr; ++ci) {
                Batch b;
                bool o0 = false;
                if ((rc = build_corr_groups(c, run, ci, b, &o0))) return rc;
                for (int j = 1; j < m.ntau; ++j)
                    given_row(b, rq.n_seqs, 0, [&](const QiwGroup &g) { return g.d_after > 0 && j == m.ntau - 1; },
                              nullptr, nullptr, &out);
            }
        } else if (call == QIW_CALL_DIFF) {
            Batch b;
            if ((rc = build_diff_batch(c, run, b))) return rc;
            for (int st = 0; st + 1 < m.ntau; ++st)
                given_row(b, rq.n_seqs, 0, [&](const QiwGroup &) { return st == 0; }, nullptr, nullptr, &out);
        } else if (call != QIW_CALL_STEP_BARE) {
            return fail(c, QIW_E_ARG, "unknown call kind");
        }
    }
    for (int64_t i = 0; i < (int64_t)out.size() && i < cap; ++i) dims[i] = out[i];
    return (int64_t)out.size();
}

extern "C" int qiw_set_sobol(qiw_ctx *c, int32_t dim, const uint32_t *m, const uint32_t *shift) {
    return guarded(c, [&] { return qiw_set_sobol_impl(c, dim, m, shift); });
}

extern "C" int qiw_set_scrambles(qiw_ctx *c, int64_t n, int32_t stride, const uint32_t *m, const uint32_t *shift) {
    return guarded(c, [&] { return qiw_set_scrambles_impl(c, n, stride, m, shift); });
}

extern "C" int qiw_set_points(qiw_ctx *c, int64_t n, int64_t n_points, int32_t stride, const double *x) {
    return guarded(c, [&] { return qiw_set_points_impl(c, n, n_points, stride, x); });
}

extern "C" int64_t qiw_scramble_dims(qiw_ctx *c, const qiw_run *run, int32_t call, int64_t cap, int32_t *dims) {
    return guarded(c, [&] { return qiw_scramble_dims_impl(c, run, call, cap, dims); });
}

extern "C" int qiw_set_ppgf(qiw_ctx *c, int32_t n_known, const double *P, const double *der0) {
    return guarded(c, [&] { return qiw_set_ppgf_impl(c, n_known, P, der0); });
}

extern "C" int qiw_get_ppgf(qiw_ctx *c, int32_t *n_known_out, double *P, double *der0) {
    return guarded(c, [&] { return qiw_get_ppgf_impl(c, n_known_out, P, der0); });
}

extern "C" int qiw_inchworm(qiw_ctx *c, const qiw_run *run, double *P_out, double *P_orders_out,
                            double *P_orders_std_out) {
    return guarded(c, [&] { return qiw_inchworm_impl(c, run, P_out, P_orders_out, P_orders_std_out); });
}

extern "C" int qiw_diff_inchworm(qiw_ctx *c, const qiw_run *run, double *P_out, double *Sigma_orders_out,
                                 double *Sigma_orders_std_out) {
    return guarded(c, [&] { return qiw_diff_inchworm_impl(c, run, P_out, Sigma_orders_out, Sigma_orders_std_out); });
}

extern "C" int qiw_inchworm_step(qiw_ctx *c, const qiw_run *run, int32_t n_w, double *value_out, double *orders_out) {
    return guarded(c, [&] { return qiw_inchworm_step_impl(c, run, n_w, value_out, orders_out); });
}

extern "C" int qiw_inchworm_step_bare(qiw_ctx *c, const qiw_run *run, double *value_out, double *orders_out) {
    return guarded(c, [&] { return qiw_inchworm_step_bare_impl(c, run, value_out, orders_out); });
}

extern "C" int qiw_correlator_2p(qiw_ctx *c, const qiw_run *run, double *corr_out) {
    return guarded(c, [&] { return qiw_correlator_2p_impl(c, run, corr_out); });
}

extern "C" int qiw_correlator_2p_std(qiw_ctx *c, const qiw_run *run, double *corr_out, double *corr_std_out) {
    return guarded(c, [&] { return qiw_correlator_2p_std_impl(c, run, corr_out, corr_std_out); });
}

extern "C" int qiw_partition_function(qiw_ctx *c, double *Z_out) {
    return guarded(c, [&] { return qiw_partition_function_impl(c, Z_out); });
}

extern "C" int qiw_density_matrix(qiw_ctx *c, double *rho_out) {
    return guarded(c, [&] { return qiw_density_matrix_impl(c, rho_out); });
}

extern "C" int qiw_sobol_points(qiw_ctx *c, int32_t dim, int64_t first, int64_t n, double *out) {
    return guarded(c, [&] { return qiw_sobol_points_impl(c, dim, first, n, out); });
}

extern "C" int qiw_simplex_points(qiw_ctx *c, int32_t d_before, int32_t d_after, double t_i, double t_w, double t_f,
                                  int64_t n, double *out) {
    return guarded(c, [&] { return qiw_simplex_points_impl(c, d_before, d_after, t_i, t_w, t_f, n, out); });
}

extern "C" int qiw_get_stats(qiw_ctx *c, qiw_stats *out) {
    return guarded(c, [&] { return qiw_get_stats_impl(c, out); });
}

extern "C" int qiw_set_graphs(qiw_ctx *c, int32_t on) {
    return guarded(c, [&] { return qiw_set_graphs_impl(c, on); });
}

extern "C" int qiw_set_tuning(qiw_ctx *c, const qiw_tuning *t) {
    return guarded(c, [&] { return qiw_set_tuning_impl(c, t); });
}

extern "C" int qiw_get_tuning(qiw_ctx *c, qiw_tuning *out) {
    return guarded(c, [&] { return qiw_get_tuning_impl(c, out); });
}

extern "C" int qiw_autotune(qiw_ctx *c, const qiw_run *run, qiw_tuning *out) {
    return guarded(c, [&] { return qiw_autotune_impl(c, run, out); });
}

extern "C" int qiw_inchworm_step_noalloc(qiw_ctx *c, const qiw_run *run, int32_t n_w, double *value_out,
                                         double *orders_out) {
    return guarded(c, [&] { return qiw_inchworm_step_noalloc_impl(c, run, n_w, value_out, orders_out); });
}
