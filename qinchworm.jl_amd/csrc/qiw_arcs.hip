// qiw_arcs.hip -- the arc walk: evaluation of open-arc programs (qiw_arcs.h) for models with
// sector blocks.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <utility>

#include "qiw_device.h"
#include "qiw_lookup.h"

namespace {

typedef float f4 __attribute__((ext_vector_type(4)));
typedef float f2 __attribute__((ext_vector_type(2)));
typedef double d2 __attribute__((ext_vector_type(2)));
template <typename T>
using ConstP = const T __attribute__((address_space(4))) *;
template <typename T>
__device__ __forceinline__ ConstP<T> as_constp(const T *p) {
    return (ConstP<T>)p;
}

constexpr uint32_t kNone = 0xFFFFFFFFu;

// A lane's vector of up to MB values and its products with a block shared by the wavefront.
//
// float: a block times the 64 lanes' vectors runs on v_mfma_f32_4x4x1_16b_f32 (16 independent
// 4x4 outer products).  Its B operand is one vector element of every lane and its result four
// rows of every lane, so a lane's vector stays where it is from product to product; the A
// operand of one (4 rows, column) slice is broadcast to all 16 products from the four lanes
// that hold it (CBSZ = 4, ABID = the slice).  A register therefore carries 16 slices of a
// block, read with one 64-lane load.
template <typename V, int MB>
struct LaneVec;

template <int MB>
struct LaneVec<float, MB> {
    static constexpr int RG = MB / 4, NV = (RG * MB + 15) / 16;
    float x[MB];
    __device__ __forceinline__ void zero() {
#pragma unroll
        for (int k = 0; k < MB; ++k) x[k] = 0.f;
    }
};

// slice s = row group * MB + column, in register s / 16 of a block, lanes 4 (s % 16) ..
template <int MB, int R, int K, int... G>
__device__ __forceinline__ void mfma_column(f4 (&acc)[MB / 4], const float *A, float y, std::integer_sequence<int, G...>) {
    ((acc[G] = __builtin_amdgcn_mfma_f32_4x4x1f32(A[(G * MB + K) / 16], y, acc[G], 4, (G * MB + K) % 16, 0)), ...);
}
// R row groups, columns below cols (uniform) in steps of KS; the columns past cols are zero
template <int MB, int R, int KS, int... K>
__device__ __forceinline__ void mfma_rows(f4 (&acc)[MB / 4], const float *A, const float *y, int cols,
                                          std::integer_sequence<int, K...>) {
    auto step = [&](auto kc) {
        constexpr int k0 = decltype(kc)::value * KS;
        if (k0 < cols) {
            mfma_column<MB, R, k0>(acc, A, y[k0], std::make_integer_sequence<int, R>{});
            if constexpr (KS > 1) mfma_column<MB, R, k0 + 1>(acc, A, y[k0 + 1], std::make_integer_sequence<int, R>{});
            if constexpr (KS > 2) {
                mfma_column<MB, R, k0 + 2>(acc, A, y[k0 + 2], std::make_integer_sequence<int, R>{});
                mfma_column<MB, R, k0 + 3>(acc, A, y[k0 + 3], std::make_integer_sequence<int, R>{});
            }
        }
    };
    (step(std::integral_constant<int, K>{}), ...);
}
template <int MB, int R = 1>
__device__ __forceinline__ void mfma_block(f4 (&acc)[MB / 4], const float *A, const float *y, int rows, int cols) {
    constexpr int KS = MB <= 8 ? 2 : 4;
    if constexpr (R < MB / 4) {
        if (rows > 4 * R) {
            mfma_block<MB, R + 1>(acc, A, y, rows, cols);
            return;
        }
    }
    mfma_rows<MB, R, KS>(acc, A, y, cols, std::make_integer_sequence<int, MB / KS>{});
}

// Joins: y (+)= w * state, the state's rows read from LDS in pairs (narrow) or fours.
template <int MB, bool FIRST>
__device__ __forceinline__ void join(float *y, float w, const float *s, int stride) {
    if (MB <= 8 && stride <= 6) {
        if (stride == 1) {
            y[0] = FIRST ? w * s[0] : fmaf(w, s[0], y[0]);
            return;
        }
#pragma unroll
        for (int k = 0; k < 6; k += 2)
            if (k < stride) {
                const f2 v = *(const f2 *)(s + k);
                y[k] = FIRST ? w * v[0] : fmaf(w, v[0], y[k]);
                y[k + 1] = FIRST ? w * v[1] : fmaf(w, v[1], y[k + 1]);
            }
        return;
    }
#pragma unroll
    for (int k = 0; k < MB; k += 4)
        if (k < stride) {
            const f4 v = *(const f4 *)(s + k);
#pragma unroll
            for (int q = 0; q < 4; ++q) y[k + q] = FIRST ? w * v[q] : fmaf(w, v[q], y[k + q]);
        }
}
template <int MB, bool FIRST>
__device__ __forceinline__ void join(double *y, double w, const double *s, int stride) {
    if (stride == 1) {
        y[0] = FIRST ? w * s[0] : fma(w, s[0], y[0]);
        return;
    }
#pragma unroll
    for (int k = 0; k < MB; k += 2)
        if (k < stride) {
            const d2 v = *(const d2 *)(s + k);
            y[k] = FIRST ? w * v[0] : fma(w, v[0], y[k]);
            y[k + 1] = FIRST ? w * v[1] : fma(w, v[1], y[k + 1]);
        }
}

template <typename V, int MB>
struct Walk;

template <int MB>
struct Walk<float, MB> {
    using L = LaneVec<float, MB>;
    static constexpr int NV = L::NV;
    f4 acc[MB / 4], out[MB / 4];
    float y[MB];
    int rk[NV];  // row | column << 8 of this lane's element of slice register v
    int lane;

    __device__ __forceinline__ void init(int lane_) {
        lane = lane_;
#pragma unroll
        for (int v = 0; v < NV; ++v) {
            const int s = 16 * v + (lane >> 2), k = s % MB, row = 4 * (s / MB) + (lane & 3);
            rk[v] = row | (k << 8);
        }
    }
    __device__ __forceinline__ void clear() {
#pragma unroll
        for (int g = 0; g < MB / 4; ++g) acc[g] = f4{0.f, 0.f, 0.f, 0.f};
    }
    __device__ __forceinline__ void clear_y() {
#pragma unroll
        for (int k = 0; k < MB; ++k) y[k] = 0.f;
    }
    // acc += O y, O in slice registers in memory
    __device__ __forceinline__ void apply_op(const float *ops, uint32_t off, int rows, int cols) {
        const int last = ((rows + 3) / 4 - 1) * MB + cols;  // slices in use
        float A[NV];
#pragma unroll
        for (int v = 0; v < NV; ++v) A[v] = 16 * v < last ? ops[off + 64 * v + lane] : 0.f;
        mfma_block<MB>(acc, A, y, rows, cols);
    }
    __device__ __forceinline__ void add_y(int rows) {
#pragma unroll
        for (int k = 0; k < MB; ++k)
            if (k < rows) acc[k / 4][k % 4] += y[k];
    }
    // out = P acc, P column-major m x m in LDS
    __device__ __forceinline__ void apply_prop(const float *P, int m) {
        const int last = ((m + 3) / 4 - 1) * MB + m;
        float A[NV];
#pragma unroll
        for (int v = 0; v < NV; ++v) {
            A[v] = 0.f;
            if (16 * v < last) {
                const int row = rk[v] & 255, k = rk[v] >> 8;
                const bool in = row < m && k < m;
                const float p = P[in ? row + k * m : 0];
                A[v] = in ? p : 0.f;
            }
        }
        float x[MB];
#pragma unroll
        for (int k = 0; k < MB; ++k) x[k] = acc[k / 4][k % 4];
#pragma unroll
        for (int g = 0; g < MB / 4; ++g) out[g] = f4{0.f, 0.f, 0.f, 0.f};
        mfma_block<MB>(out, A, x, m, m);
    }
    __device__ __forceinline__ void keep() {
#pragma unroll
        for (int g = 0; g < MB / 4; ++g) out[g] = acc[g];
    }
    __device__ __forceinline__ void store(float *d, int stride) const {
        if (MB <= 8 && stride <= 6) {
            if (stride == 1) {
                d[0] = out[0][0];
                return;
            }
#pragma unroll
            for (int k = 0; k < 6; k += 2)
                if (k < stride) *(f2 *)(d + k) = f2{out[k / 4][k % 4], out[(k + 1) / 4][(k + 1) % 4]};
            return;
        }
#pragma unroll
        for (int g = 0; g < MB / 4; ++g)
            if (4 * g < stride) *(f4 *)(d + 4 * g) = out[g];
    }
};

// double: the block's elements are wavefront-uniform multiplicands (operators through the
// scalar cache, propagators as LDS broadcasts) of ordinary multiply-adds; the matrix cores
// have no more float64 rate than the vector units.
template <int MB>
struct Walk<double, MB> {
    double acc[MB], out[MB], y[MB];
    int lane;
    __device__ __forceinline__ void init(int lane_) { lane = lane_; }
    __device__ __forceinline__ void clear() {
#pragma unroll
        for (int k = 0; k < MB; ++k) acc[k] = 0.0;
    }
    __device__ __forceinline__ void clear_y() {
#pragma unroll
        for (int k = 0; k < MB; ++k) y[k] = 0.0;
    }
    __device__ __forceinline__ void apply_op(const double *ops, uint32_t off, int rows, int cols) {
        const ConstP<double> O = as_constp(ops) + off;  // column-major, padded past the end
#pragma unroll
        for (int k = 0; k < MB; ++k)
            if (k < cols) {
#pragma unroll
                for (int i = 0; i < MB; i += 2)
                    if (i < rows) {
                        acc[i] = fma(O[k * rows + i], y[k], acc[i]);
                        acc[i + 1] = fma(i + 1 < rows ? O[k * rows + i + 1] : 0.0, y[k], acc[i + 1]);
                    }
            }
    }
    __device__ __forceinline__ void add_y(int rows) {
#pragma unroll
        for (int k = 0; k < MB; ++k)
            if (k < rows) acc[k] += y[k];
    }
    __device__ __forceinline__ void apply_prop(const double *P, int m) {
#pragma unroll
        for (int k = 0; k < MB; ++k) out[k] = 0.0;
#pragma unroll
        for (int k = 0; k < MB; ++k)
            if (k < m) {
#pragma unroll
                for (int i = 0; i < MB; i += 2)
                    if (i < m) {
                        out[i] = fma(P[k * m + i], acc[k], out[i]);
                        out[i + 1] = fma(i + 1 < m ? P[k * m + i + 1] : 0.0, acc[k], out[i + 1]);
                    }
            }
    }
    __device__ __forceinline__ void keep() {
#pragma unroll
        for (int k = 0; k < MB; ++k) out[k] = acc[k];
    }
    __device__ __forceinline__ void store(double *d, int stride) const {
        if (stride == 1) {
            d[0] = out[0];
            return;
        }
#pragma unroll
        for (int k = 0; k < MB; k += 2)
            if (k < stride) *(d2 *)(d + k) = d2{out[k], out[k + 1]};
    }
};

// i*P element e of the cell c from the float64 table.
__device__ __forceinline__ double prop_element(const double *ptab, int bt, const GridCell &c, int e) {
    const double *r0 = ptab + (int64_t)c.d * bt;
    return cell_value(c, c.d > 0 ? r0[e - bt] : 0.0, r0[e], r0[e + bt]);
}

// The arc walk.  What bounds it: the products with the operator blocks (two thirds of the
// floating-point work) and the LDS gathers that feed them; a stage's tiles are spread over
// the workgroup's wavefronts, with one barrier per stage.  Why a workgroup per sample: the
// states of one sample and column take up to 100 KB (order 4, blocks 1 4 6 4 1, float32), so
// a lane cannot own a sample; states of one sector share operator and propagator, so both
// are wavefront-uniform.  Measured against the walk of the assignment tries (one pass per
// diagram): two-orbital step orders 0:4 at N = 2^11, float32 639 -> 43.6 ms; orders 0:3 at
// N = 2^12, float64 144 -> 18.2 ms; three-orbital step orders 0:3 at N = 2^9, float32
// 399 -> 54.8 ms.
//
// One workgroup: the samples of a task one after the other; per sample the times, arc values
// and propagators go to LDS once, then every segment (initial sector) of the task is walked
// level by level.  The wavefronts share the tiles of a stage; a lane holds one column of one
// state.  The closed state's columns are multiplied by the last propagator in float64.
template <typename V, int MB, int NT>
__global__ __launch_bounds__(NT) void k_eval_arcs_t(ArcArgs aa) {
    extern __shared__ __attribute__((aligned(16))) char lds[];
    const EvalArgs &a = aa.e;
    const int tid = threadIdx.x, nt = blockDim.x;
    const int lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), nw = nt >> 6;
    const QiwTask task = a.tasks[blockIdx.x];
    const QiwGroup g = a.groups[task.group];
    const int n = g.n_nodes, bt = aa.bt;
    const double inv_h = 1.0 / a.h;
    const ConstP<uint32_t> b = as_constp(reinterpret_cast<const uint32_t *>(a.prog + g.prog_off));
    const uint32_t *words = reinterpret_cast<const uint32_t *>(a.prog + g.prog_off);
    double *tl = reinterpret_cast<double *>(lds);
    double *fin = reinterpret_cast<double *>(lds + b[4]);
    V *dv = reinterpret_cast<V *>(lds + b[5]);
    V *pl = reinterpret_cast<V *>(lds + b[6]);
    V *st = reinterpret_cast<V *>(lds + b[7]);
    const V *ops = reinterpret_cast<const V *>(aa.ops);
    const V *ops_cm = reinterpret_cast<const V *>(aa.ops_cm);
    const StepTimes T = step_times(a, g, task.tau_index);
    double *prow = a.partial + (int64_t)task.out_index * bt;
    const int seg0 = task.chunk < 0 ? 0 : task.chunk, seg1 = task.chunk < 0 ? (int)b[0] : seg0 + task.pad_;
    const bool bare = g.kind == QIW_G_BARE;
    const int skip_w = (int)b[2];
    for (int e = tid; e < bt; e += nt) prow[e] = 0.0;

    Walk<V, MB> w;
    w.init(lane);
    const int n_here = g.sampled ? min(a.spt, g.n_samples - task.first_sample) : 1;
    for (int sr = 0; sr < n_here; ++sr) {
        const int64_t sample = (int64_t)task.first_sample + sr;
        const double *u = a.ut + g.ut_off + (int64_t)task.tau_index * a.ut_row_stride + sample;
        // ---- times of the configuration positions ----
        if (tid < 16) {
            double t = 0.0;
            if (tid == n)
                t = T.tau_f;
            else if (!bare && tid == g.pos_w)
                t = T.tau_w;
            else if (tid > 1 && tid < n && g.sampled) {
                const bool after = bare || tid > g.pos_w;
                const int j = after ? n - 1 - tid : g.d_after + g.pos_w - 1 - tid;
                const double v = u[(int64_t)j * g.n_samples];
                t = after ? v * (T.tau_f - T.tau_w) + T.tau_w : v * T.tau_w;
            }
            tl[tid] = t;
        }
        // the leaves' sign (-1)^order, and (-1)^n_after for the external arc of a correlator
        // (src/diagrammatics.jl:288-303)
        const bool odd = (g.order + (g.kind == QIW_G_CORR ? g.n_after : 0)) & 1;
        const double wt = (odd ? -1.0 : 1.0) * (g.weighted ? u[(int64_t)(g.d_before + g.d_after) * g.n_samples] : 1.0);
        __syncthreads();
        // ---- arc values +-i*Delta and propagators i*P of segments 2 .. n - 1 ----
        const int na = (int)b[1];
        for (int i = tid; i < na + 1; i += nt) {
            if (i == na) {
                dv[0] = (V)0;
                dv[1] = (V)1;
                continue;
            }
            const uint32_t arc = words[b[3] + i];
            const ArcPos ap = arc_pos(tl[(arc >> 8) & 255], tl[arc & 255], inv_h, a.n_tau);
            const V v = (V)delta_value(a.dtab, (int)(arc >> 16), ap);
            dv[2 + 2 * i] = v;
            dv[3 + 2 * i] = -v;
        }
        for (int L = 2; L < n; ++L) {
            V *dst = pl + (L - 2) * bt;
            if (bare) {
                double dt = tl[L] - tl[L - 1];
                dt = dt > 0.0 ? dt : 0.0;
                for (int e = tid; e < bt; e += nt) dst[e] = aa.emask[e] ? (V)exp(-dt * aa.ediag[e]) : (V)0;
            } else {
                const GridCell c = grid_cell(tl[L], tl[L - 1], inv_h, a.n_tau);
                for (int e = tid; e < bt; e += nt) dst[e] = (V)prop_element(a.ptab, bt, c, e);
            }
        }
        __syncthreads();
        if (skip_w) {  // the node at tau_w is the identity: one propagator for its two segments
            const V *Pa = pl + (skip_w - 2) * bt, *Pb = pl + (skip_w - 1) * bt;
            V *dst = pl + (n - 2) * bt;
            for (int e = tid; e < bt; e += nt) {
                const int s = aa.sector_of[e], m = aa.dims[s], o = aa.bt_off[s], i = (e - o) % m, j = (e - o) / m;
                V v = (V)0;
                for (int q = 0; q < m; ++q) v = fma(Pb[o + i + q * m], Pa[o + q + j * m], v);
                dst[e] = v;
            }
            __syncthreads();
        }
        double mag = 0.0;
        for (int sg = seg0; sg < seg1; ++sg) {
            const ConstP<uint32_t> h = b + b[8 + sg];
            const uint32_t h0 = h[0];
            const int s0 = (int)(h0 & 255), m0 = (int)((h0 >> 8) & 255), lg = (int)(h0 >> 16), cg = 1 << lg;
            const int n_stages = (int)h[1], m1 = (int)(h[2] & 255), str1 = (int)(h[2] >> 8);
            const uint32_t rblk = h[3], rprop = h[4];
            const int col = lane & (cg - 1), sl = lane >> lg;
            for (int c0 = 0; c0 < m0; c0 += cg) {
                if (wave == 0) {  // position 1: unit columns, or columns of the operator B
                    w.clear();
                    w.clear_y();
                    const int c = c0 + col;
#pragma unroll
                    for (int k = 0; k < MB; ++k) {
                        V v = (V)0;
                        if (k < m1 && c < m0) v = rblk == kNone ? (k == c ? (V)1 : (V)0) : ops_cm[rblk + c * m1 + k];
                        w.y[k] = v;
                    }
                    w.add_y(MB);
                    if (rprop != kNone)
                        w.apply_prop(pl + rprop, m1);
                    else
                        w.keep();
                    if (lane < cg) w.store(st + h[5] + lane * str1, str1);
                }
                __syncthreads();
                for (int s = 0; s < n_stages; ++s) {
                    const int n_tiles = (int)h[8 + 2 * s];
                    const ConstP<uint32_t> tiles = b + h[8 + 2 * s + 1];
                    for (int ti = wave; ti < n_tiles; ti += nw) {
                        const uint32_t t0 = tiles[4 * ti], t1 = tiles[4 * ti + 1], t2 = tiles[4 * ti + 2];
                        const ConstP<uint32_t> op = b + tiles[4 * ti + 3];
                        const int n_ops = (int)(t0 & 255), rows = (int)((t0 >> 8) & 255), ns = (int)((t0 >> 16) & 255);
                        const int str = (int)(t0 >> 24);
                        const int sq = sl < ns ? sl : ns - 1;
                        w.clear();
                        w.clear_y();
                        for (int oi = 0; oi < n_ops; ++oi) {
                            const uint32_t blk = op[4 * oi], o1 = op[4 * oi + 1], wo = op[4 * oi + 2];
                            const int ms = (int)(o1 & 255), ss = (int)((o1 >> 8) & 255), ne = (int)(o1 >> 16);
                            const uint32_t *jw = words + wo + sq;
                            uint32_t q = jw[0];
                            for (int e = 0; e < ne; ++e) {
                                const uint32_t qn = e + 1 < ne ? jw[(e + 1) * ns] : 0u;
                                const V dvv = dv[q >> 20];
                                const V *src = st + (q & 0xFFFFFu) + col * ss;
                                if (e == 0)
                                    join<MB, true>(w.y, dvv, src, ss);
                                else
                                    join<MB, false>(w.y, dvv, src, ss);
                                q = qn;
                            }
                            if (blk == kNone)
                                w.add_y(ms);
                            else
                                w.apply_op(ops, blk, rows, ms);
                        }
                        if (t2 != kNone)
                            w.apply_prop(pl + t2, rows);
                        else
                            w.keep();
                        if (lane < ns * cg) w.store(st + t1 + lane * str, str);
                    }
                    __syncthreads();
                }
                // the closed state's columns, its parts added in float64
                const int np = (int)h[6];
                const ConstP<uint32_t> parts = b + h[7];
                const int stf = n_stages == 0 ? str1 : aa.stride[s0];
                for (int i = tid; i < m0 * cg; i += nt) {
                    const int c = i / m0, r = i - c * m0;
                    if (c0 + c >= m0) continue;
                    double v = 0.0;
                    for (int p = 0; p < np; ++p) v += (double)st[parts[p] + c * stf + r];
                    fin[(c0 + c) * m0 + r] = v;
                }
                __syncthreads();
            }
            // out[s0] += weight * iP_n[s0] * closed state, in float64
            const int o = aa.bt_off[s0];
            const GridCell cn = grid_cell(tl[n], tl[n - 1], inv_h, a.n_tau);
            double dtn = tl[n] - tl[n - 1];
            dtn = dtn > 0.0 ? dtn : 0.0;
            for (int i = tid; i < m0 * m0; i += nt) {
                const int c = i / m0, r = i - c * m0;
                double v = 0.0;
                if (bare) {
                    v = exp(-dtn * aa.ediag[o + r * (m0 + 1)]) * fin[i];
                } else {
                    for (int q = 0; q < m0; ++q)
                        v = fma(prop_element(a.ptab, bt, cn, o + r + q * m0), fin[c * m0 + q], v);
                }
                mag += fabs(v);
                prow[o + i] += wt * v;
            }
            __syncthreads();
        }
        if (a.per_sample) {
#pragma unroll
            for (int d = 32; d > 0; d >>= 1) mag += __shfl_xor(mag, d, 64);
            if (lane == 0) tl[wave] = mag;
            __syncthreads();
            if (tid == 0) {
                double s = 0.0;
                for (int i = 0; i < nw; ++i) s += tl[i];
                a.per_sample[g.ps_off + sample] = s;
            }
            __syncthreads();
        }
    }
}

template <typename V, int MB, int NT>
hipError_t launch(hipStream_t st, const ArcArgs &a, int n_tasks, int waves, size_t lds) {
    if (waves * 64 > NT || waves < 1) return hipErrorInvalidValue;
    hipLaunchKernelGGL((k_eval_arcs_t<V, MB, NT>), dim3(n_tasks), dim3(64 * waves), lds, st, a);
    return hipGetLastError();
}

}  // namespace

// Vector length of the instantiation for blocks up to mb, and the most wavefronts a
// workgroup of it can have (its registers).
int qiw_arc_rows(int mb) { return mb <= 8 ? 8 : mb <= 20 ? 20 : 32; }
int qiw_arc_waves(int mb, int fp32) { return mb <= 8 ? 16 : (mb <= 20 && fp32) ? 16 : 8; }

hipError_t qiw_launch_eval_arcs(hipStream_t st, const ArcArgs &a, int n_tasks, int mb, int fp32, int waves, size_t lds) {
    if (n_tasks < 1 || mb > 32 || a.e.n_tau < 2) return hipErrorInvalidValue;
    if (mb <= 8) return fp32 ? launch<float, 8, 1024>(st, a, n_tasks, waves, lds) : launch<double, 8, 1024>(st, a, n_tasks, waves, lds);
    if (mb <= 20) return fp32 ? launch<float, 20, 1024>(st, a, n_tasks, waves, lds) : launch<double, 20, 512>(st, a, n_tasks, waves, lds);
    return fp32 ? launch<float, 32, 512>(st, a, n_tasks, waves, lds) : launch<double, 32, 512>(st, a, n_tasks, waves, lds);
}
