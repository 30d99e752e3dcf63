// qiw_arcs.hip -- the arc walk: evaluation of open-arc programs (qiw_arcs.h) for models with
// sector blocks.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <utility>

#include "qiw_arcs.h"
#include "qiw_device.h"
#include "qiw_dpp.h"
#include "qiw_lookup.h"

using namespace qiwi;

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

constexpr uint32_t kNone = ARC_NONE;
__device__ __forceinline__ uint32_t rlane(uint32_t v, int l) { return __builtin_amdgcn_readlane(v, l); }
// the word at a byte offset of a uniform base (one load with a 32-bit vector offset)
__device__ __forceinline__ uint32_t word_at(const uint32_t *base, uint32_t byte) {
    return *reinterpret_cast<const uint32_t *>(reinterpret_cast<const char *>(base) + byte);
}
// source state (column offset coff) and arc value of a join word
template <typename V>
__device__ __forceinline__ const V *state_at(const char *lds, uint32_t q, uint32_t coff) {
    return reinterpret_cast<const V *>(lds + ((q & 0xFFFFu) * 4u + coff));
}
__device__ __forceinline__ double value_at(const char *lds, uint32_t q) {  // bits 16-19 are clear
    return *reinterpret_cast<const double *>(lds + kArcValuesAt + (q >> 17));
}

// A lane's vector of up to MB values and its products with a block shared by the wavefront.
// The walk of a slot branches once on the stride C of its source and once on the stride R of
// its states; all below is straight code for them (branches on every row and column took two
// thirds of the time).
//
// float: a block times the 64 lanes' vectors runs on v_mfma_f32_4x4x1_16b_f32 (16 independent
// 4x4 outer products).  Its B operand is one vector element of every lane and its result four
// rows of every lane, so a lane's vector stays where it is from product to product; the A
// operand of one (4 rows, column) slice is broadcast to all 16 products from the four lanes
// that hold it (CBSZ = 4, ABID = the slice).  A register therefore carries 16 slices of a
// block, read with one 64-lane load.  Only the products are in float32: the sums over joins and
// over the operators of a tile are in float64 (as the sums over diagrams of the vector and
// matrix-core walks are) and rounded once, where they enter a product, so a result is no less
// accurate than the float64 sum of float32 chains.  What they cost against sums in float32: 21.1 ->
// 23.4 ms in the two-orbital step of orders 0:4 at N = 2^11, 31.1 -> 39.7 in the three-orbital one of
// orders 0:3 at N = 2^9 (conversions and float64 additions issue at half the rate of float32
// ones, and the sums take registers).  Every slot ends with its product, so that no sum of
// joins is kept from slot to slot (27.7 and 42.7 ms with it kept).
//
// double: multiply-adds whose block element is broadcast from its lane by the instruction
// itself (v_fmac_f64 with DPP row_newbcast; every row of 16 lanes holds the same 16
// elements), so a register pair carries 16 elements.  The float64 matrix instructions have
// no more rate than the vector units.
template <typename V, int MB>
struct Walk;

// y += w s, s a state of C elements in LDS (a stride of arc_stride: 16-byte aligned from 4
// floats on, but for 6).  The sums are in float64 for both types of state (FIRST: y = w s).
template <int C, bool FIRST>
__device__ __forceinline__ void join(double *y, double w, const float *s) {
    auto add = [&](int k, float v) { y[k] = FIRST ? w * (double)v : fma(w, (double)v, y[k]); };
    if constexpr (C == 1) {
        add(0, s[0]);
    } else if constexpr (C % 4 == 0) {
#pragma unroll
        for (int k = 0; k < C; k += 4) {
            const f4 v = *(const f4 *)(s + k);
#pragma unroll
            for (int q = 0; q < 4; ++q) add(k + q, v[q]);
        }
    } else {
#pragma unroll
        for (int k = 0; k < C; k += 2) {
            const f2 v = *(const f2 *)(s + k);
            add(k, v[0]);
            add(k + 1, v[1]);
        }
    }
}
template <int C>
__device__ __forceinline__ void join(double *y, double w, const double *s) {
    if constexpr (C == 1) {
        y[0] = fma(w, s[0], y[0]);
    } else {
#pragma unroll
        for (int k = 0; k < C; k += 2) {
            const d2 v = *(const d2 *)(s + k);
            y[k] = fma(w, v[0], y[k]);
            y[k + 1] = fma(w, v[1], y[k + 1]);
        }
    }
}

template <int C>
__device__ __forceinline__ void store_sum(double *d, const double *v) {
    if constexpr (C == 1) {
        d[0] = v[0];
    } else {
#pragma unroll
        for (int k = 0; k < C; k += 2) *(d2 *)(d + k) = d2{v[k], v[k + 1]};
    }
}

// slice s = row group * MB + column, in register s / 16 of a block, lanes 4 (s % 16) ..
template <int MB, int G, int K, int... R>
__device__ __forceinline__ void mfma_column(f4 (&acc)[MB / 4], const float *A, float y, std::integer_sequence<int, R...>) {
    ((acc[R] = __builtin_amdgcn_mfma_f32_4x4x1f32(A[(R * MB + K) / 16], y, acc[R], 4, (R * MB + K) % 16, 0)), ...);
}
// G row groups, the columns K
template <int MB, int G, int... K>
__device__ __forceinline__ void mfma_block(f4 (&acc)[MB / 4], const float *A, const float *y,
                                           std::integer_sequence<int, K...>) {
    (mfma_column<MB, G, K>(acc, A, y[K], std::make_integer_sequence<int, G>{}), ...);
}

template <int MB>
struct Walk<float, MB> {
    static constexpr int NV = (MB / 4 * MB + 15) / 16;  // slice registers of a block
    static constexpr int SL = arc_slots(MB);
    double sum[MB];                 // of the products of a tile
    float A[SL][NV], next[SL][NV];  // blocks of the packet and of the next one
    int rk[NV];                     // row | column << 8 of this lane's element of slice register v
    int lane;

    __device__ __forceinline__ void init(int lane_) {
        lane = lane_;
#pragma unroll
        for (int v = 0; v < NV; ++v) {
            const int s = 16 * v + (lane >> 2), k = s % MB, row = 4 * (s / MB) + (lane & 3);
            rk[v] = row | (k << 8);
#pragma unroll
            for (int o = 0; o < SL; ++o) A[o][v] = next[o][v] = 0.f;
        }
        clear();
    }
    __device__ __forceinline__ void clear() {
#pragma unroll
        for (int k = 0; k < MB; ++k) sum[k] = 0.0;
    }
    static __device__ __forceinline__ void zero(f4 (&acc)[MB / 4]) {
#pragma unroll
        for (int g = 0; g < MB / 4; ++g) acc[g] = f4{0.f, 0.f, 0.f, 0.f};
    }
    // blocks in slice registers in memory; str: rows that are computed, ss: columns
    template <int O>
    __device__ __forceinline__ void fetch_op(const float *ops, uint32_t off, int str, int ss) {
        const int last = ((str + 3) / 4 - 1) * MB + ss;  // slices in use
#pragma unroll
        for (int v = 0; v < NV; ++v)
            if (NV == 1 || 16 * v < last) next[O][v] = ops[off + 64 * v + lane];
    }
    __device__ __forceinline__ void rotate() {
#pragma unroll
        for (int o = 0; o < SL; ++o)
#pragma unroll
            for (int v = 0; v < NV; ++v) A[o][v] = next[o][v];
    }
    // sum += O y, the product in float32
    template <int O, int C>
    __device__ __forceinline__ void product(const double (&y)[C], int str) {
        float x[C];
#pragma unroll
        for (int k = 0; k < C; ++k) x[k] = (float)y[k];
        rows<C, 1>(A[O], x, str);
    }
    template <int C, int G>
    __device__ __forceinline__ void rows(const float *a, const float (&x)[C], int str) {
        if constexpr (G < MB / 4) {
            if (str > 4 * G) {
                rows<C, G + 1>(a, x, str);
                return;
            }
        }
        f4 acc[MB / 4];
        zero(acc);
        mfma_block<MB, G>(acc, a, x, std::make_integer_sequence<int, C>{});
        // (downwards, so that the branches of all G end with the same addresses: upwards the
        // compiler joins their last stores over a pointer, and the array goes to memory)
#pragma unroll
        for (int k = 4 * G - 1; k >= 0; --k) sum[k] += (double)acc[k / 4][k % 4];
    }
    // d = P sum, P column-major m x m in LDS, C its padded size; sum = 0
    template <int C>
    __device__ __forceinline__ void finish(const float *pl, int m, float *d, bool lanes) {
        f4 acc[MB / 4];
        propagate<C>(acc, pl, m);
        if (lanes) store<C>(acc, d);
        clear();
    }
    // d = sum; sum = 0
    template <int C>
    __device__ __forceinline__ void close(double *d, bool lanes) {
        if (lanes) store_sum<C>(d, sum);
        clear();
    }
    template <int C>
    __device__ __forceinline__ void propagate(f4 (&acc)[MB / 4], const float *pl, int m) const {
        constexpr int last = ((C + 3) / 4 - 1) * MB + C;
        float P[NV], x[C];
#pragma unroll
        for (int v = 0; v < NV; ++v)
            if (16 * v < last) {
                const int row = rk[v] & 255, k = rk[v] >> 8;
                const bool in = row < m && k < m;
                const float p = pl[in ? row + k * m : 0];
                P[v] = in ? p : 0.f;
            }
#pragma unroll
        for (int k = 0; k < C; ++k) x[k] = (float)sum[k];
        zero(acc);
        mfma_block<MB, (C + 3) / 4>(acc, P, x, std::make_integer_sequence<int, C>{});
    }
    template <int C>
    static __device__ __forceinline__ void store(const f4 (&acc)[MB / 4], float *d) {
        if constexpr (C == 1) {
            d[0] = acc[0][0];
        } else if constexpr (C % 4 == 0) {
#pragma unroll
            for (int g = 0; g < C / 4; ++g) *(f4 *)(d + 4 * g) = acc[g];
        } else {
#pragma unroll
            for (int k = 0; k < C; k += 2) *(f2 *)(d + k) = f2{acc[k / 4][k % 4], acc[(k + 1) / 4][(k + 1) % 4]};
        }
    }
};

// R rows of one column, element E of the chunk onwards
template <int E, int R>
__device__ __forceinline__ void fmac_rows(double *c, const double *a, double y) {
    fmac_bcast<E % 16, R>(c, a[E / 16], y);
    if constexpr (R > 4) fmac_rows<E + 4, R - 4>(c + 4, a, y);
}
// rows I .. I + R - 1 of the chunk's columns K
template <int MB, int I, int R, int... K>
__device__ __forceinline__ void fmac_block(double *acc, const double *a, const double *y, std::integer_sequence<int, K...>) {
    (fmac_rows<K * MB + I, R>(acc + I, a, y[K]), ...);
}

template <int MB>
struct Walk<double, MB> {
    static constexpr int CH = MB <= 8 ? 8 : 4;  // columns of a chunk
    static constexpr int NV = CH * MB / 16;     // register pairs of a chunk
    static constexpr int SL = arc_slots(MB);
    double acc[MB], y[MB], A[SL][NV], next[SL][NV];  // first chunks of the packet and of the next one
    int rk[NV];  // row | column of the chunk << 8 of this lane's element of register pair v
    int lane;
    __device__ __forceinline__ void init(int lane_) {
        lane = lane_;
#pragma unroll
        for (int v = 0; v < NV; ++v) {
            const int e = 16 * v + (lane & 15);
            rk[v] = (e % MB) | ((e / MB) << 8);
#pragma unroll
            for (int o = 0; o < SL; ++o) A[o][v] = next[o][v] = 0.0;
        }
#pragma unroll
        for (int k = 0; k < MB; ++k) y[k] = 0.0;
        clear();
    }
    __device__ __forceinline__ void clear() {
#pragma unroll
        for (int k = 0; k < MB; ++k) acc[k] = 0.0;
    }
    // operator blocks: MB x MB column-major, zeros past the block; columns c0 .. of it into a
    __device__ __forceinline__ void read_op(double (&a)[NV], const double *ops, uint32_t off, int c0, int cols) const {
#pragma unroll
        for (int v = 0; v < NV; ++v)
            if (c0 + 16 * v / MB < cols) a[v] = ops[off + c0 * MB + 16 * v + (lane & 15)];
    }
    template <int O>
    __device__ __forceinline__ void fetch_op(const double *ops, uint32_t off, int, int ss) {
        read_op(next[O], ops, off, 0, ss);
    }
    __device__ __forceinline__ void rotate() {
#pragma unroll
        for (int o = 0; o < SL; ++o)
#pragma unroll
            for (int v = 0; v < NV; ++v) A[o][v] = next[o][v];
    }
    // acc += (C columns of the chunk in a) x
    template <int C, int R>
    __device__ __forceinline__ void rows(const double (&a)[NV], const double *x, int str) {
        constexpr auto columns = std::make_integer_sequence<int, C>{};
        if constexpr (MB <= 8) {
            if (str == 4)
                fmac_block<MB, 0, 4>(acc, a, x, columns);
            else if (str == 6)
                fmac_block<MB, 0, 6>(acc, a, x, columns);
            else if (str == 1)
                fmac_block<MB, 0, 1>(acc, a, x, columns);
            else if (str == 2)
                fmac_block<MB, 0, 2>(acc, a, x, columns);
            else
                fmac_block<MB, 0, 8>(acc, a, x, columns);
        } else if constexpr (R < MB) {  // rows in fours
            if (R < str) {
                fmac_block<MB, R, 4>(acc, a, x, columns);
                rows<C, R + 4>(a, x, str);
            }
        }
    }
    template <int O, int C, int K = 0>
    __device__ __forceinline__ void product(const double *ops, uint32_t off, int str) {
        if constexpr (K < C) {
            if constexpr (K > 0) read_op(A[O], ops, off, K, C);
            rows<(C < CH ? C : CH), 0>(A[O], y + K, str);
            product<O, C, K + CH>(ops, off, str);
        } else {
#pragma unroll
            for (int k = 0; k < C; ++k) y[k] = 0.0;
        }
    }
    template <int C>
    __device__ __forceinline__ void finish(const double *pl, int m, double *d, bool lanes) {
        propagate<C>(pl, m);
        close<C>(d, lanes);
    }
    template <int C>
    __device__ __forceinline__ void close(double *d, bool lanes) {
        if (lanes) store_sum<C>(d, acc);
        clear();
    }
    template <int C>
    __device__ __forceinline__ void propagate(const double *pl, int m) {
        double x[C];
#pragma unroll
        for (int k = 0; k < C; ++k) x[k] = acc[k];
        clear();
        prop_chunks<C, 0>(pl, x, m);
    }
    template <int C, int K>
    __device__ __forceinline__ void prop_chunks(const double *pl, const double *x, int m) {
        if constexpr (K < C) {
            double P[NV];
#pragma unroll
            for (int v = 0; v < NV; ++v)
                if (K + 16 * v / MB < C) {
                    const int row = rk[v] & 255, k = K + (rk[v] >> 8);
                    const bool in = row < m && k < m;
                    const double p = pl[in ? row + k * m : 0];
                    P[v] = in ? p : 0.0;
                }
            if constexpr (MB <= 8)
                fmac_block<MB, 0, C>(acc, P, x, std::make_integer_sequence<int, C>{});
            else
                rows<CH, 0>(P, x + K, C);
            prop_chunks<C, K + CH>(pl, x, m);
        }
    }
};

// Join words of a packet: first and second steps of its slots.
template <int SL>
struct Joins {
    uint32_t first[SL], second[SL];
    // byte: of the lane's first word; step: from one block of joins to the next
    __device__ __forceinline__ void load(const uint32_t *words, uint32_t byte, uint32_t step, bool two) {
#pragma unroll
        for (int o = 0; o < SL; ++o) first[o] = word_at(words, byte + 4u * o);
        if (two) {
#pragma unroll
            for (int o = 0; o < SL; ++o) second[o] = word_at(words, byte + step + 4u * o);
        }
    }
};

// The blocks of the packet whose records are in hd, into next (one register: read without
// asking whether the slot has a block, the first one then).
template <typename W, typename V, int O>
__device__ __forceinline__ void fetch_ops(W &w, const V *ops, uint32_t hd) {
    if constexpr (O < W::SL) {
        const uint32_t shape = rlane(hd, 8 * O + 1);
        if (W::NV == 1 || (rlane(hd, 8 * O) & ARC_TIMES))
            w.template fetch_op<O>(ops, rlane(hd, 8 * O + 2), (int)((shape >> 8) & 255), (int)(shape >> 16));
        fetch_ops<W, V, O + 1>(w, ops, hd);
    }
}

// What a slot needs besides its record.
template <typename V>
struct SlotArgs {
    const char *lds;
    V *st;
    double *closed;  // the closed state by the offsets of the states
    const V *pl, *ops;
    int col, lg;
};

// Joins and product of slot O, sources of stride C.
template <typename V, int MB, int O, int C>
__device__ __forceinline__ void slot_joins(Walk<V, MB> &w, const Joins<Walk<V, MB>::SL> &jw, const SlotArgs<V> &x,
                                           uint32_t fl, uint32_t blk, int str) {
    const uint32_t coff = (uint32_t)(x.col * C) * (uint32_t)sizeof(V), q = jw.first[O], r = jw.second[O];
    if constexpr (sizeof(V) == 4) {  // every slot ends with its product
        double y[C];
        join<C, true>(y, value_at(x.lds, q), state_at<V>(x.lds, q, coff));
        if (fl & ARC_SECOND) join<C, false>(y, value_at(x.lds, r), state_at<V>(x.lds, r, coff));
        w.template product<O, C>(y, str);
    } else {
        join<C>(w.y, value_at(x.lds, q), state_at<V>(x.lds, q, coff));
        if (fl & ARC_SECOND) join<C>(w.y, value_at(x.lds, r), state_at<V>(x.lds, r, coff));
        if (fl & ARC_TIMES) w.template product<O, C>(x.ops, blk, str);
    }
}
// The end of a tile of stride C: propagator and store.
template <typename V, int MB, int C>
__device__ __forceinline__ void slot_store(Walk<V, MB> &w, const SlotArgs<V> &x, uint32_t prop, int rows, uint32_t to,
                                           int lanes) {
    const int lane = threadIdx.x & 63;
    if (prop != kNone)
        w.template finish<C>(x.pl + prop, rows, x.st + to + lane * C, lane < lanes);
    else
        w.template close<C>(x.closed + to + lane * C, lane < lanes);
}

// Slots O .. of a packet; false after the segment's last one.
template <typename V, int MB, int O>
__device__ __forceinline__ bool run_slots(Walk<V, MB> &w, const Joins<Walk<V, MB>::SL> &jw, uint32_t hd,
                                          const SlotArgs<V> &x) {
    if constexpr (O < Walk<V, MB>::SL) {
        const uint32_t fl = rlane(hd, 8 * O), shape = rlane(hd, 8 * O + 1), blk = rlane(hd, 8 * O + 2);
        const int str = (int)((shape >> 8) & 255), ss = (int)(shape >> 16);
        if (fl & (ARC_BARRIER | ARC_END | ARC_IDLE)) {
            if (fl & ARC_BARRIER) __syncthreads();
            if (fl & ARC_END) return false;
        }
#define QIW_STRIDE(S, CALL)                     \
  {                                             \
    if constexpr (MB <= 8) {                    \
        if (S == 4) CALL(4);                    \
        else if (S == 6) CALL(6);               \
        else if (S == 1) CALL(1);               \
        else if (S == 2) CALL(2);               \
        else CALL(8);                           \
    } else if constexpr (MB <= 20) {            \
        if (S == 20) CALL(20);                  \
        else if (S == 16) CALL(16);             \
        else if (S == 8) CALL(8);               \
        else if (S == 4) CALL(4);               \
        else CALL(12);                          \
    } else {                                    \
        if (S <= 8) {                           \
            if (S == 4) CALL(4);                \
            else CALL(8);                       \
        } else if (S <= 16) {                   \
            if (S == 12) CALL(12);              \
            else CALL(16);                      \
        } else if (S <= 24) {                   \
            if (S == 20) CALL(20);              \
            else CALL(24);                      \
        } else if (S == 28) CALL(28);           \
        else CALL(32);                          \
    }                                           \
  }
#define QIW_JOINS(C) slot_joins<V, MB, O, C>(w, jw, x, fl, blk, str)
        if (!(fl & ARC_IDLE)) QIW_STRIDE(ss, QIW_JOINS)
        if (fl & ARC_STORE) {
            const uint32_t to = rlane(hd, 8 * O + 3), prop = rlane(hd, 8 * O + 4);
            const int rows = (int)(shape & 255), lanes = (int)(rlane(hd, 8 * O + 5) << x.lg);
#define QIW_STORE(C) slot_store<V, MB, C>(w, x, prop, rows, to, lanes)
            QIW_STRIDE(str, QIW_STORE)
        }
#undef QIW_JOINS
#undef QIW_STORE
#undef QIW_STRIDE
        return run_slots<V, MB, O + 1>(w, jw, hd, x);
    }
    return true;
}

// Grid cell of a segment in LDS.
struct ArcCell {
    double wp, wm;
    int d, pad_;
};
static_assert(kArcCellsAt + 16 * sizeof(ArcCell) <= kArcValuesAt, "LDS of the cells");

// i*P element e of the cell c from the float64 table.
__device__ __forceinline__ double prop_element(const double *ptab, int bt, const GridCell &c, int e) {
    const double *r0 = ptab + (int64_t)c.d * bt;
    return cell_value(c, c.d > 0 ? r0[e - bt] : 0.0, r0[e], r0[e + bt]);
}

// The arc walk.  What bounds it: issue of the products (vector units 50 % busy, matrix cores
// 30 to 40 % for float32), the LDS gathers that feed them (20 %) and the stages' barriers.  Why
// a workgroup per sample: the states of one sample and column take up to 100 KB (order 4,
// blocks 1 4 6 4 1, float32), so a lane cannot own a sample; states of one sector share
// operator and propagator, so both are wavefront-uniform.  Measured against the walk of the
// assignment tries (one pass per diagram): two-orbital solve on 50 points, orders 0:2 at
// N = 2^10, float64 451 -> 15.4 ms; two-orbital step, orders 0:4 at N = 2^11, float32 643 -> 23.4
// ms; orders 0:3 at N = 2^12, float64 144 -> 8.8 ms; three-orbital step, orders 0:3 at N =
// 2^9, float32 399 -> 39.7 ms; orders 0:2 at N = 2^8, float64 63.8 -> 3.2 ms.  Of these the
// first form of the walk reached 29.9, 43.6, 18.2, 54.8 and 28.8 ms: what it lost were branches
// on every row and column (one in five instructions), operator blocks and joins read when they
// were wanted (a load's whole latency each), stages waiting for one wavefront with a tile of
// many operators, for float64 operator elements through the scalar cache, the last propagator's
// gathers in every segment, and the workgroup shapes.
//
// One workgroup: the samples of a task one after the other; per sample the times, arc values
// and propagators go to LDS once, then every segment (initial sector) of the task is walked
// level by level.  The wavefronts share the tiles of a stage; a lane holds one column of one
// state.  The closed states of all segments are multiplied by the last propagator in float64
// at the end (segment by segment its gathers and the sums in memory were waited for each time).
// Wavefronts per SIMD: float64 at MB = 8 takes three (168 registers, what spills is outside the
// slots; two-orbital step 8.7 ms, 11.0 with two and 11.1 with four), float32 at MB = 20 two
// (three-orbital step 39.7 ms, 41.7 with three).
template <typename V, int MB, int NT>
__global__ __launch_bounds__(NT, MB == 8 && sizeof(V) == 8 ? 3 : 2) void k_eval_arcs_t(ArcArgs aa) {
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
    double *dv = reinterpret_cast<double *>(lds + kArcValuesAt);
    V *pl = reinterpret_cast<V *>(lds + b[6]);
    V *st = reinterpret_cast<V *>(lds + b[7]);
    const V *ops = reinterpret_cast<const V *>(aa.ops);
    const V *ops_cm = reinterpret_cast<const V *>(aa.ops_cm);
    const StepTimes T = step_times(a, g, task.tau_index);
    double *prow = a.partial + (int64_t)task.out_index * bt;
    const int seg0 = task.chunk < 0 ? 0 : task.chunk, seg1 = task.chunk < 0 ? (int)b[0] : seg0 + task.pad_;
    const bool bare = g.kind == QIW_G_BARE;
    const int skip_w = (int)b[2];
    ArcCell *cells = reinterpret_cast<ArcCell *>(lds + kArcCellsAt);

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
        for (int e = tid; e < bt; e += nt) fin[e] = 0.0;
        // the leaves' sign (-1)^order, and (-1)^n_after for the external arc of a correlator
        // (src/diagrammatics.jl:288-303)
        const bool odd = (g.order + (g.kind == QIW_G_CORR ? g.n_after : 0)) & 1;
        const double wt = (odd ? -1.0 : 1.0) * (g.weighted ? u[(int64_t)(g.d_before + g.d_after) * g.n_samples] : 1.0);
        __syncthreads();
        // ---- arc values +-i*Delta, and the grid cells of the segments ----
        const int na = (int)b[1];
        for (int i = tid; i < na + 1; i += nt) {
            if (i == na) {
                dv[0] = 0.0;
                dv[1] = 1.0;
                continue;
            }
            const uint32_t arc = words[b[3] + i];
            const ArcPos ap = arc_pos(tl[(arc >> 8) & 255], tl[arc & 255], inv_h, a.n_tau);
            const double v = delta_value(a.dtab, (int)(arc >> 16), ap);
            dv[2 + 2 * i] = v;
            dv[3 + 2 * i] = -v;
        }
        if (tid >= nt - 16 && !bare) {  // (the last threads: the first ones have the arcs)
            const int L = 2 + tid - (nt - 16);
            if (L <= n) {
                const GridCell c = grid_cell(tl[L], tl[L - 1], inv_h, a.n_tau);
                cells[L - 2] = ArcCell{c.wp, c.wm, c.d, 0};
            }
        }
        __syncthreads();
        // ---- propagators i*P of segments 2 .. n - 1 ----
        for (int L = 2; L < n; ++L) {
            V *p = pl + (L - 2) * bt;
            if (bare) {
                double dt = tl[L] - tl[L - 1];
                dt = dt > 0.0 ? dt : 0.0;
                for (int e = tid; e < bt; e += nt) p[e] = aa.emask[e] ? (V)exp(-dt * aa.ediag[e]) : (V)0;
            } else {
                const GridCell c{cells[L - 2].d, cells[L - 2].wp, cells[L - 2].wm};
                for (int e = tid; e < bt; e += nt) p[e] = (V)prop_element(a.ptab, bt, c, e);
            }
        }
        __syncthreads();
        if (skip_w) {  // the node at tau_w is the identity: one propagator for its two segments
            const V *Pa = pl + (skip_w - 2) * bt, *Pb = pl + (skip_w - 1) * bt;
            V *dst = pl + (n - 2) * bt;
            for (int e = tid; e < bt; e += nt) {
                const uint32_t at = aa.element[e];
                const int o = (int)(at & 0xFFFFu), i = (int)((at >> 16) & 31u), j = (int)((at >> 21) & 31u), m = 1 + (int)(at >> 26);
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
            const int m1 = (int)(h[1] & 255), str1 = (int)(h[1] >> 8);
            const uint32_t rblk = h[2], rprop = h[3];
            const int o = aa.bt_off[s0];
            double *closed = reinterpret_cast<double *>(st + h[7]) - h[7];
            constexpr int SL = Walk<V, MB>::SL;
            const int col = lane & (cg - 1);
            const uint32_t jstep = 4u * (SL * (64u >> lg));  // bytes of a block of joins
            for (int c0 = 0; c0 < m0; c0 += cg) {
                // the first packet and the second one's records, read ahead of the root
                uint32_t rec = 4u * h[8 + 2 * wave] + 4u * lane;  // byte offsets in the program
                uint32_t jat = 4u * h[9 + 2 * wave] + 4u * (SL * ((uint32_t)lane >> lg));
                uint32_t hd = word_at(words, rec), hn = word_at(words, rec + 32u * SL);
                const uint32_t part = lane < (int)h[5] ? words[h[6] + lane] : 0u;
                Joins<SL> jw, jn;
                bool two = rlane(hd, 6) != 0;
                jw.load(words, jat, jstep, two);
                Walk<V, MB> w;
                w.init(lane);
                fetch_ops<Walk<V, MB>, V, 0>(w, ops, hd);
                w.rotate();
                const SlotArgs<V> sa{lds, st, closed, pl, ops, col, lg};
                // position 1: unit columns, or columns of the operator B, times the propagator
                // that follows
                for (int i = tid; i < cg * str1; i += nt) {
                    const int cc = i / str1, k = i - cc * str1, c = c0 + cc;
                    V v = (V)0;
                    if (k < m1 && c < m0) {
                        if (rblk == kNone)
                            v = rprop == kNone ? (k == c ? (V)1 : (V)0) : pl[rprop + k + c * m1];
                        else if (rprop == kNone)
                            v = ops_cm[rblk + c * m1 + k];
                        else
                            for (int j = 0; j < m1; ++j) v = fma(pl[rprop + k + j * m1], ops_cm[rblk + c * m1 + j], v);
                    }
                    if (rprop == kNone)
                        closed[h[4] + i] = (double)v;
                    else
                        st[h[4] + i] = v;
                }
                for (;;) {
                    // the next packet, and the records of the one after it
                    rec += 32u * SL;
                    jat += two ? 2u * jstep : jstep;
                    two = rlane(hn, 6) != 0;
                    const uint32_t h2 = word_at(words, rec + 32u * SL);
                    jn.load(words, jat, jstep, two);
                    fetch_ops<Walk<V, MB>, V, 0>(w, ops, hn);
                    if (!run_slots<V, MB, 0>(w, jw, hd, sa)) break;
                    hd = hn;
                    hn = h2;
                    jw = jn;
                    w.rotate();
                }
                // the closed state's columns, its parts (one per lane) added in float64; no other
                // state lies where the closed ones do, so the next pass may start
                const int np = (int)h[5], stf = aa.stride[s0];
                for (int i = wave; i < m0 * cg; i += nw) {
                    const int c = i / m0, r = i - c * m0;
                    if (c0 + c >= m0) break;
                    double v = lane < np ? closed[part + c * stf + r] : 0.0;
                    for (int p = lane + 64; p < np; p += 64) v += closed[words[h[6] + p] + c * stf + r];
#pragma unroll
                    for (int d = 32; d > 0; d >>= 1) v += __shfl_xor(v, d, 64);
                    if (lane == 0) fin[o + (c0 + c) * m0 + r] += v;
                }
            }
            __syncthreads();  // the next segment's states may lie where these closed ones do
        }
        // out[s0] = weight * iP_n[s0] * closed state, in float64; iP_n where the states were
        double *last = reinterpret_cast<double *>(st);
        if (!bare) {
            const GridCell c{cells[n - 2].d, cells[n - 2].wp, cells[n - 2].wm};
            for (int e = tid; e < bt; e += nt) last[e] = prop_element(a.ptab, bt, c, e);
            __syncthreads();
        }
        double dtn = tl[n] - tl[n - 1];
        dtn = dtn > 0.0 ? dtn : 0.0;
        for (int e = tid; e < bt; e += nt) {
            const uint32_t at = aa.element[e];
            const int o = (int)(at & 0xFFFFu), r = (int)((at >> 16) & 31u), c = (int)((at >> 21) & 31u), m = 1 + (int)(at >> 26);
            double v = 0.0;
            if (bare) {
                v = exp(-dtn * aa.ediag[o + r * (m + 1)]) * fin[e];
            } else {
                for (int q = 0; q < m; ++q) v = fma(last[o + r + q * m], fin[o + c * m + q], v);
            }
            mag += fabs(v);
            prow[e] = sr == 0 ? wt * v : prow[e] + wt * v;
        }
        __syncthreads();
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

// ---------------------------------------------------------------------------------------
// The scalar arc walk (all sectors 1x1; programs of ScalarPacker, qiw_arcs.h)
//
// What bounds it: for the order-4 programs of the single orbital (1900 words) the issue of six
// to ten instructions per word, two of them scalar; for all smaller programs (16 to 400 words)
// the set-up of the rows, whose gathers keep the address unit of the CU half busy.  Why states
// in registers read through the VGPR index mode: the order-4 states of 64 samples (47 at a
// time) would fill 24 KB of LDS per wavefront and double the LDS reads; an indexed multiply-add
// takes its source slot without a move.  The compiler has no register array of 64 float64
// values with a run-time index (its tuples end at 16), so the loop is one assembly block on
// fixed registers:
//   v[32:] slots, v[14:15] accumulator, v[16:23] v[24:31] the rows of four words each, v10 v13
//   row addresses, v11 lane offset, v12 row mask; s[40:55] a ring of four times four words.
// Rows and words of the next fours are read while four words are at work; every load's wait is
// inside the block.
//
// SLOTS: programs of up to 24 slots (all but order 4 of the single orbital and order 6 of the
// single level) run in 80 registers, six wavefronts per SIMD, the others in 168, three.
// Measured against the walk of the assignment tries: single-orbital solve (199 steps, orders
// 0:4, N = 2^14) 64.9 -> 17.0 ms, its evaluator 0.31 -> 0.076 ms per step; single-level step of
// orders 0:5 at N = 2^15 7.4 -> 0.18 ms, its evaluator 0.10.  Of these the walk with one register
// count, rows and gathers one after the other took 0.084 and 0.15 ms; three correlators of orders
// 0:3 on 200 points at N = 2^14 went from 10.3 to 7.1 ms with both (3.3 in one launch), a
// randomized step of the single level (orders 0:4, eight times 2^12) from 67 to 36 us.  Keeping
// intervals and fractions of the times instead cost LDS (41 us).  A launch takes one
// instantiation for all its groups: with two launches of a step the small programs' own launch
// cost more than it gained (single orbital 85 instead of 78 us per step).
// ---------------------------------------------------------------------------------------
constexpr int kScalarFew = 24;
#define QIW_SARC_FEW                                                                                                \
    "v10", "v11", "v12", "v13", "v14", "v15", "v16", "v17", "v18", "v19", "v20", "v21", "v22", "v23", "v24", \
    "v25", "v26", "v27", "v28", "v29", "v30", "v31", "v32", "v33", "v34", "v35", "v36", "v37", "v38", "v39", \
    "v40", "v41", "v42", "v43", "v44", "v45", "v46", "v47", "v48", "v49", "v50", "v51", "v52", "v53", "v54", \
    "v55", "v56", "v57", "v58", "v59", "v60", "v61", "v62", "v63", "v64", "v65", "v66", "v67", "v68", "v69", \
    "v70", "v71", "v72", "v73", "v74", "v75", "v76", "v77", "v78", "v79"
#define QIW_SARC_MANY                                                                                               \
    QIW_SARC_FEW, "v80", "v81", "v82", "v83", "v84",                                                          \
    "v85", "v86", "v87", "v88", "v89", "v90", "v91", "v92", "v93", "v94", "v95", "v96", "v97", "v98", "v99", \
    "v100", "v101", "v102", "v103", "v104", "v105", "v106", "v107", "v108", "v109", "v110", "v111", "v112", \
    "v113", "v114", "v115", "v116", "v117", "v118", "v119", "v120", "v121", "v122", "v123", "v124", "v125", \
    "v126", "v127", "v128", "v129", "v130", "v131", "v132", "v133", "v134", "v135", "v136", "v137", "v138", \
    "v139", "v140", "v141", "v142", "v143", "v144", "v145", "v146", "v147", "v148", "v149", "v150", "v151", \
    "v152", "v153", "v154", "v155", "v156", "v157", "v158", "v159"
#define QIW_ROW(w, a, lo, hi)                            \
    "v_and_or_b32 v" #a ", s" #w ", v12, v11\n"          \
    "ds_read_b64 v[" #lo ":" #hi "], v" #a "\n"
#define QIW_ROWS_A(w0, w1, w2, w3) \
    QIW_ROW(w0, 10, 16, 17) QIW_ROW(w1, 13, 18, 19) QIW_ROW(w2, 10, 20, 21) QIW_ROW(w3, 13, 22, 23)
#define QIW_ROWS_B(w0, w1, w2, w3) \
    QIW_ROW(w0, 10, 24, 25) QIW_ROW(w1, 13, 26, 27) QIW_ROW(w2, 10, 28, 29) QIW_ROW(w3, 13, 30, 31)
// a positive TERM falls through; the others run out of line and come back.  The index mode
// stays on for first sources, which are slots only in the terms.
#define QIW_WORD(w, lo, hi)                                       \
    "s_bitcmp1_b32 s" #w ", 31\n"                                 \
    "s_cbranch_scc1 .Lsp" #w "_%=\n"                              \
    "s_set_gpr_idx_idx s" #w "\n"                                 \
    "v_fma_f64 v[14:15], v[32:33], v[" #lo ":" #hi "], v[14:15]\n" \
    ".Lnx" #w "_%=:\n"
#define QIW_WORDS_A(w0, w1, w2, w3) QIW_WORD(w0, 16, 17) QIW_WORD(w1, 18, 19) QIW_WORD(w2, 20, 21) QIW_WORD(w3, 22, 23)
#define QIW_WORDS_B(w0, w1, w2, w3) QIW_WORD(w0, 24, 25) QIW_WORD(w1, 26, 27) QIW_WORD(w2, 28, 29) QIW_WORD(w3, 30, 31)
#define QIW_SPECIAL(w, lo, hi)                                    \
    ".Lsp" #w "_%=:\n"                                            \
    "s_bitcmp1_b32 s" #w ", 30\n"                                 \
    "s_cbranch_scc1 .Lmi" #w "_%=\n"                              \
    "s_set_gpr_idx_on s" #w ", gpr_idx(DST)\n"                    \
    "v_mul_f64 v[32:33], v[14:15], v[" #lo ":" #hi "]\n"          \
    "s_set_gpr_idx_on s" #w ", gpr_idx(SRC0)\n"                   \
    "v_mov_b32 v14, 0\n"                                          \
    "v_mov_b32 v15, 0\n"                                          \
    "s_branch .Lnx" #w "_%=\n"                                    \
    ".Lmi" #w "_%=:\n"                                            \
    "s_set_gpr_idx_idx s" #w "\n"                                 \
    "v_fma_f64 v[14:15], v[32:33], -v[" #lo ":" #hi "], v[14:15]\n" \
    "s_branch .Lnx" #w "_%=\n"
#define QIW_SPECIALS_A(w0, w1, w2, w3) \
    QIW_SPECIAL(w0, 16, 17) QIW_SPECIAL(w1, 18, 19) QIW_SPECIAL(w2, 20, 21) QIW_SPECIAL(w3, 22, 23)
#define QIW_SPECIALS_B(w0, w1, w2, w3) \
    QIW_SPECIAL(w0, 24, 25) QIW_SPECIAL(w1, 26, 27) QIW_SPECIAL(w2, 28, 29) QIW_SPECIAL(w3, 30, 31)
#define QIW_ZERO(r) "v_mov_b32 v" #r ", 0\n"
#define QIW_OUT(lo, hi, off) "ds_write_b64 v11, v[" #lo ":" #hi "] offset:" #off "\n"
#define QIW_SARC_WORDS                                                                                        \
    "s_mov_b32 s59, m0\n"                                                                                     \
    QIW_ZERO(14) QIW_ZERO(15) QIW_ZERO(32) QIW_ZERO(33) QIW_ZERO(34) QIW_ZERO(35) QIW_ZERO(36) QIW_ZERO(37)   \
    QIW_ZERO(38) QIW_ZERO(39) QIW_ZERO(40) QIW_ZERO(41) QIW_ZERO(42) QIW_ZERO(43) QIW_ZERO(44) QIW_ZERO(45)   \
    QIW_ZERO(46) QIW_ZERO(47) QIW_ZERO(48) QIW_ZERO(50) QIW_ZERO(51)                                          \
    "v_mov_b32 v49, 0x3ff00000\n"                                                                             \
    "v_mov_b32 v11, %2\n"                                                                                     \
    "v_mov_b32 v12, 0x3fe00\n"                                                                                \
    "s_mov_b64 s[56:57], %0\n"                                                                                \
    "s_mov_b32 s58, %1\n"                                                                                     \
    "s_cmp_eq_u32 s58, 0\n"                                                                                   \
    "s_cbranch_scc1 .Lend_%=\n"                                                                               \
    "s_load_dwordx8 s[40:47], s[56:57], 0x0\n"                                                                \
    "s_waitcnt lgkmcnt(0)\n"                                                                                  \
    QIW_ROWS_A(40, 41, 42, 43)                                                                                \
    "s_set_gpr_idx_on s40, gpr_idx(SRC0)\n"                                                                   \
    ".Lloop_%=:\n"                                                                                            \
    "s_waitcnt lgkmcnt(0)\n"                                                                                  \
    "s_load_dwordx4 s[48:51], s[56:57], 0x20\n"                                                               \
    QIW_ROWS_B(44, 45, 46, 47)                                                                                \
    QIW_WORDS_A(40, 41, 42, 43)                                                                               \
    "s_waitcnt lgkmcnt(0)\n"                                                                                  \
    "s_load_dwordx4 s[52:55], s[56:57], 0x30\n"                                                               \
    QIW_ROWS_A(48, 49, 50, 51)                                                                                \
    QIW_WORDS_B(44, 45, 46, 47)                                                                               \
    "s_waitcnt lgkmcnt(0)\n"                                                                                  \
    "s_load_dwordx4 s[40:43], s[56:57], 0x40\n"                                                               \
    QIW_ROWS_B(52, 53, 54, 55)                                                                                \
    QIW_WORDS_A(48, 49, 50, 51)                                                                               \
    "s_waitcnt lgkmcnt(0)\n"                                                                                  \
    "s_load_dwordx4 s[44:47], s[56:57], 0x50\n"                                                               \
    QIW_ROWS_A(40, 41, 42, 43)                                                                                \
    QIW_WORDS_B(52, 53, 54, 55)                                                                               \
    "s_add_u32 s56, s56, 64\n"                                                                                \
    "s_addc_u32 s57, s57, 0\n"                                                                                \
    "s_sub_u32 s58, s58, 1\n"                                                                                 \
    "s_cmp_lg_u32 s58, 0\n"                                                                                   \
    "s_cbranch_scc1 .Lloop_%=\n"                                                                              \
    "s_set_gpr_idx_off\n"                                                                                     \
    "s_branch .Lend_%=\n"                                                                                     \
    QIW_SPECIALS_A(40, 41, 42, 43) QIW_SPECIALS_B(44, 45, 46, 47)                                             \
    QIW_SPECIALS_A(48, 49, 50, 51) QIW_SPECIALS_B(52, 53, 54, 55)                                             \
    ".Lend_%=:\n"                                                                                             \
    "s_waitcnt vmcnt(0) lgkmcnt(0)\n"                                                                         \
    "s_barrier\n"                                                                                             \
    "v_add_u32 v11, %3, v11\n"                                                                                \
    QIW_OUT(32, 33, 0) QIW_OUT(34, 35, 512)                                                                   \
    "s_cmp_lt_u32 %4, 4\n"                                                                                    \
    "s_cbranch_scc1 .Lout_%=\n"                                                                               \
    QIW_OUT(36, 37, 1024) QIW_OUT(38, 39, 1536)                                                               \
    "s_cmp_lt_u32 %4, 8\n"                                                                                    \
    "s_cbranch_scc1 .Lout_%=\n"                                                                               \
    QIW_OUT(40, 41, 2048) QIW_OUT(42, 43, 2560) QIW_OUT(44, 45, 3072) QIW_OUT(46, 47, 3584)                   \
    ".Lout_%=:\n"                                                                                             \
    "s_mov_b32 m0, s59\n"                                                                                     \
    "s_waitcnt lgkmcnt(0)\n"

// Runs `blocks` blocks of 16 words from `prog` (eight words and the rows of four past the end
// are read too) on the rows at LDS address 0, lane_off = 8 * lane; then, after a workgroup
// barrier, stores the results of sectors 0 .. n_out - 1 (2, 4 or 8) at out_off + 512 s.
template <int SLOTS>
__device__ __forceinline__ void sarc_words(const uint32_t *prog, int blocks, uint32_t lane_off, uint32_t out_off, int n_out) {
    if constexpr (SLOTS <= kScalarFew)
        asm volatile(QIW_SARC_WORDS
                     :
                     : "s"(prog), "s"(blocks), "v"(lane_off), "s"(out_off), "s"(n_out)
                     : "memory", "scc", "s40", "s41", "s42", "s43", "s44", "s45", "s46", "s47", "s48", "s49", "s50", "s51",
                       "s52", "s53", "s54", "s55", "s56", "s57", "s58", "s59", QIW_SARC_FEW);
    else
        asm volatile(QIW_SARC_WORDS
                     :
                     : "s"(prog), "s"(blocks), "v"(lane_off), "s"(out_off), "s"(n_out)
                     : "memory", "scc", "s40", "s41", "s42", "s43", "s44", "s45", "s46", "s47", "s48", "s49", "s50", "s51",
                       "s52", "s53", "s54", "s55", "s56", "s57", "s58", "s59", QIW_SARC_MANY);
}

// The sum over the wavefront, in lane 63.
template <int CTRL, int ROWS>
__device__ __forceinline__ double add_dpp(double v) {
    const int lo = __builtin_amdgcn_update_dpp(0, __double2loint(v), CTRL, ROWS, 0xf, false);
    const int hi = __builtin_amdgcn_update_dpp(0, __double2hiint(v), CTRL, ROWS, 0xf, false);
    return v + __hiloint2double(hi, lo);
}
__device__ __forceinline__ double wave_sum(double v) {
    v = add_dpp<0x111, 0xf>(v);  // row_shr 1, 2, 4, 8
    v = add_dpp<0x112, 0xf>(v);
    v = add_dpp<0x114, 0xf>(v);
    v = add_dpp<0x118, 0xf>(v);
    v = add_dpp<0x142, 0xa>(v);  // row_bcast 15, 31
    return add_dpp<0x143, 0xc>(v);
}

// Sectors s and s + 1 (one of them if !two) of the propagator table at a cell: three loads.
typedef double d2u __attribute__((ext_vector_type(2), aligned(8)));
struct PairLoad {
    d2u gm, g0, gp;
    __device__ __forceinline__ void load(const double *ptab, int ns, const GridCell &c, int s, bool two) {
        const uint32_t at = (uint32_t)(c.d * ns + s), back = c.d > 0 ? at - (uint32_t)ns : at;
        if (two) {
            gm = *reinterpret_cast<const d2u *>(ptab + back);
            g0 = *reinterpret_cast<const d2u *>(ptab + at);
            gp = *reinterpret_cast<const d2u *>(ptab + at + ns);
        } else {
            gm = d2u{ptab[back], 0.0};
            g0 = d2u{ptab[at], 0.0};
            gp = d2u{ptab[at + ns], 0.0};
        }
    }
    __device__ __forceinline__ d2u value(const GridCell &c) const {
        return d2u{cell_value(c, gm[0], g0[0], gp[0]), cell_value(c, gm[1], g0[1], gp[1])};
    }
};

// grid_cell of two times in units of the grid step.
__device__ __forceinline__ GridCell cell_between(double x1, double x2, int n_tau) {
    x1 = x1 > x2 ? x1 : x2;
    const int i1 = min(max((int)x1, 0), n_tau - 2), i2 = min(max((int)x2, 0), n_tau - 2);
    const double a = x1 - (double)i1, b = x2 - (double)i2;
    return GridCell{i1 - i2, a * (1.0 - b), (1.0 - a) * b};
}

// GRID: every table is a grid container, and no bare group: the times are kept in units of the
// grid step, which halves the instructions of a cell.  The set-up reads all records with
// the first loads, one per lane, and gathers for UA arcs and UP propagators at a time: with one
// after the other a wavefront waited for nine tenths of its time.
template <bool GRID, bool DLR, int SLOTS>
__global__ __launch_bounds__(256, SLOTS > kScalarFew ? 3 : DLR ? 4 : 6) void k_eval_sarcs_t(EvalArgs a) {
    extern __shared__ __attribute__((aligned(16))) char lds[];
    constexpr int UA = GRID ? 3 : SLOTS <= kScalarFew ? 1 : 2, UP = 2;
    double *tab = reinterpret_cast<double *>(lds);  // rows, LDS address 0
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const QiwTask task = a.tasks[blockIdx.x];
    const QiwGroup g = a.groups[task.group];
    const int n = g.n_nodes, ns = a.ns;
    double *tl = tab + g.n_pslots * 64;  // times of the positions (GRID: in grid steps)
    const double inv_h = 1.0 / a.h;
    const uint32_t *words = reinterpret_cast<const uint32_t *>(a.prog + g.prog_off);
    const ConstP<uint32_t> b = as_constp(words);
    const StepTimes T = step_times(a, g, task.tau_index);
    const bool bare = !GRID && g.kind == QIW_G_BARE;
    const int na = (int)b[2], np = (int)b[4];
    if (!(b[12] | b[13] | b[14] | b[15])) {  // no diagram: zeros
        if (tid < a.n_out) a.partial[(int64_t)task.out_index * a.n_out + tid] = 0.0;
        if (a.per_sample && wave == 0 && task.first_sample + lane < g.n_samples)
            a.per_sample[g.ps_off + task.first_sample + lane] = 0.0;
        return;
    }
    // ---- times of the configuration positions, and the records of the rows ----
    {
        const int64_t sample = (int64_t)task.first_sample + lane;
        const double *u = a.ut + g.ut_off + (int64_t)task.tau_index * a.ut_row_stride + (sample < g.n_samples ? sample : 0);
        double v[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int p = wave + 4 * i;
            const bool after = bare || p > g.pos_w;
            const int j = after ? n - 1 - p : g.d_after + g.pos_w - 1 - p;
            v[i] = 0.0;
            if (p > 1 && p < n && g.sampled && (bare || p != g.pos_w)) v[i] = u[(int64_t)j * g.n_samples];
        }
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int p = wave + 4 * i;
            if (p > n) break;
            double t = 0.0;
            if (p == n)
                t = T.tau_f;
            else if (!bare && p == g.pos_w)
                t = T.tau_w;
            else if (p > 1 && g.sampled)
                t = bare || p > g.pos_w ? v[i] * (T.tau_f - T.tau_w) + T.tau_w : v[i] * T.tau_w;
            tl[p * 64 + lane] = GRID ? t * inv_h : t;
        }
    }
    auto cell = [&](int later, int earlier) {  // of two positions
        if constexpr (GRID)
            return cell_between(tl[later * 64 + lane], tl[earlier * 64 + lane], a.n_tau);
        else
            return grid_cell(tl[later * 64 + lane], tl[earlier * 64 + lane], inv_h, a.n_tau);
    };
    uint32_t rec[3] = {0u, 0u, 0u}, prec[2] = {0u, 0u};
    auto arc_records = [&](int first) {
        if (first + lane < na) {
            const uint32_t *r = words + b[3] + 3 * (first + lane);
            rec[0] = r[0];
            rec[1] = r[1];
            rec[2] = r[2];
        }
    };
    arc_records(0);
    if (lane < np) {
        const uint32_t *r = words + b[5] + 2 * lane;
        prec[0] = r[0];
        prec[1] = r[1];
    }
    __syncthreads();
    // ---- rows: constants, arc values, propagators ----
    {
        const ConstP<uint32_t> c = b + b[1];
        for (int i = wave; i < (int)b[0]; i += 4)
            tab[i * 64 + lane] = __hiloint2double((int)c[2 * i + 1], (int)c[2 * i]);
    }
    for (int c0 = 0; c0 < na; c0 += 64) {  // records of up to 64 arcs
        const int nc = min(64, na - c0);
        if (c0 > 0) arc_records(c0);
        for (int i0 = wave; i0 < nc; i0 += 4 * UA) {
            ArcPos ap[UA];
#pragma unroll
            for (int q = 0; q < UA; ++q) {  // past the last arc: the last one again
                const uint32_t ends = rlane(rec[0], min(i0 + 4 * q, nc - 1));
                if constexpr (GRID)
                    ap[q].c = cell((int)(ends >> 8), (int)(ends & 255));
                else
                    ap[q] = arc_pos(tl[(ends >> 8) * 64 + lane], tl[(ends & 255) * 64 + lane], inv_h, a.n_tau);
            }
            for (int tb = 0; tb < a.dtab.n_tables; tb += 2) {
                double c[UA][2][GRID ? 3 : 4];
                uint32_t rows[UA];
#pragma unroll
                for (int q = 0; q < UA; ++q) {
                    rows[q] = i0 + 4 * q < nc ? rlane(tb ? rec[2] : rec[1], i0 + 4 * q) : 0xFFFFFFFFu;
#pragma unroll
                    for (int t = 0; t < 2; ++t) {
                        if (((rows[q] >> (16 * t)) & 0xFFFFu) == 0xFFFFu) continue;
                        if (DLR && ((a.dtab.dlr_mask >> (tb + t)) & 1)) continue;
                        const double *co = a.dtab.coef + (int64_t)(tb + t) * (a.n_tau - 1) * 4;
                        const uint32_t at = 4u * (uint32_t)(GRID || ((a.dtab.grid_mask >> (tb + t)) & 1) ? ap[q].c.d : ap[q].j);
#pragma unroll
                        for (int k = 0; k < (GRID ? 3 : 4); ++k) c[q][t][k] = co[at + k];
                    }
                }
#pragma unroll
                for (int q = 0; q < UA; ++q)
#pragma unroll
                    for (int t = 0; t < 2; ++t) {
                        const uint32_t r = (rows[q] >> (16 * t)) & 0xFFFFu;
                        if (r == 0xFFFFu) continue;
                        double v;
                        if (DLR && ((a.dtab.dlr_mask >> (tb + t)) & 1))
                            v = delta_value<DLR>(a.dtab, tb + t, ap[q]);
                        else if (GRID || ((a.dtab.grid_mask >> (tb + t)) & 1))
                            v = c[q][t][0] + ap[q].c.wp * c[q][t][1] - ap[q].c.wm * c[q][t][2];
                        else
                            v = c[q][t][0] + ap[q].u * (c[q][t][1] + ap[q].u * (c[q][t][2] + ap[q].u * c[q][t][GRID ? 2 : 3]));
                        tab[r * 64 + lane] = v;
                    }
            }
        }
    }
    if (bare) {
        for (int i = wave; i < np; i += 4) {
            const uint32_t w = rlane(prec[0], i), seg = rlane(prec[1], i);
            const int r = (int)(w & 0xFFFFu), s = (int)((w >> 16) & 255u), L = (int)(seg & 255u);
            double dt = tl[L * 64 + lane] - tl[(L - 1) * 64 + lane];
            dt = dt > 0.0 ? dt : 0.0;
            tab[r * 64 + lane] = exp(-dt * a.e_shift[s]);
            if (w >> 24) tab[(r + 1) * 64 + lane] = exp(-dt * a.e_shift[s + 1]);
        }
    } else {
        for (int i0 = wave; i0 < np; i0 += 4 * UP) {
            GridCell c[UP];
            PairLoad x[UP];
#pragma unroll
            for (int q = 0; q < UP; ++q) {
                const int i = min(i0 + 4 * q, np - 1), L = (int)(rlane(prec[1], i) & 255u);
                c[q] = cell(L, L - 1);
            }
#pragma unroll
            for (int q = 0; q < UP; ++q) {
                const uint32_t w = rlane(prec[0], min(i0 + 4 * q, np - 1));
                x[q].load(a.ptab, ns, c[q], (int)((w >> 16) & 255u), (w >> 24) != 0);
            }
#pragma unroll
            for (int q = 0; q < UP; ++q) {
                const int i = i0 + 4 * q;
                if (i >= np) break;
                const uint32_t w = rlane(prec[0], i), seg = rlane(prec[1], i);
                const int r = (int)(w & 0xFFFFu), s = (int)((w >> 16) & 255u), L = (int)(seg & 255u), L2 = (int)(seg >> 8);
                d2u v = x[q].value(c[q]);
                if (L2) {  // times the propagator after the left-out node at tau_w
                    const GridCell c2 = cell(L2, L);
                    PairLoad y;
                    y.load(a.ptab, ns, c2, s, (w >> 24) != 0);
                    v *= y.value(c2);
                }
                tab[r * 64 + lane] = v[0];
                if (w >> 24) tab[(r + 1) * 64 + lane] = v[1];
            }
        }
    }
    __syncthreads();
    if (b[6]) {  // rows times a constant (operator elements other than +-1)
        const ConstP<uint32_t> sc = b + b[7];
        for (int i = wave; i < (int)b[6]; i += 4)
            tab[sc[3 * i] * 64 + lane] = tab[sc[3 * i + 1] * 64 + lane] * tab[sc[3 * i + 2] * 64 + lane];
        __syncthreads();
    }
    // ---- each wavefront's program; results in row n_out * wave + s ----
    const int n_res = a.n_out, n_out = scalar_out_rows(n_res);
    sarc_words<SLOTS>(words + b[8 + wave], (int)b[12 + wave], (uint32_t)lane * 8u, (uint32_t)(wave * n_out) * 512u, n_out);
    __syncthreads();
    // the leaves' sign (-1)^order, and (-1)^n_after for the external arc of a correlator
    // (src/diagrammatics.jl:288-303)
    const int64_t sample = (int64_t)task.first_sample + lane;
    const bool active = sample < g.n_samples;
    const bool odd = (g.order + (g.kind == QIW_G_CORR ? g.n_after : 0)) & 1;
    double wt = odd ? -1.0 : 1.0;
    if (g.weighted) {
        const double *u = a.ut + g.ut_off + (int64_t)task.tau_index * a.ut_row_stride + (active ? sample : 0);
        wt *= u[(int64_t)(g.d_before + g.d_after) * g.n_samples];
    }
    for (int s = wave; s < n_res; s += 4) {
        double v = 0.0;
#pragma unroll
        for (int w = 0; w < 4; ++w) v += tab[(n_out * w + s) * 64 + lane];
        if (a.per_sample) tl[s * 64 + lane] = fabs(v);
        v = wave_sum(active ? v * wt : 0.0);
        if (lane == 63) a.partial[(int64_t)task.out_index * n_res + s] = v;
    }
    if (a.per_sample) {
        __syncthreads();
        if (wave == 0 && active) {
            double m = 0.0;
            for (int s = 0; s < n_res; ++s) m += tl[s * 64 + lane];
            a.per_sample[g.ps_off + sample] = m;
        }
    }
}

template <int SLOTS>
void launch_sarcs(hipStream_t st, const EvalArgs &a, int n_tasks, bool bare, size_t lds) {
    const dim3 grid(n_tasks), block(256);
    if (a.dtab.dlr_mask)
        hipLaunchKernelGGL((k_eval_sarcs_t<false, true, SLOTS>), grid, block, lds, st, a);
    else if (!bare && a.dtab.grid_mask == (1 << a.dtab.n_tables) - 1)
        hipLaunchKernelGGL((k_eval_sarcs_t<true, false, SLOTS>), grid, block, lds, st, a);
    else
        hipLaunchKernelGGL((k_eval_sarcs_t<false, false, SLOTS>), grid, block, lds, st, a);
}

}  // namespace

// Vector length of the instantiation for blocks up to mb, and the most wavefronts a
// workgroup of it can have (its registers).
int qiw_arc_rows(int mb) { return mb <= 8 ? 8 : mb <= 20 ? 20 : 32; }
int qiw_arc_waves(int mb, int fp32) { return fp32 && mb <= 8 ? 16 : 8; }

hipError_t qiw_launch_eval_arcs(hipStream_t st, const ArcArgs &a, int n_tasks, int mb, int fp32, int waves, size_t lds) {
    if (n_tasks < 1 || mb > 32 || a.e.n_tau < 2) return hipErrorInvalidValue;
    if (mb <= 8) return fp32 ? launch<float, 8, 1024>(st, a, n_tasks, waves, lds) : launch<double, 8, 512>(st, a, n_tasks, waves, lds);
    if (mb <= 20) return fp32 ? launch<float, 20, 512>(st, a, n_tasks, waves, lds) : launch<double, 20, 512>(st, a, n_tasks, waves, lds);
    return fp32 ? launch<float, 32, 512>(st, a, n_tasks, waves, lds) : launch<double, 32, 512>(st, a, n_tasks, waves, lds);
}

// slots: register slots of the programs; bare: its groups are bare ones; lds: scalar_lds_rows of the
// largest group, 512 bytes each.
hipError_t qiw_launch_eval_sarcs(hipStream_t st, const EvalArgs &a, int n_tasks, int slots, bool bare, size_t lds) {
    if (n_tasks < 1 || a.ns > 8 || a.n_out < 1 || a.n_out > 8 || a.dtab.n_tables > 4 || slots > kScalarSlots) return hipErrorInvalidValue;
    if (slots <= kScalarFew)
        launch_sarcs<kScalarFew>(st, a, n_tasks, bare, lds);
    else
        launch_sarcs<kScalarSlots>(st, a, n_tasks, bare, lds);
    return hipGetLastError();
}
int qiw_sarc_slots(int slots) { return slots <= kScalarFew ? kScalarFew : kScalarSlots; }
