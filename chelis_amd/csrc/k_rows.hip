// Row regions on gfx950: softmax, causal scaled softmax, softmax adjoint and
// layer norm over the last axis, each as ONE kernel that reads its row once
// from HBM into registers and writes its result once.
//
// Layout of a row in registers. A row of n elements is treated as the
// power-of-two capacity CAP = S * 64W * V >= n, padded past n. The row is
// cut into S segments of 64W*V elements; in segment s, thread t holds the
// V consecutive elements starting at s*64W*V + t*V, loaded with one 16-byte
// vector load, so each load instruction of a wave covers one contiguous
// 1 KiB span (fully coalesced).
//
// Canonical sum tree ([05-OP-30]). Every (segment, thread) block is an
// aligned power-of-two run of leaves, so the adjacent-pair tree over the
// padded row is: an in-register tree over the V leaves, then a wave64
// butterfly (xor 1,2,...,32: step m joins the aligned blocks of 2^m
// threads), then a tree over the W waves through LDS, then a tree over the
// S segments. Padding leaves are -0.0, the exact additive identity
// (x + -0 = x for every x under round-to-nearest), and a power-of-two tree
// over the padded row has the same value as the adjacent-pair tree with an
// odd carry over the n real leaves. IEEE addition is commutative, so both
// butterfly partners hold the same bits.
//
// max_reduce ([05-OP-12]) combines with max_first in index order: in-lane
// left to right, butterfly with the lower lane as the left operand,
// waves and segments in order. Padding is -inf, which never displaces an
// earlier element.
#include "chain.h"

#include <initializer_list>

namespace chelis {
namespace {

// 16-byte native vectors (the nontemporal builtins take clang vector types).
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef double f64x2 __attribute__((ext_vector_type(2)));
template <typename T, int V>
struct VecT;
template <>
struct VecT<float, 4> {
    using type = f32x4;
};
template <>
struct VecT<double, 2> {
    using type = f64x2;
};

// Streaming rows are read once and written once: NT selects the
// nontemporal (streaming) cache policy for them; vectors shared by every row
// (layer norm's gamma and beta) use the default policy. The access is
// aligned to the element only: a 16-byte global access needs no more on
// gfx950, so rows of any length and start move as vectors.
template <bool NT, typename T, int V>
__device__ inline typename VecT<T, V>::type vload(const T *p) {
    typedef T Q __attribute__((ext_vector_type(V), aligned(sizeof(T))));
    if constexpr (NT) return __builtin_nontemporal_load(reinterpret_cast<const Q *>(p));
    else return *reinterpret_cast<const Q *>(p);
}
template <typename T, int V>
__device__ inline void vstore(typename VecT<T, V>::type v, T *p) {
    typedef T Q __attribute__((ext_vector_type(V), aligned(sizeof(T))));
    __builtin_nontemporal_store(v, reinterpret_cast<Q *>(p));
}

template <typename T>
__device__ inline T neg_inf() {
    return -__builtin_huge_val();
}
template <>
__device__ inline float neg_inf<float>() {
    return -__builtin_huge_valf();
}

template <typename T>
__device__ inline T exp_leaf(T v);
template <>
__device__ inline float exp_leaf<float>(float v) {
    return expf_cr(v);
}
template <>
__device__ inline double exp_leaf<double>(double v) {
    return leaf_exp<double>(v);
}

// 2^(j/64), j = 0..63, held one entry per lane (lane j holds T[j]); a
// lookup is a wave64 shuffle, so every lane of the wave must be active.
struct ExpTableLanes {
    double t;
    __device__ explicit ExpTableLanes(int lane) : t(chelis_exp2_64_tab[lane][0]) {}
    __device__ double operator()(int j) const { return __shfl(t, j, 64); }
};

// 2^(j/64) as a double-double, read from the block's LDS copy: one 16-byte
// LDS read per lookup where a lane-held copy took four lane shuffles and
// four registers (the f64 softmax row: 58 against 64-68 us for [4096, 4096]
// on one box, bit-identical).
struct Exp2TableLds {
    const double2 *t;
    __device__ void operator()(int j, double &h, double &l) const {
        const double2 e = t[j];
        h = e.x;
        l = e.y;
    }
    // the high part alone (the faithful exp)
    __device__ double operator()(int j) const { return t[j].x; }
};

// The exp table of each dtype, built before the row loads so waiting for it
// never waits for a row: binary32 holds it one entry per lane, binary64 in
// LDS (filled by the kernel's first wave).
template <typename T>
struct RowExpTab;
template <>
struct RowExpTab<float> {
    using type = ExpTableLanes;
    __device__ static type make(int lane, const double2 *) { return type(lane); }
};
template <>
struct RowExpTab<double> {
    using type = Exp2TableLds;
    __device__ static type make(int, const double2 *lds) { return type{lds}; }
};

// Which of a lane's NE exp results need the correctly rounded fallback.
// Up to 16 per lane: one wave-uniform lane mask per element (scalar
// registers, set straight from the compare); beyond that: a per-lane bit set.
template <int NE, bool UNIFORM = (NE <= 16)>
struct SlowSet;
template <int NE>
struct SlowSet<NE, true> {
    uint64_t lanes[NE];
    uint64_t all = 0;
    __device__ void set(int k, bool slow) {
        lanes[k] = __ballot(slow);
        all |= lanes[k];
    }
    __device__ bool any() const { return all != 0; }
    __device__ bool has(int k, int lane) const { return (lanes[k] >> lane) & 1u; }
};
template <int NE>
struct SlowSet<NE, false> {
    static_assert(NE <= 64, "one bit per element");
    uint32_t bits[2] = {0, 0};
    __device__ void set(int k, bool slow) { bits[k >> 5] |= (uint32_t)slow << (k & 31); }
    // the lane's next flagged element, or -1, taken out of the set
    __device__ int take() {
        const int h = bits[0] ? 0 : 1;
        const uint32_t b = bits[h];
        bits[h] = b & (b - 1);
        return b ? 32 * h + __builtin_ctz(b) : -1;
    }
    __device__ bool any() const { return __any((bits[0] | bits[1]) != 0); }
    __device__ bool has(int k, int) const { return (bits[k >> 5] >> (k & 31)) & 1u; }
};

// The rare correctly rounded fallback stays out of line: inlined 16 times it
// would dominate the kernel's code.
__device__ __noinline__ float expf_slow(float x) { return expf_cr_dd(x); }

// Per-row geometry: which row this wave group owns and where it starts. A
// row has W waves of 64 lanes, or (W = 1) L = 16 lanes of a wave that holds
// four rows. Lanes of a short row past the last one repeat it (every lane of
// the wave takes part in its lane exchanges) and do not store.
template <int W, int R, int L>
struct RowCoord {
    static_assert(L == 64 || (L == 16 && W == 1), "whole waves, or a quarter of one");
    int lane, wave_in_row, row_in_block, tid_in_row;
    int64_t row;
    bool live;
    __device__ explicit RowCoord(int64_t rows) {
        const int tid = threadIdx.x;
        lane = tid & 63;
        const int wave = tid >> 6;
        wave_in_row = wave % W;
        row_in_block = wave / W;
        tid_in_row = L == 64 ? wave_in_row * 64 + lane : lane % L;
        row = (int64_t)blockIdx.x * R + row_in_block;
        if (L < 64) row = row * (64 / L) + lane / L;
        live = row < rows;
        if (L < 64 && !live) row = rows - 1;
    }
};

// Canonical tree sum and plain maximum of one value per lane over the L
// lanes of a row; every lane gets the result.
template <int L, typename T>
__device__ inline T lanes_tree_sum(T x) {
    if constexpr (L == 64) return wave_tree_sum(x);
    x = x + dpp_perm<kDppXor1>(x);
    x = x + dpp_perm<kDppXor2>(x);
    x = x + dpp_perm<kDppHalfMirror>(x);
    return x + dpp_perm<kDppMirror>(x);
}
template <int L, typename T>
__device__ inline T lanes_vmax(T x) {
    if constexpr (L == 64) return wave_vmax(x);
    x = vmax(x, dpp_perm<kDppXor1>(x));
    x = vmax(x, dpp_perm<kDppXor2>(x));
    x = vmax(x, dpp_perm<kDppHalfMirror>(x));
    return vmax(x, dpp_perm<kDppMirror>(x));
}

// A row's n elements, padded past n, in two halves: issue() sends the loads,
// take() waits for them, so a kernel that reads several rows has all of them
// in flight before it waits for the first. Neither has a branch around a
// load (a branch there made the compiler wait for one load before the next:
// layer norm of [20000, 1000] 34.3 against 31.6 us): a lane past the end
// reads the row's last V elements again. RAGGED serves row lengths that are
// no multiple of V; there the lane that straddles the end moves those down
// to its own place. Without PAD an element past n may hold anything.
template <typename T, int V, int S, int W, int L, bool RAGGED, bool NT = true, bool PAD = true>
struct RowLoad {
    static constexpr int SEG = L * W * V;
    using Q = typename VecT<T, V>::type;
    const T *p;
    int n, tid;
    Q q[S];
    __device__ RowLoad(const T *row, int count, int tid_in_row) : p(row), n(count), tid(tid_in_row) {}
    __device__ void issue() {
        if (RAGGED && n < V) return;
#pragma unroll
        for (int s = 0; s < S; ++s) {
            const int base = s * SEG + tid * V;
            q[s] = vload<NT, T, V>(p + (base < n - V ? base : n - V));
        }
    }
    __device__ void take(T pad, T (&v)[S][V]) {
        if (RAGGED && n < V) {
#pragma unroll
            for (int s = 0; s < S; ++s)
#pragma unroll
                for (int i = 0; i < V; ++i) {
                    const int j = s * SEG + tid * V + i;
                    v[s][i] = j < n ? p[j] : pad;
                }
            return;
        }
#pragma unroll
        for (int s = 0; s < S; ++s) {
            const int base = s * SEG + tid * V;
            if constexpr (!RAGGED) {
#pragma unroll
                for (int i = 0; i < V; ++i) v[s][i] = !PAD || base < n ? q[s][i] : pad;
            } else {
                // d elements of the lane's vector lie past the end
                const int d = base > n - V ? base - (n - V) : 0;
#pragma unroll
                for (int i = 0; i < V; ++i) {
                    v[s][i] = pad;
#pragma unroll
                    for (int u = V - 1; u >= i; --u) v[s][i] = i + d == u ? q[s][u] : v[s][i];
                }
            }
        }
    }
};

// DENSE: the row is exactly the register capacity.
template <typename T, int V, int S, int W, int L>
__device__ inline void load_dense(const T *__restrict__ p, int tid_in_row, T (&v)[S][V]) {
#pragma unroll
    for (int s = 0; s < S; ++s) {
        const typename VecT<T, V>::type q =
            vload<true, T, V>(p + s * L * W * V + tid_in_row * V);
#pragma unroll
        for (int i = 0; i < V; ++i) v[s][i] = q[i];
    }
}

template <typename T, int V, int S, int W, int L, bool RAGGED>
__device__ inline void store_row(T *__restrict__ p, int n, int tid_in_row, const T (&v)[S][V]) {
    constexpr int SEG = L * W * V;
#pragma unroll
    for (int s = 0; s < S; ++s) {
        const int base = s * SEG + tid_in_row * V;
        if (base + V <= n) {
            typename VecT<T, V>::type q;
#pragma unroll
            for (int i = 0; i < V; ++i) q[i] = v[s][i];
            vstore<T, V>(q, p + base);
        } else if constexpr (RAGGED) {
#pragma unroll
            for (int i = 0; i < V; ++i)
                if (base + i < n) p[base + i] = v[s][i];
        }
    }
}

// Canonical tree over the padded row of leaves leaf(s, i); every thread of
// the row gets the total.
template <typename T, int V, int S, int W, int R, int L, class F>
__device__ inline T row_tree_sum(F leaf, T *lds, const RowCoord<W, R, L> &c) {
    T seg[S];
#pragma unroll
    for (int s = 0; s < S; ++s) {
        T a[V];
#pragma unroll
        for (int i = 0; i < V; ++i) a[i] = leaf(s, i);
#pragma unroll
        for (int w = V; w > 1; w >>= 1)
#pragma unroll
            for (int i = 0; i < w / 2; ++i) a[i] = a[2 * i] + a[2 * i + 1];
        seg[s] = lanes_tree_sum<L>(a[0]);
    }
    if constexpr (S * W >= 32 && W > 1) {
        // the (segment, wave) totals in order are the leaves of the row's top
        // subtree: each lane joins its run of them and the wave joins the
        // lanes (-0 past the end). Each thread reading all S * W totals held
        // too many registers for rows of sixteen waves.
        constexpr int N = S * W, P = N > 64 ? N / 64 : 1;
        T *top = lds + c.row_in_block * N;
        if (c.lane == 0)
#pragma unroll
            for (int s = 0; s < S; ++s) top[s * W + c.wave_in_row] = seg[s];
        __syncthreads();
        T a[P];
#pragma unroll
        for (int i = 0; i < P; ++i) a[i] = c.lane * P + i < N ? top[c.lane * P + i] : T(-0.0);
#pragma unroll
        for (int w = P; w > 1; w >>= 1)
#pragma unroll
            for (int i = 0; i < w / 2; ++i) a[i] = a[2 * i] + a[2 * i + 1];
        const T total = wave_tree_sum(a[0]);
        __syncthreads();
        return total;
    } else if constexpr (W > 1) {
        if (c.lane == 0)
#pragma unroll
            for (int s = 0; s < S; ++s) lds[(c.row_in_block * W + c.wave_in_row) * S + s] = seg[s];
        __syncthreads();
#pragma unroll
        for (int s = 0; s < S; ++s) {
            T p[W];
#pragma unroll
            for (int w = 0; w < W; ++w) p[w] = lds[(c.row_in_block * W + w) * S + s];
#pragma unroll
            for (int w = W; w > 1; w >>= 1)
#pragma unroll
                for (int i = 0; i < w / 2; ++i) p[i] = p[2 * i] + p[2 * i + 1];
            seg[s] = p[0];
        }
        __syncthreads();
    }
#pragma unroll
    for (int w = S; w > 1; w >>= 1)
#pragma unroll
        for (int i = 0; i < w / 2; ++i) seg[i] = seg[2 * i] + seg[2 * i + 1];
    return seg[0];
}
template <typename T, int V, int S, int W, int R, int L>
__device__ inline T row_tree_sum(const T (&v)[S][V], T *lds, const RowCoord<W, R, L> &c) {
    return row_tree_sum<T, V, S, W, R, L>([&](int s, int i) { return v[s][i]; }, lds, c);
}

// Plain IEEE maximum over the padded row (v_max: a NaN operand yields the
// other one, and +0/-0 ties are unordered). Softmax uses it in place of
// [05-OP-12]'s first-NaN / first-representation rule because the two give
// identical softmax bits: a NaN anywhere in the row makes that element's
// x - m NaN, hence the tree sum NaN and every output the canonical NaN under
// either rule; and a zero maximum enters only through x - m, where
// x - (+0) and x - (-0) differ at most in the sign of a zero, which exp maps
// to the same 1.
template <typename T, int V, int S, int W, int R, int L>
__device__ inline T row_max_plain(const T (&v)[S][V], T *lds, const RowCoord<W, R, L> &c) {
    T x = v[0][0];
#pragma unroll
    for (int s = 0; s < S; ++s)
#pragma unroll
        for (int i = 0; i < V; ++i) x = vmax(x, v[s][i]);
    x = lanes_vmax<L>(x);
    if constexpr (W > 1) {
        if (c.lane == 0) lds[c.row_in_block * W + c.wave_in_row] = x;
        __syncthreads();
#pragma unroll
        for (int w = 0; w < W; ++w) x = vmax(x, lds[c.row_in_block * W + w]);
        __syncthreads();
    }
    return x;
}

// v / total at the dtype. binary32: the quotient is formed as
// (double)v * (1 / (double)total) and rounded once to binary32. That is the
// correctly rounded v / total: the exact quotient of two binary32 values is
// never closer than 2^-49 relative to a binary32 rounding midpoint (it is
// X 2^a / (T 2^b) with 24-bit X, T against a midpoint M 2^c with 25-bit M,
// and X 2^a - T M 2^(b+c) is a nonzero multiple of 2^min(a, b+c); the
// subnormal range keeps an absolute gap of at least 2^-150 / T), while the
// binary64 product is within 2^-52 relative of it.
template <typename T>
struct RowDiv {
    T total;
    double inv;
    __device__ explicit RowDiv(T t) : total(t), inv(1.0 / (double)t) {}
    __device__ T operator()(T v) const { return canon(quot_f32(v, inv)); }
};

__device__ __noinline__ double div_full(double v, double t) { return v / t; }

// binary64: the steps of the device's IEEE division (v_div_scale_f64 of
// both operands, v_rcp_f64 with two Newton steps, product, residual, fma,
// v_div_fixup_f64), with the reciprocal - which depends only on the
// divisor - formed once per row. The steps are taken as they are where the
// scale steps are the identity: a divisor in [1, 2^20] (the row totals)
// and a dividend that is 0 or at least 2^-960 (v_div_scale_f64 scales a
// dividend whose biased exponent is at most 53, or whose quotient would be
// subnormal); any other element takes the full division.
template <>
struct RowDiv<double> {
    double total, rcp;
    bool fast;
    __device__ explicit RowDiv(double t) : total(t), fast(t >= 1.0 && t <= 0x1p20) {
        double r = __builtin_amdgcn_rcp(t);
        double e = fma(-t, r, 1.0);
        r = fma(r, e, r);
        e = fma(-t, r, 1.0);
        rcp = fma(r, e, r);
    }
    __device__ double operator()(double v) const {
        if (fast && (v == 0.0 || v >= 0x1p-960)) {
            const double q = v * rcp;
            const double r = fma(-total, q, v);
            return canon(__builtin_amdgcn_div_fixup(fma(r, rcp, q), total, v));
        }
        return canon(div_full(v, total));
    }
};

// The value softmax takes x - max of: element j of a row, optionally
// as where(j <= qi, x * scale, -inf) (masked 1: causal, masked 2: scale only).
template <typename T>
__device__ inline T softmax_arg(T raw, int j, int qi, int masked, T scale) {
    if (!masked) return raw;
    const T sc = canon(raw * scale);
    return (masked == 2 || j <= qi) ? sc : neg_inf<T>();
}

// One row: v holds the raw row (padding -inf) on entry and the softmax on
// exit; xr is the row in memory (re-read only by the rare exp fallback, which
// may use the result row yr as its working space).
// FAITHFUL (binary64 only): the faithful exp and one reciprocal per row in
// place of the correctly rounded exp and the IEEE division.
template <typename T, int V, int S, int W, int R, int L, bool FAITHFUL = false>
__device__ inline void softmax_row(T (&v)[S][V], const T *xr, T *yr, int64_t row, int n, int masked, T scale,
                                   int64_t q_len, T *lds, const RowCoord<W, R, L> &c,
                                   const typename RowExpTab<T>::type &tab) {
    constexpr int SEG = L * W * V;
    const int qi = masked ? (int)(row % q_len) : 0;
    if (masked) {
#pragma unroll
        for (int s = 0; s < S; ++s)
#pragma unroll
            for (int i = 0; i < V; ++i) {
                const int j = s * SEG + c.tid_in_row * V + i;
                if (j < n) v[s][i] = softmax_arg(v[s][i], j, qi, masked, scale);
            }
    }
    const T m = row_max_plain<T, V, S, W, R, L>(v, lds, c);
    const bool full = n == S * SEG;
    if constexpr (sizeof(T) == 4) {
        // exp(x - m) in place: the branch-free fast path for every element
        // (2^(j/64) from the lane-held table), then one wave-uniform pass of
        // the correctly rounded core over the few flagged elements, whose
        // argument is formed again from the row in memory. x - m is <= 0 or
        // NaN (m is the row maximum), so the NONPOS path applies.
        SlowSet<S * V> flagged;
#pragma unroll
        for (int s = 0; s < S; ++s)
#pragma unroll
            for (int i = 0; i < V; ++i) {
                bool slow;
                v[s][i] = expf_fast<true>(v[s][i] - m, tab, slow);
                flagged.set(s * V + i, slow);
                // long rows: a segment at a time, for registers
                if (S * V > 16 && i == V - 1) __builtin_amdgcn_sched_barrier(0);
            }
        if constexpr (S * V <= 16) {
            if (flagged.any()) {
#pragma unroll
                for (int s = 0; s < S; ++s)
#pragma unroll
                    for (int i = 0; i < V; ++i) {
                        const int j = s * SEG + c.tid_in_row * V + i;
                        if (flagged.has(s * V + i, c.lane) && (full || j < n))
                            v[s][i] = expf_slow(softmax_arg(xr[j], j, qi, masked, scale) - m);
                    }
            }
        } else if (flagged.any()) {
            // many elements per lane: the flagged elements are finished in the
            // result row in memory (each lane its own), where the others wait,
            // so no register is held across the core; an element not yet
            // finished keeps its input there when the call is in place. A
            // call of the core per element left the row in scratch memory
            // ([1000, 32003] binary32: 3.5 ms, 3600 bytes of it per lane).
#pragma unroll
            for (int s = 0; s < S; ++s)
#pragma unroll
                for (int i = 0; i < V; ++i) {
                    const int j = s * SEG + c.tid_in_row * V + i;
                    if (j < n && !flagged.has(s * V + i, c.lane)) yr[j] = v[s][i];
                }
            while (flagged.any()) {
                const int k = flagged.take();
                const int j = (k / V) * SEG + c.tid_in_row * V + k % V;
                if (k >= 0 && j < n) yr[j] = expf_cr_dd(softmax_arg(xr[j], j, qi, masked, scale) - m);
            }
#pragma unroll
            for (int s = 0; s < S; ++s)
#pragma unroll
                for (int i = 0; i < V; ++i) {
                    const int j = s * SEG + c.tid_in_row * V + i;
                    v[s][i] = j < n ? yr[j] : T(-0.0);
                }
        }
        if (!full) {
#pragma unroll
            for (int s = 0; s < S; ++s)
#pragma unroll
                for (int i = 0; i < V; ++i) {
                    const int j = s * SEG + c.tid_in_row * V + i;
                    if (j >= n) v[s][i] = T(-0.0);
                }
        }
        const T total = row_tree_sum<T, V, S, W, R, L>(v, lds, c);
        if (total != total) {
            // a NaN total makes every quotient the canonical NaN
#pragma unroll
            for (int s = 0; s < S; ++s)
#pragma unroll
                for (int i = 0; i < V; ++i) v[s][i] = canon(total);
        } else {
            // total >= 1 (the maximum contributes exp(0)) or +inf: finite
            // e / total needs no NaN finalization
            const double inv = 1.0 / (double)total;
#pragma unroll
            for (int s = 0; s < S; ++s)
#pragma unroll
                for (int i = 0; i < V; ++i) v[s][i] = quot_f32(v[s][i], inv);
        }
    } else if constexpr (FAITHFUL) {
        // the default binary64 row: exp(x - m) faithful (within 1 ulp, no
        // fallback pass), the canonical tree total, then e * (1 / total):
        // within a few ulps of the correctly rounded quotients. A NaN
        // argument yields a NaN exp, hence a NaN total and every output the
        // canonical NaN, as in the exact row.
#pragma unroll
        for (int s = 0; s < S; ++s)
#pragma unroll
            for (int i = 0; i < V; ++i) v[s][i] = exp_nonpos_faithful(v[s][i] - m, tab);
        if (!full) {
#pragma unroll
            for (int s = 0; s < S; ++s)
#pragma unroll
                for (int i = 0; i < V; ++i) {
                    const int j = s * SEG + c.tid_in_row * V + i;
                    if (j >= n) v[s][i] = T(-0.0);
                }
        }
        const T total = row_tree_sum<T, V, S, W, R, L>(v, lds, c);
        if (total != total) {
#pragma unroll
            for (int s = 0; s < S; ++s)
#pragma unroll
                for (int i = 0; i < V; ++i) v[s][i] = canon(total);
        } else {
            // 1 <= total <= n: every product is finite
            const T inv = T(1) / total;
#pragma unroll
            for (int s = 0; s < S; ++s)
#pragma unroll
                for (int i = 0; i < V; ++i) v[s][i] = v[s][i] * inv;
        }
    } else {
        // exp(x - m) in place, as for binary32: the binary64 fast path for
        // every element (2^(j/64) as a double-double from the lane-held
        // table), then one wave-uniform pass of the fixed-point path over the
        // flagged elements (about one in 2^19, and NaN arguments).
        SlowSet<S * V> flagged;
#pragma unroll
        for (int s = 0; s < S; ++s)
#pragma unroll
            for (int i = 0; i < V; ++i) {
                bool slow;
                v[s][i] = exp_fast<true>(v[s][i] - m, tab, slow);
                flagged.set(s * V + i, slow);
            }
        if constexpr (S * V <= 16) {
            if (flagged.any()) {
#pragma unroll
                for (int s = 0; s < S; ++s)
#pragma unroll
                    for (int i = 0; i < V; ++i) {
                        const int j = s * SEG + c.tid_in_row * V + i;
                        if (flagged.has(s * V + i, c.lane) && (full || j < n))
                            v[s][i] = exp_slow64(softmax_arg(xr[j], j, qi, masked, scale) - m);
                    }
            }
        } else if (flagged.any()) {
#pragma unroll
            for (int s = 0; s < S; ++s)
#pragma unroll
                for (int i = 0; i < V; ++i) {
                    const int j = s * SEG + c.tid_in_row * V + i;
                    if (j < n && !flagged.has(s * V + i, c.lane)) yr[j] = v[s][i];
                }
            while (flagged.any()) {
                const int k = flagged.take();
                const int j = (k / V) * SEG + c.tid_in_row * V + k % V;
                if (k >= 0 && j < n) yr[j] = exp_cr_slow(softmax_arg(xr[j], j, qi, masked, scale) - m);
            }
#pragma unroll
            for (int s = 0; s < S; ++s)
#pragma unroll
                for (int i = 0; i < V; ++i) {
                    const int j = s * SEG + c.tid_in_row * V + i;
                    v[s][i] = j < n ? yr[j] : T(-0.0);
                }
        }
        if (!full) {
#pragma unroll
            for (int s = 0; s < S; ++s)
#pragma unroll
                for (int i = 0; i < V; ++i) {
                    const int j = s * SEG + c.tid_in_row * V + i;
                    if (j >= n) v[s][i] = T(-0.0);
                }
        }
        const RowDiv<T> div(canon(row_tree_sum<T, V, S, W, R, L>(v, lds, c)));
#pragma unroll
        for (int s = 0; s < S; ++s)
#pragma unroll
            for (int i = 0; i < V; ++i) v[s][i] = div(v[s][i]);
    }
}

// softmax over the last axis, optionally of where(j <= i, x * scale, -inf)
// (causal != 0, q_len = rows per score matrix). DENSE instances serve the
// common case (no mask, row length equal to the register capacity S*L*W*V)
// with every bound test folded away. FAITHFUL as for
// softmax_row.
template <typename T, int V, int S, int W, int R, int L, bool DENSE, bool RAGGED, bool FAITHFUL = false>
__global__ __launch_bounds__(64 * W * R, W == 16 && S == 8 && (sizeof(T) == 4 || FAITHFUL) ? 8 : 1) void softmax_kernel(const T *x, T *y,
                                                              int64_t rows, int n_arg, int64_t ldx, int64_t ldy,
                                                              int masked_arg, T scale, int64_t q_len) {
    __shared__ T lds[R * W * S];
    constexpr int SEG = L * W * V;
    const int n = DENSE ? S * SEG : n_arg;
    const int masked = DENSE ? 0 : masked_arg;
    __shared__ double2 exp_tab[sizeof(T) == 8 ? 64 : 1];
    if constexpr (sizeof(T) == 8) {
        if (threadIdx.x < 64) exp_tab[threadIdx.x] = double2{chelis_exp2_64_tab[threadIdx.x][0], chelis_exp2_64_tab[threadIdx.x][1]};
        __syncthreads();
    }
    RowCoord<W, R, L> c(rows);
    if (L == 64 && !c.live) return;  // whole row groups exit together (R rows per block, W waves each)
    const T *xr = x + c.row * ldx;
    const typename RowExpTab<T>::type tab = RowExpTab<T>::make(c.lane, exp_tab);
    T v[S][V];
    // causal rows read only j <= qi: the mask turns every later element into
    // -inf whatever it holds, which is the padding value
    if constexpr (DENSE) {
        load_dense<T, V, S, W, L>(xr, c.tid_in_row, v);
    } else {
        const int need = masked == 1 ? (int)(c.row % q_len) + 1 : n, up = (need + V - 1) / V * V;
        const int n_load = up < n ? up : n;
        RowLoad<T, V, S, W, L, RAGGED> lx(xr, n_load, c.tid_in_row);
        lx.issue();
        lx.take(neg_inf<T>(), v);
    }
    softmax_row<T, V, S, W, R, L, FAITHFUL>(v, xr, y + c.row * ldy, c.row, n, masked, scale, q_len, lds, c, tab);
    if (c.live) store_row<T, V, S, W, L, RAGGED>(y + c.row * ldy, n, c.tid_in_row, v);
}

// dx = y * (g - sum(g * y)) over the last axis. Rows of sixteen segments
// (two of them are more than a lane's registers) are read again for the
// second half, from the caches where they fit.
template <typename T, int V, int S, int W, int R, int L, bool RAGGED>
__global__ __launch_bounds__(64 * W * R) void softmax_adjoint_kernel(const T *__restrict__ y,
                                                                      const T *__restrict__ g, T *__restrict__ dx,
                                                                      int64_t rows, int n, int64_t ldy,
                                                                      int64_t ldg, int64_t ldd) {
    __shared__ T lds[R * W * S];
    RowCoord<W, R, L> c(rows);
    if (L == 64 && !c.live) return;
    constexpr int SEG = L * W * V;
    const T *yr = y + c.row * ldy, *gr = g + c.row * ldg;
    T *dr = dx + c.row * ldd;
    auto product = [](T a, T b) { return canon(a * b); };
    if constexpr (S < 16) {
        T yv[S][V], gv[S][V];
        RowLoad<T, V, S, W, L, RAGGED> ly(yr, n, c.tid_in_row), lg(gr, n, c.tid_in_row);
        ly.issue();
        lg.issue();
        ly.take(T(-0.0), yv);
        lg.take(T(-0.0), gv);
        const T total = canon(row_tree_sum<T, V, S, W, R, L>(
            [&](int s, int i) {
                return s * SEG + c.tid_in_row * V + i < n ? product(gv[s][i], yv[s][i]) : T(-0.0);
            },
            lds, c));
#pragma unroll
        for (int s = 0; s < S; ++s)
#pragma unroll
            for (int i = 0; i < V; ++i) gv[s][i] = canon(yv[s][i] * canon(gv[s][i] - total));
        if (c.live) store_row<T, V, S, W, L, RAGGED>(dr, n, c.tid_in_row, gv);
    } else {
        // in place (dx is y or g) is safe: every read of the row precedes
        // the barrier below or is of the lane's own elements
        T t[S][V];
#pragma unroll
        for (int s = 0; s < S; ++s)
#pragma unroll
            for (int i = 0; i < V; ++i) {
                const int j = s * SEG + c.tid_in_row * V + i;
                t[s][i] = j < n ? product(gr[j], yr[j]) : T(-0.0);
            }
        const T total = canon(row_tree_sum<T, V, S, W, R, L>(t, lds, c));
#pragma unroll
        for (int s = 0; s < S; ++s)
#pragma unroll
            for (int i = 0; i < V; ++i) {
                const int j = s * SEG + c.tid_in_row * V + i;
                if (j < n) dr[j] = canon(yr[j] * canon(gr[j] - total));
            }
    }
}

// layer_norm: mean = tree(x)/n; c = x - mean; var = tree(c*c)/n;
// y = (c / sqrt(var + eps)) * gamma + beta, every primitive finalized.
template <typename T, int V, int S, int W, int R, int L, bool RAGGED>
__global__ __launch_bounds__(64 * W * R) void layer_norm_kernel(const T *__restrict__ x, const T *__restrict__ gamma,
                                                                 const T *__restrict__ beta, T *__restrict__ y,
                                                                 int64_t rows, int n, int64_t ldx, int64_t ldy,
                                                                 T eps) {
    __shared__ T lds[R * W * S];
    RowCoord<W, R, L> c(rows);
    if (L == 64 && !c.live) return;
    // gamma/beta are [n] vectors shared by every row: their loads go out with
    // the row's, ahead of the reductions' barriers (after them each row waited
    // out two more cache round trips: [65536,1024] 90.8 -> 88.5 us); rows of
    // sixteen waves have no registers to hold them that long
    constexpr bool EARLY = sizeof(T) == 4 ? S * W < 128 : S < 8;
    T v[S][V], gm[EARLY ? S : 1][V], bt[EARLY ? S : 1][V];
    RowLoad<T, V, S, W, L, RAGGED> lx(x + c.row * ldx, n, c.tid_in_row);
    if constexpr (EARLY) {
        RowLoad<T, V, S, W, L, RAGGED, false, false> lg(gamma, n, c.tid_in_row), lb(beta, n, c.tid_in_row);
        lx.issue();
        lg.issue();
        lb.issue();
        lx.take(T(-0.0), v);
        lg.take(T(0), gm);
        lb.take(T(0), bt);
    } else {
        lx.issue();
        lx.take(T(-0.0), v);
    }
    const T extent = (T)n;
    const T mean = canon(canon(row_tree_sum<T, V, S, W, R, L>(v, lds, c)) / extent);
    constexpr int SEG = L * W * V;
#pragma unroll
    for (int s = 0; s < S; ++s)
#pragma unroll
        for (int i = 0; i < V; ++i) v[s][i] = canon(v[s][i] - mean);
    const T var = canon(canon(row_tree_sum<T, V, S, W, R, L>(
                            [&](int s, int i) {
                                return s * SEG + c.tid_in_row * V + i < n ? canon(v[s][i] * v[s][i]) : T(-0.0);
                            },
                            lds, c)) /
                        extent);
    const T denom = canon_bits(sqrt(canon(var + eps)));
#pragma unroll
    for (int s = 0; s < S; ++s) {
        if constexpr (EARLY) {
#pragma unroll
            for (int i = 0; i < V; ++i) v[s][i] = canon(canon(v[s][i] / denom) * gm[s][i]);
#pragma unroll
            for (int i = 0; i < V; ++i) v[s][i] = canon(v[s][i] + bt[s][i]);
        } else {
            T gs[1][V], bs[1][V];
            const int off = s * SEG < n ? s * SEG : 0;
            RowLoad<T, V, 1, W, L, RAGGED, false, false> lg(gamma + off, n - off, c.tid_in_row), lb(beta + off, n - off, c.tid_in_row);
            lg.issue();
            lb.issue();
            lg.take(T(0), gs);
            lb.take(T(0), bs);
#pragma unroll
            for (int i = 0; i < V; ++i) v[s][i] = canon(canon(canon(v[s][i] / denom) * gs[0][i]) + bs[0][i]);
            __builtin_amdgcn_sched_barrier(0);
        }
    }
    if (c.live) store_row<T, V, S, W, L, RAGGED>(y + c.row * ldy, n, c.tid_in_row, v);
}

// ---------------------------------------------------------------- dispatch
// Instantiated shapes: (S, W, R) per capacity. V is 16 bytes of T.
enum class RowOp { Softmax, SoftmaxAdjoint, LayerNorm };

struct RowArgs {
    const void *a, *b, *c;
    void *out;
    int64_t rows, n, lda, ldb, ldo;
    int masked;
    double scale;
    int64_t q_len;
    double eps;
};

template <typename T, int V, int S, int W, int R, int L, bool DENSE, bool RAGGED>
void launch_softmax(const RowArgs &a, unsigned grid, hipStream_t st) {
    const dim3 block(64 * W * R);
    // binary64 outside the exact mode: the faithful row
    if constexpr (sizeof(T) == 8) {
        if (!exact_mode()) {
            softmax_kernel<T, V, S, W, R, L, DENSE, RAGGED, true><<<grid, block, 0, st>>>(
                (const T *)a.a, (T *)a.out, a.rows, (int)a.n, a.lda, a.ldo, a.masked, (T)a.scale, a.q_len);
            return;
        }
    }
    softmax_kernel<T, V, S, W, R, L, DENSE, RAGGED><<<grid, block, 0, st>>>(
        (const T *)a.a, (T *)a.out, a.rows, (int)a.n, a.lda, a.ldo, a.masked, (T)a.scale, a.q_len);
}

template <typename T, int V, int S, int W, int R, int L, bool RAGGED>
void launch_pair(RowOp op, const RowArgs &a, unsigned grid, hipStream_t st) {
    const dim3 block(64 * W * R);
    if (op == RowOp::SoftmaxAdjoint)
        softmax_adjoint_kernel<T, V, S, W, R, L, RAGGED><<<grid, block, 0, st>>>(
            (const T *)a.a, (const T *)a.b, (T *)a.out, a.rows, (int)a.n, a.lda, a.ldb, a.ldo);
    else
        layer_norm_kernel<T, V, S, W, R, L, RAGGED><<<grid, block, 0, st>>>(
            (const T *)a.a, (const T *)a.b, (const T *)a.c, (T *)a.out, a.rows, (int)a.n, a.lda, a.ldo, (T)a.eps);
}

template <typename T, int V, int S, int W, int R, int L>
int32_t launch_shape(RowOp op, const RowArgs &a, hipStream_t st) {
    const unsigned grid = grid_for(a.rows, R * (64 / L));
    if (!grid_fits(grid, 64 * W * R)) return set_error(CHELIS_HIP_EUNSUPPORTED, "rows: %lld rows exceed one launch",
                                                       (long long)a.rows);
    const bool ragged = a.n % V != 0;
    if (op == RowOp::Softmax) {
        if (ragged) launch_softmax<T, V, S, W, R, L, false, true>(a, grid, st);
        else if (!a.masked && a.n == (int64_t)S * L * W * V) launch_softmax<T, V, S, W, R, L, true, false>(a, grid, st);
        else launch_softmax<T, V, S, W, R, L, false, false>(a, grid, st);
    } else if (ragged) {
        launch_pair<T, V, S, W, R, L, true>(op, a, grid, st);
    } else {
        launch_pair<T, V, S, W, R, L, false>(op, a, grid, st);
    }
    CHELIS_LAUNCH_CHECK();
    return CHELIS_HIP_OK;
}

// Capacity ladder: CAP = S * 64W * V, smallest power of two >= n.
template <typename T>
int32_t launch_rows(RowOp op, const RowArgs &a) {
    constexpr int V = 16 / sizeof(T);
    hipStream_t st = stream();
    if (!st) return set_error(CHELIS_HIP_EHIP, "no HIP device");
    const int64_t seg1 = 64 * V;  // one wave, one segment
    const int64_t n = a.n;
    // rows of at most half a wave's vectors: four rows per wave, sixteen lanes
    // each (one row per wave leaves most lanes idle: softmax and adjoint of
    // [363636, 33] binary32 206 -> 65 us, [120000, 100] 84 -> 48; layer norm
    // 118 -> 36 and 49 -> 23)
    if (n <= 16 * V) return launch_shape<T, V, 1, 1, 4, 16>(op, a, st);
    if (n <= 32 * V) return launch_shape<T, V, 2, 1, 4, 16>(op, a, st);
    if (n <= seg1) return launch_shape<T, V, 1, 1, 4, 64>(op, a, st);
    if (n <= 2 * seg1) return launch_shape<T, V, 2, 1, 4, 64>(op, a, st);
    // binary32 rows of 513-1024: two waves per row, two segments each
    // (23.4 against 24.2 us for [16384, 1024] with one wave of four
    // segments, same box: the shorter per-wave dependency chain keeps more
    // stores in flight); other rows of this bucket: one row per 64-lane
    // block, so blocks retire independently and the waves of a CU drift
    // apart, one wave's loads overlapping another's arithmetic
    if (n <= 4 * seg1) {
        if constexpr (sizeof(T) == 4) return launch_shape<T, V, 2, 2, 1, 64>(op, a, st);
        if (op == RowOp::LayerNorm) return launch_shape<T, V, 4, 1, 4, 64>(op, a, st);
        return launch_shape<T, V, 4, 1, 1, 64>(op, a, st);
    }
    // binary64 layer norm: two waves (gamma and beta fit beside the row;
    // [23391, 513] 64.4 -> 60.9 us)
    if (n <= 8 * seg1 && sizeof(T) == 8 && op == RowOp::LayerNorm) return launch_shape<T, V, 4, 2, 1, 64>(op, a, st);
    if (n <= 8 * seg1) return launch_shape<T, V, 8, 1, 2, 64>(op, a, st);
    if (n <= 16 * seg1) return launch_shape<T, V, 4, 4, 1, 64>(op, a, st);
    if (n <= 32 * seg1) return launch_shape<T, V, 8, 4, 1, 64>(op, a, st);
    if (n <= 64 * seg1) return launch_shape<T, V, 8, 8, 1, 64>(op, a, st);
    if (n <= 128 * seg1) return launch_shape<T, V, 8, 16, 1, 64>(op, a, st);
    if (n <= 256 * seg1) return launch_shape<T, V, 16, 16, 1, 64>(op, a, st);
    return set_error(CHELIS_HIP_EUNSUPPORTED, "row length %lld exceeds the in-register row capacity %lld",
                     (long long)n, (long long)(256 * seg1));
}

int32_t dispatch(chelis_dtype dt, RowOp op, const RowArgs &a) {
    if (a.rows == 0 || a.n == 0) return CHELIS_HIP_OK;
    return dt == CHELIS_DTYPE_F32 ? launch_rows<float>(op, a) : launch_rows<double>(op, a);
}

int32_t check_rows_pair(const chelis_gpu_tensor *x, const chelis_gpu_tensor *y, RowView *vx, RowView *vy,
                        const char *what) {
    int32_t s;
    if ((s = check_tensor(x, "x")) || (s = check_tensor(y, "y"))) return s;
    if (!is_float(x->dtype) || x->dtype != y->dtype)
        return set_error(CHELIS_HIP_EDOMAIN, "%s: x and y must share an f32 or f64 dtype", what);
    if (!same_shape(x, y)) return set_error(CHELIS_HIP_EDOMAIN, "%s: x and y shapes differ", what);
    if (!row_view(x, vx) || !row_view(y, vy))
        return set_error(CHELIS_HIP_EUNSUPPORTED, "%s: last axis must be contiguous with uniform row stride", what);
    return CHELIS_HIP_OK;
}

// ---------------------------------------------------------------- long rows
// Rows longer than the register capacity (64 * 256 * 16 / sizeof(T): 65 536
// binary32 or 32 768 binary64 values) run as the graph the region stands
// for, one launch per reduction and per elementwise pass, in the same
// primitive order as the row kernels: the reductions take the canonical
// tree over the whole row (aligned segment totals joined pass by pass), the
// chains finalize every primitive, so the results are bit-identical to what
// the row kernels would give (and to the C lane's).
constexpr int64_t kRowCapacityBytes = 64 * 256 * 16;

struct Rows2 {
    int64_t shape[2], strides[2];
    chelis_gpu_tensor t{};
    Rows2(void *data, chelis_dtype dt, int64_t rows, int64_t n, int64_t s_row, int64_t s_col, int64_t cap) {
        shape[0] = rows, shape[1] = n, strides[0] = s_row, strides[1] = s_col;
        t.data = data;
        t.dtype = dt;
        t.rank = 2;
        t.shape = shape;
        t.strides = strides;
        t.count = rows * n;
        t.byte_capacity = cap;
    }
};
struct Vec1 {
    int64_t shape[1], strides[1];
    chelis_gpu_tensor t{};
    Vec1(void *data, chelis_dtype dt, int64_t n) {
        shape[0] = n, strides[0] = 1;
        t.data = data;
        t.dtype = dt;
        t.rank = 1;
        t.shape = shape;
        t.strides = strides;
        t.count = n;
        t.byte_capacity = n * dtype_width(dt);
    }
};

chelis_fused_step fstep(int op, int32_t a0, int32_t a1 = 0, double imm = 0.0) {
    chelis_fused_step st{};
    st.op = (uint8_t)op;
    st.args[0] = a0;
    st.args[1] = a1;
    st.imm = imm;
    return st;
}
constexpr int32_t prv(int32_t k) { return -(k + 1); }
chelis_fused_chain fchain(std::initializer_list<chelis_fused_step> steps) {
    chelis_fused_chain c{};
    for (const chelis_fused_step &st : steps) c.steps[c.n_steps++] = st;
    return c;
}

// Per-row scratch vectors, released (stream-ordered) at scope exit.
struct RowScratch {
    void *p = nullptr;
    size_t bytes = 0;
    explicit RowScratch(size_t b) : p(scratch_alloc(b)), bytes(b) {}
    ~RowScratch() { scratch_free(p, bytes); }
};

int32_t long_softmax(const chelis_gpu_tensor *x, const chelis_gpu_tensor *y, const RowView &vx, const RowView &vy) {
    const chelis_dtype dt = x->dtype;
    const int64_t w = dtype_width(dt), R = vx.rows, n = vx.n;
    RowScratch m(R * w), sum(R * w);
    if (!m.p || !sum.p) return set_error(CHELIS_HIP_EHIP, "softmax: row scratch of %lld bytes", (long long)(2 * R * w));
    const Rows2 X(x->data, dt, R, n, vx.ld, 1, x->byte_capacity), Y(y->data, dt, R, n, vy.ld, 1, y->byte_capacity);
    const Vec1 M(m.p, dt, R), S(sum.p, dt, R);
    const Rows2 Mb(m.p, dt, R, n, 1, 0, R * w), Sb(sum.p, dt, R, n, 1, 0, R * w);
    // m = max over the row; s = tree(exp(x - m)); y = exp(x - m) / s
    const chelis_gpu_tensor *in1[1] = {&X.t};
    if (int32_t st = chelis_hip_reduce(CHELIS_REDUCE_MAX, nullptr, in1, 1, 1, &M.t)) return st;
    const chelis_fused_chain e = fchain({fstep(CHELIS_FUSED_SUB, 0, 1), fstep(CHELIS_FUSED_EXP, prv(0))});
    const chelis_gpu_tensor *in2[2] = {&X.t, &Mb.t};
    if (int32_t st = chelis_hip_reduce(CHELIS_REDUCE_SUM, &e, in2, 2, 1, &S.t)) return st;
    const chelis_fused_chain q = fchain(
        {fstep(CHELIS_FUSED_SUB, 0, 1), fstep(CHELIS_FUSED_EXP, prv(0)), fstep(CHELIS_FUSED_DIV, prv(1), 2)});
    const chelis_gpu_tensor *in3[3] = {&X.t, &Mb.t, &Sb.t};
    return chelis_hip_fused_elementwise(&q, in3, 3, &Y.t);
}

int32_t long_softmax_adjoint(const chelis_gpu_tensor *y, const chelis_gpu_tensor *g, const chelis_gpu_tensor *dx,
                             const RowView &vy, const RowView &vg, const RowView &vd) {
    const chelis_dtype dt = y->dtype;
    const int64_t w = dtype_width(dt), R = vy.rows, n = vy.n;
    RowScratch tot(R * w);
    if (!tot.p) return set_error(CHELIS_HIP_EHIP, "softmax_adjoint: row scratch of %lld bytes", (long long)(R * w));
    const Rows2 Yv(y->data, dt, R, n, vy.ld, 1, y->byte_capacity), G(g->data, dt, R, n, vg.ld, 1, g->byte_capacity),
        D(dx->data, dt, R, n, vd.ld, 1, dx->byte_capacity);
    const Vec1 T(tot.p, dt, R);
    const Rows2 Tb(tot.p, dt, R, n, 1, 0, R * w);
    // t = tree(g * y); dx = y * (g - t)
    const chelis_fused_chain gy = fchain({fstep(CHELIS_FUSED_MUL, 0, 1)});
    const chelis_gpu_tensor *in2[2] = {&G.t, &Yv.t};
    if (int32_t st = chelis_hip_reduce(CHELIS_REDUCE_SUM, &gy, in2, 2, 1, &T.t)) return st;
    const chelis_fused_chain d = fchain({fstep(CHELIS_FUSED_SUB, 1, 2), fstep(CHELIS_FUSED_MUL, 0, prv(0))});
    const chelis_gpu_tensor *in3[3] = {&Yv.t, &G.t, &Tb.t};
    return chelis_hip_fused_elementwise(&d, in3, 3, &D.t);
}

int32_t long_layer_norm(const chelis_gpu_tensor *x, const chelis_gpu_tensor *gamma, const chelis_gpu_tensor *beta,
                        double eps, const chelis_gpu_tensor *y, const RowView &vx, const RowView &vy) {
    const chelis_dtype dt = x->dtype;
    const int64_t w = dtype_width(dt), R = vx.rows, n = vx.n;
    RowScratch tmp(R * w), mean(R * w), den(R * w);
    if (!tmp.p || !mean.p || !den.p)
        return set_error(CHELIS_HIP_EHIP, "layer_norm: row scratch of %lld bytes", (long long)(3 * R * w));
    const Rows2 X(x->data, dt, R, n, vx.ld, 1, x->byte_capacity), Y(y->data, dt, R, n, vy.ld, 1, y->byte_capacity);
    const Vec1 Tv(tmp.p, dt, R), Mv(mean.p, dt, R), Dv(den.p, dt, R);
    const Rows2 Mb(mean.p, dt, R, n, 1, 0, R * w), Db(den.p, dt, R, n, 1, 0, R * w);
    const Rows2 Gb(gamma->data, dt, R, n, 0, 1, gamma->byte_capacity), Bb(beta->data, dt, R, n, 0, 1, beta->byte_capacity);
    const double extent = (double)n;
    // mean = tree(x) / n
    const chelis_gpu_tensor *in1[1] = {&X.t};
    if (int32_t st = chelis_hip_reduce(CHELIS_REDUCE_SUM, nullptr, in1, 1, 1, &Tv.t)) return st;
    const chelis_fused_chain by_n = fchain({fstep(CHELIS_FUSED_CONST, 0, 0, extent), fstep(CHELIS_FUSED_DIV, 0, prv(0))});
    const chelis_gpu_tensor *t1[1] = {&Tv.t};
    if (int32_t st = chelis_hip_fused_elementwise(&by_n, t1, 1, &Mv.t)) return st;
    // var = tree((x - mean)^2) / n; denom = sqrt(var + eps)
    const chelis_fused_chain sq = fchain({fstep(CHELIS_FUSED_SUB, 0, 1), fstep(CHELIS_FUSED_MUL, prv(0), prv(0))});
    const chelis_gpu_tensor *in2[2] = {&X.t, &Mb.t};
    if (int32_t st = chelis_hip_reduce(CHELIS_REDUCE_SUM, &sq, in2, 2, 1, &Tv.t)) return st;
    const chelis_fused_chain dn = fchain({fstep(CHELIS_FUSED_CONST, 0, 0, extent), fstep(CHELIS_FUSED_DIV, 0, prv(0)),
                                          fstep(CHELIS_FUSED_CONST, 0, 0, eps), fstep(CHELIS_FUSED_ADD, prv(1), prv(2)),
                                          fstep(CHELIS_FUSED_SQRT, prv(3))});
    if (int32_t st = chelis_hip_fused_elementwise(&dn, t1, 1, &Dv.t)) return st;
    // y = ((x - mean) / denom) * gamma + beta
    const chelis_fused_chain out = fchain({fstep(CHELIS_FUSED_SUB, 0, 1), fstep(CHELIS_FUSED_DIV, prv(0), 2),
                                           fstep(CHELIS_FUSED_MUL, prv(1), 3), fstep(CHELIS_FUSED_ADD, prv(2), 4)});
    const chelis_gpu_tensor *in5[5] = {&X.t, &Mb.t, &Db.t, &Gb.t, &Bb.t};
    return chelis_hip_fused_elementwise(&out, in5, 5, &Y.t);
}

bool long_rows(chelis_dtype dt, int64_t n) { return n > kRowCapacityBytes / dtype_width(dt); }

}  // namespace
}  // namespace chelis

using namespace chelis;

extern "C" int32_t chelis_hip_softmax(const chelis_gpu_tensor *x, const chelis_gpu_tensor *y) {
    RowView vx, vy;
    if (int32_t s = check_rows_pair(x, y, &vx, &vy, "softmax")) return s;
    if (vx.rows && long_rows(x->dtype, vx.n)) return long_softmax(x, y, vx, vy);
    RowArgs a{x->data, nullptr, nullptr, y->data, vx.rows, vx.n, vx.ld, 0, vy.ld, 0, 1.0, 1, 0.0};
    return dispatch(x->dtype, RowOp::Softmax, a);
}

extern "C" int32_t chelis_hip_scaled_masked_softmax(const chelis_gpu_tensor *x, double scale, int32_t causal,
                                                    const chelis_gpu_tensor *y) {
    RowView vx, vy;
    if (int32_t s = check_rows_pair(x, y, &vx, &vy, "scaled_masked_softmax")) return s;
    if (x->rank < 2) return set_error(CHELIS_HIP_EDOMAIN, "scaled_masked_softmax: scores need rank >= 2");
    const int64_t q_len = x->shape[x->rank - 2];
    if (causal && q_len != vx.n)
        return set_error(CHELIS_HIP_EDOMAIN, "scaled_masked_softmax: causal mask needs square score matrices");
    RowArgs a{x->data, nullptr, nullptr, y->data, vx.rows, vx.n, vx.ld, 0, vy.ld, causal ? 1 : 2, scale, q_len > 0 ? q_len : 1, 0.0};
    return dispatch(x->dtype, RowOp::Softmax, a);
}

extern "C" int32_t chelis_hip_softmax_adjoint(const chelis_gpu_tensor *y, const chelis_gpu_tensor *g,
                                              const chelis_gpu_tensor *dx) {
    RowView vy, vg, vd;
    if (int32_t s = check_rows_pair(y, dx, &vy, &vd, "softmax_adjoint")) return s;
    if (int32_t s = check_tensor(g, "g")) return s;
    if (g->dtype != y->dtype || !same_shape(g, y) || !row_view(g, &vg))
        return set_error(CHELIS_HIP_EDOMAIN, "softmax_adjoint: g must match y");
    if (vy.rows && long_rows(y->dtype, vy.n)) return long_softmax_adjoint(y, g, dx, vy, vg, vd);
    RowArgs a{y->data, g->data, nullptr, dx->data, vy.rows, vy.n, vy.ld, vg.ld, vd.ld, 0, 1.0, 1, 0.0};
    return dispatch(y->dtype, RowOp::SoftmaxAdjoint, a);
}

extern "C" int32_t chelis_hip_layer_norm(const chelis_gpu_tensor *x, const chelis_gpu_tensor *gamma,
                                         const chelis_gpu_tensor *beta, double epsilon,
                                         const chelis_gpu_tensor *y) {
    RowView vx, vy;
    if (int32_t s = check_rows_pair(x, y, &vx, &vy, "layer_norm")) return s;
    int32_t s;
    if ((s = check_tensor(gamma, "gamma")) || (s = check_tensor(beta, "beta"))) return s;
    for (const chelis_gpu_tensor *p : {gamma, beta})
        if (p->dtype != x->dtype || p->rank != 1 || p->shape[0] != vx.n || (vx.n > 1 && p->strides[0] != 1))
            return set_error(CHELIS_HIP_EDOMAIN, "layer_norm: gamma/beta must be contiguous [hidden]");
    if (vx.n == 0) return set_error(CHELIS_HIP_EDOMAIN, "layer_norm: hidden extent must be positive");
    if (vx.rows && long_rows(x->dtype, vx.n)) return long_layer_norm(x, gamma, beta, epsilon, y, vx, vy);
    RowArgs a{x->data, gamma->data, beta->data, y->data, vx.rows, vx.n, vx.ld, 0, vy.ld, 0, 1.0, 1, epsilon};
    return dispatch(x->dtype, RowOp::LayerNorm, a);
}
