// Generic neighbourhood-attention kernels: every rank (as three padded axes),
// dtype (fp32 / fp16 / bf16), kernel size, dilation, stride, causal mask and
// GQA ratio.  Vector-ALU (FMA) kernels with fp32 accumulation (split gathers
// of fp32 operands: fp64).
//
// Work mapping: a "group" of LPQ consecutive lanes owns one query (or one key,
// for the key-centric gradient kernels); each lane owns DPL consecutive head
// dims, so a group covers up to DPL*LPQ dims and dot products finish with a
// log2(LPQ)-step butterfly.  Queries are enumerated (b, o0, o1, o2, h) with the
// head fastest, so one wave reads whole [H, D] token rows.  K/V neighbours are
// read straight from global memory; the overlap between neighbouring windows
// is served by L1/L2 (blocks are remapped so each XCD walks a contiguous
// range).
//
// Bound by instruction issue and the L1 (each neighbour's row is read once per
// query).  What took the time beside the products, and was taken out: 64-bit
// position products and divisions in every step, sums through the LDS
// crossbar, one store per logit, selects on every element for lanes past the
// head dim, and on the key side loads waited for one by one.  us, before ->
// after: fp32 fused 2 x 64 x 64 x 4, dim 64, 11 x 11, dilation 2: 115 / 108 /
// 260 -> 80 / 85 / 152 (forward / dQ / dK dV); bfloat16 2 x 12 x 20 x 24 x 4,
// dim 48, 3 x 5 x 5: 130 / 239 / 262 -> 77 / 156 / 145; fp32 split ops 4 x 45
// x 61 x 4, dim 32, 7 x 7: query side 25 each, key side 66 -> 22-25 and 33.
#include <algorithm>
#include <cstdlib>
#include <type_traits>

#include "na_launch.h"

namespace na {

namespace {

struct QPos {
    int b, h, o0, o1, o2, i0, i1, i2;
};

__device__ __forceinline__ QPos decode_query(const Prob& p, long long qi) {
    QPos r;
    r.h = static_cast<int>(qi % p.Hq);
    long long t = qi / p.Hq;
    r.o2 = static_cast<int>(t % p.ax[2].out); t /= p.ax[2].out;
    r.o1 = static_cast<int>(t % p.ax[1].out); t /= p.ax[1].out;
    r.o0 = static_cast<int>(t % p.ax[0].out);
    r.b = static_cast<int>(t / p.ax[0].out);
    r.i0 = r.o0 * p.ax[0].st;
    r.i1 = r.o1 * p.ax[1].st;
    r.i2 = r.o2 * p.ax[2].st;
    return r;
}

struct KPos {
    int b, h, m0, m1, m2;
};

__device__ __forceinline__ KPos decode_key(const Prob& p, long long ki, int heads) {
    KPos r;
    r.h = static_cast<int>(ki % heads);
    long long t = ki / heads;
    r.m2 = static_cast<int>(t % p.ax[2].len); t /= p.ax[2].len;
    r.m1 = static_cast<int>(t % p.ax[1].len); t /= p.ax[1].len;
    r.m0 = static_cast<int>(t % p.ax[0].len);
    r.b = static_cast<int>(t / p.ax[0].len);
    return r;
}

__device__ __forceinline__ long long group_index(int lpq) {
    const int blk = xcd_block(blockIdx.x, gridDim.x);
    return (static_cast<long long>(blk) * blockDim.x + threadIdx.x) / lpq;
}

// Variable-length problems: lens[b * 3 + a] is sample b's extent on padded
// axis a (stride 1).  It replaces the problem's (maximum) extent in the window
// rule; positions past it are padding.  A sample whose extents fall outside
// [kernel * dilation, maximum], or hit the even-kernel-equal-to-length case,
// is all padding.  False: (i0, i1, i2) is padding for its sample.
__device__ __forceinline__ bool sample_extent(Prob& p, const int* __restrict__ lens, int b, int i0, int i1,
                                              int i2) {
    int L[3];
    bool ok = true;
#pragma unroll
    for (int a = 0; a < 3; ++a) {
        const Axis& A = p.ax[a];
        L[a] = lens[b * 3 + a];
        ok = ok && L[a] >= A.k * A.dil && L[a] <= A.len &&
             !(!A.causal && A.dil == 1 && (A.k % 2) == 0 && A.k == L[a]);
    }
    if (!ok || i0 >= L[0] || i1 >= L[1] || i2 >= L[2]) return false;
#pragma unroll
    for (int a = 0; a < 3; ++a) p.ax[a].len = p.ax[a].out = L[a];
    return true;
}

// Sum over the LPQ consecutive lanes of a group, on the vector ALU: pairs and
// quads by quad permutes, then mirrored halves (each quad, then each half row
// holds one value by then).  Shuffles through the LDS crossbar put two or
// three LDS latencies into every step's chain.
template <int LPQ>
__device__ __forceinline__ float lane_sum(float v) {
    const auto dpp = [&](auto ctrl) {
        return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), decltype(ctrl)::value,
                                                                     0xf, 0xf, true));
    };
    if constexpr (LPQ >= 2) v += dpp(std::integral_constant<int, 0xB1>{});    // quad_perm [1, 0, 3, 2]
    if constexpr (LPQ >= 4) v += dpp(std::integral_constant<int, 0x4E>{});    // quad_perm [2, 3, 0, 1]
    if constexpr (LPQ >= 8) v += dpp(std::integral_constant<int, 0x141>{});   // row_half_mirror
    if constexpr (LPQ >= 16) v += dpp(std::integral_constant<int, 0x140>{});  // row_mirror
    static_assert(LPQ <= 16);
    return v;
}

// The DPL head dims of a group's lane, as registers.  On 16-byte aligned rows
// (`vec`: D is a multiple of DPL) they are 16-byte pieces dealt to the lanes in
// turn, so that every load of a group reads one contiguous run: with a lane's
// dims side by side, the two loads of an fp32 row each spanned the whole row
// and the L1 served them at half its rate.  Other rows: DPL dims side by side,
// one element at a time.
template <typename T, int DPL, int LPQ>
struct Run {
    static constexpr int EPP = 16 / static_cast<int>(sizeof(T)), NW = DPL / EPP;
    static_assert(NW >= 1);
    struct Raw {
        uint4 w[NW];
    };

    static __device__ __forceinline__ int dim(int lane, int w) { return (w * LPQ + lane) * EPP; }

    // Issues the loads.  Pieces past the head dim read the row start; their
    // values meet only `dot`, which drops them, and registers never stored.
    static __device__ __forceinline__ Raw fetch(const T* __restrict__ p, int lane, int D) {
        Raw r;
#pragma unroll
        for (int w = 0; w < NW; ++w) {
            const int d = dim(lane, w);
            r.w[w] = *reinterpret_cast<const uint4*>(p + (d < D ? d : 0));
        }
        return r;
    }
    static __device__ __forceinline__ void unpack(const Raw& r, float (&out)[DPL]) {
        const T* e = reinterpret_cast<const T*>(r.w);
#pragma unroll
        for (int j = 0; j < DPL; ++j) out[j] = to_f(e[j]);
    }
    static __device__ __forceinline__ void load(const T* __restrict__ p, int lane, int D, int vec, float (&out)[DPL]) {
        if (vec) {
            unpack(fetch(p, lane, D), out);
        } else {
#pragma unroll
            for (int j = 0; j < DPL; ++j) out[j] = lane * DPL + j < D ? to_f(p[lane * DPL + j]) : 0.f;
        }
    }
    static __device__ __forceinline__ void store(T* __restrict__ p, int lane, int D, int vec, const float (&in)[DPL]) {
        if (vec) {
#pragma unroll
            for (int w = 0; w < NW; ++w) {
                const int d = dim(lane, w);
                if (d >= D) continue;
                T e[EPP];
#pragma unroll
                for (int j = 0; j < EPP; ++j) e[j] = from_f<T>(in[w * EPP + j]);
                *reinterpret_cast<uint4*>(p + d) = *reinterpret_cast<const uint4*>(e);
            }
        } else {
#pragma unroll
            for (int j = 0; j < DPL; ++j)
                if (lane * DPL + j < D) p[lane * DPL + j] = from_f<T>(in[j]);
        }
    }
    // The lane's part of a . b over D dims.
    static __device__ __forceinline__ float dot(const float (&a)[DPL], const float (&b)[DPL], int lane, int D,
                                                int vec) {
        float sum = 0.f;
#pragma unroll
        for (int w = 0; w < NW; ++w) {
            float s = 0.f;
#pragma unroll
            for (int j = 0; j < EPP; ++j) s = fmaf(a[w * EPP + j], b[w * EPP + j], s);
            sum += !vec || dim(lane, w) < D ? s : 0.f;
        }
        return sum;
    }
    static __device__ __forceinline__ void zero(T* g, int lane, int D, int vec) {
        float z[DPL];
#pragma unroll
        for (int j = 0; j < DPL; ++j) z[j] = 0.f;
        store(g, lane, D, vec, z);
    }
};

// ---------------------------------------------------------------------------
// Pipelined walks.  A group's walk over its neighbours (or attending
// queries) waits on each step's loads; with `walk_*_pipelined` the loads of
// the next U steps are already in flight.  `fetch` issues a step's loads and
// returns the raw registers (no use of the loaded values, so no wait), `use`
// consumes them, in the same order as the plain walk.  fetch(offsets, e) gets
// the neighbour's offsets in the walk's operands and its index, use(step, e,
// valid, u) its registers (u: step within its block of U); masked (causal)
// neighbours load from a clamped position and are skipped by `use`.  Only for
// 16-byte aligned runs and, on the key side, strides of 1 (`VEC` where a kernel
// has an instance of its own for them: their registers would take up to half
// of the waves from the plain walk's callers).  dK/dV, bfloat16, 8 x 8 heads,
// us, one kernel for both walks -> two: 12 x 24 x 24, 3 x 3 x 3, dim 20 1011 ->
// 610; 96 x 96, 3 x 3, stride 2, dim 72 762 -> 463; QK of 130 x 150, 5 x 5, dim
// 44, 2 heads 59 -> 40.  (Forward, AV and dQ keep one: apart they were level,
// or slower for more waves on the same L1.)
// ---------------------------------------------------------------------------
// Steps in flight: about 8 runs of 16 bytes per lane.
template <typename T, int DPL, int RUNS>
constexpr int pipe_depth() {
    constexpr int w = DPL * static_cast<int>(sizeof(T)) / 16 * RUNS;
    return w >= 4 ? 2 : 8 / w;
}

// Keeps what follows in a branch of its own: turned into selects, a new row's
// products or a step's products would be paid on every step.
__device__ __forceinline__ void keep_branch() { asm volatile(""); }

// Offsets of one step in NT operands.  The walks below carry them from step
// to step by additions: computed from the position, each was three 64-bit
// products, which run at a quarter of the rate and took most of the time.
template <int NT>
struct Offsets {
    long long o[NT];
};

template <int U, int NT, class Fetch, class Use>
__device__ __forceinline__ void walk_neighbors_pipelined(const Prob& p, int b, int h, int i0, int i1, int i2, int sp,
                                                         int split, const Lay (&l)[NT], Fetch&& fetch, Use&& use) {
    const Axis &A0 = p.ax[0], &A1 = p.ax[1], &A2 = p.ax[2];
    const int f0 = axis_first(A0, i0), f1 = axis_first(A1, i1), f2 = axis_first(A2, i2);
    const int sa = split_axis(p);
    const int x0 = sa == 0 ? sp : 0, xs = sa == 0 ? split : 1;
    const int y0 = sa == 1 ? sp : 0, ys = sa == 1 ? split : 1;
    const int z0 = sa == 2 ? sp : 0, zs = sa == 2 ? split : 1;
    const int nx = x0 < A0.k ? (A0.k - x0 + xs - 1) / xs : 0;
    const int ny = y0 < A1.k ? (A1.k - y0 + ys - 1) / ys : 0;
    const int nz = z0 < A2.k ? (A2.k - z0 + zs - 1) / zs : 0;
    const int total = nx * ny * nz;
    using P = decltype(fetch(Offsets<NT>{}, 0));
    int x = x0, y = y0, z = z0, e = 0;
    bool ok = false;
    Offsets<NT> row, col, dcol;
#pragma unroll
    for (int t = 0; t < NT; ++t) dcol.o[t] = static_cast<long long>(zs) * A2.dil * l[t].s2;
    const auto start_row = [&] {
        const int j0 = f0 + x * A0.dil, j1 = f1 + y * A1.dil;
        ok = (j0 >= 0) & (j1 >= 0);
        e = (x * A1.k + y) * A2.k;
#pragma unroll
        for (int t = 0; t < NT; ++t) {
            row.o[t] = l[t].at(b, j0 < 0 ? 0 : j0, j1 < 0 ? 0 : j1, 0, h);
            col.o[t] = static_cast<long long>(f2 + z0 * A2.dil) * l[t].s2;
        }
    };
    start_row();
    // blocks of U steps: every fetch of a block is issued before the first
    // use, unconditionally (past the end the cursor stays on the last step),
    // so the compiler waits for each step's loads with the rest in flight
    for (int i = 0; i < total; i += U) {
        P buf[U];
        int eb[U];
        bool okb[U];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int j2 = f2 + z * A2.dil;
            okb[u] = ok & (j2 >= 0);
            eb[u] = e + z;
            Offsets<NT> at;
#pragma unroll
            for (int t = 0; t < NT; ++t) at.o[t] = row.o[t] + (j2 < 0 ? 0 : col.o[t]);
            buf[u] = fetch(at, eb[u]);
            if (i + u + 1 < total) {
                z += zs;
#pragma unroll
                for (int t = 0; t < NT; ++t) col.o[t] += dcol.o[t];
                if (z >= A2.k) {
                    keep_branch();
                    z = z0;
                    if ((y += ys) >= A1.k) {
                        y = y0;
                        x += xs;
                    }
                    start_row();
                }
            }
        }
#pragma unroll
        for (int u = 0; u < U; ++u)
            if (i + u < total) use(buf[u], eb[u], okb[u], u);
    }
}

// The attending queries of key (m0, m1, m2), in for_each_query_split's order:
// fetch(offsets, e) and use(step, e).  Strides of 1 only: positions and
// windows come from the key's residue class.
template <int U, int NT, class Fetch, class Use>
__device__ __forceinline__ void walk_queries_pipelined(const Prob& p, int b, int h, int m0, int m1, int m2, int sp,
                                                       int split, const Lay (&l)[NT], Fetch&& fetch, Use&& use) {
    int lo[3], hi[3], key[3];
    const int m[3] = {m0, m1, m2};
    ClassAxis c[3];
    bool any = true;
#pragma unroll
    for (int a = 0; a < 3; ++a) {
        const Axis& A = p.ax[a];
        key[a] = m[a] / A.dil;
        c[a] = class_axis(A, m[a] - key[a] * A.dil);
        class_span(c[a], key[a], lo[a], hi[a]);
        while (hi[a] >= lo[a] && m[a] + (hi[a] - key[a]) * A.dil >= A.out) --hi[a];
        any = any && lo[a] <= hi[a];
    }
    if (!any) return;
    const Axis &A0 = p.ax[0], &A1 = p.ax[1], &A2 = p.ax[2];
    const int sa = split_axis(p);
    const int s0 = sa == 0 ? split : 1, s1 = sa == 1 ? split : 1, s2 = sa == 2 ? split : 1;
    const int b0 = lo[0] + (sa == 0 ? sp : 0), b1 = lo[1] + (sa == 1 ? sp : 0), b2 = lo[2] + (sa == 2 ? sp : 0);
    const int n0 = hi[0] >= b0 ? (hi[0] - b0) / s0 + 1 : 0, n1 = hi[1] >= b1 ? (hi[1] - b1) / s1 + 1 : 0;
    const int n2 = hi[2] >= b2 ? (hi[2] - b2) / s2 + 1 : 0;
    const int total = n0 * n1 * n2;
    if (total == 0) return;
    using P = decltype(fetch(Offsets<NT>{}, 0));
    int j0 = b0, j1 = b1, j2 = b2, e = 0;
    Offsets<NT> at, dcol;
#pragma unroll
    for (int t = 0; t < NT; ++t) dcol.o[t] = static_cast<long long>(s2) * A2.dil * l[t].s2;
    const auto start_row = [&] {
        e = ((key[0] - class_ws(c[0], j0)) * A1.k + key[1] - class_ws(c[1], j1)) * A2.k + key[2];
#pragma unroll
        for (int t = 0; t < NT; ++t)
            at.o[t] = l[t].at(b, m0 + (j0 - key[0]) * A0.dil, m1 + (j1 - key[1]) * A1.dil,
                              m2 + (b2 - key[2]) * A2.dil, h);
    };
    start_row();
    for (int i = 0; i < total; i += U) {
        P buf[U];
        int eb[U];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            eb[u] = e - class_ws(c[2], j2);
            buf[u] = fetch(at, eb[u]);
            if (i + u + 1 < total) {
                j2 += s2;
#pragma unroll
                for (int t = 0; t < NT; ++t) at.o[t] += dcol.o[t];
                if (j2 > hi[2]) {
                    keep_branch();
                    j2 = b2;
                    if ((j1 += s1) > hi[1]) {
                        j1 = b1;
                        j0 += s0;
                    }
                    start_row();
                }
            }
        }
#pragma unroll
        for (int u = 0; u < U; ++u)
            if (i + u < total) {
                keep_branch();
                use(buf[u], eb[u]);
            }
    }
}

// Instances whose registers sit just past a step of the waves per SIMD (head
// dims above 128) are built for the waves below it.
template <typename T, int DPL>
constexpr bool kWide16 = DPL == 16 && sizeof(T) == 2;
template <typename T, int DPL>
constexpr bool kWide32 = DPL == 16 && sizeof(T) == 4;

__host__ __device__ inline bool unit_strides(const Prob& p) {
    return p.ax[0].st == 1 && p.ax[1].st == 1 && p.ax[2].st == 1;
}

// ---------------------------------------------------------------------------
// Fused forward with online softmax.
// ---------------------------------------------------------------------------
template <typename T, int DPL, int LPQ>
__global__ __launch_bounds__(256, (kWide16<T, DPL> ? 4 : 1)) void k_forward(Prob p, int vec, int split, const int* __restrict__ lens,
                                                 const T* __restrict__ q, Lay lq,
                                                 const T* __restrict__ k, Lay lk,
                                                 const T* __restrict__ v, Lay lv,
                                                 T* __restrict__ out, Lay lo,
                                                 float* __restrict__ lse, Lay ll) {
    const long long qi = group_index(LPQ * split);
    if (qi >= static_cast<long long>(p.B) * p.nout * p.Hq) return;
    using R = Run<T, DPL, LPQ>;
    const int ln = threadIdx.x % LPQ;
    const int sp = (threadIdx.x / LPQ) % split;
    const QPos Q = decode_query(p, qi);
    const int hk = Q.h / p.rep;
    if (lens && !sample_extent(p, lens, Q.b, Q.i0, Q.i1, Q.i2)) {
        if (sp == 0) R::zero(out + lo.at(Q.b, Q.o0, Q.o1, Q.o2, Q.h), ln, p.Dv, vec);
        if (sp == 0 && ln == 0) lse[ll.at(Q.b, Q.o0, Q.o1, Q.o2, Q.h)] = 0.f;
        return;
    }

    float qv[DPL];
    R::load(q + lq.at(Q.b, Q.i0, Q.i1, Q.i2, Q.h), ln, p.Dqk, vec, qv);
    float m = -INFINITY, l = 0.f, acc[DPL];
#pragma unroll
    for (int j = 0; j < DPL; ++j) acc[j] = 0.f;

    const auto step = [&](const float (&kv)[DPL], const float (&vv)[DPL]) {
        const float s = lane_sum<LPQ>(R::dot(qv, kv, ln, p.Dqk, vec)) * p.scale;
        if (s > m) {
            const float c = expf(m - s);
            l *= c;
#pragma unroll
            for (int j = 0; j < DPL; ++j) acc[j] *= c;
            m = s;
        }
        const float e = expf(s - m);
        l += e;
#pragma unroll
        for (int j = 0; j < DPL; ++j) acc[j] = fmaf(e, vv[j], acc[j]);
    };
    if (vec) {
        struct Step {
            typename R::Raw k, v;
        };
        walk_neighbors_pipelined<pipe_depth<T, DPL, 2>(), 2>(
            p, Q.b, hk, Q.i0, Q.i1, Q.i2, sp, split, {lk, lv},
            [&](const Offsets<2>& at, int) {
                return Step{R::fetch(k + at.o[0], ln, p.Dqk), R::fetch(v + at.o[1], ln, p.Dv)};
            },
            [&](const Step& st, int, bool ok, int) {
                if (!ok) return;
                keep_branch();
                float kv[DPL], vv[DPL];
                R::unpack(st.k, kv);
                R::unpack(st.v, vv);
                step(kv, vv);
            });
    } else {
        for_each_neighbor_split(p, Q.i0, Q.i1, Q.i2, sp, split, [&](int j0, int j1, int j2, int, bool ok) {
            if (!ok) return;
            float kv[DPL], vv[DPL];
            R::load(k + lk.at(Q.b, j0, j1, j2, hk), ln, p.Dqk, vec, kv);
            R::load(v + lv.at(Q.b, j0, j1, j2, hk), ln, p.Dv, vec, vv);
            step(kv, vv);
        });
    }

    if (split > 1) {
        // merge the groups' softmax states (a group may have seen no neighbour)
        const float mall = split_max<LPQ>(m, split);
        const float c = m == -INFINITY ? 0.f : expf(m - mall);
        l = split_sum<LPQ>(l * c, split);
#pragma unroll
        for (int j = 0; j < DPL; ++j) acc[j] = split_sum<LPQ>(acc[j] * c, split);
        m = mall;
    }
#pragma unroll
    for (int j = 0; j < DPL; ++j) acc[j] = acc[j] / l;
    if (sp == 0) R::store(out + lo.at(Q.b, Q.o0, Q.o1, Q.o2, Q.h), ln, p.Dv, vec, acc);
    if (sp == 0 && ln == 0) lse[ll.at(Q.b, Q.o0, Q.o1, Q.o2, Q.h)] = m + logf(l);
}

// Row elements of a query, one per step, collected so that the group's lanes
// store up to LPQ of them at once (of one block of U steps).
template <typename T, int LPQ, int U>
struct RowPut {
    T* row;
    int at = -1;
    T val{};
    __device__ __forceinline__ void add(int lane, int u, int e, T v) {
        if (u % LPQ == lane) {
            at = e;
            val = v;
        }
        if (u % LPQ == LPQ - 1 || u == U - 1) flush();
    }
    __device__ __forceinline__ void flush() {
        if (at >= 0) row[at] = val;
        at = -1;
    }
};

// ---------------------------------------------------------------------------
// Split QK: logits per neighbour (unscaled unless has_scale), -inf if invalid.
// ---------------------------------------------------------------------------
template <typename T, int DPL, int LPQ, bool VEC>
__global__ __launch_bounds__(256) void k_qk(Prob p, int split,
                                            const T* __restrict__ q, Lay lq,
                                            const T* __restrict__ k, Lay lk,
                                            T* __restrict__ attn, Lay la) {
    const long long qi = group_index(LPQ * split);
    if (qi >= static_cast<long long>(p.B) * p.nout * p.Hq) return;
    using R = Run<T, DPL, LPQ>;
    constexpr int vec = VEC;
    const int ln = threadIdx.x % LPQ;
    const int sp = (threadIdx.x / LPQ) % split;
    const QPos Q = decode_query(p, qi);
    float qv[DPL];
    R::load(q + lq.at(Q.b, Q.i0, Q.i1, Q.i2, Q.h), ln, p.Dqk, vec, qv);
    T* row = attn + la.at(Q.b, Q.o0, Q.o1, Q.o2, Q.h);
    if constexpr (VEC) {
        RowPut<T, LPQ, pipe_depth<T, DPL, 1>()> put{row};
        walk_neighbors_pipelined<pipe_depth<T, DPL, 1>(), 1>(
            p, Q.b, Q.h, Q.i0, Q.i1, Q.i2, sp, split, {lk},
            [&](const Offsets<1>& at, int) { return R::fetch(k + at.o[0], ln, p.Dqk); },
            [&](const typename R::Raw& r, int e, bool ok, int u) {
                float kv[DPL];
                R::unpack(r, kv);
                const float acc = R::dot(qv, kv, ln, p.Dqk, vec);
                float s = ok ? lane_sum<LPQ>(acc) : -INFINITY;
                if (p.has_scale) s *= p.scale;
                put.add(ln, u, e, from_f<T>(s));
            });
        put.flush();
        return;
    }
    for_each_neighbor_split(p, Q.i0, Q.i1, Q.i2, sp, split, [&](int j0, int j1, int j2, int e, bool ok) {
        float s = -INFINITY;
        if (ok) {
            float kv[DPL];
            R::load(k + lk.at(Q.b, j0, j1, j2, Q.h), ln, p.Dqk, vec, kv);
            const float acc = R::dot(qv, kv, ln, p.Dqk, vec);
            s = lane_sum<LPQ>(acc);
        }
        if (p.has_scale) s *= p.scale;
        if (ln == 0) row[e] = from_f<T>(s);
    });
}

// Accumulator of the split ops' gathers (AV output, dq, dk, dv): a sum over
// a whole window (or over every query attending a key), hundreds of products
// in 3-D.  For fp32 operands it runs in double -- a product of two fp32
// values is exact there, so the result is the correctly rounded sum, and no
// summation-order noise of fp32 (which passes 1e-5 relative at 3-D window
// sizes) reaches the output; 16-bit operands keep fp32 accumulators.
template <typename T>
struct GatherAcc {
    using type = float;
};
template <>
struct GatherAcc<float> {
    using type = double;
};

template <typename A>
__device__ __forceinline__ A gather_fma(float a, float b, A acc) {
    return static_cast<A>(a) * static_cast<A>(b) + acc;
}

// The groups' sum of acc (times mul) rounded to float.
template <int LPQ, typename A, int DPL>
__device__ __forceinline__ void gather_out(const A (&acc)[DPL], int split, float mul, float (&out)[DPL]) {
#pragma unroll
    for (int j = 0; j < DPL; ++j) {
        A v = acc[j];
        for (int m = split >> 1; m >= 1; m >>= 1) v += __shfl_xor(v, m * LPQ);
        out[j] = static_cast<float>(v * static_cast<A>(mul));
    }
}

// ---------------------------------------------------------------------------
// Split AV: out = sum_valid attn * v.
// ---------------------------------------------------------------------------
template <typename T, int DPL, int LPQ>
__global__ __launch_bounds__(256) void k_av(Prob p, int vec, int split,
                                            const T* __restrict__ attn, Lay la,
                                            const T* __restrict__ v, Lay lv,
                                            T* __restrict__ out, Lay lo) {
    const long long qi = group_index(LPQ * split);
    if (qi >= static_cast<long long>(p.B) * p.nout * p.Hq) return;
    using R = Run<T, DPL, LPQ>;
    const int ln = threadIdx.x % LPQ;
    const int sp = (threadIdx.x / LPQ) % split;
    const QPos Q = decode_query(p, qi);
    const T* row = attn + la.at(Q.b, Q.o0, Q.o1, Q.o2, Q.h);
    using A = typename GatherAcc<T>::type;
    A acc[DPL];
#pragma unroll
    for (int j = 0; j < DPL; ++j) acc[j] = 0;
    if (vec) {
        struct Step {
            typename R::Raw v;
            T a;
        };
        walk_neighbors_pipelined<pipe_depth<T, DPL, 1>(), 1>(
            p, Q.b, Q.h, Q.i0, Q.i1, Q.i2, sp, split, {lv},
            [&](const Offsets<1>& at, int e) {
                return Step{R::fetch(v + at.o[0], ln, p.Dv), row[e]};
            },
            [&](const Step& st, int, bool ok, int) {
                if (!ok) return;
                keep_branch();
                const float a = to_f(st.a);
                float vv[DPL];
                R::unpack(st.v, vv);
#pragma unroll
                for (int j = 0; j < DPL; ++j) acc[j] = gather_fma(a, vv[j], acc[j]);
            });
    } else {
        for_each_neighbor_split(p, Q.i0, Q.i1, Q.i2, sp, split, [&](int j0, int j1, int j2, int e, bool ok) {
            if (!ok) return;
            const float a = to_f(row[e]);
            float vv[DPL];
            R::load(v + lv.at(Q.b, j0, j1, j2, Q.h), ln, p.Dv, vec, vv);
#pragma unroll
            for (int j = 0; j < DPL; ++j) acc[j] = gather_fma(a, vv[j], acc[j]);
        });
    }
    float res[DPL];
    gather_out<LPQ>(acc, split, 1.f, res);
    if (sp == 0) R::store(out + lo.at(Q.b, Q.o0, Q.o1, Q.o2, Q.h), ln, p.Dv, vec, res);
}

// ---------------------------------------------------------------------------
// Fused backward, query side: delta = dO.O - dlse, and
// dq = scale * sum_k P (dO.v_k - delta) k_k with P = exp(scale q.k - lse).
// ---------------------------------------------------------------------------
template <typename T, int DPL, int LPQ>
__global__ __launch_bounds__(256, (kWide32<T, DPL> ? 3 : 1)) void k_bwd_dq(Prob p, int vec, int split, const int* __restrict__ lens,
                                                const T* __restrict__ q, Lay lq,
                                                const T* __restrict__ k, Lay lk,
                                                const T* __restrict__ v, Lay lv,
                                                const T* __restrict__ o, Lay lo,
                                                const T* __restrict__ dout, Lay ldo,
                                                const float* __restrict__ lse, Lay ll,
                                                const float* __restrict__ dlse, Lay ldl,
                                                T* __restrict__ dq, Lay ldq,
                                                float* __restrict__ delta, Lay lde) {
    const long long qi = group_index(LPQ * split);
    if (qi >= static_cast<long long>(p.B) * p.nout * p.Hq) return;
    using R = Run<T, DPL, LPQ>;
    const int ln = threadIdx.x % LPQ;
    const int sp = (threadIdx.x / LPQ) % split;
    const QPos Q = decode_query(p, qi);
    const int hk = Q.h / p.rep;
    if (lens && !sample_extent(p, lens, Q.b, Q.i0, Q.i1, Q.i2)) {
        if (sp == 0) R::zero(dq + ldq.at(Q.b, Q.i0, Q.i1, Q.i2, Q.h), ln, p.Dqk, vec);
        if (sp == 0 && ln == 0) delta[lde.at(Q.b, Q.o0, Q.o1, Q.o2, Q.h)] = 0.f;
        return;
    }

    float qv[DPL], dov[DPL];
    R::load(q + lq.at(Q.b, Q.i0, Q.i1, Q.i2, Q.h), ln, p.Dqk, vec, qv);
    R::load(dout + ldo.at(Q.b, Q.o0, Q.o1, Q.o2, Q.h), ln, p.Dv, vec, dov);
    const float L = lse[ll.at(Q.b, Q.o0, Q.o1, Q.o2, Q.h)];
    // use(key, value) for each valid neighbour
    const auto walk = [&](auto&& use) {
        if (vec) {
            struct Step {
                typename R::Raw k, v;
            };
            walk_neighbors_pipelined<pipe_depth<T, DPL, 2>(), 2>(
                p, Q.b, hk, Q.i0, Q.i1, Q.i2, sp, split, {lk, lv},
                [&](const Offsets<2>& at, int) {
                    return Step{R::fetch(k + at.o[0], ln, p.Dqk), R::fetch(v + at.o[1], ln, p.Dv)};
                },
                [&](const Step& st, int, bool ok, int) {
                    if (!ok) return;
                    keep_branch();
                    float kv[DPL], vv[DPL];
                    R::unpack(st.k, kv);
                    R::unpack(st.v, vv);
                    use(kv, vv);
                });
        } else {
            for_each_neighbor_split(p, Q.i0, Q.i1, Q.i2, sp, split, [&](int j0, int j1, int j2, int, bool ok) {
                if (!ok) return;
                float kv[DPL], vv[DPL];
                R::load(k + lk.at(Q.b, j0, j1, j2, hk), ln, p.Dqk, vec, kv);
                R::load(v + lv.at(Q.b, j0, j1, j2, hk), ln, p.Dv, vec, vv);
                use(kv, vv);
            });
        }
    };
    float di = 0.f;
    if constexpr (sizeof(T) == 4) {
        // delta = dO . O: exact enough when O was stored in fp32.
        float ov[DPL];
        R::load(o + lo.at(Q.b, Q.o0, Q.o1, Q.o2, Q.h), ln, p.Dv, vec, ov);
        di = lane_sum<LPQ>(R::dot(dov, ov, ln, p.Dv, vec));
    } else {
        // 16-bit O carries ~2^-9 relative rounding; use the equivalent
        // delta = sum_k P_k (dO . v_k) from an extra pass instead.
        walk([&](const float (&kv)[DPL], const float (&vv)[DPL]) {
            const float s = lane_sum<LPQ>(R::dot(qv, kv, ln, p.Dqk, vec)) * p.scale;
            const float dp = lane_sum<LPQ>(R::dot(dov, vv, ln, p.Dv, vec));
            di = fmaf(expf(s - L), dp, di);
        });
        di = split_sum<LPQ>(di, split);
    }
    if (dlse) di -= dlse[ldl.at(Q.b, Q.o0, Q.o1, Q.o2, Q.h)];
    if (sp == 0 && ln == 0) delta[lde.at(Q.b, Q.o0, Q.o1, Q.o2, Q.h)] = di;

    float acc[DPL];
#pragma unroll
    for (int j = 0; j < DPL; ++j) acc[j] = 0.f;
    const auto step = [&](const float (&kv)[DPL], const float (&vv)[DPL]) {
        const float s = lane_sum<LPQ>(R::dot(qv, kv, ln, p.Dqk, vec)) * p.scale;
        const float dp = lane_sum<LPQ>(R::dot(dov, vv, ln, p.Dv, vec));
        const float ds = expf(s - L) * (dp - di);
#pragma unroll
        for (int j = 0; j < DPL; ++j) acc[j] = fmaf(ds, kv[j], acc[j]);
    };
    walk(step);
#pragma unroll
    for (int j = 0; j < DPL; ++j) acc[j] = split_sum<LPQ>(acc[j], split) * p.scale;
    if (sp == 0) R::store(dq + ldq.at(Q.b, Q.i0, Q.i1, Q.i2, Q.h), ln, p.Dqk, vec, acc);
}

// ---------------------------------------------------------------------------
// Fused backward, key side: for each key/value position and kv head, gather
// over the queries (of every q head in the GQA group) whose windows hold it:
// dv = sum P dO,  dk = scale * sum P (dO.v - delta) q.  Deterministic (no
// atomics); recomputes P from q, k and lse.
// ---------------------------------------------------------------------------
template <typename T, int DPL, int LPQ, bool VEC>
__global__ __launch_bounds__(256, (kWide32<T, DPL> ? 2 : 1)) void k_bwd_dkdv(Prob p, int aligned, int split, const int* __restrict__ lens,
                                                  const T* __restrict__ q, Lay lq,
                                                  const T* __restrict__ k, Lay lk,
                                                  const T* __restrict__ v, Lay lv,
                                                  const T* __restrict__ dout, Lay ldo,
                                                  const float* __restrict__ lse, Lay ll,
                                                  const float* __restrict__ delta, Lay lde,
                                                  T* __restrict__ dk, Lay ldk,
                                                  T* __restrict__ dv, Lay ldv) {
    const long long ki = group_index(LPQ * split);
    if (ki >= static_cast<long long>(p.B) * p.nkey * p.Hkv) return;
    using R = Run<T, DPL, LPQ>;
    const int vec = VEC ? 1 : aligned;
    const int ln = threadIdx.x % LPQ;
    const int sp = (threadIdx.x / LPQ) % split;
    const KPos K = decode_key(p, ki, p.Hkv);
    if (lens && !sample_extent(p, lens, K.b, K.m0, K.m1, K.m2)) {
        if (sp == 0) R::zero(dk + ldk.at(K.b, K.m0, K.m1, K.m2, K.h), ln, p.Dqk, vec);
        if (sp == 0) R::zero(dv + ldv.at(K.b, K.m0, K.m1, K.m2, K.h), ln, p.Dv, vec);
        return;
    }

    float kv[DPL], vv[DPL], gk[DPL], gv[DPL];
    R::load(k + lk.at(K.b, K.m0, K.m1, K.m2, K.h), ln, p.Dqk, vec, kv);
    R::load(v + lv.at(K.b, K.m0, K.m1, K.m2, K.h), ln, p.Dv, vec, vv);
#pragma unroll
    for (int j = 0; j < DPL; ++j) { gk[j] = 0.f; gv[j] = 0.f; }

    const auto add = [&](const float (&qv)[DPL], const float (&dov)[DPL], float L, float di) {
        const float s = lane_sum<LPQ>(R::dot(qv, kv, ln, p.Dqk, vec)) * p.scale;
        const float dp = lane_sum<LPQ>(R::dot(dov, vv, ln, p.Dv, vec));
        const float pr = expf(s - L);
        const float ds = pr * (dp - di);
#pragma unroll
        for (int j = 0; j < DPL; ++j) {
            gv[j] = fmaf(pr, dov[j], gv[j]);
            gk[j] = fmaf(ds, qv[j], gk[j]);
        }
    };
    if constexpr (VEC) {
        struct Step {
            typename R::Raw q, g;
            float L, di;
        };
        for (int r = 0; r < p.rep; ++r) {
            walk_queries_pipelined<pipe_depth<T, DPL, 2>(), 4>(
                p, K.b, K.h * p.rep + r, K.m0, K.m1, K.m2, sp, split, {lq, ldo, ll, lde},
                [&](const Offsets<4>& at, int) {
                    return Step{R::fetch(q + at.o[0], ln, p.Dqk), R::fetch(dout + at.o[1], ln, p.Dv),
                                lse[at.o[2]], delta[at.o[3]]};
                },
                [&](const Step& st, int) {
                    float qv[DPL], dov[DPL];
                    R::unpack(st.q, qv);
                    R::unpack(st.g, dov);
                    add(qv, dov, st.L, st.di);
                });
        }
    } else {
        for_each_query_split(p, K.m0, K.m1, K.m2, sp, split, [&](int o0, int o1, int o2, int i0, int i1, int i2, int) {
            for (int r = 0; r < p.rep; ++r) {
                const int h = K.h * p.rep + r;
                float qv[DPL], dov[DPL];
                R::load(q + lq.at(K.b, i0, i1, i2, h), ln, p.Dqk, vec, qv);
                R::load(dout + ldo.at(K.b, o0, o1, o2, h), ln, p.Dv, vec, dov);
                add(qv, dov, lse[ll.at(K.b, o0, o1, o2, h)], delta[lde.at(K.b, o0, o1, o2, h)]);
            }
        });
    }
#pragma unroll
    for (int j = 0; j < DPL; ++j) {
        gk[j] = split_sum<LPQ>(gk[j], split) * p.scale;
        gv[j] = split_sum<LPQ>(gv[j], split);
    }
    if (sp == 0) R::store(dk + ldk.at(K.b, K.m0, K.m1, K.m2, K.h), ln, p.Dqk, vec, gk);
    if (sp == 0) R::store(dv + ldv.at(K.b, K.m0, K.m1, K.m2, K.h), ln, p.Dv, vec, gv);
}

// ---------------------------------------------------------------------------
// Split QK backward.  dq (query side) and dk (key side); grad of an invalid
// entry is zero, and both carry the logit scale when has_scale.
// ---------------------------------------------------------------------------
template <typename T, int DPL, int LPQ>
__global__ __launch_bounds__(256) void k_qk_bwd_q(Prob p, int vec, int split,
                                                  const T* __restrict__ da, Lay lda,
                                                  const T* __restrict__ k, Lay lk,
                                                  T* __restrict__ dq, Lay ldq) {
    const long long qi = group_index(LPQ * split);
    if (qi >= static_cast<long long>(p.B) * p.nout * p.Hq) return;
    using R = Run<T, DPL, LPQ>;
    const int ln = threadIdx.x % LPQ;
    const int sp = (threadIdx.x / LPQ) % split;
    const QPos Q = decode_query(p, qi);
    const T* row = da + lda.at(Q.b, Q.o0, Q.o1, Q.o2, Q.h);
    using A = typename GatherAcc<T>::type;
    A acc[DPL];
#pragma unroll
    for (int j = 0; j < DPL; ++j) acc[j] = 0;
    if (vec) {
        struct Step {
            typename R::Raw k;
            T g;
        };
        walk_neighbors_pipelined<pipe_depth<T, DPL, 1>(), 1>(
            p, Q.b, Q.h, Q.i0, Q.i1, Q.i2, sp, split, {lk},
            [&](const Offsets<1>& at, int e) {
                return Step{R::fetch(k + at.o[0], ln, p.Dqk), row[e]};
            },
            [&](const Step& st, int, bool ok, int) {
                if (!ok) return;
                keep_branch();
                const float g = to_f(st.g);
                float kv[DPL];
                R::unpack(st.k, kv);
#pragma unroll
                for (int j = 0; j < DPL; ++j) acc[j] = gather_fma(g, kv[j], acc[j]);
            });
    } else {
        for_each_neighbor_split(p, Q.i0, Q.i1, Q.i2, sp, split, [&](int j0, int j1, int j2, int e, bool ok) {
            if (!ok) return;
            const float g = to_f(row[e]);
            float kv[DPL];
            R::load(k + lk.at(Q.b, j0, j1, j2, Q.h), ln, p.Dqk, vec, kv);
#pragma unroll
            for (int j = 0; j < DPL; ++j) acc[j] = gather_fma(g, kv[j], acc[j]);
        });
    }
    float res[DPL];
    gather_out<LPQ>(acc, split, p.has_scale ? p.scale : 1.f, res);
    if (sp == 0) R::store(dq + ldq.at(Q.b, Q.i0, Q.i1, Q.i2, Q.h), ln, p.Dqk, vec, res);
}

template <typename T, int DPL, int LPQ, bool VEC>
__global__ __launch_bounds__(256) void k_qk_bwd_k(Prob p, int aligned, int split,
                                                  const T* __restrict__ da, Lay lda,
                                                  const T* __restrict__ q, Lay lq,
                                                  T* __restrict__ dk, Lay ldk) {
    const long long ki = group_index(LPQ * split);
    if (ki >= static_cast<long long>(p.B) * p.nkey * p.Hkv) return;
    using R = Run<T, DPL, LPQ>;
    const int vec = VEC ? 1 : aligned;
    const int ln = threadIdx.x % LPQ;
    const int sp = (threadIdx.x / LPQ) % split;
    const KPos K = decode_key(p, ki, p.Hkv);
    using A = typename GatherAcc<T>::type;
    A acc[DPL];
#pragma unroll
    for (int j = 0; j < DPL; ++j) acc[j] = 0;
    if constexpr (VEC) {
        struct Step {
            typename R::Raw x;
            T w;
        };
        walk_queries_pipelined<pipe_depth<T, DPL, 1>(), 2>(
            p, K.b, K.h, K.m0, K.m1, K.m2, sp, split, {lq, lda},
            [&](const Offsets<2>& at, int e) {
                return Step{R::fetch(q + at.o[0], ln, p.Dqk), da[at.o[1] + e]};
            },
            [&](const Step& st, int) {
                const float w = to_f(st.w);
                float xv[DPL];
                R::unpack(st.x, xv);
#pragma unroll
                for (int j = 0; j < DPL; ++j) acc[j] = gather_fma(w, xv[j], acc[j]);
            });
    } else {
        for_each_query_split(p, K.m0, K.m1, K.m2, sp, split, [&](int o0, int o1, int o2, int i0, int i1, int i2, int e) {
            const float g = to_f(da[lda.at(K.b, o0, o1, o2, K.h) + e]);
            float qv[DPL];
            R::load(q + lq.at(K.b, i0, i1, i2, K.h), ln, p.Dqk, vec, qv);
#pragma unroll
            for (int j = 0; j < DPL; ++j) acc[j] = gather_fma(g, qv[j], acc[j]);
        });
    }
    float res[DPL];
    gather_out<LPQ>(acc, split, p.has_scale ? p.scale : 1.f, res);
    if (sp == 0) R::store(dk + ldk.at(K.b, K.m0, K.m1, K.m2, K.h), ln, p.Dqk, vec, res);
}

// ---------------------------------------------------------------------------
// Split AV backward: dattn (query side) and dv (key side).
// ---------------------------------------------------------------------------
template <typename T, int DPL, int LPQ, bool VEC>
__global__ __launch_bounds__(256) void k_av_bwd_a(Prob p, int split,
                                                  const T* __restrict__ dout, Lay ldo,
                                                  const T* __restrict__ v, Lay lv,
                                                  T* __restrict__ da, Lay lda) {
    const long long qi = group_index(LPQ * split);
    if (qi >= static_cast<long long>(p.B) * p.nout * p.Hq) return;
    using R = Run<T, DPL, LPQ>;
    constexpr int vec = VEC;
    const int ln = threadIdx.x % LPQ;
    const int sp = (threadIdx.x / LPQ) % split;
    const QPos Q = decode_query(p, qi);
    float dov[DPL];
    R::load(dout + ldo.at(Q.b, Q.o0, Q.o1, Q.o2, Q.h), ln, p.Dv, vec, dov);
    T* row = da + lda.at(Q.b, Q.o0, Q.o1, Q.o2, Q.h);
    if constexpr (VEC) {
        RowPut<T, LPQ, pipe_depth<T, DPL, 1>()> put{row};
        walk_neighbors_pipelined<pipe_depth<T, DPL, 1>(), 1>(
            p, Q.b, Q.h, Q.i0, Q.i1, Q.i2, sp, split, {lv},
            [&](const Offsets<1>& at, int) { return R::fetch(v + at.o[0], ln, p.Dv); },
            [&](const typename R::Raw& r, int e, bool ok, int u) {
                float vv[DPL];
                R::unpack(r, vv);
                const float acc = R::dot(dov, vv, ln, p.Dv, vec);
                const float g = ok ? lane_sum<LPQ>(acc) : 0.f;
                put.add(ln, u, e, from_f<T>(g));
            });
        put.flush();
        return;
    }
    for_each_neighbor_split(p, Q.i0, Q.i1, Q.i2, sp, split, [&](int j0, int j1, int j2, int e, bool ok) {
        float g = 0.f;
        if (ok) {
            float vv[DPL];
            R::load(v + lv.at(Q.b, j0, j1, j2, Q.h), ln, p.Dv, vec, vv);
            const float acc = R::dot(dov, vv, ln, p.Dv, vec);
            g = lane_sum<LPQ>(acc);
        }
        if (ln == 0) row[e] = from_f<T>(g);
    });
}

template <typename T, int DPL, int LPQ, bool VEC>
__global__ __launch_bounds__(256) void k_av_bwd_v(Prob p, int aligned, int split,
                                                  const T* __restrict__ dout, Lay ldo,
                                                  const T* __restrict__ attn, Lay la,
                                                  T* __restrict__ dv, Lay ldv) {
    const long long ki = group_index(LPQ * split);
    if (ki >= static_cast<long long>(p.B) * p.nkey * p.Hkv) return;
    using R = Run<T, DPL, LPQ>;
    const int vec = VEC ? 1 : aligned;
    const int ln = threadIdx.x % LPQ;
    const int sp = (threadIdx.x / LPQ) % split;
    const KPos K = decode_key(p, ki, p.Hkv);
    using A = typename GatherAcc<T>::type;
    A acc[DPL];
#pragma unroll
    for (int j = 0; j < DPL; ++j) acc[j] = 0;
    if constexpr (VEC) {
        struct Step {
            typename R::Raw x;
            T w;
        };
        walk_queries_pipelined<pipe_depth<T, DPL, 1>(), 2>(
            p, K.b, K.h, K.m0, K.m1, K.m2, sp, split, {ldo, la},
            [&](const Offsets<2>& at, int e) {
                return Step{R::fetch(dout + at.o[0], ln, p.Dv), attn[at.o[1] + e]};
            },
            [&](const Step& st, int) {
                const float w = to_f(st.w);
                float xv[DPL];
                R::unpack(st.x, xv);
#pragma unroll
                for (int j = 0; j < DPL; ++j) acc[j] = gather_fma(w, xv[j], acc[j]);
            });
    } else {
        for_each_query_split(p, K.m0, K.m1, K.m2, sp, split, [&](int o0, int o1, int o2, int, int, int, int e) {
            const float a = to_f(attn[la.at(K.b, o0, o1, o2, K.h) + e]);
            float dov[DPL];
            R::load(dout + ldo.at(K.b, o0, o1, o2, K.h), ln, p.Dv, vec, dov);
#pragma unroll
            for (int j = 0; j < DPL; ++j) acc[j] = gather_fma(a, dov[j], acc[j]);
        });
    }
    float res[DPL];
    gather_out<LPQ>(acc, split, 1.f, res);
    if (sp == 0) R::store(dv + ldv.at(K.b, K.m0, K.m1, K.m2, K.h), ln, p.Dv, vec, res);
}

// ---------------------------------------------------------------------------
// Neighbourhood map export (one thread per (query position, neighbour)).
// ---------------------------------------------------------------------------
__global__ __launch_bounds__(256) void k_map(Prob p, int64_t* __restrict__ flat, uint8_t* __restrict__ valid) {
    const long long t = static_cast<long long>(blockIdx.x) * blockDim.x + threadIdx.x;
    if (t >= static_cast<long long>(p.nout) * p.kv) return;
    const int e = static_cast<int>(t % p.kv);
    long long oq = t / p.kv;
    const int o2 = static_cast<int>(oq % p.ax[2].out); oq /= p.ax[2].out;
    const int o1 = static_cast<int>(oq % p.ax[1].out); oq /= p.ax[1].out;
    const int o0 = static_cast<int>(oq);
    const int z = e % p.ax[2].k, y = (e / p.ax[2].k) % p.ax[1].k, x = e / (p.ax[2].k * p.ax[1].k);
    const int os[3] = {o0, o1, o2}, ks[3] = {x, y, z};
    long long f = 0;
    bool ok = true;
    for (int a = 0; a < 3; ++a) {
        const Axis& A = p.ax[a];
        const int i = os[a] * A.st;
        int j = axis_first(A, i) + ks[a] * A.dil;
        if (A.causal) {
            ok = ok && (j >= 0) && (j <= i);
            j = j < 0 ? 0 : (j > A.len - 1 ? A.len - 1 : j);
        }
        f = f * A.len + j;
    }
    flat[t] = f;
    valid[t] = ok ? 1 : 0;
}

}  // namespace

// ---------------------------------------------------------------------------
// Launchers.
// ---------------------------------------------------------------------------

namespace {

// Lanes-per-query / dims-per-lane configurations, chosen from the head dim.
template <template <typename, int, int> class Launch, typename T, typename... Args>
hipError_t by_dim(int D, Args&&... args) {
    if (D <= 8) return Launch<T, 8, 1>::run(args...);
    if (D <= 16) return Launch<T, 8, 2>::run(args...);
    if (D <= 32) return Launch<T, 8, 4>::run(args...);
    if (D <= 64) return Launch<T, 8, 8>::run(args...);
    if (D <= 128) return Launch<T, 8, 16>::run(args...);
    return Launch<T, 16, 16>::run(args...);
}

template <template <typename, int, int> class Launch, typename... Args>
hipError_t by_type(int dtype, int D, Args&&... args) {
    switch (dtype) {
        case NATTEN_F32: return by_dim<Launch, float>(D, args...);
        case NATTEN_F16: return by_dim<Launch, f16>(D, args...);
        default: return by_dim<Launch, bf16>(D, args...);
    }
}

inline unsigned grid_for(long long groups, int lpq) {
    const long long threads = groups * lpq;
    return static_cast<unsigned>((threads + 255) / 256);
}

// Lane groups per query (key).  Each group walks its neighbours (attending
// queries) one after another, so a small problem (few groups) is bound by that
// chain.  Splitting the walk over up to 8 groups shortens it, until the launch
// fills a 256-CU device: past that the walks are bound by issue and L1 and the
// groups' own overhead shows.  Over 3500 timed kernels (1-D to 3-D, head dims 10
// to 256, splits of 1 to 8 forced) the best split reaches about 1.5 waves per
// SIMD on the query side, 2 for the key side's pipelined walk and 3 for its
// plain one, which waits on every step's loads; a group of a pipelined walk
// needs a block of loads (8 neighbours) of its own.  By this rule they take 0.5
// to 3.4 % more than at their best split (at 1.5 waves throughout 1.2 to 6.4 %;
// dK/dV, bfloat16, 8 x 6 x 12 x 14 x 8, 3 x 5 x 5, dim 12: 350 -> 213 us, AV of
// 2 x 300 x 4, 7, dim 72: 7.5 -> 5.7).  Groups stay within one wave (lpq * split
// <= 64) and never outnumber the split axis's kernel positions.
// NATTEN_HIP_SPLIT=n fixes it (tuning).
inline int choose_split(const Prob& p, long long groups, int lpq, bool piped, bool key) {
    static const int forced = [] {
        const char* e = std::getenv("NATTEN_HIP_SPLIT");
        return e ? std::atoi(e) : 0;
    }();
    int kmax = p.ax[split_axis(p)].k;
    if (piped) kmax = std::min(kmax, p.kv / 8);
    const long long target = 256LL * (!key ? 6 : piped ? 8 : 12);
    int split = 1;
    if (forced > 0) {
        while (split * 2 <= forced && split * 2 * lpq <= 64) split *= 2;
        return split;
    }
    const long long waves = (groups * lpq + 63) / 64;
    while (split < 8 && split * 2 * lpq <= 64 && split * 2 <= kmax && waves * split < target) split *= 2;
    return split;
}

template <typename T, int DPL, int LPQ>
struct LForward {
    static hipError_t run(const Prob& p, int vec, const int* lens, const void* q, Lay lq, const void* k, Lay lk,
                          const void* v, Lay lv, void* o, Lay lo, float* lse, Lay ll, hipStream_t s) {
        const long long n = static_cast<long long>(p.B) * p.nout * p.Hq;
        const int split = choose_split(p, n, LPQ, vec != 0, false);
        NA_LAUNCH(lens ? "na_varlen_forward" : "na_forward", (k_forward<T, DPL, LPQ>),
                  dim3(grid_for(n, LPQ * split)), dim3(256), 0, s, p, vec, split, lens, (const T*)q, lq, (const T*)k, lk, (const T*)v, lv, (T*)o, lo, lse,
                  ll);
        return hipGetLastError();
    }
};

template <typename T, int DPL, int LPQ>
struct LQK {
    static hipError_t run(const Prob& p, int vec, const void* q, Lay lq, const void* k, Lay lk, void* a, Lay la,
                          hipStream_t s) {
        const long long n = static_cast<long long>(p.B) * p.nout * p.Hq;
        const int split = choose_split(p, n, LPQ, vec != 0, false);
        const auto kern = vec ? k_qk<T, DPL, LPQ, true> : k_qk<T, DPL, LPQ, false>;
        NA_LAUNCH("na_qk", kern, dim3(grid_for(n, LPQ * split)), dim3(256), 0, s, p, split, (const T*)q, lq,
                           (const T*)k, lk, (T*)a, la);
        return hipGetLastError();
    }
};

template <typename T, int DPL, int LPQ>
struct LAV {
    static hipError_t run(const Prob& p, int vec, const void* a, Lay la, const void* v, Lay lv, void* o, Lay lo,
                          hipStream_t s) {
        const long long n = static_cast<long long>(p.B) * p.nout * p.Hq;
        const int split = choose_split(p, n, LPQ, vec != 0, false);
        NA_LAUNCH("na_av", (k_av<T, DPL, LPQ>), dim3(grid_for(n, LPQ * split)), dim3(256), 0, s, p, vec, split, (const T*)a, la,
                           (const T*)v, lv, (T*)o, lo);
        return hipGetLastError();
    }
};

template <typename T, int DPL, int LPQ>
struct LBackward {
    static hipError_t run(const Prob& p, int vec, const int* lens, const void* q, Lay lq, const void* k, Lay lk,
                          const void* v, Lay lv, const void* o, Lay lo, const void* dout, Lay ldo, const float* lse,
                          Lay ll, const float* dlse, Lay ldl, void* dq, Lay ldq, void* dk, Lay ldk, void* dv,
                          Lay ldv, float* delta, Lay lde, hipStream_t s) {
        const long long nq = static_cast<long long>(p.B) * p.nout * p.Hq;
        const int sq = choose_split(p, nq, LPQ, vec != 0, false);
        NA_LAUNCH(lens ? "na_varlen_bwd_dq" : "na_bwd_dq", (k_bwd_dq<T, DPL, LPQ>), dim3(grid_for(nq, LPQ * sq)),
                  dim3(256), 0, s, p, vec, sq, lens, (const T*)q, lq, (const T*)k, lk, (const T*)v, lv, (const T*)o, lo,
                  (const T*)dout, ldo, lse, ll, dlse, ldl, (T*)dq, ldq, delta, lde);
        hipError_t e = hipGetLastError();
        if (e != hipSuccess) return e;
        const long long nk = static_cast<long long>(p.B) * p.nkey * p.Hkv;
        const int sk = choose_split(p, nk, LPQ, vec && unit_strides(p), true);
        const auto kern_k = vec && unit_strides(p) ? k_bwd_dkdv<T, DPL, LPQ, true> : k_bwd_dkdv<T, DPL, LPQ, false>;
        NA_LAUNCH(lens ? "na_varlen_bwd_dkdv" : "na_bwd_dkdv", kern_k,
                  dim3(grid_for(nk, LPQ * sk)), dim3(256), 0, s, p, vec, sk, lens, (const T*)q, lq, (const T*)k, lk,
                  (const T*)v, lv, (const T*)dout, ldo, lse, ll, (const float*)delta, lde, (T*)dk, ldk, (T*)dv,
                  ldv);
        return hipGetLastError();
    }
};

template <typename T, int DPL, int LPQ>
struct LQKBwd {
    static hipError_t run(const Prob& p, int vec, const void* da, Lay lda, const void* q, Lay lq, const void* k,
                          Lay lk, void* dq, Lay ldq, void* dk, Lay ldk, int sides, hipStream_t s) {
        if (sides & kQuerySide) {
            const long long nq = static_cast<long long>(p.B) * p.nout * p.Hq;
            const int split = choose_split(p, nq, LPQ, vec != 0, false);
            NA_LAUNCH("na_qk_bwd_q", (k_qk_bwd_q<T, DPL, LPQ>), dim3(grid_for(nq, LPQ * split)), dim3(256), 0, s, p, vec, split,
                      (const T*)da, lda, (const T*)k, lk, (T*)dq, ldq);
            const hipError_t e = hipGetLastError();
            if (e != hipSuccess) return e;
        }
        if (!(sides & kKeySide)) return hipSuccess;
        const long long nk = static_cast<long long>(p.B) * p.nkey * p.Hkv;
        const int split = choose_split(p, nk, LPQ, vec && unit_strides(p), true);
        const auto kern = vec && unit_strides(p) ? k_qk_bwd_k<T, DPL, LPQ, true> : k_qk_bwd_k<T, DPL, LPQ, false>;
        NA_LAUNCH("na_qk_bwd_k", kern, dim3(grid_for(nk, LPQ * split)), dim3(256), 0, s, p, vec, split,
                           (const T*)da, lda, (const T*)q, lq, (T*)dk, ldk);
        return hipGetLastError();
    }
};

template <typename T, int DPL, int LPQ>
struct LAVBwd {
    static hipError_t run(const Prob& p, int vec, const void* dout, Lay ldo, const void* a, Lay la, const void* v,
                          Lay lv, void* da, Lay lda, void* dv, Lay ldv, int sides, hipStream_t s) {
        if (sides & kQuerySide) {
            const long long nq = static_cast<long long>(p.B) * p.nout * p.Hq;
            const int split = choose_split(p, nq, LPQ, vec != 0, false);
            const auto kern = vec ? k_av_bwd_a<T, DPL, LPQ, true> : k_av_bwd_a<T, DPL, LPQ, false>;
            NA_LAUNCH("na_av_bwd_a", kern, dim3(grid_for(nq, LPQ * split)), dim3(256), 0, s, p, split,
                      (const T*)dout, ldo, (const T*)v, lv, (T*)da, lda);
            const hipError_t e = hipGetLastError();
            if (e != hipSuccess) return e;
        }
        if (!(sides & kKeySide)) return hipSuccess;
        const long long nk = static_cast<long long>(p.B) * p.nkey * p.Hkv;
        const int split = choose_split(p, nk, LPQ, vec && unit_strides(p), true);
        const auto kern = vec && unit_strides(p) ? k_av_bwd_v<T, DPL, LPQ, true> : k_av_bwd_v<T, DPL, LPQ, false>;
        NA_LAUNCH("na_av_bwd_v", kern, dim3(grid_for(nk, LPQ * split)), dim3(256), 0, s, p, vec, split,
                           (const T*)dout, ldo, (const T*)a, la, (T*)dv, ldv);
        return hipGetLastError();
    }
};

}  // namespace

hipError_t generic_forward(const Prob& p, int vec, const void* q, Lay lq, const void* k, Lay lk, const void* v,
                           Lay lv, void* o, Lay lo, float* lse, Lay ll, int dtype, hipStream_t s, const int* lens) {
    return by_type<LForward>(dtype, p.Dqk > p.Dv ? p.Dqk : p.Dv, p, vec, lens, q, lq, k, lk, v, lv, o, lo, lse, ll,
                             s);
}

hipError_t generic_qk(const Prob& p, int vec, const void* q, Lay lq, const void* k, Lay lk, void* a, Lay la,
                      int dtype, hipStream_t s) {
    return by_type<LQK>(dtype, p.Dqk, p, vec, q, lq, k, lk, a, la, s);
}

hipError_t generic_av(const Prob& p, int vec, const void* a, Lay la, const void* v, Lay lv, void* o, Lay lo,
                      int dtype, hipStream_t s) {
    return by_type<LAV>(dtype, p.Dv, p, vec, a, la, v, lv, o, lo, s);
}

hipError_t generic_backward(const Prob& p, int vec, const void* q, Lay lq, const void* k, Lay lk, const void* v,
                            Lay lv, const void* o, Lay lo, const void* dout, Lay ldo, const float* lse, Lay ll,
                            const float* dlse, Lay ldl, void* dq, Lay ldq, void* dk, Lay ldk, void* dv, Lay ldv,
                            float* delta, Lay lde, int dtype, hipStream_t s, const int* lens) {
    return by_type<LBackward>(dtype, p.Dqk > p.Dv ? p.Dqk : p.Dv, p, vec, lens, q, lq, k, lk, v, lv, o, lo, dout,
                              ldo, lse, ll, dlse, ldl, dq, ldq, dk, ldk, dv, ldv, delta, lde, s);
}

hipError_t generic_qk_backward(const Prob& p, int vec, const void* da, Lay lda, const void* q, Lay lq,
                               const void* k, Lay lk, void* dq, Lay ldq, void* dk, Lay ldk, int dtype,
                               hipStream_t s, int sides) {
    return by_type<LQKBwd>(dtype, p.Dqk, p, vec, da, lda, q, lq, k, lk, dq, ldq, dk, ldk, sides, s);
}

hipError_t generic_av_backward(const Prob& p, int vec, const void* dout, Lay ldo, const void* a, Lay la,
                               const void* v, Lay lv, void* da, Lay lda, void* dv, Lay ldv, int dtype,
                               hipStream_t s, int sides) {
    return by_type<LAVBwd>(dtype, p.Dv, p, vec, dout, ldo, a, la, v, lv, da, lda, dv, ldv, sides, s);
}

hipError_t neighborhood_map(const Prob& p, int64_t* flat, uint8_t* valid, hipStream_t s) {
    const long long n = static_cast<long long>(p.nout) * p.kv;
    if (n == 0) return hipSuccess;
    NA_LAUNCH("na_map", k_map, dim3(static_cast<unsigned>((n + 255) / 256)), dim3(256), 0, s, p, flat, valid);
    return hipGetLastError();
}

}  // namespace na
