// Band kernels (gfx950, bf16 / fp16, head dim 32 / 64 / 128, stride 1):
// fused forward, backward dQ and backward dK/dV for windows whose staged
// union is too large for the other tile kernels to hold at once.
//
// The 8x8 tile kernels (na_lean.hip) stop at kernel 9, and the general tile
// kernels (na_mfma.hip) stage a whole plane of the union: at kernel 13 x 13
// and head dim 64 only a 16-query tile fits, which stages 23 rows of K and V
// per query and runs one wave per workgroup.  Here a workgroup of 8 waves
// owns 128 queries (keys) of one class pair and one (batch, head) -- a box
// of 128 / T2 rows of T2 = 8 or 16 columns, 16 items per wave -- and walks
// the union a band of NC chunks (32 slots each) at a time, so that LDS holds
// two bands whatever the kernel size:
//
// * The next band's rows are requested into registers before the current
//   band is computed, and stored to the other LDS buffer after it: loads
//   overlap the products, with one barrier per band.  (Loads straight to
//   LDS cannot be used that way: the compiler waits for all of them before
//   any LDS read.)
// * A union row takes one chunk: 32 slots, which every union's columns fit
//   (band_columns in na_common.h).
// * A wave computes only the chunks that its own items' windows reach; its
//   online softmax rescales once per band.
//
// What bounds it: LDS reads (a chunk's 8 KB of K and V rows per 16 queries)
// and the latency of a wave's score -> maximum -> exponential -> product
// chain; 8 waves and bands of 4 rows measured as fast as 4 waves or bands of
// 2 (16 waves: 28 % slower).  Measured, general tile (or, *, vector) kernels
// -> these: 13 x 13, head dim 64, fp16, 4 x 135 x 241, 8 heads, forward 2350
// -> 252 us; bf16 4 x 64 x 64, 8 heads, forward 275 -> 35, dQ 981* -> 70,
// dK/dV 968* -> 81 us; head dim 128, 4 heads 501* / 1043* / 998* -> 40 / 82 /
// 82 us; 11 x 11, head dim 32, 4 x 61 x 130, 8 heads 103 / 139 / 128 -> 46 /
// 81 / 62 us.  (*: the two-term products of band_sides.)
//
// The geometry is computed in the kernel (no tables): every call, captured
// or not, runs the same code.  MFMA lane layouts, the swizzle and the masks
// are those of na_mfma.hip.
#include <algorithm>
#include <cstdio>
#include <cstdlib>
#include <cstring>

#include "na_tile.h"

namespace na {

namespace {

typedef unsigned int u32x4_t __attribute__((ext_vector_type(4)));

constexpr int kBandWaves = 8;
constexpr int kBandThreads = 64 * kBandWaves;
constexpr uint32_t kBandOOR = 0x40000000u;  // past every staged plane (planes < 2^30 bytes)

// Chunks per band: two 16-byte pieces per thread and operand at head dims
// 64 and 128, one at 32.
template <int D>
constexpr int kBandChunks = D == 128 ? 2 : 4;

// LDS bytes of one operand's band, and of one buffer of two operands.
template <int D>
constexpr int kBandOp = kBandChunks<D> * 32 * D * 2;

// Tile shape: log2 of the box's columns and rows, tiles per class and axis,
// and the divisors that decode a workgroup's index.
struct BandGeo {
    int sh1, sh2;
    int lenmod[3];                            // (axes 1 and 2, as the next two)
    FastDiv heads, tiles, rep, nt[3], dil[3];
};

template <typename T>
struct BandArgs {
    Prob p;
    BandGeo g;
    const T *q, *k, *v, *o, *dout;
    const float *lse, *dlse, *delta;
    T *out, *dq, *dk, *dv;
    float *lse_out, *delta_out;
    LayK lq, lk, lv, lo, ldo, ldq, ldk, ldv, ll, lde, ldl;
    uint32_t ab, bb;  // byte ranges of one plane of the two staged operands
};

// A workgroup's tile: batch, head (kv head on the key side), the tile's
// geometry on axes 1 and 2 (with this wave's box), residues.
struct BandTile {
    int b, h, r[3];
    AxisGeo a[3];
    __device__ __forceinline__ bool tile_ok() const { return a[1].tile_ok && a[2].tile_ok; }
    __device__ __forceinline__ bool wave_ok() const { return a[1].wave_ok && a[2].wave_ok; }
};

template <bool KEY>
__device__ __forceinline__ BandTile band_tile(const Prob& p, const BandGeo& g, int wave) {
    BandTile t;
    const int x = xcd_block(blockIdx.x, gridDim.x);
    const int bt = fdiv(x, g.heads);
    t.h = x - bt * static_cast<int>(g.heads.d);
    t.b = fdiv(bt, g.tiles);
    int s = bt - t.b * static_cast<int>(g.tiles.d);
    int tt[3];
#pragma unroll
    for (int a = 2; a >= 1; --a) {
        int q = fdiv(s, g.nt[a]);
        tt[a] = s - q * static_cast<int>(g.nt[a].d);
        s = q;
        q = fdiv(s, g.dil[a]);
        t.r[a] = s - q * static_cast<int>(g.dil[a].d);
        s = q;
    }
    const int T[3] = {1, 1 << g.sh1, 1 << g.sh2};
    // the wave's items 16 w .. 16 w + 15 in row-major order: whole rows (T2 <= 16)
    const int e1 = wave * 16 >> g.sh2;
    const int wl[3] = {0, e1, 0}, wh[3] = {0, e1 + (16 >> g.sh2) - 1, T[2] - 1};
#pragma unroll
    for (int a = 1; a < 3; ++a) {
        const Axis& A = p.ax[a];
        t.a[a] = axis_geometry(A.len, A.k, A.dil, A.causal, g.lenmod[a], 1, A.len, T[a], tt[a], t.r[a], wl[a], wh[a],
                               KEY, g.dil[a]);
    }
    return t;
}

__device__ __forceinline__ ClassAxis band_class(const Axis& A, const AxisGeo& g) {
    return ClassAxis{g.n, A.k, A.k >> 1, g.B, A.causal, 1};
}

// The lane's item: validity, position, and its window (key side: attending
// queries) relative to the union -- rows [rlo, rlo + rn) and columns [clo,
// clo + cn); rn = 0 for lanes past the tile.
struct BandLane {
    bool valid;
    int pos[3], rlo, rn, clo, cn;
};

template <bool KEY>
__device__ __forceinline__ BandLane band_lane(const Prob& p, const BandGeo& g, const BandTile& t, int wave, int col) {
    const int f = wave * 16 + col;
    const int e[3] = {0, f >> g.sh2, f & ((1 << g.sh2) - 1)};
    BandLane l;
    l.valid = e[1] < t.a[1].E && e[2] < t.a[2].E;
    l.pos[0] = 0;
    int lo[3], hi[3];
#pragma unroll
    for (int a = 1; a < 3; ++a) {
        const int j = t.a[a].J + (l.valid ? e[a] : 0);
        l.pos[a] = t.r[a] + j * p.ax[a].dil;
        item_box(band_class(p.ax[a], t.a[a]), j, KEY, lo[a], hi[a]);
    }
    l.rlo = lo[1] - t.a[1].lo;
    l.rn = l.valid ? imax(hi[1] - lo[1] + 1, 0) : 0;
    l.clo = lo[2] - t.a[2].lo;
    l.cn = imax(hi[2] - lo[2] + 1, 0);
    return l;
}

// Column mask of the lane's 8 slots of a chunk, as the score product's
// accumulator input.
__device__ __forceinline__ void band_colbias(const BandLane& l, int grp, f32x4_t (&bias)[2]) {
    const int c0 = 8 * grp - l.clo;
#pragma unroll
    for (int e = 0; e < 8; ++e)
        bias[e >> 2][e & 3] = static_cast<unsigned>(c0 + e) < static_cast<unsigned>(l.cn) ? 0.f : -INFINITY;
}

template <typename T>
__device__ __forceinline__ __amdgpu_buffer_rsrc_t band_rsrc(const T* p, uint32_t bytes) {
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<T*>(p), static_cast<short>(0), static_cast<int>(bytes),
                                             0x00020000);
}

// XOR swizzle of the 16-byte pieces of LDS row `row` (D / 8 pieces per row).
// LDS has 64 4-byte banks and serves 256 bytes per pass.  A 16-byte read runs
// in four passes of 16 lanes -- {0-3, 12-15, 20-27}, {4-11, 16-19, 28-31} and
// the same plus 32 -- and a transposing 8-byte read in two of 32 consecutive
// lanes (measured from pairs of lanes made to collide).  With slot = 8x + 4b
// + y, a score-operand pass covers x = 0, 3 of one lane group and x = 1, 2 of
// the next, and a transposing pass x = 0, 1 or x = 2, 3 of all y, two
// neighbouring pieces each: both are free of conflicts when the swizzle's
// bits above 0 take every value over (x % 2, y) and bit 0 stays clear.  With
// swz (na_tile.h) the transposing reads take two passes more, which shows
// little: dK/dV 11 x 11, head dim 32, 63.5 -> 61.9 us, 13 x 13, head dim 128,
// 82.3 -> 81.6, but 9 x 9, head dim 64, 106 -> 107 us.
template <int D>
__host__ __device__ constexpr int band_swz(int row) {
    if constexpr (D == 32) return ((row >> 3) & 1) << 1;
    else if constexpr (D == 64) return (((row >> 3) & 1) << 2) | (((row >> 1) & 1) << 1);
    else return (((row >> 3) & 1) << 3) | ((row & 3) << 1);
}

// Staging of two operands' bands: thread t moves 16-byte piece t % P of
// slots t / P + j * SPT, j < NP, of each operand (SPT slots, whole union rows,
// per round of the workgroup).  Columns past the union and rows past it load
// from outside the buffer (zeros).
template <typename T, int D>
struct BandStage {
    static constexpr int P = D / 8, NP = kBandChunks<D> * 32 * P / kBandThreads, SPT = kBandThreads / P;
    static_assert(SPT % 32 == 0, "rounds of whole rows; the swizzle repeats every 32 slots");
    int row0, dst;                // first union row (wave-uniform); LDS byte offset of round 0
    uint32_t ca, cb;              // lane part of the global offsets
    int base_a, base_b, step_a, step_b;
    uint4 ra[NP], rb[NP];

    __device__ __forceinline__ void init(const Prob& p, const BandTile& t, const LayK& la, const LayK& lb) {
        const int tid = threadIdx.x, pp = tid % P, slot = tid / P, c = slot % 32;
        row0 = __builtin_amdgcn_readfirstlane(slot / 32);
        const int d1 = p.ax[1].dil, d2 = p.ax[2].dil;
        dst = slot * D * 2 + ((pp ^ band_swz<D>(slot)) << 4);
        const bool in = c < t.a[2].U;
        ca = in ? static_cast<uint32_t>(c * d2 * la.s2 * 2 + pp * 16) : kBandOOR;
        cb = in ? static_cast<uint32_t>(c * d2 * lb.s2 * 2 + pp * 16) : kBandOOR;
        const int p1 = t.r[1] + t.a[1].lo * d1, p2 = t.r[2] + t.a[2].lo * d2;
        base_a = (p1 * la.s1 + p2 * la.s2) * 2;
        base_b = (p1 * lb.s1 + p2 * lb.s2) * 2;
        step_a = d1 * la.s1 * 2;
        step_b = d1 * lb.s1 * 2;
    }

    // request band `bi` of the planes at pa / pb
    __device__ __forceinline__ void load(__amdgpu_buffer_rsrc_t pa, __amdgpu_buffer_rsrc_t pb, int bi, int U1) {
#pragma unroll
        for (int j = 0; j < NP; ++j) {
            const int row = bi * kBandChunks<D> + row0 + j * (SPT / 32);
            const uint32_t oa = row < U1 ? static_cast<uint32_t>(base_a + row * step_a) : kBandOOR;
            const uint32_t ob = row < U1 ? static_cast<uint32_t>(base_b + row * step_b) : kBandOOR;
            ra[j] = __builtin_bit_cast(uint4, __builtin_amdgcn_raw_buffer_load_b128(pa, ca + oa, 0, 0));
            rb[j] = __builtin_bit_cast(uint4, __builtin_amdgcn_raw_buffer_load_b128(pb, cb + ob, 0, 0));
        }
    }

    // store the requested band into the buffer at `buf`
    __device__ __forceinline__ void store(unsigned char* buf) const {
#pragma unroll
        for (int j = 0; j < NP; ++j) {
            unsigned char* x = buf + dst + j * (kBandThreads * 16);
            *reinterpret_cast<uint4*>(x) = ra[j];
            *reinterpret_cast<uint4*>(x + kBandOp<D>) = rb[j];
        }
    }
};

// LDS byte offsets (from an operand's band) of the lane's A operands of
// chunk 0: the score product's (rows = slots) and, transposed, the product's
// over slots (na_tile.h, score_chunk and accumulate_chunk).
template <int D>
struct BandOff {
    int a[2][D / 32], t[2][D / 16];
    __device__ __forceinline__ void init(int lane) {
        const int col = lane & 15, grp = lane >> 4;
#pragma unroll
        for (int b = 0; b < 2; ++b) {
            const int slot = 8 * (col >> 2) + 4 * b + (col & 3);
#pragma unroll
            for (int ks = 0; ks < D / 32; ++ks) a[b][ks] = slot * D * 2 + (((ks * 4 + grp) ^ band_swz<D>(slot)) << 4);
        }
#pragma unroll
        for (int hi = 0; hi < 2; ++hi) {
            const int r = 8 * grp + (col >> 2) + 4 * hi;
#pragma unroll
            for (int db = 0; db < D / 16; ++db)
                t[hi][db] = r * D * 2 + (((2 * db + ((col & 3) >> 1)) ^ band_swz<D>(r)) << 4) + (col & 1) * 8;
        }
    }
};

template <typename T, int D>
__device__ __forceinline__ void band_score(const unsigned char* X, const BandOff<D>& o, int c,
                                           const uint4 (&frag)[D / 32], const f32x4_t (&bias)[2], f32x4_t (&out)[2]) {
#pragma unroll
    for (int b = 0; b < 2; ++b) {
        f32x4_t acc = bias[b];
#pragma unroll
        for (int ks = 0; ks < D / 32; ++ks) {
            const u32x4_t a = *reinterpret_cast<const u32x4_t*>(X + o.a[b][ks] + c * 32 * D * 2);
            acc = Mma<T>::run(__builtin_bit_cast(uint4, a), frag[ks], acc);
        }
        out[b] = acc;
    }
}

// What rounding v to `packed` left over, packed in turn.
template <typename T>
__device__ __forceinline__ uint4 pack_rest(const f32x4_t (&v)[2], uint4 packed) {
    const uint32_t w[4] = {packed.x, packed.y, packed.z, packed.w};
    f32x4_t r[2];
#pragma unroll
    for (int i = 0; i < 8; ++i) {
        const uint32_t h = w[i >> 1] >> (16 * (i & 1)) & 0xffffu;
        float f;
        if constexpr (std::is_same_v<T, bf16>)
            f = __uint_as_float(h << 16);
        else
            f = static_cast<float>(__builtin_bit_cast(f16, static_cast<uint16_t>(h)));
        r[i >> 2][i & 3] = v[i >> 2][i & 3] - f;
    }
    return pack8<T>(r);
}

// Two fp16 terms share fp16's exponents: their sum stops at 2^-25 absolute,
// where bfloat16's keeps 16 bits of every value.  So fp16 pairs are scaled by
// powers of two, exact to apply and to take out: P of the key side by 2^15 (P
// <= 1 up to rounding), dS by a factor of its item's own.  Unscaled, dQ and dK
// lost up to 7 times their rounding error at dO ~ 1e-3 (97 x 16, head dim
// 32); scaled, none.  Time: 4 x 64 x 64 x 8, dim 64, 13 x 13, fp16 68 -> 71 us
// (dQ) and 80 -> 88 us (dK/dV).
template <typename T, bool TWO>
constexpr bool kScaled = TWO && std::is_same_v<T, f16>;
constexpr float kScaleP = 32768.f;
// Values of a scaled item stay below this (their factor puts a new maximum
// in [2^13, 2^14)).
constexpr float kScaleLimit = 32768.f;

// The power of two that moves m >= 0 into [2^13, 2^14); within 2^+-96, so
// that it and its reciprocal are normal.
__device__ __forceinline__ float scale_for(float m) {
    const int e = static_cast<int>(__float_as_uint(m) >> 23 & 0xffu);
    const int k = 140 - e < 96 ? 140 - e : 96;
    return __uint_as_float(static_cast<uint32_t>(k < -96 ? 127 - 96 : 127 + k) << 23);
}

// 1 / x of a power of two from scale_for.
__device__ __forceinline__ float inv_pow2(float x) { return __uint_as_float((254u << 23) - __float_as_uint(x)); }

// Largest |v| of 8, at least m; NaNs (a masked slot's 0 times infinity) drop out.
__device__ __forceinline__ float abs_max8(const f32x4_t (&v)[2], float m) {
#pragma unroll
    for (int i = 0; i < 8; ++i) m = fmaxf(m, __builtin_fabsf(v[i >> 2][i & 3]));
    return m;
}

// Maximum over the four 16-lane rows of the wave, NaNs dropping out.
__device__ __forceinline__ float max_rows_num(float v) {
    const auto a = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    v = fmaxf(__uint_as_float(a[0]), __uint_as_float(a[1]));
    const auto b = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    return fmaxf(__uint_as_float(b[0]), __uint_as_float(b[1]));
}

// acc += X^T of chunk c times v, v as one 16-bit term or (TWO) as two.
template <typename T, int D, bool TWO>
__device__ __forceinline__ void band_accumulate(const unsigned char* X, const BandOff<D>& o, int c,
                                                const f32x4_t (&v)[2], f32x4_t (&acc)[D / 16]) {
    const uint4 packed = pack8<T>(v);
    uint4 rest;
    if constexpr (TWO) rest = pack_rest<T>(v, packed);
#pragma unroll
    for (int db = 0; db < D / 16; ++db) {
        const i16x4_t lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_i16x4_t*)(X + o.t[0][db] + c * 32 * D * 2));
        const i16x4_t hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_i16x4_t*)(X + o.t[1][db] + c * 32 * D * 2));
        const uint2 l2 = __builtin_bit_cast(uint2, lo), h2 = __builtin_bit_cast(uint2, hi);
        const uint4 x = make_uint4(l2.x, l2.y, h2.x, h2.y);
        acc[db] = Mma<T>::run(x, packed, acc[db]);
        if constexpr (TWO) acc[db] = Mma<T>::run(x, rest, acc[db]);
    }
}

// Chunks of a band whose code the backward kernels lay side by side.  With two
// terms at head dim 64 that spilled 12 to 47 registers; one after another, 0
// to 12 (13 x 13, 4 x 135 x 241 x 8, bfloat16, dQ 586 -> 546, dK/dV 1040 -> 685
// us).
template <int D, bool TWO>
constexpr int kBandUnroll = TWO && D == 64 ? 1 : kBandChunks<D>;

// Waves per SIMD the kernels are built for: two workgroups of 8 waves fit a
// CU's LDS; at head dim 128 the backward kernels need the registers of one.
constexpr int band_waves(int D, bool backward) { return D == 128 && backward ? 2 : 4; }
#define NA_BAND_OCC(D, BWD) __attribute__((amdgpu_waves_per_eu(band_waves(D, BWD))))

template <typename T, int D>
__device__ __forceinline__ void band_redo_fwd(const void* kargs, int b, int h, int hk, int p0, int p1, int p2,
                                              int grp) {
    const BandArgs<T>& A = *static_cast<const BandArgs<T>*>(kargs);
    const int pos[3] = {p0, p1, p2};
    ExactAxis x[3];
    for (int a = 0; a < 3; ++a) x[a] = exact_axis(A.p.ax[a], pos[a]);
    f32x4_t acc[D / 16];
    float lse_v;
    exact_forward<T, D>(A.p.scale, x, bh_ptr(A.q, A.lq, b, h) + vol_off(A.lq, pos), bh_ptr(A.k, A.lk, b, hk),
                        strides3(A.lk), bh_ptr(A.v, A.lv, b, hk), strides3(A.lv), grp, acc, lse_v);
    store_rows<T, D>(bh_ptr(A.out, A.lo, b, h), vol_off(A.lo, pos), grp, acc, 1.f);
    if (grp == 0) bh_ptr(A.lse_out, A.ll, b, h)[vol_off(A.ll, pos)] = lse_v;
}

template <typename T, int D, bool TWO>
__global__ __launch_bounds__(kBandThreads) NA_BAND_OCC(D, false) void k_band_fwd(BandArgs<T> args) {
    constexpr int NC = kBandChunks<D>, BUF = 2 * kBandOp<D>;
    const Prob& p = args.p;
    unsigned char* smem = lds_base();
    const int lane = threadIdx.x & 63, col = lane & 15, grp = lane >> 4;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const BandTile t = band_tile<false>(p, args.g, wave);
    if (!t.tile_ok()) return;
    const int hk = args.g.rep.d == 1 ? t.h : fdiv(t.h, args.g.rep);
    const T* kb = bh_ptr(args.k, args.lk, t.b, hk);
    const T* vb = bh_ptr(args.v, args.lv, t.b, hk);
    BandStage<T, D> st;
    st.init(p, t, args.lk, args.lv);
    const int U1 = t.a[1].U, nb = (U1 + NC - 1) / NC;
    const auto load = [&](int bi) { st.load(band_rsrc(kb, args.ab), band_rsrc(vb, args.bb), bi, U1); };
    load(0);

    const BandLane ln = band_lane<false>(p, args.g, t, wave, col);
    uint4 qf[D / 32];
    load_frags<T, D>(bh_ptr(args.q, args.lq, t.b, t.h), vol_off(args.lq, ln.pos), ln.valid, grp, qf);
    f32x4_t cb[2];
    band_colbias(ln, grp, cb);
    BandOff<D> off;
    off.init(lane);
    const float sc2 = p.scale * kLog2e;
    // the wave's chunks
    const int wc0 = t.a[1].glo, wc1 = t.wave_ok() ? t.a[1].ghi : -1;
    const uint4 ones = make_uint4(Mma<T>::kOnes, Mma<T>::kOnes, Mma<T>::kOnes, Mma<T>::kOnes);

    f32x4_t acc[D / 16], lacc = f32x4_t{0.f, 0.f, 0.f, 0.f};
    float m = -INFINITY, lpart = 0.f;
#pragma unroll
    for (int db = 0; db < D / 16; ++db) acc[db] = f32x4_t{0.f, 0.f, 0.f, 0.f};
    int bi = 0;
    // one band: publish it in buffer B, request the next one, compute
    const auto step = [&](auto BC) {
        constexpr int B = decltype(BC)::value;
        st.store(smem + B * BUF);
        lds_publish_barrier();
        const int c0 = bi * NC;
        const bool more = ++bi < nb;
        if (more) load(bi);
        if (c0 + NC - 1 >= wc0 && c0 <= wc1) {
            const unsigned char* Kb = smem + B * BUF;
            const unsigned char* Vb = Kb + kBandOp<D>;
            f32x4_t s[NC][2];
            bool rv[NC];
            float cm = -INFINITY;
#pragma unroll
            for (int c = 0; c < NC; ++c) {
                if (c0 + c >= wc0 && c0 + c <= wc1) {
                    const int row = c0 + c - ln.rlo;
                    rv[c] = static_cast<unsigned>(row) < static_cast<unsigned>(ln.rn);
                    band_score<T, D>(Kb, off, c, qf, cb, s[c]);
                    cm = fmaxp(cm, rv[c] ? max8(s[c]) : -INFINITY);
                }
            }
            const float mnew = fmaxp(m, max_rows(cm) * sc2);
            const float mref = mnew == -INFINITY ? 0.f : mnew;
            const float corr = __builtin_amdgcn_exp2f(m - mref);
            m = mnew;
            if constexpr (TWO) lpart *= corr;
            else lacc *= corr;
#pragma unroll
            for (int db = 0; db < D / 16; ++db) acc[db] *= corr;
#pragma unroll
            for (int c = 0; c < NC; ++c) {
                if (c0 + c >= wc0 && c0 + c <= wc1) {
                    const float o = rv[c] ? -mref : -INFINITY;
#pragma unroll
                    for (int bb = 0; bb < 2; ++bb)
#pragma unroll
                        for (int i = 0; i < 4; ++i) s[c][bb][i] = __builtin_amdgcn_exp2f(fmaf(s[c][bb][i], sc2, o));
                    band_accumulate<T, D, TWO>(Vb, off, c, s[c], acc);
                    // the row sum: of the rounded values that the product took, or
                    // (two terms, the rest far below the result's rounding) in fp32
                    if constexpr (TWO)
                        lpart += ((s[c][0][0] + s[c][0][1]) + (s[c][0][2] + s[c][0][3])) +
                                 ((s[c][1][0] + s[c][1][1]) + (s[c][1][2] + s[c][1][3]));
                    else
                        lacc = Mma<T>::run(ones, pack8<T>(s[c]), lacc);
                }
            }
        }
        return more;
    };
#pragma unroll 1
    while (step(std::integral_constant<int, 0>{}) && step(std::integral_constant<int, 1>{})) {
    }
    const float lsum = TWO ? sum_rows(lpart) : lacc[0];
    const bool redo = ln.valid && item_nonfinite(lane_sum(acc, lsum));
    if (ln.valid) {
        store_rows<T, D>(bh_ptr(args.out, args.lo, t.b, t.h), vol_off(args.lo, ln.pos), grp, acc, 1.f / lsum);
        if (grp == 0) bh_ptr(args.lse_out, args.ll, t.b, t.h)[vol_off(args.ll, ln.pos)] = (m + __log2f(lsum)) * kLn2;
    }
    if (redo)
        band_redo_fwd<T, D>(kernargs(), t.b, t.h, hk, opaque(ln.pos[0]), opaque(ln.pos[1]), opaque(ln.pos[2]), grp);
}

// Backward, query side: as k_bwd_q_mfma.  A first walk takes delta =
// sum over the window of P dP (= dO . O) from the kernel's own products
// (where that is not finite, dO . O from the rows), a second one forms dS =
// P (dP - delta) and dq.
template <typename T, int D>
__device__ __forceinline__ void band_redo_bwd_q(const void* kargs, int b, int h, int hk, int p0, int p1, int p2,
                                                int grp) {
    const BandArgs<T>& A = *static_cast<const BandArgs<T>*>(kargs);
    const int pos[3] = {p0, p1, p2};
    ExactAxis x[3];
    for (int a = 0; a < 3; ++a) x[a] = exact_axis(A.p.ax[a], pos[a]);
    const T* do_row = bh_ptr(A.dout, A.ldo, b, h) + vol_off(A.ldo, pos);
    float di = exact_dot<T, D>(do_row, bh_ptr(A.o, A.lo, b, h) + vol_off(A.lo, pos));
    if (A.dlse) di -= bh_ptr(A.dlse, A.ldl, b, h)[vol_off(A.ldl, pos)];
    f32x4_t acc[D / 16];
    exact_backward_q<T, D>(A.p.scale, x, bh_ptr(A.q, A.lq, b, h) + vol_off(A.lq, pos), do_row,
                           bh_ptr(A.lse, A.ll, b, h)[vol_off(A.ll, pos)], di, bh_ptr(A.k, A.lk, b, hk),
                           strides3(A.lk), bh_ptr(A.v, A.lv, b, hk), strides3(A.lv), grp, acc);
    store_rows<T, D>(bh_ptr(A.dq, A.ldq, b, h), vol_off(A.ldq, pos), grp, acc, A.p.scale);
}

template <typename T, int D, bool TWO>
__global__ __launch_bounds__(kBandThreads) NA_BAND_OCC(D, true) void k_band_bwd_q(BandArgs<T> args) {
    constexpr int NC = kBandChunks<D>, BUF = 2 * kBandOp<D>;
    const Prob& p = args.p;
    unsigned char* smem = lds_base();
    const int lane = threadIdx.x & 63, col = lane & 15, grp = lane >> 4;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const BandTile t = band_tile<false>(p, args.g, wave);
    if (!t.tile_ok()) return;
    const int hk = args.g.rep.d == 1 ? t.h : fdiv(t.h, args.g.rep);
    const T* kb = bh_ptr(args.k, args.lk, t.b, hk);
    const T* vb = bh_ptr(args.v, args.lv, t.b, hk);
    BandStage<T, D> st;
    st.init(p, t, args.lk, args.lv);
    const int U1 = t.a[1].U, nb = (U1 + NC - 1) / NC;
    const auto load = [&](int bi) { st.load(band_rsrc(kb, args.ab), band_rsrc(vb, args.bb), bi, U1); };
    load(0);

    const BandLane ln = band_lane<false>(p, args.g, t, wave, col);
    uint4 qf[D / 32], gf[D / 32];
    load_frags<T, D>(bh_ptr(args.q, args.lq, t.b, t.h), vol_off(args.lq, ln.pos), ln.valid, grp, qf);
    load_frags<T, D>(bh_ptr(args.dout, args.ldo, t.b, t.h), vol_off(args.ldo, ln.pos), ln.valid, grp, gf);
    const float L2 = ln.valid ? bh_ptr(args.lse, args.ll, t.b, t.h)[vol_off(args.ll, ln.pos)] * kLog2e : 0.f;
    const float dl = ln.valid && args.dlse ? bh_ptr(args.dlse, args.ldl, t.b, t.h)[vol_off(args.ldl, ln.pos)] : 0.f;
    f32x4_t cb[2];
    band_colbias(ln, grp, cb);
    BandOff<D> off;
    off.init(lane);
    const float sc2 = p.scale * kLog2e;
    const int wc0 = t.a[1].glo, wc1 = t.wave_ok() ? t.a[1].ghi : -1;
    const f32x4_t zero[2] = {f32x4_t{0.f, 0.f, 0.f, 0.f}, f32x4_t{0.f, 0.f, 0.f, 0.f}};

    f32x4_t acc[D / 16];
#pragma unroll
    for (int db = 0; db < D / 16; ++db) acc[db] = f32x4_t{0.f, 0.f, 0.f, 0.f};
    float part = 0.f, di = 0.f;
    float pmax = 0.f, gs = 1.f;  // scaled: largest |P dP|, and dS's factor
    int bi = 0, pass = 0;
    const auto step = [&](auto BC) {
        constexpr int B = decltype(BC)::value;
        st.store(smem + B * BUF);
        lds_publish_barrier();
        const int c0 = bi * NC, cpass = pass;
        if (++bi == nb) {
            bi = 0;
            ++pass;
        }
        const bool more = pass < 2;
        if (more) load(bi);
        const unsigned char* Kb = smem + B * BUF;
        const unsigned char* Vb = Kb + kBandOp<D>;
#pragma unroll kBandUnroll<D, TWO>
        for (int c = 0; c < NC; ++c) {
            if (c0 + c < wc0 || c0 + c > wc1) continue;
            const int row = c0 + c - ln.rlo;
            const float o = static_cast<unsigned>(row) < static_cast<unsigned>(ln.rn) ? -L2 : -INFINITY;
            f32x4_t s[2], dp[2];
            band_score<T, D>(Kb, off, c, qf, cb, s);
            band_score<T, D>(Vb, off, c, gf, zero, dp);
            if (cpass == 0) {
                if constexpr (kScaled<T, TWO>) {
#pragma unroll
                    for (int i = 0; i < 8; ++i) {
                        const float e = __builtin_amdgcn_exp2f(fmaf(s[i >> 2][i & 3], sc2, o)), x = dp[i >> 2][i & 3];
                        part = fmaf(e, x, part);
                        pmax = fmaxf(pmax, __builtin_fabsf(e * x));
                    }
                } else {
                    part = delta_part(s, dp, sc2, o, part);
                }
            } else {
#pragma unroll
                for (int bb = 0; bb < 2; ++bb)
#pragma unroll
                    for (int i = 0; i < 4; ++i)
                        s[bb][i] = __builtin_amdgcn_exp2f(fmaf(s[bb][i], sc2, o)) *
                                   (kScaled<T, TWO> ? fmaf(dp[bb][i], gs, -gs * di) : dp[bb][i] - di);
                band_accumulate<T, D, TWO>(Kb, off, c, s, acc);
            }
        }
        if (pass == 1 && cpass == 0) {
            di = sum_rows(part) - dl;
            if (ln.valid && !(__builtin_fabsf(di) <= __FLT_MAX__))
                di = exact_dot<T, D>(bh_ptr(args.dout, args.ldo, t.b, t.h) + vol_off(args.ldo, ln.pos),
                                     bh_ptr(args.o, args.lo, t.b, t.h) + vol_off(args.lo, ln.pos)) -
                     dl;
            if (ln.valid && grp == 0) bh_ptr(args.delta_out, args.lde, t.b, t.h)[vol_off(args.lde, ln.pos)] = di;
            // |dS| <= |P dP| + |delta|, as P <= 1
            if constexpr (kScaled<T, TWO>) gs = scale_for(max_rows_num(pmax) + __builtin_fabsf(di));
        }
        return more;
    };
#pragma unroll 1
    while (step(std::integral_constant<int, 0>{}) && step(std::integral_constant<int, 1>{})) {
    }
    const bool redo = ln.valid && item_nonfinite(lane_sum(acc, 0.f));
    if (ln.valid)
        store_rows<T, D>(bh_ptr(args.dq, args.ldq, t.b, t.h), vol_off(args.ldq, ln.pos), grp, acc,
                         kScaled<T, TWO> ? p.scale * inv_pow2(gs) : p.scale);
    if (redo)
        band_redo_bwd_q<T, D>(kernargs(), t.b, t.h, hk, opaque(ln.pos[0]), opaque(ln.pos[1]), opaque(ln.pos[2]), grp);
}

// Backward, key side: as k_bwd_kv_mfma; the walk covers every q head of the
// kv head's group.  Per slot of a band: -lse log2 e and -delta in LDS, and 8
// -inf entries that lanes failing the row test read instead.
template <typename T, int D>
__device__ __forceinline__ void band_redo_bwd_kv(const void* kargs, int b, int hk, int p0, int p1, int p2, int grp) {
    const BandArgs<T>& A = *static_cast<const BandArgs<T>*>(kargs);
    const int pos[3] = {p0, p1, p2};
    ExactAxis x[3];
    for (int a = 0; a < 3; ++a) x[a] = exact_axis(A.p.ax[a], pos[a]);
    const T* kr = bh_ptr(A.k, A.lk, b, hk) + vol_off(A.lk, pos);
    const T* vr = bh_ptr(A.v, A.lv, b, hk) + vol_off(A.lv, pos);
    const int rep = A.p.rep;
    f32x4_t g[D / 16];
    exact_zero(g);
#pragma unroll 1
    for (int h = hk * rep; h < (hk + 1) * rep; ++h)
        exact_backward_kv<T, D, true>(A.p.scale, x, kr, vr, bh_ptr(A.q, A.lq, b, h), strides3(A.lq),
                                      bh_ptr(A.dout, A.ldo, b, h), strides3(A.ldo), bh_ptr(A.lse, A.ll, b, h),
                                      strides3(A.ll), bh_ptr(A.delta, A.lde, b, h), strides3(A.lde), grp, g);
    store_rows<T, D>(bh_ptr(A.dv, A.ldv, b, hk), vol_off(A.ldv, pos), grp, g, 1.f);
    exact_zero(g);
#pragma unroll 1
    for (int h = hk * rep; h < (hk + 1) * rep; ++h)
        exact_backward_kv<T, D, false>(A.p.scale, x, kr, vr, bh_ptr(A.q, A.lq, b, h), strides3(A.lq),
                                       bh_ptr(A.dout, A.ldo, b, h), strides3(A.ldo), bh_ptr(A.lse, A.ll, b, h),
                                       strides3(A.ll), bh_ptr(A.delta, A.lde, b, h), strides3(A.lde), grp, g);
    store_rows<T, D>(bh_ptr(A.dk, A.ldk, b, hk), vol_off(A.ldk, pos), grp, g, A.p.scale);
}

template <typename T, int D, bool TWO>
__global__ __launch_bounds__(kBandThreads) NA_BAND_OCC(D, true) void k_band_bwd_kv(BandArgs<T> args) {
    constexpr int NC = kBandChunks<D>, BUF = 2 * kBandOp<D>, NS = NC * 32;
    const Prob& p = args.p;
    unsigned char* smem = lds_base();
    float* scal = reinterpret_cast<float*>(smem + 2 * BUF);  // per buffer NS (-lse), NS (-delta); then 8 x -inf
    const int lane = threadIdx.x & 63, col = lane & 15, grp = lane >> 4;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const BandTile t = band_tile<true>(p, args.g, wave);
    if (!t.tile_ok()) return;
    const BandLane ln = band_lane<true>(p, args.g, t, wave, col);
    const int U1 = t.a[1].U, U2 = t.a[2].U;
    f32x4_t gk[D / 16], gv[D / 16];
#pragma unroll
    for (int db = 0; db < D / 16; ++db) gk[db] = gv[db] = f32x4_t{0.f, 0.f, 0.f, 0.f};
    float gs = scale_for(0.f);  // scaled: the factor of P' dP' = 2^15 dS
    const auto store = [&]() {
        constexpr bool S = kScaled<T, TWO>;
        store_rows<T, D>(bh_ptr(args.dk, args.ldk, t.b, t.h), vol_off(args.ldk, ln.pos), grp, gk,
                         S ? p.scale * (1.f / kScaleP) * inv_pow2(gs) : p.scale);
        store_rows<T, D>(bh_ptr(args.dv, args.ldv, t.b, t.h), vol_off(args.ldv, ln.pos), grp, gv,
                         S ? 1.f / kScaleP : 1.f);
    };
    if (U1 == 0 || U2 == 0) {  // no query attends these keys
        if (ln.valid) store();
        return;
    }
    const int rep = static_cast<int>(args.g.rep.d);
    BandStage<T, D> st;
    st.init(p, t, args.lq, args.ldo);
    const int nb = (U1 + NC - 1) / NC;
    // the thread's slot of a band (threads past NS load slot 0's scalars and drop them)
    const int sslot = threadIdx.x < NS ? static_cast<int>(threadIdx.x) : 0;
    const int srow = sslot / 32, scol = sslot % 32;
    const bool sin = scol < U2;
    const int q2 = t.r[2] + (t.a[2].lo + (sin ? scol : 0)) * p.ax[2].dil;
    const int sl2 = q2 * args.ll.s2, sd2 = q2 * args.lde.s2;
    float pl, pd;
    bool pin;
    int h = t.h * rep, bi = 0;
    const auto load = [&]() {
        const int row = bi * NC + srow;
        pin = sin && row < U1;
        const int p1 = t.r[1] + (t.a[1].lo + (pin ? row : 0)) * p.ax[1].dil;
        pl = bh_ptr(args.lse, args.ll, t.b, h)[p1 * args.ll.s1 + sl2];
        pd = bh_ptr(args.delta, args.lde, t.b, h)[p1 * args.lde.s1 + sd2];
        st.load(band_rsrc(bh_ptr(args.q, args.lq, t.b, h), args.ab),
                band_rsrc(bh_ptr(args.dout, args.ldo, t.b, h), args.bb), bi, U1);
    };
    load();

    uint4 kf[D / 32], vf[D / 32];
    load_frags<T, D>(bh_ptr(args.k, args.lk, t.b, t.h), vol_off(args.lk, ln.pos), ln.valid, grp, kf);
    load_frags<T, D>(bh_ptr(args.v, args.lv, t.b, t.h), vol_off(args.lv, ln.pos), ln.valid, grp, vf);
    if (threadIdx.x < 8) scal[4 * NS + threadIdx.x] = -INFINITY;
    f32x4_t cb[2];
    band_colbias(ln, grp, cb);
    BandOff<D> off;
    off.init(lane);
    const float sc2 = p.scale * kLog2e;
    const int wc0 = t.a[1].glo, wc1 = t.wave_ok() ? t.a[1].ghi : -1;
    const int hend = (t.h + 1) * rep;
    const float* ninf = scal + 4 * NS;
    const auto step = [&](auto BC) {
        constexpr int B = decltype(BC)::value;
        st.store(smem + B * BUF);
        if (threadIdx.x < NS) {
            scal[B * 2 * NS + threadIdx.x] = pin ? -pl * kLog2e : 0.f;
            scal[B * 2 * NS + NS + threadIdx.x] = pin ? -pd : 0.f;
        }
        lds_publish_barrier();
        const int c0 = bi * NC;
        if (++bi == nb) {
            bi = 0;
            ++h;
        }
        const bool more = h < hend;
        if (more) load();
        const unsigned char* Qb = smem + B * BUF;
        const unsigned char* Gb = Qb + kBandOp<D>;
#pragma unroll kBandUnroll<D, TWO>
        for (int c = 0; c < NC; ++c) {
            if (c0 + c < wc0 || c0 + c > wc1) continue;
            const int row = c0 + c - ln.rlo;
            const float* sc = scal + B * 2 * NS + 32 * c + 8 * grp;
            const float* nlc = static_cast<unsigned>(row) < static_cast<unsigned>(ln.rn) ? sc : ninf;
            const f32x4_t nl[2] = {*reinterpret_cast<const f32x4_t*>(nlc),
                                   *reinterpret_cast<const f32x4_t*>(nlc + 4)};
            const f32x4_t nd[2] = {*reinterpret_cast<const f32x4_t*>(sc + NS),
                                   *reinterpret_cast<const f32x4_t*>(sc + NS + 4)};
            f32x4_t s[2], dp[2];
            band_score<T, D>(Qb, off, c, kf, cb, s);
            band_score<T, D>(Gb, off, c, vf, nd, dp);
#pragma unroll
            for (int bb = 0; bb < 2; ++bb)
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    s[bb][i] = __builtin_amdgcn_exp2f(fmaf(s[bb][i], sc2, nl[bb][i]));
                    if constexpr (kScaled<T, TWO>) s[bb][i] *= kScaleP;
                    dp[bb][i] *= s[bb][i];
                }
            if constexpr (kScaled<T, TWO>) {
                // a new maximum past the limit lowers the item's factor (and what
                // it has gathered), as the forward's online softmax does
                const float mx = abs_max8(dp, 0.f);
                if (__any(mx * gs >= kScaleLimit)) {
                    const float m = max_rows_num(mx), ng = m * gs >= kScaleLimit ? scale_for(m) : gs;
                    const float corr = ng * inv_pow2(gs);
                    gs = ng;
#pragma unroll
                    for (int db = 0; db < D / 16; ++db) gk[db] *= corr;
                }
#pragma unroll
                for (int i = 0; i < 8; ++i) dp[i >> 2][i & 3] *= gs;
            }
            band_accumulate<T, D, TWO>(Gb, off, c, s, gv);
            band_accumulate<T, D, TWO>(Qb, off, c, dp, gk);
        }
        return more;
    };
#pragma unroll 1
    while (step(std::integral_constant<int, 0>{}) && step(std::integral_constant<int, 1>{})) {
    }
    const bool redo = ln.valid && item_nonfinite(lane_sum(gk, lane_sum(gv, 0.f)));
    if (ln.valid) store();
    if (redo)
        band_redo_bwd_kv<T, D>(kernargs(), t.b, t.h, opaque(ln.pos[0]), opaque(ln.pos[1]), opaque(ln.pos[2]), grp);
}

// ---------------------------------------------------------------------------
// Host side.
// ---------------------------------------------------------------------------

BandGeo band_geo(const Prob& p, int sh2, int heads) {
    BandGeo g{};
    g.sh2 = sh2;
    g.sh1 = log2_of(kBandWaves * 16) - sh2;
    const int T[3] = {1, 1 << g.sh1, 1 << g.sh2};
    long long tiles = 1;
    for (int a = 1; a < 3; ++a) {
        const int n = (n_class_h(p.ax[a], 0) + T[a] - 1) / T[a];
        g.lenmod[a] = p.ax[a].len % p.ax[a].dil;
        g.nt[a] = make_fastdiv(static_cast<uint32_t>(n));
        g.dil[a] = make_fastdiv(static_cast<uint32_t>(p.ax[a].dil));
        tiles *= static_cast<long long>(n) * p.ax[a].dil;
    }
    g.tiles = make_fastdiv(static_cast<uint32_t>(tiles));
    g.heads = make_fastdiv(static_cast<uint32_t>(heads));
    g.rep = make_fastdiv(static_cast<uint32_t>(p.rep));
    return g;
}

long long band_blocks(const Prob& p, const BandGeo& g) {
    return static_cast<long long>(p.B) * g.heads.d * g.tiles.d;
}

uint32_t band_plane(const Prob& p, const Lay& l, int D) {
    return static_cast<uint32_t>(((static_cast<long long>(p.ax[1].len) - 1) * l.s1 +
                                  (static_cast<long long>(p.ax[2].len) - 1) * l.s2 + D) * 2);
}

template <typename T, int D>
constexpr size_t kBandLds = kLdsPad + 4 * kBandOp<D>;
template <typename T, int D>
constexpr size_t kBandLdsKv = kBandLds<T, D> + (4 * kBandChunks<D> * 32 + 8) * sizeof(float);

template <typename T, int D>
void band_audit_dim(LdsAudit& a) {
    audit_one(k_band_fwd<T, D, false>, "k_band_fwd", a);
    audit_one(k_band_fwd<T, D, true>, "k_band_fwd", a);
    audit_one(k_band_bwd_q<T, D, false>, "k_band_bwd_q", a);
    audit_one(k_band_bwd_q<T, D, true>, "k_band_bwd_q", a);
    audit_one(k_band_bwd_kv<T, D, false>, "k_band_bwd_kv", a);
    audit_one(k_band_bwd_kv<T, D, true>, "k_band_bwd_kv", a);
}

// No static LDS in any instance (see lds_base): checked once per process.
bool band_static_lds_ok() {
    static const bool ok = [] {
        LdsAudit a;
        band_audit_dim<bf16, 32>(a);
        band_audit_dim<bf16, 64>(a);
        band_audit_dim<bf16, 128>(a);
        band_audit_dim<f16, 32>(a);
        band_audit_dim<f16, 64>(a);
        band_audit_dim<f16, 128>(a);
        return a.bad == 0;
    }();
    return ok;
}

// NATTEN_HIP_BAND: 0 keeps every call off these kernels, 1 puts every call
// that they can serve on them (tuning, tests); else band_pays decides.
int band_forced() {
    const char* e = std::getenv("NATTEN_HIP_BAND");
    return !e ? -1 : std::strcmp(e, "0") == 0 ? 0 : std::strcmp(e, "1") == 0 ? 1 : -1;
}

template <typename T, int D>
hipError_t band_fwd_run(const Prob& p, const void* q, Lay lq, const void* k, Lay lk, const void* v, Lay lv, void* o,
                        Lay lo, float* lse, Lay ll, bool two, hipStream_t s) {
    BandArgs<T> a{};
    a.p = p;
    a.g = band_geo(p, band_columns(p.ax[2].k, false), p.Hq);
    a.q = static_cast<const T*>(q);
    a.k = static_cast<const T*>(k);
    a.v = static_cast<const T*>(v);
    a.out = static_cast<T*>(o);
    a.lse_out = lse;
    a.lq = to_k(lq);
    a.lk = to_k(lk);
    a.lv = to_k(lv);
    a.lo = to_k(lo);
    a.ll = to_k(ll);
    a.ab = band_plane(p, lk, D);
    a.bb = band_plane(p, lv, D);
    auto kern = two ? k_band_fwd<T, D, true> : k_band_fwd<T, D, false>;
    const hipError_t e = allow_lds(kern, kBandLds<T, D>);
    if (e != hipSuccess) return e;
    NA_LAUNCH("na_fwd_band", kern, dim3(static_cast<unsigned>(band_blocks(p, a.g))), dim3(kBandThreads),
              (kBandLds<T, D>), s, a);
    return hipGetLastError();
}

template <typename T, int D>
hipError_t band_bwd_run(const Prob& p, const void* q, Lay lq, const void* k, Lay lk, const void* v, Lay lv,
                        const void* o, Lay lo, const void* dout, Lay ldo, const float* lse, Lay ll, const float* dlse,
                        Lay ldl, void* dq, Lay ldq, void* dk, Lay ldk, void* dv, Lay ldv, float* delta, Lay lde,
                        int sides, bool two, hipStream_t s) {
    BandArgs<T> a{};
    a.p = p;
    a.g = band_geo(p, band_columns(p.ax[2].k, false), p.Hq);
    a.q = static_cast<const T*>(q);
    a.k = static_cast<const T*>(k);
    a.v = static_cast<const T*>(v);
    a.o = static_cast<const T*>(o);
    a.dout = static_cast<const T*>(dout);
    a.lse = lse;
    a.dlse = dlse;
    a.delta = delta;
    a.delta_out = delta;
    a.dq = static_cast<T*>(dq);
    a.dk = static_cast<T*>(dk);
    a.dv = static_cast<T*>(dv);
    a.lq = to_k(lq);
    a.lk = to_k(lk);
    a.lv = to_k(lv);
    a.lo = to_k(lo);
    a.ldo = to_k(ldo);
    a.ldq = to_k(ldq);
    a.ldk = to_k(ldk);
    a.ldv = to_k(ldv);
    a.ll = to_k(ll);
    a.lde = to_k(lde);
    a.ldl = to_k(ldl);
    a.ab = band_plane(p, lk, D);
    a.bb = band_plane(p, lv, D);
    hipError_t e;
    if (sides & kQuerySide) {
        auto kq = two ? k_band_bwd_q<T, D, true> : k_band_bwd_q<T, D, false>;
        if ((e = allow_lds(kq, kBandLds<T, D>)) != hipSuccess) return e;
        NA_LAUNCH("na_bwd_q_band", kq, dim3(static_cast<unsigned>(band_blocks(p, a.g))), dim3(kBandThreads),
                  (kBandLds<T, D>), s, a);
        if ((e = hipGetLastError()) != hipSuccess) return e;
    }
    if (!(sides & kKeySide)) return hipSuccess;
    a.g = band_geo(p, band_columns(p.ax[2].k, true), p.Hkv);
    a.ab = band_plane(p, lq, D);
    a.bb = band_plane(p, ldo, D);
    auto kk = two ? k_band_bwd_kv<T, D, true> : k_band_bwd_kv<T, D, false>;
    if ((e = allow_lds(kk, kBandLdsKv<T, D>)) != hipSuccess) return e;
    NA_LAUNCH("na_bwd_kv_band", kk, dim3(static_cast<unsigned>(band_blocks(p, a.g))), dim3(kBandThreads),
              (kBandLdsKv<T, D>), s, a);
    return hipGetLastError();
}

#define NA_BAND_DISPATCH(RUN, ...)                              \
    if (dtype == NATTEN_BF16) {                                 \
        if (p.Dqk == 32) return RUN<bf16, 32>(__VA_ARGS__);     \
        if (p.Dqk == 64) return RUN<bf16, 64>(__VA_ARGS__);     \
        return RUN<bf16, 128>(__VA_ARGS__);                     \
    }                                                           \
    if (p.Dqk == 32) return RUN<f16, 32>(__VA_ARGS__);          \
    if (p.Dqk == 64) return RUN<f16, 64>(__VA_ARGS__);          \
    return RUN<f16, 128>(__VA_ARGS__)

}  // namespace

// The sides of a problem that run on these kernels: 2-D (axis 0 of extent 1)
// at stride 1, 16-bit, head dim 32 / 64 / 128 for q, k and v, in-plane
// kernel of 2 to 16 columns (so that a tile's union fits 32), and
// * both sides for 10 to 16 columns (past the 8x8 tile kernels), and at head
//   dim 128 from 8: there the general tiles' border unions cross 16 columns
//   and their rows double (9 x 9, 8 x 64 x 64 x 4 heads: forward 97 -> 54
//   us, the backward left the tiles, 995 + 950 -> 124 + 111 us; at 7 x 7 both
//   are level, 57 + 76 + 90 against 58 + 99 + 87);
// * the key side alone where the 8x8 tiles serve the query side but some key
//   tile's union does not fit them (`lean`: they take the problem; 9 x 9, 8 x
//   64 x 64 x 8: dK/dV 222 -> 49 us at head dim 32, 613 -> 107 at 64; 7 x 7
//   on 32 x 22 x 22 x 8: 57 -> 37).
// Where the general tiles hold the problem too, band_pays decides per kernel.
// Where the general tiles cannot hold the problem either, the alternative is
// the vector kernels, whose probabilities and their gradients stay in fp32:
// there they enter the matrix products as two 16-bit terms (TWO; the rest
// after rounding is the second), which keeps 16 (fp16, scaled: 22) of their
// bits, and the row sums stay in fp32.  The callers ask for it (`two`).
// `lays`: every 16-bit operand and fp32 row operand of the call.  The answer
// depends on the problem alone, never on which tables exist.
int band_sides(const Prob& p, int dtype, bool aligned, bool lean, std::initializer_list<Lay> lays) {
    if (!aligned || dtype == NATTEN_F32 || !(p.scale > 0.f)) return 0;
    if (p.Dqk != p.Dv || (p.Dqk != 32 && p.Dqk != 64 && p.Dqk != 128)) return 0;
    if (p.ax[0].len != 1 || p.ax[0].k != 1) return 0;
    for (int a = 0; a < 3; ++a)
        if (p.ax[a].st != 1 || p.ax[a].len >= (1 << 24)) return 0;
    if (band_columns(p.ax[2].k, true) < 0) return 0;
    // a tile has at least 8 rows: fewer would leave its waves idle
    if (n_class_h(p.ax[1], 0) < 8) return 0;
    const bool both = p.ax[2].k >= (p.Dqk == 128 ? 8 : 10);
    if (!both && !(lean && !lean_key_tiles_fit(p))) return 0;
    if (!offsets_fit(p, lays)) return 0;
    for (const Lay& l : lays)
        if (band_plane(p, l, p.Dqk) >= kBandOOR) return 0;
    const long long tiles = ((static_cast<long long>(p.ax[1].len) + 7) / 8 + p.ax[1].dil) *
                            ((static_cast<long long>(p.ax[2].len) + 7) / 8 + p.ax[2].dil);
    if (tiles * p.B * p.Hq >= (1LL << 31) || !band_static_lds_ok() || band_forced() == 0) return 0;
    return both ? kQuerySide | kKeySide : kKeySide;
}

// A workgroup here owns 128 items and walks rows of 32 slots, 16 of them idle
// where a class is that narrow, so small grids, short windows and small
// classes are faster on the general tiles.  The line, over 4080 timed pairs (a
// kernel each; 16 x 16 to 128 x 128 at dilation 1 to 4, windows of 3 x 8 to
// 16 x 16, 1 to 256 heads in all, bf16):
// * the general tiles stage enough in all: below 300 / 150 / 130 thousand slots
//   (head dim 32 / 64 / 128) both are bound by one workgroup's latency, which
//   is longer here (one 64 x 64 image, 1 head, dim 64, 13 x 13 under dilation
//   4: forward 6.8 against 11.1 us, backward 16 against 35);
// * their tile is past 64 KB of LDS (one workgroup per CU, nothing overlaps)
//   and they stage more slots than these kernels, or at dim 128 about as many
//   (forward, 256 heads of 20 x 20, 9 x 9: 100 against 58 us at 0.94 of the
//   slots), but not dQ, whose registers leave one workgroup per CU here too;
// * or it has fallen to 32 items or fewer and they stage 1.5 times the slots
//   (backward: 2.1 times).
// Over those pairs the choice is within 0.9 % of the faster kernel's time on
// average (kernel by kernel), and above the general tiles' by more than 5 %
// in 8 of them (at most 23 %).
bool band_pays(const Prob& p, FusedKernel kernel, const TileLoad& general) {
    if (band_forced() == 1) return true;
    const bool key = kernel == kFusedKey;
    if (general.slots <= (p.Dqk == 32 ? 300000 : p.Dqk == 64 ? 150000 : 130000)) return false;
    const BandGeo g = band_geo(p, band_columns(p.ax[2].k, key), key ? p.Hkv : p.Hq);
    const long long slots = band_blocks(p, g) * 32 * union_extent(p.ax[1], 1 << g.sh1, key) * (key ? p.rep : 1);
    if (general.lds > 64 * 1024) {
        const bool wide = p.Dqk == 128 && kernel != kFusedQuery;
        return 20 * general.slots > (wide ? 17 : 22) * slots;
    }
    return general.items <= 32 && 10 * general.slots > (kernel == kFusedForward ? 15 : 21) * slots;
}

hipError_t band_forward(const Prob& p, const void* q, Lay lq, const void* k, Lay lk, const void* v, Lay lv, void* o,
                        Lay lo, float* lse, Lay ll, int dtype, hipStream_t s, bool two) {
    NA_BAND_DISPATCH(band_fwd_run, p, q, lq, k, lk, v, lv, o, lo, lse, ll, two, s);
}

hipError_t band_backward(const Prob& p, const void* q, Lay lq, const void* k, Lay lk, const void* v, Lay lv,
                         const void* o, Lay lo, const void* dout, Lay ldo, const float* lse, Lay ll, const float* dlse,
                         Lay ldl, void* dq, Lay ldq, void* dk, Lay ldk, void* dv, Lay ldv, float* delta, Lay lde,
                         int dtype, hipStream_t s, int sides, bool two) {
    NA_BAND_DISPATCH(band_bwd_run, p, q, lq, k, lk, v, lv, o, lo, dout, ldo, lse, ll, dlse, ldl, dq, ldq, dk, ldk, dv,
                     ldv, delta, lde, sides, two, s);
}

}  // namespace na
