// Pair tiles over the dense nodes (gfx950).
//
// Every dense node is held by a sizeable share of the samples, so every pair
// block visits it: the kernels are dense contractions with |x_i - x_j| in
// place of the product, which no matrix instruction forms.  They are laid out
// like a vector-ALU GEMM: a tile is a workgroup of 2 x 2 waves, a lane holding its
// rows and columns in groups of 16 bytes, a group apart from the next lane's, so that
// its operands are ds_read_b128 of 8 distinct contiguous pieces (no bank conflicts,
// each piece broadcast to 8 lanes).  Node rows go from memory to LDS by
// global_load_lds, 16 bytes per lane, a stage of nodes ahead.  Only the scaled FP32
// weighted kernel waits for them at the barrier: in the others the next nodes' indices
// and lengths (or, with a rolled node loop, the first read of a stage buffer that the
// compiler cannot tell from the other one) have a wave wait before its terms, and what
// overlaps the loads are the terms of the CU's other waves.
#include "ssu_devmath.hpp"
#include "ssu_tiles.hpp"

#include <algorithm>

namespace ssu {

namespace {

constexpr uint32_t N_XCDS = 8;

#define SSU_GLOBAL(p) ((const __attribute__((address_space(1))) void*)(p))
#define SSU_LDS(p) ((__attribute__((address_space(3))) void*)(p))

// nodes [a, b) of part p of np: whole stages of eb nodes
__device__ __forceinline__ void part_range(uint32_t nd, uint32_t eb, uint32_t p, uint32_t np, uint32_t& a, uint32_t& b) {
    const uint32_t st = (nd + eb - 1) / eb;
    a = (uint32_t)((uint64_t)st * p / np) * eb;
    b = min(nd, (uint32_t)((uint64_t)st * (p + 1) / np) * eb);
    a = min(a, nd);
}

// ------------------------------------------------------------------ terms
//
// An operation says what a lane holds and how a node's values enter a pair:
//   V        operand type; FP32 sums are merged into FP64 every MERGE nodes
//   RL, CL   rows and columns a lane holds, so a tile has 16 RL x 16 CL pairs, WAVES of them per SIMD
//            (8 x 8 at two waves; with two sums per pair 4 x 4 at three or four, which hide the
//            transcendentals' latency: 8 rows by 4 at two took 15 to 20% longer for the VAW terms)
//   EB       nodes per LDS stage (two stages are resident), UNROLL of them in one loop body
//   TWO      a denominator is summed beside the numerator
//   LEN      the node's length is staged too (otherwise U's rows are scaled by it)
//   COUNTS   the samples' counts are staged in the last of PANELS panels, and the pair's totals used (VAW)
//   prep     what a lane does to a value it reads
constexpr uint32_t MERGE = 64;

// the distance from numerator and denominator and the rare nodes' shares of them
// (0 / 0, no node held by either sample: NaN)
__device__ __forceinline__ double ratio(double nm, double dn, double share, double share2, bool normalized) {
    nm += share;
    nm = nm < 0.0 ? 0.0 : nm;   // the shares' rounding can undershoot 0
    return normalized ? nm / (dn + share2) : nm;
}

// FP32 weighted: |l u - l v|, two instructions at the full FP32 rate (register
// operands only: an SGPR operand halves it, as do min, max and v_sad_u32).
// Bound by VALU issue: 16,384 samples x 9,790 dense nodes in 44.9 ms, 2.94e13
// terms/s of the 3.1e13 that sub + add reach in registers at two waves per SIMD;
// 32 x 64 pairs per wave with lengths in the term, three LDS reads for 32 terms,
// took 70.4 ms.  SCALED = false: l |u - v| of plain rows, for trees with a negative
// length, whose sign |l u - l v| would lose.
template <bool SCALED> struct OpW32 {
    typedef float V;
    static constexpr int RL = 8, CL = 8, WAVES = 2, EB = 16, UNROLL = 16;
    static constexpr bool TWO = false, LEN = !SCALED, COUNTS = false, FLAGS = false;
    static constexpr uint32_t PANELS = 1;
    static __device__ __forceinline__ float prep(float u) { return u; }
    static __device__ __forceinline__ void term(float u, float v, float l, float& num) {
        if constexpr (SCALED) num += __builtin_fabsf(u - v);
        else num = __builtin_fmaf(__builtin_fabsf(u - v), l, num);
    }
    // d from the tile's sums x, y and the rare nodes' shares of them
    static __device__ __forceinline__ double distance(double x, double, double share, double, double tot,
                                                      bool normalized) {
        x += share;
        x = x < 0.0 ? 0.0 : x;   // the share's rounding can undershoot 0; NaN (empty samples) passes
        return normalized ? x / tot : x;
    }
};

// FP64 weighted: M = sum of l min(u, v), of which the distance is S_i + S_j - 2 M
// (u, v >= 0; v_min_f64 without the NaN quieting the compiler adds for values it
// does not see produced).  3,001 samples x 3,700 dense nodes in 1.62 ms, 1.1e13
// terms/s: 58% of the 1.9e13 at which the two instructions issue (half the FP32 rate);
// the rest are the waits for a v_min's result in the instruction after it and for the
// next stage.  64 x 64 blocks of one wave took 2.66 ms; 131 samples 0.37 -> 0.04 ms,
// the parts filling the device.
struct OpW64 {
    typedef double V;
    static constexpr int RL = 8, CL = 8, WAVES = 2, EB = 8, UNROLL = 8;
    static constexpr bool TWO = false, LEN = true, COUNTS = false, FLAGS = false;
    static constexpr uint32_t PANELS = 1;
    static __device__ __forceinline__ double prep(double u) { return u; }
    static __device__ __forceinline__ void term(double u, double v, double l, double& num) {
        double m;
        asm("v_min_f64 %0, %1, %2" : "=v"(m) : "v"(u), "v"(v));
        num = __builtin_fma(m, l, num);
    }
    static __device__ __forceinline__ double distance(double m, double, double share, double, double tot,
                                                      bool normalized) {
        double x = tot - 2.0 * (m + share);
        x = x < 0.0 ? 0.0 : x;
        return normalized ? x / tot : x;
    }
};

// s^(a-1) for s >= 0, finite at s = 0 (the terms it weighs are 0 there).  AL
// picks the power: 0 any a (FP32: hardware log2 / exp2), 1 a = 1/2 (reciprocal
// square root), 2 a = 1.
template <int AL> __device__ __forceinline__ float pow_less_one(float s, float a) {
    const float ss = fmaxf(s, 1.17549435e-38f);
    if constexpr (AL == 2) return 1.0f;
    else if constexpr (AL == 1) return __builtin_amdgcn_rsqf(ss);
    else return __builtin_amdgcn_exp2f((a - 1.0f) * __builtin_amdgcn_logf(ss));
}
template <int AL> __device__ __forceinline__ double pow_less_one(double s, double a) {
    const double ss = s > 0.0 ? s : 1.0;
    if constexpr (AL == 2) return 1.0;
    else if constexpr (AL == 1) return rsqrt_nr<2>(ss);
    else return dpow64(ss, a - 1.0);
}

// Generalized (src/unifrac_task_impl.hpp:1016-1024): num += l s^a |u - v| / s,
// den += l s^a with s = u + v, both from the one power s^(a-1) (its error is
// then the same in both and largely leaves the ratio).  Bound by VALU issue, the
// transcendental at a quarter of the add's rate: 4,000 samples x 1,930 dense
// nodes, a = 1/2 in 3.76 ms, a = 1 in 1.25 ms, other a in 4.3 ms (several pairs'
// powers in step measured the same).  32 x 64 pairs per wave with two powers per
// term took 1.8 times as long.
template <class T, int AL> struct OpGen {
    typedef T V;
    static constexpr int RL = 4, CL = 4, WAVES = 4, EB = sizeof(T) == 4 ? 16 : 8, UNROLL = 1;
    static constexpr bool TWO = true, LEN = true, COUNTS = false, FLAGS = false;
    static constexpr uint32_t PANELS = 1;
    static __device__ __forceinline__ T prep(T u) { return u; }
    static __device__ __forceinline__ void term(T u, T v, T l, T alpha, T& num, T& den) {
        const T s = u + v;
        const T q = pow_less_one<AL>(s, alpha);
        num = __builtin_elementwise_fma(__builtin_elementwise_abs(u - v) * q, l, num);
        den = __builtin_elementwise_fma(s * q, l, den);
    }
    static __device__ __forceinline__ double distance(double x, double y, double share, double share2, double, bool) {
        return ratio(x, y, share, share2, true);
    }
};

// VAW (src/unifrac_task_impl.hpp:881-893, 1098-1109, 1817-1829): each node's
// terms over vaw = sqrt(mi (m - mi)), mi = c_i + c_j, m = T_i + T_j, and 0 where
// that is 0.  KIND 1: weighted, 2: presence (the counts are the one panel: a
// sample holds the node where its count is positive), 3: generalized (0 <= alpha
// <= 1: the weighted terms' quotients in the generalized terms).  Bound by VALU
// issue: 4,000 samples x 3,550 dense nodes in 7.8 ms (FP32), 1,500 samples 1.36 ms
// against 2.2 ms in whole 64 x 64 tiles (300 workgroups, node counts and totals in
// registers).
template <class T, int KIND, int AL = 0> struct OpVaw {
    typedef T V;
    static constexpr int RL = 4, CL = 4, WAVES = 3, EB = sizeof(T) == 4 ? 16 : 8, UNROLL = 1;
    static constexpr bool TWO = true, LEN = true, COUNTS = true, FLAGS = KIND == 1;
    static constexpr uint32_t PANELS = KIND == 2 ? 1 : 2;
    static __device__ __forceinline__ T prep(T u) { return KIND == 2 ? (u > T(0) ? T(1) : T(0)) : u; }
    static __device__ __forceinline__ float rsqrt(float x) { return __builtin_amdgcn_rsqf(x); }
    static __device__ __forceinline__ double rsqrt(double x) { return rsqrt_nr<2>(x); }
    // m - mi.  FP32 (whole counts, any two totals below 2^24: exact either way): from what
    // each sample's total leaves of its count, once per sample and node; FP64: m - mi itself
    // (the totals opaque here, or their 32 sums would be kept in registers across the nodes)
    static __device__ __forceinline__ float other(float t, float c) { return t - c; }
    static __device__ __forceinline__ double other(double t, double) {
        asm volatile("" : "+v"(t));
        return t;
    }
    static __device__ __forceinline__ float rest(float eu, float ev, float) { return eu + ev; }
    static __device__ __forceinline__ double rest(double tu, double tv, double mi) { return (tu + tv) - mi; }
    static __device__ __forceinline__ void term(T u, T v, T cu, T cv, T tu, T tv, T l, T alpha, T& num, T& den) {
        const T mi = cu + cv;
        const T x = mi * rest(tu, tv, mi);
        const T rv = rsqrt(x);   // (x = 0: not finite, and not taken)
        const T r = x > T(0) ? rv : T(0);
        if constexpr (KIND == 3) {
            const T s1 = (u + v) * r, d1 = __builtin_elementwise_abs(u - v) * r;
            const T q = pow_less_one<AL>(s1, alpha);
            num = __builtin_elementwise_fma(d1 * q, l, num);
            den = __builtin_elementwise_fma(s1 * q, l, den);
        } else {
            const T t = l * r;
            num = __builtin_elementwise_fma(__builtin_elementwise_abs(u - v), t, num);
            const T o = KIND == 2 ? (u > v ? u : v) : u + v;
            den = __builtin_elementwise_fma(o, t, den);
        }
    }
    static __device__ __forceinline__ double distance(double x, double y, double share, double share2, double,
                                                      bool normalized) {
        return ratio(x, y, share, share2, normalized);
    }
};

template <class OP> struct Shape {
    typedef typename OP::V V;
    static constexpr uint32_t ROWS = 16 * OP::RL, COLS = 16 * OP::CL;   // of a tile: 2 x 2 waves
    static constexpr uint32_t WAVE_ROWS = 8 * OP::RL, WAVE_COLS = 8 * OP::CL;
    static constexpr uint32_t NODE = ROWS + COLS;               // staged values of a node (and as many counts)
    static constexpr uint32_t PAIRS = OP::RL * OP::CL;          // of a lane
    static constexpr uint32_t SLOT = PAIRS * (OP::TWO ? 2 : 1) * 256;   // doubles of a workspace slot
    static constexpr bool MIXED = sizeof(V) == 4;
    static constexpr uint32_t G = 16 / sizeof(V);               // values of one 16-byte LDS read
    static_assert(SLOT * sizeof(double) == tile_slot_bytes(ROWS), "the workspace is sized by the tile's rows");
    // the lane's q-th row in its wave's rows (l = li), or column in its wave's columns (l = lj)
    static __device__ __forceinline__ uint32_t at(uint32_t l, uint32_t q) { return q / G * (8 * G) + l * G + q % G; }
    // a lane's N values at(l, 0 .. N - 1) of a staged panel
    template <int N> static __device__ __forceinline__ void read(V (&x)[N], const V* panel, uint32_t l) {
        typedef __attribute__((ext_vector_type(G))) V vec;
#pragma unroll
        for (int h = 0; h < N / (int)G; ++h) {
            const vec v = *reinterpret_cast<const vec*>(panel + at(l, h * G));
#pragma unroll
            for (int z = 0; z < (int)G; ++z) x[h * G + z] = v[z];
        }
    }
};

// the distance of pair i < j, written to both triangles
template <class OP>
__device__ __forceinline__ void write_pair(const TileArgs& g, size_t i, size_t j, double x, double y) {
    typedef typename OP::V V;
    V* out = (V*)g.out;
    double share = 0.0, share2 = 0.0;   // the rare nodes', from the posting walk
    if (g.add_partial) {
        share = (double)out[i * g.n + j];
        if constexpr (OP::TWO) share2 = (double)((const V*)g.out2)[i * g.n + j];
    }
    const double tot = OP::TWO ? 0.0 : g.S[i] + g.S[j];
    const double d = OP::distance(x, y, share, share2, tot, g.normalized);
    if constexpr (OP::FLAGS) {
        // unnormalised: near-duplicates (distance below flag_tau of the pair's VAW
        // denominator) marked for the FP64 recomputation
        if (g.flags && g.band.has((uint32_t)(j - i)) && d < (double)g.flag_tau * (y + share2)) {
            g.flags[1 + i] = 1u;
            g.flags[1 + j] = 1u;
            atomicAdd(g.flags, 1u);
        }
    }
    out[i * g.n + j] = (V)d;
    out[j * g.n + i] = (V)d;
}

template <class OP>
__global__ void __launch_bounds__(256, OP::WAVES) k_tiles(TileArgs g) {
    typedef Shape<OP> SH;
    typedef typename OP::V V;
    constexpr int RL = OP::RL, CL = OP::CL;
    constexpr uint32_t EB = OP::EB, PANELS = OP::PANELS;
    const uint32_t seq = (blockIdx.x % N_XCDS) * g.per_xcd + blockIdx.x / N_XCDS;
    if (seq >= g.n_units) return;
    const uint32_t bij = g.units[seq].bij, part = g.units[seq].part;
    if (bij == TILE_NONE) return;
    const uint32_t bi = bij >> 16, bj = bij & 0xffffu;
    const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
    const uint32_t li = lane >> 3, lj = lane & 7, wr = (wave >> 1) * SH::WAVE_ROWS, wc = (wave & 1) * SH::WAVE_COLS;
    __shared__ __attribute__((aligned(16))) V sv[2][EB][PANELS][SH::NODE];   // a node: its rows, then its columns
    __shared__ V sl[2][EB];
    __shared__ __attribute__((aligned(16))) V st[OP::COUNTS ? SH::NODE : 1];

    const uint32_t nd = g.dlist[0];
    const uint32_t np = (part & 63u) + 1;
    uint32_t ka, kb;
    part_range(nd, EB, (part >> 6) & 63u, np, ka, kb);

    V num[RL][CL], den[OP::TWO ? RL : 1][OP::TWO ? CL : 1];
    double num64[SH::MIXED ? RL : 1][SH::MIXED ? CL : 1], den64[SH::MIXED && OP::TWO ? RL : 1][SH::MIXED && OP::TWO ? CL : 1];
#pragma unroll
    for (int r = 0; r < RL; ++r)
#pragma unroll
        for (int c = 0; c < CL; ++c) {
            num[r][c] = V(0);
            if constexpr (OP::TWO) den[r][c] = V(0);
            if constexpr (SH::MIXED) num64[r][c] = 0.0;
            if constexpr (SH::MIXED && OP::TWO) den64[r][c] = 0.0;
        }

    // wave w stages nodes w, w + 4, ..: 16 bytes per lane, rows then columns
    constexpr uint32_t VEC = 16 / sizeof(V), RLANES = SH::ROWS / VEC, CLANES = SH::COLS / VEC;
    const uint32_t* dl = g.dlist + 1;
    const uint32_t i0 = bi * SH::ROWS, j0 = bj * SH::COLS;
    if constexpr (OP::COUNTS) {   // the samples' totals (read again at each node: registers are short)
        for (uint32_t q = threadIdx.x; q < SH::NODE; q += 256) {
            const uint32_t smp = q < SH::ROWS ? i0 + q : j0 + q - SH::ROWS;
            st[q] = smp < g.n ? (V)g.totals[smp] : V(0);
        }
    }
    // the rows of the wave's nodes of the stage after the next one to be loaded, read ahead of their use
    uint32_t row_next[EB / 4];
    V len_next = V(0);
    auto index = [&](uint32_t k0) __attribute__((always_inline)) {
#pragma unroll
        for (uint32_t e = 0; e < EB / 4; ++e) row_next[e] = dl[min(k0 + wave + 4 * e, kb - 1)];
        if (g.rows) {
#pragma unroll
            for (uint32_t e = 0; e < EB / 4; ++e) row_next[e] = (uint32_t)g.rows[row_next[e]];
        }
        if constexpr (OP::LEN) len_next = threadIdx.x < EB ? (V)g.len[dl[min(k0 + threadIdx.x, kb - 1)]] : V(0);
    };
    // stages nodes k0 .. and reads the indices of the next ones
    auto stage = [&](int buf, uint32_t k0) __attribute__((always_inline)) {
#pragma unroll
        for (uint32_t e = 0; e < EB / 4; ++e) {
            const uint32_t ee = wave + 4 * e;
#pragma unroll
            for (uint32_t p = 0; p < PANELS; ++p) {
                const V* u = (const V*)(p == PANELS - 1 && OP::COUNTS ? g.C : g.U) + (size_t)row_next[e] * g.ldn;
                V* to = &sv[buf][ee][p][0];
                if constexpr (RLANES + CLANES <= 64) {
                    const V* src = u + (lane < RLANES ? i0 + lane * VEC : j0 + (lane - RLANES) * VEC);
                    if (RLANES + CLANES == 64 || lane < RLANES + CLANES)
                        __builtin_amdgcn_global_load_lds(SSU_GLOBAL(src), SSU_LDS(to), 16, 0, 0);
                } else {
                    static_assert(CLANES == 64 && RLANES <= 64, "a node is staged by one or two instructions");
                    if (RLANES == 64 || lane < RLANES)
                        __builtin_amdgcn_global_load_lds(SSU_GLOBAL(u + i0 + lane * VEC), SSU_LDS(to), 16, 0, 0);
                    __builtin_amdgcn_global_load_lds(SSU_GLOBAL(u + j0 + lane * VEC), SSU_LDS(to + SH::ROWS), 16, 0, 0);
                }
            }
        }
        if constexpr (OP::LEN) if (threadIdx.x < EB) sl[buf][threadIdx.x] = len_next;
        if (k0 + EB < kb) index(k0 + EB);
    };
    auto node = [&](int buf, uint32_t e) __attribute__((always_inline)) {
        V a[RL], b[CL], ca[OP::COUNTS ? RL : 1], cb[OP::COUNTS ? CL : 1], ea[OP::COUNTS ? RL : 1], eb[OP::COUNTS ? CL : 1];
        SH::read(a, &sv[buf][e][0][wr], li);
        SH::read(b, &sv[buf][e][0][SH::ROWS + wc], lj);
        if constexpr (OP::COUNTS) {   // (the last panel: the only one for presence terms)
            SH::read(ca, &sv[buf][e][PANELS - 1][wr], li);
            SH::read(cb, &sv[buf][e][PANELS - 1][SH::ROWS + wc], lj);
            SH::read(ea, &st[wr], li);
            SH::read(eb, &st[SH::ROWS + wc], lj);
#pragma unroll
            for (int r = 0; r < RL; ++r) ea[r] = OP::other(ea[r], ca[r]);
#pragma unroll
            for (int c = 0; c < CL; ++c) eb[c] = OP::other(eb[c], cb[c]);
        }
#pragma unroll
        for (int r = 0; r < RL; ++r) a[r] = OP::prep(a[r]);
#pragma unroll
        for (int c = 0; c < CL; ++c) b[c] = OP::prep(b[c]);
        const V l = OP::LEN ? sl[buf][e] : V(0);
        const V alpha = (V)g.alpha;
#pragma unroll
        for (int r = 0; r < RL; ++r)
#pragma unroll
            for (int c = 0; c < CL; ++c) {
                if constexpr (OP::COUNTS)
                    OP::term(a[r], b[c], ca[r], cb[c], ea[r], eb[c], l, alpha, num[r][c], den[r][c]);
                else if constexpr (OP::TWO) OP::term(a[r], b[c], l, alpha, num[r][c], den[r][c]);
                else OP::term(a[r], b[c], l, num[r][c]);
            }
    };
    auto merge = [&]() __attribute__((always_inline)) {
        if constexpr (SH::MIXED) {
#pragma unroll
            for (int r = 0; r < RL; ++r)
#pragma unroll
                for (int c = 0; c < CL; ++c) {
                    num64[r][c] += (double)num[r][c];
                    num[r][c] = V(0);
                    if constexpr (OP::TWO) { den64[r][c] += (double)den[r][c]; den[r][c] = V(0); }
                }
        }
    };

    if (ka < kb) {   // uniform
        index(ka);
        stage(0, ka);
        __syncthreads();
        int buf = 0;
        uint32_t span = 0;
        for (uint32_t k0 = ka; k0 < kb; k0 += EB) {
            if (k0 + EB < kb) stage(buf ^ 1, k0 + EB);
            else if (k0 + EB > kb) {   // (uniform) the last, partial stage: its missing nodes zero, which add nothing
                for (uint32_t q = (kb - k0) * PANELS * SH::NODE + threadIdx.x; q < EB * PANELS * SH::NODE; q += 256)
                    (&sv[buf][0][0][0])[q] = V(0);
                __syncthreads();
            }
#pragma unroll OP::UNROLL
            for (uint32_t e = 0; e < EB; ++e) node(buf, e);
            span += EB;
            if (span == MERGE) { merge(); span = 0; }
            __syncthreads();
            buf ^= 1;
        }
        merge();
    }

    auto sum = [&](int r, int c) { if constexpr (SH::MIXED) return num64[r][c]; else return num[r][c]; };
    auto sum2 = [&](int r, int c) {
        if constexpr (!OP::TWO) return 0.0;
        else if constexpr (SH::MIXED) return den64[r][c];
        else return den[r][c];
    };
    if (np > 1) {   // this part's sums to its slot, [pair of the lane][thread], for k_tiles_finish
        double* w = g.ws + (size_t)(part >> 12) * SH::SLOT + threadIdx.x;
#pragma unroll
        for (int r = 0; r < RL; ++r)
#pragma unroll
            for (int c = 0; c < CL; ++c) {
                w[(r * CL + c) * 256] = sum(r, c);
                if constexpr (OP::TWO) w[(SH::PAIRS + r * CL + c) * 256] = sum2(r, c);
            }
        return;
    }
#pragma unroll
    for (int r = 0; r < RL; ++r)
#pragma unroll
        for (int c = 0; c < CL; ++c) {
            const size_t i = i0 + wr + SH::at(li, r), j = j0 + wc + SH::at(lj, c);
            if (i < j && j < g.n) write_pair<OP>(g, i, j, sum(r, c), sum2(r, c));
            else if (i == j && i < g.n) ((V*)g.out)[i * g.n + i] = V(0);
        }
}

// The tiles cut into parts: the parts' sums in order, then the distances.
// blockIdx.y: one of the lane's rows.
template <class OP>
__global__ void __launch_bounds__(256) k_tiles_finish(TileArgs g) {
    typedef Shape<OP> SH;
    typedef typename OP::V V;
    constexpr int CL = OP::CL;
    const uint32_t bij = g.split[blockIdx.x].bij, part = g.split[blockIdx.x].part;
    const uint32_t bi = bij >> 16, bj = bij & 0xffffu, np = (part & 63u) + 1, r = blockIdx.y;
    const uint32_t wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const uint32_t li = lane >> 3, lj = lane & 7, wr = (wave >> 1) * SH::WAVE_ROWS, wc = (wave & 1) * SH::WAVE_COLS;
    const double* w = g.ws + (size_t)(part >> 12) * SH::SLOT + threadIdx.x;
    double x[CL], y[CL];
#pragma unroll
    for (int c = 0; c < CL; ++c) x[c] = y[c] = 0.0;
#pragma unroll 2
    for (uint32_t p = 0; p < np; ++p)
#pragma unroll
        for (int c = 0; c < CL; ++c) {
            x[c] += w[(size_t)p * SH::SLOT + (r * CL + c) * 256];
            if constexpr (OP::TWO) y[c] += w[(size_t)p * SH::SLOT + (SH::PAIRS + r * CL + c) * 256];
        }
#pragma unroll
    for (int c = 0; c < CL; ++c) {
        const size_t i = bi * SH::ROWS + wr + SH::at(li, r), j = bj * SH::COLS + wc + SH::at(lj, c);
        if (i < j && j < g.n) write_pair<OP>(g, i, j, x[c], y[c]);
        else if (i == j && i < g.n) ((V*)g.out)[i * g.n + i] = V(0);
    }
}

// ------------------------------------------------------------------ dense list
// One workgroup: a thread counts the bits of its run of words, an exclusive sum
// over the threads gives its first place, then it writes its nodes.
constexpr uint32_t DL_T = 1024;
__global__ void __launch_bounds__(DL_T) k_dense_list(uint32_t* __restrict__ dlist, const uint32_t* __restrict__ dmask,
                                                     uint32_t Kw) {
    __shared__ uint32_t wsum[DL_T / 64];
    const uint32_t t = threadIdx.x, lane = t & 63, w = t >> 6;
    const uint32_t per = (Kw + DL_T - 1) / DL_T;
    const uint32_t a = min(Kw, t * per), b = min(Kw, a + per);
    uint32_t c = 0;
    for (uint32_t q = a; q < b; ++q) c += __popc(dmask[q]);
    uint32_t incl = c;
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
        const uint32_t y = __shfl_up(incl, d, 64);
        if ((int)lane >= d) incl += y;
    }
    if (lane == 63) wsum[w] = incl;
    __syncthreads();
    uint32_t before = 0, total = 0;
    for (uint32_t q = 0; q < DL_T / 64; ++q) {
        before += q < w ? wsum[q] : 0u;
        total += wsum[q];
    }
    if (t == 0) dlist[0] = total;
    uint32_t* o = dlist + 1 + before + incl - c;
    for (uint32_t q = a; q < b; ++q)
        for (uint32_t m = dmask[q]; m; m &= m - 1) *o++ = q * 32 + (uint32_t)(__ffs(m) - 1);
}

}  // namespace

// ------------------------------------------------------------------ work lists

// Each XCD gets an equal run of tiles.  Whole rounds of `resident` tiles stay
// whole; the tiles left over, which would leave most of the XCD idle for one
// more round, are cut into np parts over the nodes, np the cheapest of
// ceil(left * np / resident) rounds of 1 / np of a tile each plus the cost of
// writing and reading the parts' sums, of those whose slots fit TILE_WS_BYTES.
TileSet tile_set(uint32_t n, uint32_t rows, uint32_t max_nodes) {
    const uint32_t resident = tile_resident(rows), cols = rows;
    TileSet t;
    const uint32_t nbi = (n + rows - 1) / rows, nbj = (n + cols - 1) / cols;
    // 1024 x 1024 samples per super-tile: about the tiles resident on one XCD
    const uint32_t SI = std::max<uint32_t>(1, 1024 / rows), SJ = std::max<uint32_t>(1, 1024 / cols);
    std::vector<uint32_t> order;
    for (uint32_t si = 0; si < nbi; si += SI)
        for (uint32_t sj = 0; sj < nbj; sj += SJ)
            for (uint32_t bi = si; bi < std::min(nbi, si + SI); ++bi)
                for (uint32_t bj = sj; bj < std::min(nbj, sj + SJ); ++bj)
                    if (bj >= bi) order.push_back(bi << 16 | bj);   // (with the diagonal)
    t.tiles = order.size();
    // a part is at least 64 nodes; writing and reading one costs about as much as 24 nodes' terms
    const uint32_t most = std::max<uint32_t>(1, std::min<uint32_t>(TILE_MAX_PARTS, max_nodes / 64));
    const double part_cost = max_nodes ? 24.0 / max_nodes : 1.0;
    const size_t most_slots = TILE_WS_BYTES / N_XCDS / tile_slot_bytes(rows);   // of an XCD
    std::vector<std::vector<TileUnit>> xcd(N_XCDS);
    size_t at = 0;
    for (uint32_t x = 0; x < N_XCDS; ++x) {
        const size_t end = order.size() * (x + 1) / N_XCDS, count = end - at;
        const size_t left = count % resident, whole = count - left;
        uint32_t np = 1;
        double best = left ? 1.0 : 0.0;
        for (uint32_t q = 2; q <= most && left && left * q <= most_slots; ++q) {
            const double cost = (double)((left * q + resident - 1) / resident) * (1.0 / q + part_cost);
            if (cost < 0.97 * best) { best = cost; np = q; }
        }
        for (size_t k = 0; k < count; ++k) {
            const uint32_t bij = order[at + k];
            if (k < whole || np == 1) { xcd[x].push_back({bij, 0u}); continue; }
            t.split.push_back({bij, t.slots << 12 | (np - 1)});
            for (uint32_t p = 0; p < np; ++p) xcd[x].push_back({bij, (t.slots + p) << 12 | p << 6 | (np - 1)});
            t.slots += np;
        }
        at = end;
        t.per_xcd = std::max<uint32_t>(t.per_xcd, (uint32_t)xcd[x].size());
    }
    for (auto& v : xcd) {
        v.resize(t.per_xcd, TileUnit{TILE_NONE, 0u});
        t.units.insert(t.units.end(), v.begin(), v.end());
    }
    return t;
}

TileSet tile_subset(const TileSet& full, const std::function<bool(uint32_t, uint32_t)>& keep) {
    TileSet t;
    auto in = [&](const TileUnit& u) { return u.bij != TILE_NONE && keep(u.bij >> 16, u.bij & 0xffffu); };
    for (const TileUnit& u : full.units)
        if (in(u)) {
            t.units.push_back(u);
            t.tiles += ((u.part >> 6) & 63u) == 0;
        }
    for (const TileUnit& u : full.split)
        if (in(u)) t.split.push_back(u);
    t.per_xcd = (uint32_t)((t.units.size() + N_XCDS - 1) / N_XCDS);
    t.slots = full.slots;
    return t;
}

// ------------------------------------------------------------------ launchers

hipError_t launch_dense_list(uint32_t* dlist, const uint32_t* dmask, uint32_t K, hipStream_t st) {
    if (!dlist || (K && !dmask)) return hipErrorInvalidValue;
    hipLaunchKernelGGL(k_dense_list, dim3(1), dim3(DL_T), 0, st, dlist, dmask, (K + 31) / 32);
    return hipGetLastError();
}

template <class OP> static hipError_t launch_tiles(const TileArgs& a, hipStream_t st) {
    constexpr uint32_t rows = Shape<OP>::ROWS;
    if (!a.n || !a.n_units) return hipSuccess;   // (a selection without a tile here)
    if ((!a.U && (!OP::COUNTS || OP::PANELS == 2)) || !a.dlist || !a.out || !a.units || (OP::TWO ? a.add_partial && !a.out2 : !a.S) ||
        (OP::COUNTS && (!a.C || !a.totals)) || (sizeof(typename OP::V) == 8 && !a.rows) || a.ldn < a.n ||
        a.ldn % rows || (a.n + rows - 1) / rows > 65535 || (a.n_split && (!a.split || !a.ws)) || (OP::LEN && !a.len))
        return hipErrorInvalidValue;
    hipLaunchKernelGGL(k_tiles<OP>, dim3(a.per_xcd * N_XCDS), dim3(256), 0, st, a);
    if (a.n_split) hipLaunchKernelGGL(k_tiles_finish<OP>, dim3(a.n_split, OP::RL), dim3(256), 0, st, a);
    return hipGetLastError();
}

hipError_t launch_tiles_weighted(bool fp64, const TileArgs& a, hipStream_t st) {
    if (fp64) return launch_tiles<OpW64>(a, st);
    return a.scaled ? launch_tiles<OpW32<true>>(a, st) : launch_tiles<OpW32<false>>(a, st);
}

template <class T> static hipError_t launch_gen(const TileArgs& a, hipStream_t st) {
    if (a.alpha == 0.5) return launch_tiles<OpGen<T, 1>>(a, st);
    if (a.alpha == 1.0) return launch_tiles<OpGen<T, 2>>(a, st);
    return launch_tiles<OpGen<T, 0>>(a, st);
}
hipError_t launch_tiles_generalized(bool fp64, const TileArgs& a, hipStream_t st) {
    return fp64 ? launch_gen<double>(a, st) : launch_gen<float>(a, st);
}

template <class T> static hipError_t launch_vaw(int kind, const TileArgs& a, hipStream_t st) {
    switch (kind) {
    case 1: return launch_tiles<OpVaw<T, 1>>(a, st);
    case 2: return launch_tiles<OpVaw<T, 2>>(a, st);
    case 3:
        if (a.alpha == 0.5) return launch_tiles<OpVaw<T, 3, 1>>(a, st);
        if (a.alpha == 1.0) return launch_tiles<OpVaw<T, 3, 2>>(a, st);
        return launch_tiles<OpVaw<T, 3, 0>>(a, st);
    default: return hipErrorInvalidValue;
    }
}
hipError_t launch_tiles_vaw(int kind, bool fp64, const TileArgs& a, hipStream_t st) {
    return fp64 ? launch_vaw<double>(kind, a, st) : launch_vaw<float>(kind, a, st);
}

}  // namespace ssu
