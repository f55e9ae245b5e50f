// PCoA (Gower centring + randomized FSVD) and PERMANOVA.  The matrix goes up
// once and everything that has its rows stays on the device: centring, probes,
// the products B X, both thin QR factorisations, the coordinates, the
// permutations and their sums.  The SVD of the small R factor runs on the host.
#include "ssu_engine.hpp"
#include "ssu_stats.hpp"

#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <limits>
#include <mutex>
#include <vector>

namespace ssu {

namespace {

#define ST_HIP(x)                                                                                    \
    do {                                                                                             \
        hipError_t e_ = (x);                                                                         \
        if (e_ != hipSuccess) {                                                                      \
            if (err) *err = std::string(#x) + ": " + hipGetErrorString(e_);                          \
            return false;                                                                            \
        }                                                                                            \
    } while (0)

// device memory from the process-wide cache
struct Buf {
    void* p = nullptr;
    size_t bytes = 0;
    ~Buf() { pool_free(p, bytes); }
    template <class T> T* as() const { return (T*)p; }
};

// after the buffers of a scope: no block goes back to the cache while a launch may use it
struct Idle {
    ~Idle() { (void)hipStreamSynchronize(nullptr); }
};

bool alloc(Buf& b, size_t bytes, std::string* err) {
    b.p = pool_alloc(std::max<size_t>(bytes, 16), &b.bytes, err);
    return b.p != nullptr;
}

constexpr uint32_t ST_T = 256;
constexpr uint32_t MAX_GRID_Y = 65535;

// Sum over the workgroup, the same order every time.
__device__ __forceinline__ double block_sum(double v, double* part) {
#pragma unroll
    for (int d = 32; d > 0; d >>= 1) v += __shfl_down(v, d, 64);
    if ((threadIdx.x & 63) == 0) part[threadIdx.x >> 6] = v;
    __syncthreads();
    double s = 0.0;
    for (uint32_t w = 0; w < ST_T / 64; ++w) s += part[w];
    __syncthreads();
    return s;
}

// rmean[i] = mean_j (-d_ij^2 / 2); upper[i] = sum_{j > i} d_ij^2
template <class T>
__global__ void __launch_bounds__(ST_T) k_row_stats(double* __restrict__ rmean, double* __restrict__ upper,
                                                    const T* __restrict__ D, uint32_t n) {
    __shared__ double part[ST_T / 64];
    const uint32_t i = blockIdx.x;
    const T* row = D + (size_t)i * n;
    double a = 0.0, u = 0.0;
    for (uint32_t j = threadIdx.x; j < n; j += ST_T) {
        const double d = (double)row[j];
        a += -0.5 * d * d;
        if (j > i) u += d * d;
    }
    a = block_sum(a, part);
    u = block_sum(u, part);
    if (threadIdx.x == 0) {
        rmean[i] = a / n;
        if (upper) upper[i] = u;
    }
}

// B_ij = -d_ij^2 / 2 - rmean_i - rmean_j + grand, in place
template <class T>
__global__ void __launch_bounds__(ST_T) k_center_apply(T* __restrict__ B, const double* __restrict__ rmean,
                                                       double grand, uint32_t n) {
    const size_t q = (size_t)blockIdx.x * ST_T + threadIdx.x;
    if (q >= (size_t)n * n) return;
    const uint32_t i = (uint32_t)(q / n), j = (uint32_t)(q % n);
    const double d = (double)B[q];
    B[q] = (T)(-0.5 * d * d - rmean[i] - rmean[j] + grand);
}

typedef double f64x4 __attribute__((ext_vector_type(4)));

// Y = B X for an n x n matrix B and n x ld matrices X, Y (row major, ld a multiple
// of 16, columns past the real ones zero), on v_mfma_f64_16x16x4_f64: one
// workgroup per 16 rows and 16 columns, its waves each a quarter of the inner
// index.  Lane (i, kq) of a wave reads four consecutive values of row i, j0 + 4 kq
// .., which are the A operands of four steps; B's operand of step s is row
// j0 + 4 kq + s of X (the inner index may come in any order).  Bound by the read of
// B (25 MB at 2,500 FP32 samples) and its latency: 23 us a product of 12 or 36
// columns, against 188 us with one row per workgroup, which read all of X for each.
constexpr uint32_t SM_WAVES = 4;
template <class T>
__global__ void __launch_bounds__(64 * SM_WAVES) k_symm_mult(double* __restrict__ Y, const T* __restrict__ B,
                                                             const double* __restrict__ X, uint32_t n, uint32_t ld) {
    typedef T vec __attribute__((ext_vector_type(4), aligned(sizeof(T))));   // (rows start at any multiple of a value)
    __shared__ double part[SM_WAVES][256];
    const uint32_t i0 = blockIdx.x * 16, c0 = blockIdx.y * 16;
    const uint32_t lane = threadIdx.x & 63, w = threadIdx.x >> 6, i = lane & 15, kq = lane >> 4;
    const T* row = B + (size_t)min(i0 + i, n - 1) * n;
    const double* xc = X + c0 + i;
    f64x4 acc = {0.0, 0.0, 0.0, 0.0};
    uint32_t j0 = 16 * w;
#pragma unroll 4
    for (; j0 + 16 <= n; j0 += 16 * SM_WAVES) {
        const vec b = *reinterpret_cast<const vec*>(row + j0 + 4 * kq);
        const double* x = xc + (size_t)(j0 + 4 * kq) * ld;
#pragma unroll
        for (uint32_t s = 0; s < 4; ++s)
            acc = __builtin_amdgcn_mfma_f64_16x16x4f64((double)b[s], x[(size_t)s * ld], acc, 0, 0, 0);
    }
    if (j0 < n) {   // (uniform per wave) the last, partial step
#pragma unroll
        for (uint32_t s = 0; s < 4; ++s) {
            const uint32_t j = j0 + 4 * kq + s;
            const double a = j < n ? (double)row[j] : 0.0, x = j < n ? xc[(size_t)j * ld] : 0.0;
            acc = __builtin_amdgcn_mfma_f64_16x16x4f64(a, x, acc, 0, 0, 0);
        }
    }
    // D: register r of lane l holds row l / 16 + 4 r, column l % 16
#pragma unroll
    for (int r = 0; r < 4; ++r) part[w][(kq + 4 * r) * 16 + i] = acc[r];
    __syncthreads();
    const uint32_t t = threadIdx.x, orow = i0 + t / 16;
    double s = 0.0;
    for (uint32_t q = 0; q < SM_WAVES; ++q) s += part[q][t];
    if (orow < n) Y[(size_t)orow * ld + c0 + t % 16] = s;
}

// columns [0, cols) of the row-major n x ld matrix R into the column-major H
__global__ void __launch_bounds__(ST_T) k_to_columns(double* __restrict__ H, const double* __restrict__ R, uint32_t n,
                                                     uint32_t ld, uint32_t cols) {
    const uint32_t i = blockIdx.x * ST_T + threadIdx.x;
    if (i >= n) return;
#pragma unroll 8
    for (uint32_t c = 0; c < cols; ++c) H[(size_t)c * n + i] = R[(size_t)i * ld + c];
}
// the reverse, columns past cols zero
__global__ void __launch_bounds__(ST_T) k_to_rows(double* __restrict__ R, const double* __restrict__ H, uint32_t n,
                                                  uint32_t ld, uint32_t cols) {
    const uint32_t i = blockIdx.x * ST_T + threadIdx.x;
    if (i >= n) return;
#pragma unroll 8
    for (uint32_t c = 0; c < ld; ++c) R[(size_t)i * ld + c] = c < cols ? H[(size_t)c * n + i] : 0.0;
}

__host__ __device__ uint64_t mix64(uint64_t z) {
    z += 0x9E3779B97F4A7C15ull;
    z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
    z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
    return z ^ (z >> 31);
}

// X[i][c] = a standard normal from two counter-based uniforms (Box-Muller), index i k + c; 0 past k
__global__ void __launch_bounds__(64) k_probes(double* __restrict__ X, uint32_t k, uint32_t ld, uint64_t seed) {
    const uint32_t i = blockIdx.x;
    for (uint32_t c = blockIdx.y * 64 + threadIdx.x; c < ld; c += gridDim.y * 64) {
        double x = 0.0;
        if (c < k) {
            const uint64_t idx = (uint64_t)i * k + c;
            const double u1 = ((mix64(seed ^ mix64(2 * idx)) >> 11) + 1) * 0x1.0p-53;   // (0, 1]
            const double u2 = (mix64(seed ^ mix64(2 * idx + 1)) >> 11) * 0x1.0p-53;
            x = sqrt(-2.0 * log(u1)) * cos(6.283185307179586 * u2);
        }
        X[(size_t)i * ld + c] = x;
    }
}

// R (q x q, column major, zero below its diagonal r) from above the diagonal of the n x q matrix A
__global__ void __launch_bounds__(ST_T) k_pack_r(double* __restrict__ R, const double* __restrict__ A,
                                                 const double* __restrict__ r, uint32_t n, uint32_t q) {
    const uint32_t c = blockIdx.x;
    for (uint32_t i = threadIdx.x; i < q; i += ST_T)
        R[(size_t)c * q + i] = i < c ? A[(size_t)c * n + i] : i == c ? r[c] : 0.0;
}

// Sums of two values over a workgroup of QR_T threads, in every thread, the same
// order every time.
constexpr uint32_t QR_T = 1024;
__device__ __forceinline__ void qr_sums(double& x, double& y, double (*part)[2]) {
#pragma unroll
    for (int d = 32; d > 0; d >>= 1) {
        x += __shfl_xor(x, d, 64);
        y += __shfl_xor(y, d, 64);
    }
    if ((threadIdx.x & 63) == 0) {
        part[threadIdx.x >> 6][0] = x;
        part[threadIdx.x >> 6][1] = y;
    }
    __syncthreads();
    x = y = 0.0;
#pragma unroll
    for (uint32_t w = 0; w < QR_T / 64; ++w) {
        x += part[w][0];
        y += part[w][1];
    }
}

// Step k of a thin QR by Householder reflections of the column-major n x m matrix A:
// v = (A[k:, k] - alpha e_k) / |..|, alpha = -sign(A_kk) |A[k:, k]|.  One workgroup per
// column: column k's writes v to column k of V (zero above k) and alpha to r[k], and
// leaves A[:, k] to the others, which take v's norm and their own product with it from
// the one pass over column k and reflect themselves, A[k:, c] -= 2 v (v . A[k:, c]).
// Bound by the launch and its two trips to memory: 2,500 x 36 takes 5.3 us a step,
// against 28 us with all the steps in one workgroup (one CU's L2 reads) and about 80 us
// on the host.
__global__ void __launch_bounds__(QR_T) k_householder(double* __restrict__ A, double* __restrict__ V,
                                                      double* __restrict__ r, uint32_t n, uint32_t k) {
    __shared__ double part[QR_T / 64][2];
    const uint32_t t = threadIdx.x, c = k + blockIdx.x;
    const double* col = A + (size_t)k * n;
    double* a = A + (size_t)c * n;
    const double ck = col[k], ak = a[k];
    double ss = 0.0, dot = 0.0;   // over i > k
#pragma unroll 4
    for (uint32_t i = k + 1 + t; i < n; i += QR_T) {
        const double x = col[i];
        ss += x * x;
        dot += x * a[i];
    }
    qr_sums(ss, dot, part);
    const double norm = sqrt(ck * ck + ss), alpha = ck >= 0.0 ? -norm : norm, vk = ck - alpha;
    const double vn = norm > 0.0 ? 1.0 / sqrt(vk * vk + ss) : 0.0;
    if (c == k) {
        double* v = V + (size_t)k * n;
        for (uint32_t i = t; i < n; i += QR_T) v[i] = i < k ? 0.0 : (i == k ? vk : col[i]) * vn;
        if (t == 0) r[k] = norm > 0.0 ? alpha : ck;
    } else {
        const double f = 2.0 * vn * vn * (dot + vk * ak);
#pragma unroll 4
        for (uint32_t i = k + 1 + t; i < n; i += QR_T) a[i] -= f * col[i];
        if (t == 0) a[k] = ak - f * vk;
    }
}

// Q = H_0 .. H_{q-1} I[:, :q], column major: one workgroup per column (reflections
// past the column's own leave it as it is)
__global__ void __launch_bounds__(QR_T) k_form_q(double* __restrict__ Q, const double* __restrict__ V, uint32_t n) {
    __shared__ double part[2][QR_T / 64][2];
    const uint32_t c = blockIdx.x, t = threadIdx.x;
    double* a = Q + (size_t)c * n;
    for (uint32_t i = t; i < n; i += QR_T) a[i] = i == c ? 1.0 : 0.0;
    for (uint32_t k = c + 1; k-- > 0;) {
        const double* v = V + (size_t)k * n;   // (zero above k)
        // (a thread reads and writes its own elements of a only)
        double dot = 0.0, none = 0.0;
#pragma unroll 4
        for (uint32_t i = t; i < n; i += QR_T) dot += v[i] * a[i];
        qr_sums(dot, none, part[k & 1]);
        dot *= 2.0;
#pragma unroll 4
        for (uint32_t i = t; i < n; i += QR_T) a[i] -= dot * v[i];
    }
}

// The same factorisation of a small A in one launch: A sits in the LDS of one
// workgroup, wave c % 16 reflects column c, and every wave takes a step's norm for
// itself, so that a step takes one barrier.  FORM_Q: the waves then form Q's columns in
// registers, without barriers.  Bound by the reductions' LDS latency; the launches of
// k_householder cost more up to there (300 samples, 36 columns: 130 us with Q
// against about 220).
constexpr uint32_t QRS_MAX_N = 512, QRS_E = QRS_MAX_N / 64;
constexpr size_t QRS_LDS = size_t(144) << 10;
__device__ __forceinline__ double wave_sum(double x) {
#pragma unroll
    for (int d = 32; d > 0; d >>= 1) x += __shfl_xor(x, d, 64);
    return x;
}
template <bool FORM_Q>
__global__ void __launch_bounds__(QR_T) k_qr_small(double* __restrict__ A, double* __restrict__ Q,
                                                   double* __restrict__ r, uint32_t n, uint32_t m, uint32_t q) {
    extern __shared__ double lds[];
    double* S = lds;                          // n x m, column major
    double* head = S + (size_t)n * m;         // per step: v_k before scaling, 2 / |v|^2
    const uint32_t t = threadIdx.x, lane = t & 63, w = t >> 6;
    for (uint32_t e = t; e < n * m; e += QR_T) S[e] = A[e];
    __syncthreads();
    double v[QRS_E], a[QRS_E];
    const auto rows = [&](double (&x)[QRS_E], const double* col) {
#pragma unroll
        for (uint32_t e = 0; e < QRS_E; ++e) {
            const uint32_t i = e * 64 + lane;
            x[e] = i < n ? col[i] : 0.0;
        }
    };
    const auto cut_above = [&](uint32_t k, double vk) {   // v: zero above k, vk at k
#pragma unroll
        for (uint32_t e = 0; e < QRS_E; ++e) {
            const uint32_t i = e * 64 + lane;
            v[e] = i < k ? 0.0 : i == k ? vk : v[e];
        }
    };
    const auto product = [&]() {
        double x = 0.0;
#pragma unroll
        for (uint32_t e = 0; e < QRS_E; ++e) x += v[e] * a[e];
        return wave_sum(x);
    };
    for (uint32_t k = 0; k < q; ++k) {
        rows(v, S + (size_t)k * n);
        const double ck = S[(size_t)k * n + k];
        cut_above(k, 0.0);
        double ss = 0.0;
#pragma unroll
        for (uint32_t e = 0; e < QRS_E; ++e) ss += v[e] * v[e];
        ss = wave_sum(ss);
        const double norm = sqrt(ck * ck + ss), alpha = ck >= 0.0 ? -norm : norm, vk = ck - alpha;
        const double f = norm > 0.0 ? 2.0 / (vk * vk + ss) : 0.0;
        cut_above(k, vk);
        if (t == 0) {
            head[2 * k] = vk;
            head[2 * k + 1] = f;
            r[k] = norm > 0.0 ? alpha : ck;
        }
        for (uint32_t c = w; c < m; c += QR_T / 64) {
            if (c <= k) continue;
            double* col = S + (size_t)c * n;
            rows(a, col);
            const double g = f * product();
#pragma unroll
            for (uint32_t e = 0; e < QRS_E; ++e) {
                const uint32_t i = e * 64 + lane;
                if (i < n) col[i] = a[e] - g * v[e];
            }
        }
        __syncthreads();
    }
    if (FORM_Q) {
        for (uint32_t c = w; c < q; c += QR_T / 64) {
#pragma unroll
            for (uint32_t e = 0; e < QRS_E; ++e) a[e] = e * 64 + lane == c ? 1.0 : 0.0;
            for (uint32_t k = c + 1; k-- > 0;) {
                rows(v, S + (size_t)k * n);
                cut_above(k, head[2 * k]);
                const double g = head[2 * k + 1] * product();
#pragma unroll
                for (uint32_t e = 0; e < QRS_E; ++e) a[e] -= g * v[e];
            }
#pragma unroll
            for (uint32_t e = 0; e < QRS_E; ++e) {
                const uint32_t i = e * 64 + lane;
                if (i < n) Q[(size_t)c * n + i] = a[e];
            }
        }
    } else {
        for (uint32_t e = t; e < n * m; e += QR_T) A[e] = S[e];   // (its upper triangle is R's)
    }
}

// samples[i][d] = (Q W)[i][d], W column major q x dims
__global__ void __launch_bounds__(ST_T) k_coordinates(double* __restrict__ samples, const double* __restrict__ Q,
                                                      const double* __restrict__ W, uint32_t n, uint32_t q,
                                                      uint32_t used, uint32_t dims) {
    const uint32_t i = blockIdx.x * ST_T + threadIdx.x;
    if (i >= n) return;
    for (uint32_t d = blockIdx.y; d < dims; d += gridDim.y) {
        double u = 0.0;
        if (d < used)
#pragma unroll 8
            for (uint32_t c = 0; c < q; ++c) u += Q[(size_t)c * n + i] * W[(size_t)d * q + c];
        samples[(size_t)i * dims + d] = u;
    }
}

// PERMANOVA permutations: row p > 0 of the labels is the p-th Fisher-Yates shuffle
// of the grouping (row 0 the grouping itself), written sample major, Lt[i * ldp + p]
// (columns past the rows: labels of no group).  One wave per row, its labels in LDS
// as bytes, 64 exchanges at a time: a lane whose positions no earlier lane of the
// batch touches is independent of those, so the lanes up to the first that is not
// exchange at once, the rest in further rounds (`tag`: the first lane to touch a
// position, by its low bits).  999 shuffles of 2,500 labels 90 us, 243 with the
// exchanges one after another (their LDS round trips), on the host 7 ms.
constexpr uint32_t SHUF_TAGS = 4096;
constexpr uint32_t SHUF_MAX_N = 65536 - 4 * SHUF_TAGS, SHUF_MAX_GROUPS = 256;   // (64 KB of LDS)
__global__ void __launch_bounds__(64) k_shuffles(uint32_t* __restrict__ Lt, const uint32_t* __restrict__ grouping,
                                                 uint32_t n, uint32_t n_lab, uint32_t ldp, uint64_t seed) {
    extern __shared__ uint32_t tag[];
    uint8_t* lab = reinterpret_cast<uint8_t*>(tag + SHUF_TAGS);
    const uint32_t p = blockIdx.x, lane = threadIdx.x;
    if (p >= n_lab) {
        for (uint32_t i = lane; i < n; i += 64) Lt[(size_t)i * ldp + p] = 0xffffffffu;
        return;
    }
    for (uint32_t i = lane; i < n; i += 64) lab[i] = (uint8_t)grouping[i];
    __syncthreads();
    if (p) {
        const uint64_t key = mix64(seed ^ mix64(p));
        for (uint32_t top = n - 1; top > 0; top = top > 64 ? top - 64 : 0) {   // exchanges i = top .. max(1, top - 63)
            const uint32_t cnt = min(64u, top), i_l = top - min(lane, cnt - 1);
            const uint32_t j_l = (uint32_t)(mix64(key + i_l) % (i_l + 1));
            for (uint32_t done = 0; done < cnt;) {   // (uniform)
                const bool on = lane >= done && lane < cnt;
                uint32_t *ti = tag + i_l % SHUF_TAGS, *tj = tag + j_l % SHUF_TAGS;
                if (on) *ti = *tj = 64;
                __syncthreads();
                if (on) {
                    atomicMin(ti, lane);
                    atomicMin(tj, lane);
                }
                __syncthreads();
                const uint64_t wait = __ballot(on && (*ti != lane || *tj != lane));   // (never the lane `done`)
                const uint32_t end = wait ? (uint32_t)__builtin_ctzll(wait) : cnt;
                if (on && lane < end) {
                    const uint8_t a = lab[i_l], b = lab[j_l];
                    lab[i_l] = b;
                    lab[j_l] = a;
                }
                __syncthreads();
                done = end;
            }
        }
        __syncthreads();
    }
    for (uint32_t i = lane; i < n; i += 64) Lt[(size_t)i * ldp + p] = lab[i];
}

// Label rows made on the host (row major, n_lab x n) into the sample-major Lt of
// k_shuffles, 64 x 64 by LDS.  (A call of 2,500 samples, 300 groups and 999 permutations
// takes 7.8 ms; 26.1 with Lt written on the host, a cache line touched per label.)
__global__ void __launch_bounds__(256) k_label_columns(uint32_t* __restrict__ Lt, const uint32_t* __restrict__ L,
                                                       uint32_t n, uint32_t n_lab, uint32_t ldp) {
    __shared__ uint32_t tile[64][65];
    const uint32_t i0 = blockIdx.x * 64, p0 = blockIdx.y * 64, c = threadIdx.x & 63;   // (ldp is a multiple of 64)
    for (uint32_t r = threadIdx.x >> 6; r < 64; r += 4)
        tile[r][c] = p0 + r < n_lab && i0 + c < n ? L[(size_t)(p0 + r) * n + i0 + c] : 0xffffffffu;
    __syncthreads();
    for (uint32_t r = threadIdx.x >> 6; r < 64 && i0 + r < n; r += 4) Lt[(size_t)(i0 + r) * ldp + p0 + c] = tile[c][r];
}

// Within-group sums: partial[u][p] = sum over rows i of row block ib and columns j of
// chunk jc, j > i, with L_p(i) == L_p(j), of d_ij^2 / size(L_p(i)); unit u = (ib, jc)
// from the list.  A workgroup owns 64 rows (its lanes) and 4 x PM_P label rows, PM_P
// per wave: a step's d^2 of the 64 rows come from LDS, the column's labels are
// uniform (scalar loads), so a pair and label row takes a compare into the exec mask
// and an add.  Bound by FP64 issue: 2,500 samples x 1,000 label rows 360 us, against
// 1,423 us with a select per pair and label row and labels in LDS.
constexpr uint32_t PM_R = 64, PM_J = 256, PM_P = 16, PM_PW = 4 * PM_P;
typedef uint32_t u32x16 __attribute__((ext_vector_type(16)));
static_assert(PM_P == 16, "a wave's labels of one column are one scalar load");
template <class T>
__global__ void __launch_bounds__(256) k_permanova(double* __restrict__ partial, const T* __restrict__ D,
                                                   const uint32_t* __restrict__ Lt, const double* __restrict__ inv_size,
                                                   const uint32_t* __restrict__ units, uint32_t n, uint32_t ldp,
                                                   uint32_t chunk) {
    __shared__ double dsq[64][PM_R + 1];   // [column][row]
    const uint32_t i0 = (units[blockIdx.x] >> 16) * PM_R, jb = (units[blockIdx.x] & 0xffffu) * chunk;
    const uint32_t lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const uint32_t p0 = blockIdx.y * PM_PW + w * PM_P;
    const uint32_t i = i0 + lane;
    uint32_t li[PM_P];
    double acc[PM_P];
#pragma unroll
    for (uint32_t q = 0; q < PM_P; ++q) {
        li[q] = i < n ? Lt[(size_t)i * ldp + p0 + q] : 0xfffffffeu;
        acc[q] = 0.0;
    }
    const uint32_t j_end = min(n, jb + chunk);
    uint32_t j0 = max(jb, i0);   // (i0 and jb are multiples of 64)
    T d[PM_R / 4];
    const auto load_d = [&](uint32_t j) {   // rows i0 + w + 4 q, column j + lane; clamped, cut to the pairs below
#pragma unroll
        for (uint32_t q = 0; q < PM_R / 4; ++q)
            d[q] = D[(size_t)min(i0 + w + 4 * q, n - 1) * n + min(j + lane, n - 1)];
    };
    load_d(j0);
    for (; j0 < j_end; j0 += 64) {
        __syncthreads();
#pragma unroll
        for (uint32_t q = 0; q < PM_R / 4; ++q) {
            const uint32_t r = w + 4 * q, jj = j0 + lane;
            const double x = jj < n && jj > i0 + r ? (double)d[q] : 0.0;   // (jj > i: rows past n have none)
            dsq[lane][r] = x * x;
        }
        __syncthreads();
        if (j0 + 64 < j_end) load_d(j0 + 64);
        const uint32_t cols = min(64u, n - j0);
        const uint32_t* lt = Lt + (size_t)j0 * ldp + p0;
        u32x16 lj = *reinterpret_cast<const u32x16*>(lt);   // (scalar loads, a column ahead)
        double d2 = dsq[0][lane];
        __builtin_amdgcn_s_waitcnt(0xc07f);   // lgkmcnt(0): nothing in flight at the loop's head but the loads ahead
#pragma unroll 2
        for (uint32_t c = 0; c < cols; ++c) {
            const uint32_t cn = min(c + 1, cols - 1);
            const u32x16 lj_n = *reinterpret_cast<const u32x16*>(lt + (size_t)cn * ldp);
            const double d2_n = dsq[cn][lane];
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (uint32_t q = 0; q < PM_P; q += 4)   // (every lane is active here)
                asm("v_cmpx_eq_u32 vcc, %5, %9\n\tv_add_f64 %0, %0, %4\n\ts_mov_b64 exec, -1\n\t"
                    "v_cmpx_eq_u32 vcc, %6, %10\n\tv_add_f64 %1, %1, %4\n\ts_mov_b64 exec, -1\n\t"
                    "v_cmpx_eq_u32 vcc, %7, %11\n\tv_add_f64 %2, %2, %4\n\ts_mov_b64 exec, -1\n\t"
                    "v_cmpx_eq_u32 vcc, %8, %12\n\tv_add_f64 %3, %3, %4\n\ts_mov_b64 exec, -1"
                    : "+v"(acc[q]), "+v"(acc[q + 1]), "+v"(acc[q + 2]), "+v"(acc[q + 3])
                    : "v"(d2), "s"(lj[q]), "s"(lj[q + 1]), "s"(lj[q + 2]), "s"(lj[q + 3]), "v"(li[q]), "v"(li[q + 1]),
                      "v"(li[q + 2]), "v"(li[q + 3])
                    : "vcc");
            __builtin_amdgcn_sched_barrier(0);
            lj = lj_n;
            d2 = d2_n;
        }
        asm volatile("s_nop 4");   // a lane read or DPP may not follow a VALU write of exec more closely
    }
    // per label row: the rows' sums weighted, then over the lanes
#pragma unroll
    for (uint32_t q = 0; q < PM_P; ++q) {
        double x = li[q] < 0xfffffffeu ? acc[q] * inv_size[li[q]] : 0.0;
#pragma unroll
        for (int d = 32; d > 0; d >>= 1) x += __shfl_xor(x, d, 64);
        if (lane == 0) partial[(size_t)blockIdx.x * ldp + p0 + q] = x;
    }
}

// sums[p] = sum over the units, in order, of partial[u][p]
__global__ void __launch_bounds__(ST_T) k_sum_units(double* __restrict__ sums, const double* __restrict__ partial,
                                                    uint32_t units, uint32_t ldp) {
    const uint32_t p = blockIdx.x * ST_T + threadIdx.x;
    if (p >= ldp) return;
    double s = 0.0;
#pragma unroll 8
    for (uint32_t u = 0; u < units; ++u) s += partial[(size_t)u * ldp + p];
    sums[p] = s;
}

// ----------------------------------------------------------- host helpers

// Power levels of the range finder.  scikit-bio's fsvd uses one; with one, the
// reference's own tolerances on its 57-sample case (src/test_ska.cpp:247-420)
// fail for some probe draws, with two they hold (measured over 40 draws).
constexpr uint32_t PCOA_LEVELS = 2;

// One-sided Jacobi (Hestenes) on the m x m matrix R (column major): singular
// values S (descending) and right singular vectors V (column major, same order).
void jacobi_svd(std::vector<double> R, size_t m, std::vector<double>& S, std::vector<double>& V) {
    V.assign(m * m, 0.0);
    for (size_t c = 0; c < m; ++c) V[c * m + c] = 1.0;
    for (int sweep = 0; sweep < 60; ++sweep) {
        double off = 0.0;
        for (size_t p = 0; p + 1 < m; ++p)
            for (size_t q = p + 1; q < m; ++q) {
                double a = 0.0, b = 0.0, g = 0.0;
                for (size_t i = 0; i < m; ++i) {
                    a += R[p * m + i] * R[p * m + i];
                    b += R[q * m + i] * R[q * m + i];
                    g += R[p * m + i] * R[q * m + i];
                }
                if (g == 0.0 || std::fabs(g) <= 1e-15 * std::sqrt(a * b)) continue;
                off = std::max(off, std::fabs(g) / std::sqrt(a * b));
                const double zeta = (b - a) / (2.0 * g);
                const double t = (zeta >= 0.0 ? 1.0 : -1.0) / (std::fabs(zeta) + std::sqrt(1.0 + zeta * zeta));
                const double c = 1.0 / std::sqrt(1.0 + t * t), s = c * t;
                for (size_t i = 0; i < m; ++i) {
                    const double x = R[p * m + i], y = R[q * m + i];
                    R[p * m + i] = c * x - s * y;
                    R[q * m + i] = s * x + c * y;
                    const double vx = V[p * m + i], vy = V[q * m + i];
                    V[p * m + i] = c * vx - s * vy;
                    V[q * m + i] = s * vx + c * vy;
                }
            }
        if (off <= 1e-15) break;
    }
    S.assign(m, 0.0);
    for (size_t c = 0; c < m; ++c) {
        double s = 0.0;
        for (size_t i = 0; i < m; ++i) s += R[c * m + i] * R[c * m + i];
        S[c] = std::sqrt(s);
    }
    std::vector<size_t> order(m);
    for (size_t c = 0; c < m; ++c) order[c] = c;
    std::stable_sort(order.begin(), order.end(), [&](size_t x, size_t y) { return S[x] > S[y]; });
    std::vector<double> S2(m), V2(m * m);
    for (size_t c = 0; c < m; ++c) {
        S2[c] = S[order[c]];
        std::copy(&V[order[c] * m], &V[order[c] * m] + m, &V2[c * m]);
    }
    S = std::move(S2);
    V = std::move(V2);
}

template <class T>
bool upload_matrix(Buf& d, const void* mat, uint32_t n, std::string* err) {
    const size_t bytes = (size_t)n * n * sizeof(T);
    return alloc(d, bytes, err) && copy_to_device(d.p, mat, bytes, nullptr, err);
}

template <class T>
bool center_on_device(Buf& dB, const void* mat, uint32_t n, std::vector<double>& rmean, double& grand,
                      std::string* err) {
    if (!upload_matrix<T>(dB, mat, n, err)) return false;
    Buf dr;
    Idle idle;
    if (!alloc(dr, n * sizeof(double), err)) return false;
    hipLaunchKernelGGL((k_row_stats<T>), dim3(n), dim3(ST_T), 0, 0, dr.as<double>(), nullptr, dB.as<const T>(),
                       n);
    ST_HIP(hipGetLastError());
    rmean.resize(n);
    ST_HIP(hipMemcpy(rmean.data(), dr.p, n * sizeof(double), hipMemcpyDeviceToHost));
    grand = 0.0;
    for (double r : rmean) grand += r;
    grand /= n;
    const size_t nn = (size_t)n * n;
    hipLaunchKernelGGL((k_center_apply<T>), dim3((uint32_t)((nn + ST_T - 1) / ST_T)), dim3(ST_T), 0, 0, dB.as<T>(),
                       dr.as<const double>(), grand, n);
    ST_HIP(hipGetLastError());
    return true;
}

// Y = B X, X and Y n x ld row major (device)
template <class T>
bool symm_mult(double* Y, const Buf& dB, const double* X, uint32_t n, uint32_t ld, std::string* err) {
    for (uint32_t c0 = 0; c0 < ld; c0 += MAX_GRID_Y * 16)
        hipLaunchKernelGGL((k_symm_mult<T>), dim3((n + 15) / 16, std::min(MAX_GRID_Y, (ld - c0) / 16)),
                           dim3(64 * SM_WAVES), 0, 0, Y + c0, dB.as<const T>(), X + c0, n, ld);
    ST_HIP(hipGetLastError());
    return true;
}

// Thin QR of the column-major n x m matrix A.  Q != nullptr: its first q columns to Q;
// otherwise R's diagonal to r and the rest of R above A's diagonal.  V, n x q: scratch.
bool thin_qr(double* A, double* Q, double* V, double* r, uint32_t n, uint32_t m, uint32_t q, std::string* err) {
    const size_t lds = ((size_t)n * m + 2 * q) * sizeof(double);
    if (n <= QRS_MAX_N && lds <= QRS_LDS) {
        const auto k = Q ? k_qr_small<true> : k_qr_small<false>;
        ST_HIP(hipFuncSetAttribute((const void*)k, hipFuncAttributeMaxDynamicSharedMemorySize, (int)QRS_LDS));
        hipLaunchKernelGGL(k, dim3(1), dim3(QR_T), lds, 0, A, Q, r, n, m, q);
    } else {
        for (uint32_t k = 0; k < q; ++k)
            hipLaunchKernelGGL(k_householder, dim3(m - k), dim3(QR_T), 0, 0, A, V, r, n, k);
        if (Q) hipLaunchKernelGGL(k_form_q, dim3(q), dim3(QR_T), 0, 0, Q, V, n);
    }
    ST_HIP(hipGetLastError());
    return true;
}

template <class T>
bool pcoa_t(const void* mat, uint32_t n, uint32_t dims, uint64_t seed, double* eig, double* samples,
            double* proportion, std::string* err) {
    std::fill(eig, eig + dims, 0.0);
    std::fill(samples, samples + (size_t)n * dims, 0.0);
    std::fill(proportion, proportion + dims, 0.0);
    if (n == 0 || dims == 0) return true;
    Buf dB;
    std::vector<double> rmean;
    double grand = 0.0;
    if (!center_on_device<T>(dB, mat, n, rmean, grand, err)) return false;
    double trace = 0.0;
    for (uint32_t i = 0; i < n; ++i) {
        const double d = (double)((const T*)mat)[(size_t)i * n + i];
        trace += -0.5 * d * d - 2.0 * rmean[i] + grand;
    }
    // probes G (n x k), H = [B G | B^3 G | B^5 G] (n x 3k)
    const uint32_t k = dims + 2, m = (PCOA_LEVELS + 1) * k, q = std::min(n, m);
    const uint32_t ldk = (k + 15) / 16 * 16, ldq = (q + 15) / 16 * 16, nb = (n + ST_T - 1) / ST_T;
    Buf dX, dY, dH, dV, dQ, dW, dS, dr, dR;
    Idle idle;
    const uint32_t ldx = std::max(ldk, ldq);
    if (!alloc(dX, (size_t)n * ldx * 8, err) || !alloc(dY, (size_t)n * ldx * 8, err) ||
        !alloc(dH, (size_t)n * m * 8, err) || !alloc(dV, (size_t)n * q * 8, err) ||
        !alloc(dQ, (size_t)n * q * 8, err) || !alloc(dr, q * 8, err) || !alloc(dR, (size_t)q * q * 8, err))
        return false;
    double *X = dX.as<double>(), *Y = dY.as<double>(), *H = dH.as<double>(), *V = dV.as<double>(), *Q = dQ.as<double>();
    double* r = dr.as<double>();
    hipLaunchKernelGGL(k_probes, dim3(n, std::min(MAX_GRID_Y, (ldk + 63) / 64)), dim3(64), 0, 0, X, k, ldk, seed);
    ST_HIP(hipGetLastError());
    for (uint32_t level = 0; level <= PCOA_LEVELS; ++level) {
        // level 0: Y = B G; then Y = B (B Y_prev)
        if (!symm_mult<T>(Y, dB, X, n, ldk, err)) return false;
        if (level > 0) {
            if (!symm_mult<T>(X, dB, Y, n, ldk, err)) return false;
            std::swap(X, Y);
        }
        hipLaunchKernelGGL(k_to_columns, dim3(nb), dim3(ST_T), 0, 0, H + (size_t)level * k * n, Y, n, ldk, k);
        ST_HIP(hipGetLastError());
        std::swap(X, Y);   // X: the latest power
    }
    // Q of H, T = B Q (n x q), R of T
    if (!thin_qr(H, Q, V, r, n, m, q, err)) return false;
    hipLaunchKernelGGL(k_to_rows, dim3(nb), dim3(ST_T), 0, 0, X, Q, n, ldq, q);
    ST_HIP(hipGetLastError());
    if (!symm_mult<T>(Y, dB, X, n, ldq, err)) return false;
    hipLaunchKernelGGL(k_to_columns, dim3(nb), dim3(ST_T), 0, 0, H, Y, n, ldq, q);
    ST_HIP(hipGetLastError());
    if (!thin_qr(H, nullptr, V, r, n, q, q, err)) return false;
    // SVD of T through its R factor: T = Q2 R, R = U S V' -> right singular vectors V
    std::vector<double> R((size_t)q * q);
    hipLaunchKernelGGL(k_pack_r, dim3(q), dim3(ST_T), 0, 0, dR.as<double>(), H, r, n, q);
    ST_HIP(hipGetLastError());
    ST_HIP(hipMemcpy(R.data(), dR.p, R.size() * 8, hipMemcpyDeviceToHost));
    std::vector<double> S, Vr;
    jacobi_svd(R, q, S, Vr);
    const uint32_t used = std::min(dims, q);
    // coordinates: eigenvectors Q V scaled by the square roots of the eigenvalues
    std::vector<double> W((size_t)q * std::max(used, 1u));
    for (uint32_t d = 0; d < used; ++d) {
        eig[d] = S[d];
        proportion[d] = trace != 0.0 ? S[d] / trace : 0.0;
        const double sq = std::sqrt(std::max(S[d], 0.0));
        for (uint32_t c = 0; c < q; ++c) W[(size_t)d * q + c] = Vr[(size_t)d * q + c] * sq;
    }
    if (!alloc(dW, W.size() * 8, err)) return false;
    ST_HIP(hipMemcpy(dW.p, W.data(), W.size() * 8, hipMemcpyHostToDevice));
    if (!alloc(dS, (size_t)n * dims * 8, err)) return false;
    hipLaunchKernelGGL(k_coordinates, dim3(nb, std::min(MAX_GRID_Y, dims)), dim3(ST_T), 0, 0, dS.as<double>(), Q, dW.as<const double>(), n, q,
                       used, dims);
    ST_HIP(hipGetLastError());
    ST_HIP(hipMemcpy(samples, dS.p, (size_t)n * dims * 8, hipMemcpyDeviceToHost));
    return true;
}

template <class T>
bool permanova_t(const void* mat, uint32_t n, const uint32_t* grouping, uint32_t n_perm, uint64_t seed,
                 double* fstat, double* pvalue, std::string* err) {
    *fstat = *pvalue = std::numeric_limits<double>::quiet_NaN();
    if (n < 2) return true;
    uint32_t groups = 0;
    for (uint32_t i = 0; i < n; ++i) groups = std::max(groups, grouping[i] + 1);
    std::vector<double> size(groups, 0.0);
    for (uint32_t i = 0; i < n; ++i) size[grouping[i]] += 1.0;
    uint32_t present = 0;
    for (double s : size) present += s > 0.0;
    if (present < 2 || present >= n) return true;   // pseudo-F undefined
    std::vector<double> inv(groups, 0.0);
    for (uint32_t g = 0; g < groups; ++g) inv[g] = size[g] > 0.0 ? 1.0 / size[g] : 0.0;
    // label rows: the grouping, then n_perm Fisher-Yates shuffles of it, sample major
    const uint32_t n_lab = n_perm + 1, ldp = (n_lab + PM_PW - 1) / PM_PW * PM_PW;
    Buf dD, dL, dg, drows, dinv, dpart, dsum, dunits, dr, du;
    Idle idle;
    if (!upload_matrix<T>(dD, mat, n, err) || !alloc(dL, (size_t)n * ldp * 4, err) || !alloc(dinv, groups * 8, err))
        return false;
    if (n <= SHUF_MAX_N && groups <= SHUF_MAX_GROUPS) {
        if (!alloc(dg, (size_t)n * 4, err)) return false;
        ST_HIP(hipMemcpy(dg.p, grouping, (size_t)n * 4, hipMemcpyHostToDevice));
        hipLaunchKernelGGL(k_shuffles, dim3(ldp), dim3(64), SHUF_TAGS * 4 + n, 0, dL.as<uint32_t>(), dg.as<const uint32_t>(), n, n_lab,
                           ldp, seed);
        ST_HIP(hipGetLastError());
    } else {   // more samples or groups than bytes in LDS hold
        std::vector<uint32_t> L((size_t)n_lab * n);
        for (uint32_t p = 0; p < n_lab; ++p) {
            uint32_t* row = &L[(size_t)p * n];
            std::copy(grouping, grouping + n, row);
            const uint64_t key = mix64(seed ^ mix64(p));
            for (uint32_t i = n - 1; p && i > 0; --i) std::swap(row[i], row[(uint32_t)(mix64(key + i) % (i + 1))]);
        }
        if (!alloc(drows, L.size() * 4, err) || !copy_to_device(drows.p, L.data(), L.size() * 4, nullptr, err)) return false;
        hipLaunchKernelGGL(k_label_columns, dim3((n + 63) / 64, ldp / 64), dim3(256), 0, 0, dL.as<uint32_t>(),
                           drows.as<const uint32_t>(), n, n_lab, ldp);
        ST_HIP(hipGetLastError());
    }
    ST_HIP(hipMemcpy(dinv.p, inv.data(), groups * 8, hipMemcpyHostToDevice));
    // units of 64 rows x `chunk` columns that hold a pair of the upper triangle; longer
    // chunks once the workgroups fill the chip many times over (the units' sums are
    // as many as the workgroups)
    const uint64_t rb = (n + PM_R - 1) / PM_R;
    uint32_t chunk = PM_J;
    while (chunk < n && rb * rb * PM_R / (2 * chunk) * (ldp / PM_PW) > 65536) chunk *= 2;
    std::vector<uint32_t> units;
    for (uint32_t ib = 0; ib < rb; ++ib)
        for (uint32_t jc = ib * PM_R / chunk; (uint64_t)jc * chunk < n; ++jc) units.push_back(ib << 16 | jc);
    const uint32_t nu = (uint32_t)units.size();
    if (!alloc(dunits, units.size() * 4, err) || !alloc(dpart, (size_t)nu * ldp * 8, err) || !alloc(dsum, ldp * 8, err))
        return false;
    ST_HIP(hipMemcpy(dunits.p, units.data(), units.size() * 4, hipMemcpyHostToDevice));
    hipLaunchKernelGGL((k_permanova<T>), dim3(nu, ldp / PM_PW), dim3(256), 0, 0, dpart.as<double>(), dD.as<const T>(),
                       dL.as<const uint32_t>(), dinv.as<const double>(), dunits.as<const uint32_t>(), n, ldp, chunk);
    hipLaunchKernelGGL(k_sum_units, dim3((ldp + ST_T - 1) / ST_T), dim3(ST_T), 0, 0, dsum.as<double>(),
                       dpart.as<const double>(), nu, ldp);
    ST_HIP(hipGetLastError());
    std::vector<double> within(ldp);
    ST_HIP(hipMemcpy(within.data(), dsum.p, ldp * 8, hipMemcpyDeviceToHost));
    // s_T over the upper triangle
    if (!alloc(dr, n * 8, err) || !alloc(du, n * 8, err)) return false;
    hipLaunchKernelGGL((k_row_stats<T>), dim3(n), dim3(ST_T), 0, 0, dr.as<double>(), du.as<double>(),
                       dD.as<const T>(), n);
    ST_HIP(hipGetLastError());
    std::vector<double> upper(n);
    ST_HIP(hipMemcpy(upper.data(), du.p, n * 8, hipMemcpyDeviceToHost));
    double sT = 0.0;
    for (double u : upper) sT += u;
    sT /= n;
    auto f_of = [&](uint32_t p) {
        const double sW = within[p];
        return ((sT - sW) / (present - 1)) / (sW / (n - present));
    };
    const double f0 = f_of(0);
    uint32_t ge = 0;
    for (uint32_t p = 1; p < n_lab; ++p) ge += f_of(p) >= f0;
    *fstat = f0;
    *pvalue = n_perm ? (double)(ge + 1) / (double)(n_perm + 1) : std::numeric_limits<double>::quiet_NaN();
    return true;
}

}  // namespace

// ---------------------------------------------------------------- allocation-free centring
// The device scratch of center_matrix_noalloc: the row means of one call at
// [0, n) and its grand mean at [NOALLOC_MAX_N].  Each GPU holds its own copy
// for the life of the process; every call on a GPU overwrites it, so calls
// that overlap on one GPU race.
static __device__ __align__(256) double scratch[NOALLOC_MAX_N + 32];

namespace {

constexpr int SCRATCH_MAX_DEVICES = 64;
std::mutex g_scratch_mu;
double* g_scratch_dev[SCRATCH_MAX_DEVICES] = {};   // per device: the address of its copy of `scratch`

// the current device's copy of `scratch` (looked up once per device)
bool scratch_of_device(double** out, std::string* err) {
    int dev = 0;
    ST_HIP(hipGetDevice(&dev));
    if (dev < 0 || dev >= SCRATCH_MAX_DEVICES) {
        if (err) *err = "device index " + std::to_string(dev) + " beyond the scratch table";
        return false;
    }
    std::lock_guard<std::mutex> lock(g_scratch_mu);
    if (!g_scratch_dev[dev]) {
        void* ptr = nullptr;
        ST_HIP(hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch)));
        g_scratch_dev[dev] = (double*)ptr;
    }
    *out = g_scratch_dev[dev];
    return true;
}

// rm[n_max] = sum_i rm[i] / n, the row means added in index order (as center_on_device does on the host)
__global__ void k_grand_mean(double* __restrict__ rm, uint32_t n) {
    if (blockIdx.x || threadIdx.x) return;
    double g = 0.0;
    for (uint32_t i = 0; i < n; ++i) g += rm[i];
    rm[NOALLOC_MAX_N] = g / n;
}

// C_ij = -D_ij^2 / 2 - rmean_i - rmean_j + grand (the arithmetic of k_center_apply), C may be D
__global__ void __launch_bounds__(ST_T) k_center_copy(double* C, const double* D, const double* __restrict__ rm,
                                                      uint32_t n) {
    const size_t q = (size_t)blockIdx.x * ST_T + threadIdx.x;
    if (q >= (size_t)n * n) return;
    const uint32_t i = (uint32_t)(q / n), j = (uint32_t)(q % n);
    const double d = D[q];
    C[q] = -0.5 * d * d - rm[i] - rm[j] + rm[NOALLOC_MAX_N];
}

}  // namespace

bool center_matrix_noalloc(const double* d_mat, uint32_t n, double* d_centred, void* stream, std::string* err) {
    if (n > NOALLOC_MAX_N) {
        if (err) *err = "ssu_center_matrix_fp64_noalloc: n = " + std::to_string(n) + " exceeds its maximum of " +
                        std::to_string(NOALLOC_MAX_N) + " samples";
        return false;
    }
    if (n == 0) return true;
    double* rm = nullptr;
    if (!scratch_of_device(&rm, err)) return false;
    hipStream_t st = (hipStream_t)stream;
    hipLaunchKernelGGL((k_row_stats<double>), dim3(n), dim3(ST_T), 0, st, rm, nullptr, d_mat, n);
    ST_HIP(hipGetLastError());
    hipLaunchKernelGGL(k_grand_mean, dim3(1), dim3(64), 0, st, rm, n);
    ST_HIP(hipGetLastError());
    const size_t nn = (size_t)n * n;
    hipLaunchKernelGGL(k_center_copy, dim3((uint32_t)((nn + ST_T - 1) / ST_T)), dim3(ST_T), 0, st, d_centred, d_mat,
                       rm, n);
    ST_HIP(hipGetLastError());
    return true;
}

bool center_matrix(const void* mat, bool in_fp64, uint32_t n, double* centred, std::string* err) {
    if (n == 0) return true;
    Buf dB;
    std::vector<double> rmean;
    double grand = 0.0;
    const size_t nn = (size_t)n * n;
    if (in_fp64) {
        if (!center_on_device<double>(dB, mat, n, rmean, grand, err)) return false;
        ST_HIP(hipMemcpy(centred, dB.p, nn * 8, hipMemcpyDeviceToHost));
    } else {
        if (!center_on_device<float>(dB, mat, n, rmean, grand, err)) return false;
        std::vector<float> tmp(nn);
        ST_HIP(hipMemcpy(tmp.data(), dB.p, nn * 4, hipMemcpyDeviceToHost));
        for (size_t q = 0; q < nn; ++q) centred[q] = tmp[q];
    }
    return true;
}

bool pcoa(const void* mat, bool in_fp64, uint32_t n, uint32_t dims, uint64_t seed, double* eigenvalues,
          double* samples, double* proportion, std::string* err) {
    return in_fp64 ? pcoa_t<double>(mat, n, dims, seed, eigenvalues, samples, proportion, err)
                   : pcoa_t<float>(mat, n, dims, seed, eigenvalues, samples, proportion, err);
}

bool permanova(const void* mat, bool in_fp64, uint32_t n, const uint32_t* grouping, uint32_t n_perm, uint64_t seed,
               double* fstat, double* pvalue, std::string* err) {
    return in_fp64 ? permanova_t<double>(mat, n, grouping, n_perm, seed, fstat, pvalue, err)
                   : permanova_t<float>(mat, n, grouping, n_perm, seed, fstat, pvalue, err);
}

}  // namespace ssu
