// kf_direct.hip -- fast diagonalisation of the shifted stencil (kf_direct.h).
#include "kf_direct.h"
#include "kf_plane.h"

#include <algorithm>
#include <cmath>

namespace kf {

using namespace fft;

// ======================================================================== one axis' modes (host)
// Eigenvalues of a symmetric tridiagonal matrix (diagonal a, off-diagonal b)
// and its eigenvectors as the rows of Z, by the implicit QR algorithm with
// Wilkinson's shift (Golub and Van Loan, Matrix Computations, 8.3).  False
// when it does not converge.
static bool tridiagonal_modes(std::vector<double> &a, std::vector<double> &b, std::vector<double> &Z)
{
    const int m = (int)a.size();
    Z.assign((size_t)m * m, 0.);
    for (int i = 0; i < m; ++i) Z[(size_t)i * m + i] = 1.;
    int hi = m - 1;
    for (long guard = 0; hi > 0; ++guard) {
        if (guard > 60L * m) return false;
        for (int i = 0; i < hi; ++i)
            if (std::fabs(b[i]) <= 1.2e-16 * (std::fabs(a[i]) + std::fabs(a[i + 1]))) b[i] = 0.;
        while (hi > 0 && b[hi - 1] == 0.) --hi;
        if (hi == 0) break;
        int lo = hi - 1;
        while (lo > 0 && b[lo - 1] != 0.) --lo;
        const double dl = 0.5 * (a[hi - 1] - a[hi]), bb = b[hi - 1];
        const double mu = a[hi] - bb * bb / (dl + std::copysign(std::hypot(dl, bb), dl));
        double x = a[lo] - mu, z = b[lo];
        for (int k = lo; k < hi; ++k) {
            const double r = std::hypot(x, z);
            const double c = r > 0. ? x / r : 1., s = r > 0. ? z / r : 0.;
            if (k > lo) b[k - 1] = r;
            const double ak = a[k], bk = b[k], ak1 = a[k + 1];
            a[k] = c * c * ak + 2. * c * s * bk + s * s * ak1;
            a[k + 1] = s * s * ak - 2. * c * s * bk + c * c * ak1;
            b[k] = c * s * (ak1 - ak) + (c * c - s * s) * bk;
            if (k + 1 < hi) {
                x = b[k];
                z = s * b[k + 1];
                b[k + 1] *= c;
            }
            double *p = &Z[(size_t)k * m], *q = p + m;
            for (int i = 0; i < m; ++i) {
                const double u = p[i], v = q[i];
                p[i] = c * u + s * v;
                q[i] = c * v - s * u;
            }
        }
    }
    return true;
}

static bool mirrored(const std::vector<double> &h, int n)
{
    for (int i = 0; i < n; ++i)
        if (!(h[i + 1] > 0.) || std::fabs(h[i + 1] - h[n - i]) > 1e-10 * h[i + 1]) return false;
    return true;
}

// The second difference of one axis, (u_{i+1} - u_i)/h_{i+1} - (u_i -
// u_{i-1})/h_i over v_i = (h_{i+1} + h_i)/2, is symmetric in the inner
// product of v: L = T diag(lam) T^-1 with T = V^-1/2 Q, T^-1 = Q^T V^1/2 and
// Q orthogonal.  Spacings that mirror about point 0 split it into even
// modes (u_{n-i} = u_i) and odd ones, each a tridiagonal matrix.
struct Modes {
    std::vector<double> lam, T, Ti;  // T[i][m], Ti[m][i]
    bool ok = true;
};
static Modes axis_modes(const std::vector<double> &hin, int n)
{
    std::vector<double> h(n + 1), v(n);
    for (int i = 0; i < n; ++i) h[i + 1] = 0.5 * (hin[i + 1] + hin[n - i]);
    h[0] = h[n];
    double vm = 0.;
    for (int i = 0; i < n; ++i) {
        v[i] = 0.5 * (h[i + 1] + h[i]);
        vm += v[i] / n;
    }
    auto S = [&](int i, int j) {  // V^1/2 L V^-1/2, periodic
        double s = 0.;
        if (i == j) s -= (1. / h[i + 1] + 1. / h[i]) / v[i];
        if (j == (i + 1) % n) s += 1. / (h[i + 1] * std::sqrt(v[i] * v[j]));
        if (i == (j + 1) % n) s += 1. / (h[j + 1] * std::sqrt(v[i] * v[j]));
        return s;
    };
    Modes M;
    M.T.assign((size_t)n * n, 0.);
    M.Ti.assign((size_t)n * n, 0.);
    for (int odd = 0; odd < 2; ++odd) {
        // basis vector of k: e_k alone when n - k = k (mod n), else (e_k +- e_{n-k})/sqrt 2
        std::vector<int> ks;
        for (int k = odd; k <= n - k; ++k)
            if (!odd || k != n - k) ks.push_back(k);
        const int m = (int)ks.size();
        if (m == 0) continue;
        const double sg = odd ? -1. : 1.;
        auto single = [&](int k) { return k == 0 || k == n - k; };
        auto dot = [&](int p, int q) {
            double s = S(p, q);
            if (!single(p)) s += sg * S(n - p, q);
            if (!single(q)) s += sg * S(p, n - q);
            if (!single(p) && !single(q)) s += S(n - p, n - q);
            return s * (single(p) ? 1. : std::sqrt(0.5)) * (single(q) ? 1. : std::sqrt(0.5));
        };
        std::vector<double> a(m), b(std::max(m - 1, 0)), Z;
        for (int q = 0; q < m; ++q) a[q] = dot(ks[q], ks[q]);
        for (int q = 0; q + 1 < m; ++q) b[q] = dot(ks[q], ks[q + 1]);
        M.ok = tridiagonal_modes(a, b, Z) && M.ok;
        for (int e = 0; e < m; ++e) {
            const size_t mode = M.lam.size();
            M.lam.push_back(std::min(a[e], 0.));
            for (int q = 0; q < m; ++q) {
                const int k = ks[q];
                const double z = Z[(size_t)e * m + q] * (single(k) ? 1. : std::sqrt(0.5));
                for (int side = 0; side < (single(k) ? 1 : 2); ++side) {
                    const int i = side ? n - k : k;
                    const double u = side ? sg * z : z, w = std::sqrt(v[i] / vm);
                    M.T[(size_t)i * n + mode] = u / w;
                    M.Ti[mode * n + i] = u * w;
                }
            }
        }
    }
    return M;
}

template <typename R>
bool Direct<R>::possible(const AxisDesc ax[3], const std::vector<double> h[3])
{
    bool uniform = true;
    for (int d = 0; d < 3; ++d) uniform = uniform && ax[d].type == 1;
    if (uniform) return grid_supported(ax[0].n, ax[1].n, ax[2].n);
    for (int d = 0; d < 3; ++d)
        if (!mirrored(h[d], ax[d].n)) return false;
    return true;
}

template <typename R>
Direct<R>::Direct(const AxisDesc ax[3], const std::vector<double> h[3], hipStream_t s, const fft::Plan<R> *like)
{
    fourier_ = true;
    for (int d = 0; d < 3; ++d) {
        n_[d] = ax[d].n;
        fourier_ = fourier_ && ax[d].type == 1;
    }
    std::vector<R> host;
    size_t at[9] = {};
    auto put = [&](int slot, const std::vector<double> &t) {
        host.resize((host.size() + 63) / 64 * 64);
        at[slot] = host.size();
        for (double x : t) host.push_back((R)x);
    };
    if (fourier_) {
        const double pi = std::acos(-1.);
        for (int d = 0; d < 3; ++d) {
            const double step = ax[d].L / n_[d];
            std::vector<double> lam(d == 2 ? n_[2] / 2 + 1 : n_[d]);
            for (size_t k = 0; k < lam.size(); ++k) {
                const double w = 2. * std::sin(pi * (double)k / n_[d]) / step;
                lam[k] = -w * w;
            }
            put(d, lam);
        }
    } else {
        Modes M[3];
        for (int d = 0; d < 3; ++d) {
            int same = -1;
            for (int e = 0; e < d; ++e)
                if (h[e] == h[d]) same = e;
            M[d] = same >= 0 ? M[same] : axis_modes(h[d], n_[d]);
            if (!M[d].ok) throw Error("the axis' eigenvalues did not converge");
            put(d, M[d].lam);
            const int n = n_[d];
            if (d == 2) {
                for (int i = 0; i < n; ++i)
                    for (int j = 0; j < i; ++j) {
                        std::swap(M[d].T[(size_t)i * n + j], M[d].T[(size_t)j * n + i]);
                        std::swap(M[d].Ti[(size_t)i * n + j], M[d].Ti[(size_t)j * n + i]);
                    }
            }
            put(3 + d, M[d].Ti);
            put(6 + d, M[d].T);
        }
    }
    try {
        KF_HIP(hipMalloc(&pool_, sizeof(R) * host.size()));
        KF_HIP(hipMemcpyAsync(pool_, host.data(), sizeof(R) * host.size(), hipMemcpyHostToDevice, s));
        KF_HIP(hipStreamSynchronize(s));
        for (int d = 0; d < 3; ++d) {
            lam_[d] = pool_ + at[d];
            fwd_[d] = pool_ + at[3 + d];
            inv_[d] = pool_ + at[6 + d];
        }
        if (fourier_) plan_init<R>(plan_, n_[0], n_[1], n_[2], s, like, false);
        else KF_HIP(hipMalloc(&tmp_, sizeof(R) * (size_t)n_[0] * n_[1] * n_[2]));
    } catch (...) {
        release();
        throw;
    }
}

template <typename R>
Direct<R>::~Direct()
{
    release();
}

template <typename R>
void Direct<R>::release()
{
    if (fourier_) plan_free<R>(plan_);
    (void)hipFree(pool_);
    (void)hipFree(tmp_);
}

// ======================================================================== equidistant grids
// The x axis both ways in one pass: forward transform of a column, division
// by lambda - c, inverse transform, the column staying in LDS between the
// two.  One read and one write of the spectrum instead of two of each, in
// place (a column is one workgroup's).  Bound by memory: at 256^3 FP32 28 us
// for 135 MB, 4.8 TB/s, the rate of a large copy on this card.
template <typename R, int N, int CB>
__global__ void __launch_bounds__(tpt_for(N) * CB)
k_direct_x(const C2<R> *__restrict__ tw_g, C2<R> *__restrict__ f, unsigned ny, unsigned nzs, unsigned nzc,
           const R *__restrict__ lx, const R *__restrict__ ly, const R *__restrict__ lz, const double *__restrict__ cp,
           R scale, const int *ctl)
{
    using C = C2<R>;
    constexpr int TPT = tpt_for(N);
    constexpr int WG = TPT * CB;
    __shared__ C lds[N * CB];
    __shared__ C tw[N];
    if (ctl && ctl[0]) return;
    const int tid = threadIdx.x;
    for (int m = tid; m < N; m += WG) tw[m] = tw_g[m];
    const int c = tid % CB, t0 = tid / CB;
    const unsigned q = xcd_block(blockIdx.x, gridDim.x) * CB + c;
    const unsigned j = q / nzs, k = q - j * nzs;
    const bool live = j < ny && k < nzc;
    const unsigned stride = ny * nzs;
    const R lyz = live ? ly[j] + lz[k] - (R)cp[0] : (R)-1;
    const ColBuf<C, N, CB> A{lds, c};
    struct Ld {
        const C *p;
        unsigned stride;
        bool live;
        __device__ __forceinline__ C ld(int t, int = 0) const
        {
            return live ? p[(size_t)t * stride] : mk<C>((R)0, (R)0);
        }
    } src{f + q, stride, live};
    struct Scaled {
        const ColBuf<C, N, CB> &A;
        const R *lx;
        R lyz, scale;
        __device__ __forceinline__ C ld(int t, int = 0) const
        {
            const C v = A.ld(t);
            return cscale(v, scale / (lx[t] + lyz));
        }
    } mid{A, lx, lyz, scale};
    struct St {
        C *p;
        unsigned stride;
        bool live;
        __device__ __forceinline__ void st(int t, C v, int = 0) const
        {
            if (live) p[(size_t)t * stride] = v;
        }
    } dst{f + q, stride, live};
    fft_io<C, N, TPT, -1, false, true>(tw, t0, src, A, A, A);
    __syncthreads();
    fft_io<C, N, TPT, +1, false, false, true>(tw, t0, mid, dst, A, A);
}

template <typename R>
void Direct<R>::x_pass(const double *c, const int *ctl, hipStream_t s)
{
    Plan<R> &p = plan_;
    const unsigned nv = (unsigned)p.nzc;
    const R scale = (R)(1.0 / (double)p.nr);
    switch (p.nx) {
#define KF_CASE(NN)                                                                                              \
    case NN: {                                                                                                   \
        constexpr int CB = cb_for<R>(NN);                                                                        \
        hipLaunchKernelGGL((k_direct_x<R, NN, CB>), dim3((unsigned)((scratch_cols_x(p) + CB - 1) / CB)),         \
                           dim3(tpt_for(NN) * CB), 0, s, p.tw_x, p.scratch, (unsigned)p.ny, (unsigned)p.nzs, nv, \
                           lam_[0], lam_[1], lam_[2], c, scale, ctl);                                            \
        break;                                                                                                   \
    }
        KF_FFT_LENGTHS(KF_CASE)
#undef KF_CASE
    default:
        throw Error("unsupported transform length " + std::to_string(p.nx));
    }
}

template <typename R>
void Direct<R>::solve_fourier(const R *b, R *x, const double *c, const int *ctl, hipStream_t s)
{
    Plan<R> &p = plan_;
    const long rows = (long)p.nx * p.ny;
    const StridedAddr ay = saddr_y(p);
    const unsigned nv = (unsigned)p.nzc;
    if (p.plane_fwd) {
        plane_r2c<R>(plane_tabs(p), PlaneIn<R>{four<const R *>(b), {}, nullptr, 0, 0}, p.scratch, s, ctl);
    } else {
        launch_zr2c<R>(p.nz / 2, rows, p.tw_m, p.tw_n, Gated<RowLoadReal<R>>{{b, p.nz}, ctl},
                       RowStoreC<R>{p.scratch, p.nzs}, s, 1000);
        launch_strided<R, -1>(p.ny, scratch_cols_y(p), p.tw_y, Gated<LoadMasked<R>>{{p.scratch, ay, nv}, ctl},
                              StoreMasked<R>{p.scratch, ay, nv}, s, 1000, p.vy);
    }
    x_pass(c, ctl, s);
    if (p.plane_inv) {
        PlaneOut<R> z{};
        z.scale = (R)1;
        z.o = four<R *>(x);
        plane_c2r<R>(plane_tabs(p), four<const C2<R> *>(p.scratch), nullptr, nullptr, z, 1, s, ctl);
        return;
    }
    launch_strided<R, +1>(p.ny, scratch_cols_y(p), p.tw_y, Gated<LoadMasked<R>>{{p.scratch, ay, nv}, ctl},
                          StoreMasked<R>{p.scratch, ay, nv}, s, 1000, p.vy);
    launch_zc2r<R>(p.nz / 2, rows, p.tw_m, p.tw_n, Gated<RowLoadC<R>>{{p.scratch, p.nzs}, ctl},
                   RowStoreReal<R>{x, p.nz, (R)1}, s, 1000);
}

// ======================================================================== stretched grids
template <typename R>
struct MfmaT;
template <>
struct MfmaT<double> {
    typedef double acc __attribute__((ext_vector_type(4)));
    static __device__ __forceinline__ acc mma(double a, double b, acc c)
    {
        return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
    }
    // row of accumulator element r of lane group g = lane / 16
    static __device__ __forceinline__ int row(int g, int r) { return 4 * r + g; }
};
template <>
struct MfmaT<float> {
    typedef float acc __attribute__((ext_vector_type(4)));
    static __device__ __forceinline__ acc mma(float a, float b, acc c)
    {
        return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
    }
    static __device__ __forceinline__ int row(int g, int r) { return 4 * g + r; }
};

// D[m][n] = sum_k A[m][k] B[k][n], batched: A rows of lda with k contiguous,
// B rows of ldb and D rows of ldd with n contiguous.  A transform along z
// takes the field's rows as A and the axis' transposed matrix as B; along
// y (one product per x plane) and x the matrix is A and the field B.
struct ModalMap {
    int M, N, K;
    long lda, ldb, ldd;   // row strides
    long sb, sd;          // batch strides of B and D (A is shared)
    int mt, nt, nfast;    // wave tiles along m and n, and which varies fastest
    unsigned tiles;       // mt * nt * batch
};

// One wavefront forms a (16 TM) x (16 TN) tile on the matrix cores straight
// from global memory: the matrix (n^2 values: 128 KB at 128 points FP64, 512
// KB at 256, 2 MB at the 512 of the longest z axis, of a 4 MB L2) and the
// field panel are read by neighbouring wavefronts of one XCD, so they come
// from its L2, and nothing needs a barrier.  At 128^3 FP64 a product is 18.9 us for 0.54
// GFLOP (28 of 72 TFLOP/s that a large FP64 product reaches; its 34 MB stay
// in the caches), at 64^3 4.7 us, where the launch bounds it.  k is contracted in an order that lets a lane
// load 16 bytes of A at once: lane group g takes k = KV g .. KV g + KV - 1
// of each 4 KV, in A and B alike.  The loads of GS such steps are in flight
// while the previous GS are multiplied.
template <typename R, int TM, int TN, bool KFULL, bool SCALE>
__global__ void __launch_bounds__(256)
k_modal(ModalMap mp, const R *__restrict__ A, const R *__restrict__ B, R *__restrict__ D, const R *__restrict__ lm,
        const R *__restrict__ ly, const R *__restrict__ lz, int nz, const double *__restrict__ cp, const int *ctl)
{
    using T = MfmaT<R>;
    using Acc = typename T::acc;
    constexpr int KV = 16 / (int)sizeof(R);
    constexpr int KS = 4 * KV;
    constexpr int GS = TM * TN == 1 ? 4 : 2;
    if (ctl && ctl[0]) return;
    const unsigned w = xcd_block(blockIdx.x, gridDim.x) * 4u + (threadIdx.x >> 6);
    if (w >= mp.tiles) return;
    const int lane = threadIdx.x & 63, i = lane & 15, g = lane >> 4;
    const unsigned per = (unsigned)(mp.mt * mp.nt);
    const unsigned bt = w / per, r = w - bt * per;
    const int tm = (int)(mp.nfast ? r / (unsigned)mp.nt : r % (unsigned)mp.mt);
    const int tn = (int)(mp.nfast ? r % (unsigned)mp.nt : r / (unsigned)mp.mt);
    const int m0 = tm * 16 * TM, n0 = tn * 16 * TN;
    const R *ap[TM], *bp[TN];
#pragma unroll
    for (int a = 0; a < TM; ++a) ap[a] = A + (long)min(m0 + 16 * a + i, mp.M - 1) * mp.lda;
#pragma unroll
    for (int b = 0; b < TN; ++b) bp[b] = B + (long)bt * mp.sb + min(n0 + 16 * b + i, mp.N - 1);
    Acc acc[TM][TN];
#pragma unroll
    for (int a = 0; a < TM; ++a)
#pragma unroll
        for (int b = 0; b < TN; ++b) acc[a][b] = Acc{(R)0, (R)0, (R)0, (R)0};
    R av[2][GS][TM][KV], bv[2][GS][TN][KV];
    const int steps = (mp.K + KS - 1) / KS;
    auto load = [&](int buf, int s0) {
#pragma unroll
        for (int s = 0; s < GS; ++s) {
            const int k0 = min(s0 + s, steps - 1) * KS + g * KV;
#pragma unroll
            for (int u = 0; u < KV; ++u) {
                const int k = KFULL ? k0 + u : min(k0 + u, mp.K - 1);
                const bool in = s0 + s < steps && (KFULL || k0 + u < mp.K);
#pragma unroll
                for (int a = 0; a < TM; ++a) {
                    const R v = ap[a][k];
                    av[buf][s][a][u] = in ? v : (R)0;
                }
#pragma unroll
                for (int b = 0; b < TN; ++b) bv[buf][s][b][u] = bp[b][(long)k * mp.ldb];
            }
        }
    };
    auto mul = [&](int buf) {
#pragma unroll
        for (int s = 0; s < GS; ++s)
#pragma unroll
            for (int u = 0; u < KV; ++u)
#pragma unroll
                for (int a = 0; a < TM; ++a)
#pragma unroll
                    for (int b = 0; b < TN; ++b)
                        acc[a][b] = T::mma(av[buf][s][a][u], bv[buf][s][b][u], acc[a][b]);
    };
    load(0, 0);
    for (int s = 0; s < steps; s += 2 * GS) {
        if (s + GS < steps) load(1, s + GS);
        mul(0);
        if (s + GS >= steps) break;
        if (s + 2 * GS < steps) load(0, s + 2 * GS);
        mul(1);
    }
    R *out = D + (long)bt * mp.sd;
    const R c = SCALE ? (R)cp[0] : (R)0;
#pragma unroll
    for (int b = 0; b < TN; ++b) {
        const int n = n0 + 16 * b + i;
        if (n >= mp.N) continue;
        R lyz = (R)0;
        if (SCALE) {
            const unsigned j = (unsigned)n / (unsigned)nz;
            lyz = ly[j] + lz[(unsigned)n - j * (unsigned)nz] - c;
        }
#pragma unroll
        for (int a = 0; a < TM; ++a)
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const int m = m0 + 16 * a + T::row(g, e);
                if (m >= mp.M) continue;
                R v = acc[a][b][e];
                if (SCALE) v /= lm[m] + lyz;
                out[(long)m * mp.ldd + n] = v;
            }
    }
}

template <typename R>
void Direct<R>::solve_modal(const R *b, R *x, const double *c, const int *ctl, hipStream_t s)
{
    const int nx = n_[0], ny = n_[1], nz = n_[2];
    const long plane = (long)ny * nz;
    auto go = [&](ModalMap m, int batch, const R *A, const R *B, R *D, bool scale) {
        // 32 x 32 tiles where they still give every SIMD two wavefronts, else 16 x 16
        const long big = (long)((m.M + 31) / 32) * ((m.N + 31) / 32) * batch;
        const int t = big >= 2048 ? 32 : 16;
        m.mt = (m.M + t - 1) / t;
        m.nt = (m.N + t - 1) / t;
        m.tiles = (unsigned)(m.mt * m.nt * batch);
        const bool full = m.K % (64 / (int)sizeof(R)) == 0;
        const dim3 grid((m.tiles + 3) / 4), blk(256);
#define KF_MODAL(TT, KF, SC)                                                                                        \
    hipLaunchKernelGGL((k_modal<R, TT, TT, KF, SC>), grid, blk, 0, s, m, A, B, D, lam_[0], lam_[1], lam_[2], nz, c, \
                       ctl)
#define KF_MODAL_T(TT)                                  \
    if (full && scale) KF_MODAL(TT, true, true);        \
    else if (full) KF_MODAL(TT, true, false);           \
    else if (scale) KF_MODAL(TT, false, true);          \
    else KF_MODAL(TT, false, false)
        if (t == 32) {
            KF_MODAL_T(2);
        } else {
            KF_MODAL_T(1);
        }
#undef KF_MODAL_T
#undef KF_MODAL
    };
    const ModalMap mz{nx * ny, nz, nz, nz, nz, nz, 0, 0, 0, 0, 1, 0};
    const ModalMap my{ny, nz, ny, ny, nz, nz, plane, plane, 0, 0, 0, 0};
    const ModalMap mx{nx, (int)plane, nx, nx, plane, plane, 0, 0, 0, 0, 0, 0};
    go(mz, 1, b, fwd_[2], tmp_, false);
    go(my, nx, fwd_[1], tmp_, x, false);
    go(mx, 1, fwd_[0], x, tmp_, true);
    go(mx, 1, inv_[0], tmp_, x, false);
    go(my, nx, inv_[1], x, tmp_, false);
    go(mz, 1, tmp_, inv_[2], x, false);
}

template <typename R>
void Direct<R>::solve(const R *b, R *x, const double *c, const int *ctl, hipStream_t s)
{
    if (fourier_) solve_fourier(b, x, c, ctl, s);
    else solve_modal(b, x, c, ctl, s);
}

template class Direct<float>;
template class Direct<double>;

}  // namespace kf
