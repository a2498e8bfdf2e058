// kf_plane.h -- the y and z passes of a 3D transform on one x plane held in
// LDS.
//
// A plane of Ny x (Nz/2+1) spectral values that fits the 160 KB of LDS takes
// both its y and its z transforms, and the real-space work between them, in
// one workgroup: one read of the x-transformed field and one write, in place
// of a pass over memory and a launch for each transform.  The butterflies,
// radices, twiddles and functors are those of the separate passes, so the
// numbers are the same bit for bit.
//
// Where a plane does not fit, or the lengths are not in the sets below, the
// separate passes run; one field's transforms take planes by plane_one.  Small grids are bound by the launches, of which an
// equidistant evaluation has 7 here in place of 35 and a stretched one 12 in
// place of 95; at 128^3 FP64 (a plane is 137 KB, one workgroup per CU) the
// passes over memory still outweigh the idle CUs.  RK4 step, separate passes
// against planes, us: equidistant FP64 1001 -> 477 (32^3), 1211 -> 642 (64^3),
// 1946 -> 1446 (96^3), 2812 -> 2788 (128^3); mixed 1200 -> 615 (64^3), 2110 ->
// 1894 (128^3); sine-stretched FP64 3449 -> 953 (64^3), 7049 -> 4730 (128^3).
//
//   k_plane_c2r   y inverse, z C2R, a ZStore
//   k_plane_prof  y inverse, z C2R, times 1/S', z R2C, y forward
//   k_plane_r2c   real rows, z R2C, y forward
//   k_plane_pen   the three products, the linear terms' blend, z R2C, y forward
#pragma once

#include "kf_fft.h"

namespace kf {
namespace fft {

template <typename T>
struct Four {
    T a, b, c, d;
    // by comparison: a run-time index into a kernel argument would copy it to scratch memory
    __device__ __forceinline__ T pick(unsigned f) const { return f == 0 ? a : (f == 1 ? b : (f == 2 ? c : d)); }
};
template <typename T>
inline Four<T> four(T a, T b = T(), T c = T(), T d = T())
{
    return Four<T>{a, b, c, d};
}

// ------------------------------------------------------------------ sizes
__host__ __device__ constexpr bool plane_len_y(int n)
{
    return n == 16 || n == 24 || n == 32 || n == 48 || n == 64 || n == 96 || n == 128;
}
__host__ __device__ constexpr bool plane_len_m(int m)
{
    return m == 8 || m == 12 || m == 16 || m == 24 || m == 32 || m == 48 || m == 64 || m == 96;
}
// the plane, its tables in 156 KB of LDS, and a row's TPT threads for every
// row within one workgroup
__host__ __device__ constexpr bool plane_fits(int ny, int m, int csize)
{
    return plane_len_y(ny) && plane_len_m(m) && ny * tpt_for(m) <= 1024 &&
           (ny * (m + 1) + ny + 2 * m + 1) * csize <= 156 * 1024;
}
// One field's launch has Nx workgroups, each a whole plane's chain of passes,
// against launches of its rows and columns: planes of up to `small` bytes are
// faster whatever Nx is, larger ones from an Nx on.  Separate / plane, us,
// FP64: forward 128x128 14.5 / 19.6 (Nx = 16), 28.0 / 27.9 (96), 34.1 / 31.5
// (128), 96x96 17.2 / 18.2 (48), 64x128 16.4 / 14.6 (48); inverse 128x128
// 13.1 / 19.8 (16), 26.8 / 29.9 (128), 34.6 / 35.2 (256), 96x96 19.1 / 20.5
// (96), 23.2 / 22.6 (128), 64x128 14.8 / 14.1 (48); a stretched derivative,
// with its x passes, 128x128 27.4 / 36.9 (16), 49.4 / 51.1 (128), 57.5 / 55.2
// (192), 96x96 35.4 / 35.3 (48).  FP32: forward 128x128 16.5 / 16.9 (48), 20.1
// / 19.4 (96), 96x128 14.0 / 12.5 (16); inverse 128x128 25.9 / 27.6 (192), 28.6
// / 27.8 (256), 96x96 15.6 / 16.3 (96), 17.8 / 17.4 (128), 128x64 12.2 / 14.0
// (48), 96x64 12.1 / 11.9 (16).
struct OnePlane {
    bool fwd, inv, mid;
};
inline OnePlane plane_one(int nx, int ny, int m, int csize)
{
    const bool dp = csize == 16;
    const int bytes = ny * (m + 1) * csize;
    OnePlane o;
    o.fwd = bytes <= (dp ? 70000 : 60000) || nx >= (dp ? 96 : 64);
    o.inv = bytes <= (dp ? 70000 : 30000) || (nx >= 128 && bytes <= (dp ? 110000 : 60000)) || nx >= 256;
    o.mid = bytes <= (dp ? 78000 : 30000) || (nx >= 96 && bytes <= (dp ? 110000 : 60000)) || nx >= 192;
    return o;
}
// threads of a plane's workgroup: its rows' or its columns', whichever are more
__host__ __device__ constexpr int plane_threads(int ny, int m)
{
    const int rows = ny * tpt_for(m), cols = (m + 1) * tpt_for(ny);
    const int t = rows > cols ? rows : (cols > 1024 ? 1024 : cols);
    return (t + 63) / 64 * 64 > 1024 ? 1024 : (t + 63) / 64 * 64;
}

// ------------------------------------------------------------------ arguments
template <typename R>
struct PlaneTabs {
    const C2<R> *twy, *twm, *twn;
    int nx, ny, nz, nzs;  // nzs: row length of the spectral planes
};
template <typename R>
inline PlaneTabs<R> plane_tabs(const Plan<R> &p, int nzs = 0)
{
    return PlaneTabs<R>{p.tw_y, p.tw_m, p.tw_n, p.nx, p.ny, p.nz, nzs ? nzs : p.nzs};
}

// k_plane_c2r: real rows of up to 4 fields (blockIdx.y) into o, by kind
//   0 scaled, 1 ln n and rho = exp(ln n) + nd, 2 the same with rho and nd in
//   FP64, 3 as 2 from an FP64 transform, ln n rounded to FP32, 4 o (+)= u v
// (the kinds of ZStore, in its arithmetic)
template <typename R>
struct PlaneOut {
    int kind;
    R scale;
    Four<R *> o;
    R *rho;
    const R *nd, *u;
    int acc;
    double *rho64;
    const double *nd64;
    float *lnf;
};
// k_plane_r2c: rows of field blockIdx.y from real values in R (a0), or from
// FP64 values rounded to R (d); with `products` of the 12 products of a
// blockIdx.y / 3 of a0 and a blockIdx.y % 3 of a1
template <typename R>
struct PlaneIn {
    Four<const R *> a0, a1;
    const double *d;
    int products;
    long dstride;  // elements between the fields' planes in dst
};
// k_plane_prof: derivative b = blockIdx.y % 3 of field blockIdx.y / 3, with
// `one` >= 0 the single axis `one` of dst in place, or with `one` = -2 plane
// set y along the axis of the y-th two bits of axes, from the field of the
// y-th four bits of srcs (h0 null: in place)
template <typename R>
struct PlaneProf {
    const C2<R> *h0;  // x-inverse of D23 F, one per field
    C2<R> *dst;       // three per field; slot 0 holds the x-inverse of i k_x D23 F
    long stride;      // elements between fields' planes
    Four<const R *> prof;
    const R *ky, *kz;
    R scale;
    int one;
    unsigned axes;
    unsigned long srcs;
};
// k_plane_pen: per field f = blockIdx.y the sources s0, s1, s2 (x-inverse
// spectra; ky and kz set: s1 times i k_y, s2 times i k_z), lin in place
template <typename R>
struct PlanePen {
    Four<const C2<R> *> s0, s1, s2;
    Four<C2<R> *> lin;
    const R *ky, *kz;
    const R *U0, *U1, *U2;
    Four<const R *> f;
    const R *mask, *bar;
    Four<R> c1;
    R c0, scale;
    Four<R *> g0, g1, g2;  // where set: the three real-space derivatives (the adjoint's capture)
};

template <typename R>
void plane_c2r(const PlaneTabs<R> &t, Four<const C2<R> *> src, const R *ky, const R *kz, const PlaneOut<R> &z,
               int fields, hipStream_t s, const int *ctl = nullptr);
template <typename R>
void plane_prof(const PlaneTabs<R> &t, const PlaneProf<R> &a, int planes, hipStream_t s);
template <typename R>
void plane_r2c(const PlaneTabs<R> &t, const PlaneIn<R> &in, C2<R> *dst, hipStream_t s, const int *ctl = nullptr,
               int fields = 1);
template <typename R>
void plane_pen(const PlaneTabs<R> &t, const PlanePen<R> &a, int fields, hipStream_t s);

}  // namespace fft
}  // namespace kf
