// sc_solve_common.h -- pieces shared by the Green-function build and the
// field transforms.
#pragma once

#include <hip/hip_runtime.h>

#include "sc_fft_dev.h"
#include "sc_fft_mix.h"
#include "sc_internal.h"

namespace sc {

constexpr double kFPEI = 299792458.0 * 299792458.0 * 1.0e-7;  // src/utils.jl:7-8

// true when L has no prime factor above 7 (the radices of the transforms)
inline bool smooth7(int L)
{
    if (L < 1) return false;
    for (int f : {2, 3, 5, 7})
        while (L % f == 0) L /= f;
    return L == 1;
}

// true when the register engines transform length L
inline bool reg_length(int L)
{
    switch (L) {
#define X(LL) case LL:
        SC_MIX_LENGTHS(X)
#undef X
        return true;
    default: return false;
    }
}

// Transform half-length of an axis of n nodes: the smallest t >= n whose 2t
// the register engines transform (sc_fft_mix.h), on axes beyond those lengths
// (n > 256) the smallest whose 2t has no prime factor above 7.  The reference
// zero-pads each axis to exactly 2n (src/mesh.jl:51-61) and FFTW transforms
// any length.  The convolution it computes is linear: output node m < n sums
// rho[j] G(m - j) over j < n, lags |m - j| <= n - 1, so any cyclic length of
// at least 2n - 1 gives the same outputs.  Other axes are therefore padded
// further, to 2t: rho stays zero beyond its n nodes, the Green function is
// built on t lags (its first n are the reference's cell integrals; it depends
// on the spacing, gamma and the image offset only, not on n), and only the n
// physical outputs are written.  Padding to the next register length beats
// transforming 2n itself on the generic engine also where the padding is
// widest (one solve, generic at 2n's own length -> register: 201^3, 402 -> 512
// points, 2994 -> 1531 us in Float32 and 4748 -> 2584 us in Float64; 101^3,
// 210 -> 256, 386 -> 162 and 549 -> 269 us; 161^3 Float64 with the cathode,
// 324 -> 384, 3377 -> 2861 us); the spectra and the Green scratch grow with the
// padding, at the worst (201^3 at 256 for 210) to 1.8 times the bytes.  Not on every
// mesh of a longer axis (padding_pays).
inline int transform_half(int n, bool smooth)
{
    int t = n;
    if (!smooth && 2 * n <= kMixMaxLength) {
        while (!reg_length(2 * t)) ++t;
        return t;
    }
    while (!smooth7(2 * t)) ++t;
    return t;
}

// Whether a mesh of an axis beyond the register lengths along z pads x and y to
// them.  The z convolution and the z pass of the Green build stay on the generic
// engine there, over more pencils, r times as many; the x and y passes gain
// less than that costs where r is large, the more so the longer z is and the more
// passes are generic anyway.  One solve, free / cathode (us), 7-smooth -> register
// lengths: Float64 131x131x300 (r = 1.14) 3158 / 6272 -> 2379 / 5142, 101x129x300
// (1.30) 2450 / 4821 -> 2112 / 4558, but 81x81x300 (1.40) 1059 / 2129 -> 1110 / 2275,
// 101x101x1024 (1.49) 8344 / 13959 -> 9976 / 16913, 64x101x600 (1.22) 2517 / 4135 ->
// 2581 / 4293, 201x300x300 (1.22, two generic axes) 12899 / 23771 -> 13378 / 25012;
// Float32 81x81x300 688 / 1248 -> 579 / 1090, 101x101x400 (1.49) 1618 / 2889 -> 1547 /
// 2700, but 51x51x600 (1.40) 717 / 1450 -> 726 / 1545, 101x101x1024 4673 / 9451 -> 4844 /
// 10125.  With z on a register engine padding always gained (300x201x201 Float64
// 7103 / 12303 -> 4674 / 10224).
inline bool padding_pays(const Mesh *m)
{
    const int nx = (int)m->n[0], ny = (int)m->n[1], nz = (int)m->n[2];
    if (2 * nz <= kMixMaxLength) return true;
    const double r = (double)transform_half(nx, false) * transform_half(ny, false) /
                     ((double)transform_half(nx, true) * transform_half(ny, true));
    const bool far = 2 * nz >= 2 * kMixMaxLength;  // a z axis of 512 nodes and more
    if (m->dtype == SC_F32) return !far || r <= 4.0 / 3.0;
    if (2 * nx > kMixMaxLength || 2 * ny > kMixMaxLength) return r <= 1.1;
    return r <= (far ? 1.2 : 4.0 / 3.0);
}

// Solves of a Float32 mesh whose rho was deposited from Float64 particles (adjoint
// solves: whose cotangents were, if any were since) keep the plain 7-smooth lengths, and with them the
// generic engine, except for unpadded powers of two.  Their caller gets the
// interpolated fields in Float64 and so sees the transforms' Float32 rounding
// itself, which any other length or radix moves by 1e-7 of the field: such fields
// are the same bits whatever ran on the mesh before.  The choice is that of the
// solve alone (choose_lengths); the workspace holds both sets of lengths.
inline bool smooth_lengths(const Mesh *m) { return m->smooth; }

// Shape of a solve.  nx, ny, nz are the transform half-lengths (the Green
// function's lags and spectral octant); mx, my, mz the mesh's nodes (the
// extent of rho, efield and the real rows the passes read and write).  They
// differ only on axes padded beyond 2n (transform_half).
struct Dims {
    int nx, ny, nz;  // transform half-lengths: L = 2n, spectral octant n + 1
    int mx, my, mz;  // mesh nodes (data extent)
    int Kx;          // nx + 1 kept x frequencies
    int Kp;          // row stride of kx-indexed arrays: Kx rounded up to 32, so that the
                     // 16-lane row segments of every transform start on a 128-byte line
    int Lx, Ly, Lz;  // padded lengths
};

inline Dims make_dims(const Mesh *m)
{
    Dims d;
    d.mx = (int)m->n[0];
    d.my = (int)m->n[1];
    d.mz = (int)m->n[2];
    const bool smooth = smooth_lengths(m) || !padding_pays(m);
    d.nx = transform_half(d.mx, smooth);
    d.ny = transform_half(d.my, smooth);
    d.nz = transform_half(d.mz, smooth);
    d.Kx = d.nx + 1;
    d.Kp = (d.Kx + 31) / 32 * 32;
    d.Lx = 2 * d.nx;
    d.Ly = 2 * d.ny;
    d.Lz = 2 * d.nz;
    return d;
}

// Engine of a transform of length L: the power-of-two register engine where no
// axis is padded (the Green passes work on the padded extents throughout and
// pass padded = false), else the mixed-radix one, else (longer axes, meshes
// with smooth_lengths, force_generic_transforms) the generic LDS engine.
enum Engine { kGeneric, kPow2, kMix };
inline Engine engine_of(const Mesh *m, int L, bool padded)
{
    if (m->generic_transforms || !reg_length(L)) return kGeneric;
    if (!padded && L >= 32 && (L & (L - 1)) == 0) return kPow2;
    return smooth_lengths(m) ? kGeneric : kMix;
}
// Whether the x and y passes run as one kernel per direction (sc_solve_plane.hip):
// two short axes of any lengths up to 64, or two equal longer ones as far as the
// plane's pencils fit a workgroup (1024 lanes, and 160 KB of LDS in Float64).  One
// solve with its Green build, separate passes / this (us): Float32 16^3 34.6 / 26.8,
// 32^3 36.7 / 31.1, 32x32x512 164 / 155, 50^3 47.6 / 41.9, 64^3 60.9 / 56.0, 64x64x256
// 129 / 121, 65x65x129 90.4 / 90.0; Float64 16^3 30.6 / 26.4, 32^3 36.1 / 32.2,
// 32x32x512 234 / 220, 50^3 56.1 / 52.8, 48x48x96 73.2 / 73.1, 48x48x256 122 / 116; and
// two launches fewer for the host.  Solves with smooth_lengths keep their bits, and
// force_generic_transforms its engine.
inline bool plane_lengths(const Mesh *m, const Dims &d)
{
    if (m->generic_transforms || smooth_lengths(m)) return false;
    auto is_short = [](int L) { return L == 16 || L == 24 || L == 32 || L == 48 || L == 64; };
    if (is_short(d.Lx) && is_short(d.Ly)) return true;
    if (d.Lx != d.Ly) return false;
    if (d.Lx == 128 || d.Lx == 144 || d.Lx == 160) return m->dtype == SC_F32;
    return d.Lx == 72 || d.Lx == 80 || d.Lx == 96 || d.Lx == 100;
}
// true when some axis is padded beyond twice its nodes
inline bool dims_padded(const Dims &d) { return d.nx != d.mx || d.ny != d.my || d.nz != d.mz; }

inline int div_up(int a, int b) { return (a + b - 1) / b; }

// Largest batch with nb*n <= cap elements, at most nbmax pencils.
inline int pick_nb(int n, int cap, int nbmax)
{
    int nb = cap / n;
    if (nb > nbmax) nb = nbmax;
    if (nb < 1) nb = 1;
    return nb;
}

// What one solve computes: the three field components in free space or with
// the cathode image charge, the scalar potential in free space, or the
// transpose of the field solve (free space or cathode): g_rho = S^T g_E.
enum SolveMode {
    kFieldFree = 0,
    kFieldCathode = 1,
    kPotential = 2,
    kAdjointFree = 3,
    kAdjointCathode = 4
};

inline bool mode_cathode(int mode) { return mode == kFieldCathode || mode == kAdjointCathode; }
inline bool mode_adjoint(int mode) { return mode == kAdjointFree || mode == kAdjointCathode; }
// The Green spectra a mode needs (the transpose uses the field's).
inline int green_mode(int mode)
{
    return mode == kPotential ? kPotential : (mode_cathode(mode) ? kFieldCathode : kFieldFree);
}

// Buffers of one solve: the real input `in` (nin components of the mesh's
// mx*my*mz nodes) is transformed along x and y into the spectra `fwd` (nin of
// them), the z convolution writes nout spectra to `inv`, and the inverse y
// and x passes write the real output `out` (nout components).  Spectra are
// [mz][Ly][Kp] complex each, consecutive.
struct SolveIO {
    int mode;
    int nin, nout;
    const void *in;
    void *out;
    void *fwd;
    void *inv;
};

// ---- grouped solves: bunches of one mesh shape, one launch per kernel ----
// Per-bunch buffers and Green geometry of a grouped solve (a table in device
// memory).  A grouped launch stacks the bunches along x: workgroup x belongs
// to bunch x / per and acts as workgroup x % per of that bunch's own launch.
// Kernels given no table (the single-bunch launch) use their arguments.
struct SBunch {
    const void *in;
    void *out, *fwd, *inv, *Gf, *Gi, *R;
    double *F;
    double dx, dy, dz, offzg;  // Green spacings (dz times gamma) and image offset times gamma
    double scale[4];
};

__device__ __forceinline__ int group_block(const SBunch *tab, int per, const SBunch *&sb)
{
    if (!tab) {
        sb = nullptr;
        return (int)blockIdx.x;
    }
    const int k = (int)blockIdx.x / per;
    sb = tab + k;
    return (int)blockIdx.x - k * per;
}

// Pencil (x block, ky) of z-convolution task `task`, with nbx x blocks per ky
// row.  The rows go in the order 0, 1, Ly-1, 2, Ly-2, ..., ny, because rows
// ky and Ly - ky read the same Green row (the spectrum is even in ky), and
// neighbouring x blocks share the 128-byte lines of that row.
__device__ __forceinline__ void zconv_pencils(int task, int nbx, int Ly, int &bx, int &ky)
{
    bx = task % nbx;
    const int u = task / nbx;
    const int kyp = (u + 1) >> 1;
    ky = u == 0 ? 0 : ((u & 1) ? kyp : Ly - kyp);
}

// Small Green builds run on the caller's stream, the others overlap the deposit
// on the side stream.  The events that fork and join the stream cost the host
// 24 us a solve, more than a small build takes on the GPU.  Measured, step of
// 10k particles on 16^3 on the side stream / inline 100 / 60 us, 100k on 32^3
// 98 / 76, 200k on 48^3 Float32 115 / 104 but Float64 116 / 124, 1M on 64^3
// 124 / 136; with the cathode 50k on 32^3 101 / 75, on 48^3 Float64 109 / 113.
// Float64 particles on a Float32 mesh have generic passes on axes that are no powers
// of two, and no fused kernel, and their builds take longer.  Two or three generic
// passes: step of 2k such particles on 20^3 95 / 90, with the cathode 96 / 94, on 24^3
// 96 / 97 and 97 / 102, 43x62x13 106 / 125, 33^3 107 / 122 (one solve 80 / 93), 21x244x23
// 134 / 155 (96 / 125).  One: 32x32x20 and 64x64x20 level, of 60k on 32x32x50 104 / 112,
// but one solve 70 / 60; on 50x64x32 99 / 116, one solve 68 / 70.
constexpr int64_t kSmallGreenBytes = 640 << 10, kSmallWideBytes = 384 << 10, kSmallGenericBytes = 80 << 10;
inline bool green_small(const Mesh *m, const Dims &d, size_t size, int cath)
{
    const int64_t nodes = (int64_t)(d.nx + 1) * (d.ny + 1) * (d.nz + 1);
    int generic = 0;
    for (const int L : {d.Lx, d.Ly, d.Lz}) generic += engine_of(m, L, false) == kGeneric;
    const int64_t most = generic > 1                            ? kSmallGenericBytes
                         : generic > 0 && smooth_lengths(m) ? kSmallWideBytes
                                                                : kSmallGreenBytes;
    return nodes * (int64_t)size * (cath ? 2 : 1) <= most;
}

// Builds the transformed Green functions for green_mode `mode` into ws.Gf
// (and ws.Gi for kFieldCathode): three field components, or the
// potential's one (stored in the first component's slot).
template <typename T>
int build_green(Mesh *m, const double dl[3], double gamma, double offz, int mode);

// Solve kernel `which` (0 forward x, 1 forward y, 2 z convolution, 3 inverse
// y, 4 inverse x) of `io` on the power-of-two (launch_fast) or mixed-radix
// (launch_mix) register engine; false when the engine does not take it
// (nothing is launched then).
template <typename T>
bool launch_fast(Mesh *m, int which, const SolveIO &io);
template <typename T>
bool launch_mix(Mesh *m, int which, const SolveIO &io);
// The x and y passes of one mesh, or (tab) of nb same-shape bunches: forward from
// `in` to `spec`, or inverse from `spec` to `out`, ncomp components.
template <typename T>
void launch_plane(const Mesh *m, const T *in, cpx<T> *spec, T *out, const SBunch *tab, int nb, int ncomp,
                  bool inverse, hipStream_t st);

// Grouped forms, on `st`, for nb bunches of the mesh shape of m0 whose
// transforms run on the register engines: the Green build (field modes) of
// every bunch, from m0's twiddles and the table's spacings, and solve
// kernel `which` of every bunch with the table's buffers.
template <typename T>
void build_green_grouped(const Mesh *m0, int nb, const SBunch *tab, double gamma, int mode,
                         hipStream_t st);
template <typename T>
void launch_fast_grouped(const Mesh *m0, int nb, const SBunch *tab, int which, int mode, int nin,
                         int nout, hipStream_t st);
template <typename T>
void launch_mix_grouped(const Mesh *m0, int nb, const SBunch *tab, int which, int mode, int nin,
                        int nout, hipStream_t st);

}  // namespace sc
