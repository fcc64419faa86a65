// sc_solve_plane.hip -- the x and y passes of a solve in one kernel, on short
// x and y axes (plane_lengths).
//
// On small meshes a pass takes 3-4 us however little it moves: the launch, one
// round trip to memory, a few barriers.  Here a workgroup takes one (x, y) plane
// through both passes; the half-transformed plane stays in LDS.  The transforms
// are those of sc_fft_mix.h, every pencil of the plane at once.  Bound by its
// dependent phases (load, two transforms, store): 6.2-7 us timed alone on 32^3 where
// two passes took 12.4-14, the inverse on 64x64x256 Float32 24 against 20.4 + 11.6.
// plane_lengths has the solves' times.
#include <hip/hip_runtime.h>

#include "sc_solve_common.h"

namespace sc {

namespace {

using mix::Shape;

// X(LX, LY) for the pairs of plane_lengths.
#define SC_PLANE_Y(X, LX) X(LX, 16) X(LX, 24) X(LX, 32) X(LX, 48) X(LX, 64)
#define SC_PLANE_PAIRS(X) \
    SC_PLANE_Y(X, 16) SC_PLANE_Y(X, 24) SC_PLANE_Y(X, 32) SC_PLANE_Y(X, 48) SC_PLANE_Y(X, 64) \
    X(72, 72) X(80, 80) X(96, 96) X(100, 100) X(128, 128) X(144, 144) \
    X(160, 160)

// Shape of a workgroup: lanes for the LY / 2 rows of the x pass and for the
// LX / 2 + 1 columns of the y pass, in whole waves.  Lanes without a pencil
// transform one of their own (zeros), so every LDS slice is theirs.
template <typename T, int LX, int LY>
struct PlaneShape {
    static constexpr int EX = Shape<T, LX>::E, TX = LX / EX;
    static constexpr int EY = Shape<T, LY>::E, TY = LY / EY;
    static constexpr int KX = LX / 2 + 1;
    static constexpr int LANES = LY / 2 * TX > KX * TY ? LY / 2 * TX : KX * TY;
    static constexpr int THREADS = (LANES + 63) / 64 * 64;
    static constexpr int NX = (THREADS + TX - 1) / TX;  // x pencils, contiguous slices
    static constexpr int NY = THREADS / TY;             // y pencils, side by side,
    static constexpr int SY = NY + 1;                   // and one for the lanes left over
    static constexpr int XS = NX * reg::padded<LX, EX>(), YS = SY * LY, PS = KX * (LY / 2);
    static constexpr int LDS = XS > YS ? (XS > PS ? XS : PS) : (YS > PS ? YS : PS);
};

// Forward: plane z of component blockIdx.y of the real input to its (kx, ky)
// spectrum, zero-padded to 2nx and 2ny.
template <typename T, int LX, int LY>
__global__ void __launch_bounds__((PlaneShape<T, LX, LY>::THREADS))
k_fwd_xy(const T *__restrict__ in, cpx<T> *__restrict__ spec, const cpx<T> *__restrict__ twxg,
         const cpx<T> *__restrict__ twyg, Dims d, const SBunch *__restrict__ tab)
{
    using S = PlaneShape<T, LX, LY>;
    constexpr int EX = S::EX, TX = S::TX, EY = S::EY, TY = S::TY, KX = S::KX;
    __shared__ cpx<T> twx[LX], twy[LY];
    __shared__ cpx<T> lds[S::LDS];
    const SBunch *sb;
    const int z = group_block(tab, d.mz, sb);
    if (sb) {
        in = static_cast<const T *>(sb->in);
        spec = static_cast<cpx<T> *>(sb->fwd);
    }
    for (int i = threadIdx.x; i < LX; i += S::THREADS) twx[i] = gld(twxg + i);
    for (int i = threadIdx.x; i < LY; i += S::THREADS) twy[i] = gld(twyg + i);
    const int mx = d.mx, my = d.my;
    const size_t plane = (size_t)blockIdx.y * d.mz + z;
    {
        const int y = threadIdx.x / TX, j = threadIdx.x % TX;
        const bool live = y < my;
        const T *row = in + (plane * my + (live ? y : 0)) * mx;
        cpx<T> v[EX];
#pragma unroll
        for (int q = 0; q < EX; ++q) {
            v[q] = cpx<T>{(T)0, (T)0};
            if (q < EX / 2) {
                const int e = j + q * TX;
                const bool on = live && e < mx;
                const T t = gld(row + (on ? e : 0));
                v[q].x = on ? t : (T)0;
            }
        }
        mix::fft<T, LX, EX, -1>(v, j, lds + y * reg::padded<LX, EX>(), 1, twx);
        __syncthreads();  // every lane past the last exchange
        if (live) {
#pragma unroll
            for (int q = 0; q <= EX / 2; ++q) {
                const int k = j + q * TX;
                if (k < KX) lds[y * KX + k] = v[q];
            }
        }
        __syncthreads();
    }
    const bool in_y = (int)threadIdx.x < S::NY * TY;
    const int kx = in_y ? threadIdx.x % S::NY : S::NY,
              j = in_y ? threadIdx.x / S::NY : threadIdx.x - S::NY * TY;
    const bool live = kx < KX;
    cpx<T> v[EY];
#pragma unroll
    for (int q = 0; q < EY; ++q) {
        v[q] = cpx<T>{(T)0, (T)0};
        if (q < EY / 2) {
            const int e = j + q * TY;
            const bool on = live && e < my;
            const cpx<T> t = lds[on ? e * KX + kx : 0];
            v[q] = on ? t : cpx<T>{(T)0, (T)0};
        }
    }
    mix::fft<T, LY, EY, -1>(v, j, lds + kx, S::SY, twy);
    if (live) {
        cpx<T> *out = spec + plane * LY * d.Kp + kx;
#pragma unroll
        for (int q = 0; q < EY; ++q) gst(out + (size_t)(j + q * TY) * d.Kp, v[q]);
    }
}

// Backward: the (kx, ky) spectrum of plane z of component blockIdx.y to the real
// output (complex to real along x, with Hermitian completion).
template <typename T, int LX, int LY>
__global__ void __launch_bounds__((PlaneShape<T, LX, LY>::THREADS))
k_inv_yx(const cpx<T> *__restrict__ spec, T *__restrict__ out, const cpx<T> *__restrict__ twxg,
         const cpx<T> *__restrict__ twyg, Dims d, const SBunch *__restrict__ tab)
{
    using S = PlaneShape<T, LX, LY>;
    constexpr int EX = S::EX, TX = S::TX, EY = S::EY, TY = S::TY, KX = S::KX;
    __shared__ cpx<T> twx[LX], twy[LY];
    __shared__ cpx<T> lds[S::LDS];
    const SBunch *sb;
    const int z = group_block(tab, d.mz, sb);
    if (sb) {
        spec = static_cast<const cpx<T> *>(sb->inv);
        out = static_cast<T *>(sb->out);
    }
    for (int i = threadIdx.x; i < LX; i += S::THREADS) twx[i] = gld(twxg + i);
    for (int i = threadIdx.x; i < LY; i += S::THREADS) twy[i] = gld(twyg + i);
    const int mx = d.mx, my = d.my;
    const size_t plane = (size_t)blockIdx.y * d.mz + z;
    {
        const bool in_y = (int)threadIdx.x < S::NY * TY;
        const int kx = in_y ? threadIdx.x % S::NY : S::NY,
                  j = in_y ? threadIdx.x / S::NY : threadIdx.x - S::NY * TY;
        const bool live = kx < KX;
        const cpx<T> *col = spec + plane * LY * d.Kp + (live ? kx : 0);
        cpx<T> v[EY];
#pragma unroll
        for (int q = 0; q < EY; ++q) v[q] = gld(col + (size_t)(j + q * TY) * d.Kp);
        mix::fft<T, LY, EY, +1>(v, j, lds + kx, S::SY, twy);
        __syncthreads();  // every lane past the last exchange
        if (live) {
#pragma unroll
            for (int q = 0; q < EY / 2; ++q) {
                const int e = j + q * TY;
                if (e < my) lds[e * KX + kx] = v[q];
            }
        }
        __syncthreads();
    }
    const int y = threadIdx.x / TX, j = threadIdx.x % TX;
    const bool live = y < my;
    const cpx<T> *row = lds + (live ? y : 0) * KX;
    cpx<T> v[EX];
#pragma unroll
    for (int q = 0; q < EX; ++q) {
        const int k = j + q * TX;
        const bool direct = k < KX;
        v[q] = row[direct ? k : LX - k];
        if (!direct) v[q].y = -v[q].y;
    }
    mix::fft<T, LX, EX, +1>(v, j, lds + y * reg::padded<LX, EX>(), 1, twx);
    if (live) {
        T *o = out + (plane * my + y) * mx;
#pragma unroll
        for (int q = 0; q < EX / 2; ++q)
            if (j + q * TX < mx) gst(o + j + q * TX, v[q].x);
    }
}

template <typename T, int LX, int LY>
void launch_pair(const Dims &d, const T *in, cpx<T> *spec, T *out, const cpx<T> *twx, const cpx<T> *twy,
                 const SBunch *tab, int nb, int ncomp, bool inverse, hipStream_t st)
{
    if constexpr (sizeof(T) == 4 || LX <= 100) {
        const dim3 grid(d.mz * nb, ncomp), block(PlaneShape<T, LX, LY>::THREADS);
        if (inverse)
            hipLaunchKernelGGL((k_inv_yx<T, LX, LY>), grid, block, 0, st, (const cpx<T> *)spec, out, twx,
                               twy, d, tab);
        else
            hipLaunchKernelGGL((k_fwd_xy<T, LX, LY>), grid, block, 0, st, in, spec, twx, twy, d, tab);
    }
}

}  // namespace

template <typename T>
void launch_plane(const Mesh *m, const T *in, cpx<T> *spec, T *out, const SBunch *tab, int nb, int ncomp,
                  bool inverse, hipStream_t st)
{
    const Dims d = make_dims(m);
    const cpx<T> *twx = static_cast<const cpx<T> *>(m->ws.twT[0]);
    const cpx<T> *twy = static_cast<const cpx<T> *>(m->ws.twT[1]);
    switch (d.Lx * 1024 + d.Ly) {
#define X(LX, LY)                                                                            \
    case LX * 1024 + LY:                                                                     \
        launch_pair<T, LX, LY>(d, in, spec, out, twx, twy, tab, nb, ncomp, inverse, st);     \
        break;
        SC_PLANE_PAIRS(X)
#undef X
    default: break;  // the caller checks plane_lengths
    }
}

#if SC_PLANE_PART == 0
template void launch_plane<float>(const Mesh *, const float *, cpx<float> *, float *, const SBunch *, int,
                                  int, bool, hipStream_t);
#else
template void launch_plane<double>(const Mesh *, const double *, cpx<double> *, double *, const SBunch *,
                                   int, int, bool, hipStream_t);
#endif

}  // namespace sc
