// sc_solve_mix.hip -- register-resident transform kernels of the field solve
// for the mixed-radix lengths of sc_fft_mix.h (axes of up to 256 nodes that are
// no unpadded powers of two, see sc_solve_fast.hip).
//
// Same data flow and layouts as the generic kernels in sc_solve.hip (which
// remain the path for longer axes), with every pencil held in registers:
// a lane loads its E elements straight from HBM, the pencil is transformed
// with one LDS exchange per pass boundary, and the lane stores straight to
// HBM.  Which inputs are zero (the padded half) and which outputs are kept
// (the physical octant, the Hermitian half) depends only on the register
// index, so the pruning is resolved at compile time; on axes padded beyond
// twice their nodes (Dims) a compare drops what lies past the mesh.
//
// Measured against the generic engine on the lengths that are no power of two:
// the eight transform and Green-transform kernels took 368 -> 120 us on 100^3 in
// Float32 (the whole step of 1M particles 387 -> 208 us) and 410 -> 131 us on
// 65x65x129 in Float64, padded to 72x72x144 (500k particles: 411 -> 214 us).
//
// The file is compiled once per part of the lengths and mesh type
// (SC_MIX_PART 0..3, see build.py), so that the parts build in parallel;
// part 0 also holds the dispatch.
#include <hip/hip_runtime.h>

#include "sc_fft_mix.h"
#include "sc_solve_common.h"

namespace sc {

namespace {

using mix::Shape;

// (Workgroups of 512 threads for the z convolution, which make each
// workgroup's Green row segment a whole 128-byte line, cut its fetched bytes
// by a quarter on MI355X but ran slower: the kernel is bound by its
// transform arithmetic, not by memory.)

// Waves per SIMD of the z convolution.  The forward pencil stays in registers
// across the three inverse transforms: 2 E complex values and the
// butterfly's temporaries.  Up to 16 Float32 or 8 Float64 values per lane
// three waves (168 VGPRs) hold them (unconstrained, the 256-point Float32
// kernel takes 169 VGPRs, two waves); with more values, or with the cathode
// image, whose spectrum is held as well, 168 VGPRs would spill to scratch.
template <typename T, int L, bool CATH>
constexpr int zconv_waves()
{
    constexpr int words = Shape<T, L>::E * (int)sizeof(T) / 4;
    return words > 32 || (CATH && (words > 20 || Shape<T, L>::E == 20)) ? 1 : CATH || words > 16 ? 2 : 3;
}

// Whether the z convolution runs here: with the cathode image a lane holds the
// image's spectrum (field) or sum (transposed) as well, three arrays of E values
// beside the butterfly's temporaries, and at many values per lane the kernel drops to
// one wave per SIMD and moves them through AGPRs; the generic kernel, which
// splits a pencil over more lanes, is faster then and takes those lengths.
// Measured (us, generic / this, 128x128 nodes across), field, Float64: 80 points
// 96 / 135, 160 230 / 319, but 96 128 / 74, 200 309 / 161, 320 564 / 580 and even on
// 90x90; in Float32 80 84 / 43, 160 143 / 155 and even on 90x90.  Transposed, Float64:
// 80 119 / 173, 96 149 / 198, 160 265 / 393, 192 323 / 456, 200 339 / 408, 288 585 / 838,
// 384 812 / 920 (320 spills two registers of 512), but 72 116 / 109, 144 247 / 249, 100
// 160 / 164, 400 926 / 851; Float32: 80 92 / 146, 160 155 / 289, 200 211 / 219, 320 352 /
// 623, 400 485 / 713, 256 (90x90) 141 / 155, but 96 101 / 39, 288 318 / 161.
template <typename T, int L>
constexpr bool zconv_here(int mode)
{
    constexpr bool f64 = sizeof(T) == 8;
    if (mode == kFieldCathode) return !(f64 && (L == 80 || L == 160));
    if (mode != kAdjointCathode) return true;
    switch (L) {
    case 80: case 160: case 200: case 320: return false;
    case 96: case 192: case 288: case 384: return !f64;
    case 256: case 400: return f64;
    default: return true;
    }
}

// x pass of the real input: rows (y, z) of component blockIdx.y, zero-padded
// to 2nx, kx in [0, nx] to that component's spectrum.
template <typename T, int L>
__global__ void __launch_bounds__((Shape<T, L>::THREADS))
k_rho_fwd_x_m(const T *__restrict__ in, cpx<T> *__restrict__ spec, const cpx<T> *__restrict__ twg,
              Dims d, const SBunch *__restrict__ tab, int per)
{
    using S = Shape<T, L>;
    constexpr int E = S::E, TPP = S::TPP, NB = S::NB;
    __shared__ cpx<T> tw[L];
    __shared__ cpx<T> lds[NB * reg::padded<L, E>()];
    const SBunch *sb;
    const int bx = group_block(tab, per, sb);
    if (sb) {
        in = static_cast<const T *>(sb->in);
        spec = static_cast<cpx<T> *>(sb->fwd);
    }
    for (int i = threadIdx.x; i < L; i += S::THREADS) tw[i] = gld(twg + i);
    const int b = threadIdx.x / TPP, j = threadIdx.x % TPP;
    const int r = bx * NB + b;
    const int nrows = d.my * d.mz, nx = d.nx, mx = d.mx;
    const bool live = r < nrows;
    const T *rho = in + ((size_t)blockIdx.y * nrows + (live ? r : 0)) * mx;
    cpx<T> *A = spec + (size_t)blockIdx.y * d.mz * d.Ly * d.Kp;
    cpx<T> v[E];
#pragma unroll
    for (int q = 0; q < E; ++q) {
        v[q] = cpx<T>{(T)0, (T)0};
        if (q < E / 2) {
            const int e = j + q * TPP;
            const bool on = live && e < mx;
            const T t = gld(rho + (on ? e : 0));
            v[q].x = on ? t : (T)0;
        }
    }
    mix::fft<T, L, E, -1>(v, j, lds + b * reg::padded<L, E>(), 1, tw);
    if (live) {
        const int y = r % d.my, z = r / d.my;
        cpx<T> *out = A + ((size_t)z * d.Ly + y) * d.Kp;
#pragma unroll
        for (int q = 0; q <= E / 2; ++q) {
            const int k = j + q * TPP;
            if (q < E / 2 || k == nx) gst(out + k, v[q]);
        }
    }
}

// y pass: pencils (kx, z < nz) of component blockIdx.z along y, ny inputs
// zero-padded to 2ny.
template <typename T, int L>
__global__ void __launch_bounds__((Shape<T, L>::THREADS))
k_rho_fwd_y_m(cpx<T> *__restrict__ A, const cpx<T> *__restrict__ twg, Dims d,
              const SBunch *__restrict__ tab, int per)
{
    using S = Shape<T, L>;
    constexpr int E = S::E, TPP = S::TPP, NB = S::NB;
    __shared__ cpx<T> tw[L];
    __shared__ cpx<T> lds[NB * L];
    const SBunch *sb;
    const int bx = group_block(tab, per, sb);
    if (sb) A = static_cast<cpx<T> *>(sb->fwd);
    for (int i = threadIdx.x; i < L; i += S::THREADS) tw[i] = gld(twg + i);
    const int b = threadIdx.x % NB, j = threadIdx.x / NB;
    const int kx = bx * NB + b, z = blockIdx.y;
    const int Kx = d.Kx, Kp = d.Kp;
    const bool live = kx < Kx;
    cpx<T> *Ap = A + ((size_t)blockIdx.z * d.mz + z) * d.Ly * Kp + (live ? kx : 0);
    cpx<T> v[E];
#pragma unroll
    for (int q = 0; q < E; ++q) {
        v[q] = cpx<T>{(T)0, (T)0};
        if (q < E / 2) {
            const int e = j + q * TPP;
            const bool on = live && e < d.my;
            const cpx<T> t = gld(Ap + (size_t)(on ? e : 0) * Kp);
            v[q] = on ? t : cpx<T>{(T)0, (T)0};
        }
    }
    mix::fft<T, L, E, -1>(v, j, lds + b, NB, tw);
    if (live) {
#pragma unroll
        for (int q = 0; q < E; ++q) gst(Ap + (size_t)(j + q * TPP) * Kp, v[q]);
    }
}

// Fused z convolution (see k_zconv in sc_solve.hip for the algebra), MODE
// a SolveMode.  With the cathode image the z-reversed pencil's spectrum is
// held as well (formed from the forward spectrum, not transformed).
template <typename T, int L, int MODE>
__global__ void __launch_bounds__((Shape<T, L>::THREADS))
__attribute__((amdgpu_waves_per_eu((zconv_waves<T, L, MODE == kFieldCathode>()))))
k_zconv_m(const cpx<T> *__restrict__ A, cpx<T> *__restrict__ B, const T *__restrict__ Gf,
          const cpx<T> *__restrict__ Gi, const cpx<T> *__restrict__ twg, Dims d,
          const SBunch *__restrict__ tab, int per)
{
    // grouped launches and the cathode mode: grid (x blocks [* bunches], Ly);
    // one bunch in free space or for the potential: a 1-D grid of per * Ly
    // workgroups in XCD order, per x blocks per row (the cathode mode, at two
    // waves per SIMD, measured 2 us slower in that order in Float64)
    const SBunch *sb = nullptr;
    int bx, ky;
    if (tab) {
        bx = group_block(tab, per, sb);
        ky = (int)blockIdx.y;
    } else if (MODE == kFieldCathode) {
        bx = (int)blockIdx.x;
        ky = (int)blockIdx.y;
    } else {
        zconv_pencils(xcd_task((int)blockIdx.x, (int)gridDim.x), per, d.Ly, bx, ky);
    }
    if (sb) {
        A = static_cast<const cpx<T> *>(sb->fwd);
        B = static_cast<cpx<T> *>(sb->inv);
        Gf = static_cast<const T *>(sb->Gf);
        Gi = static_cast<const cpx<T> *>(sb->Gi);
    }
    constexpr bool CATH = MODE == kFieldCathode, POT = MODE == kPotential;
    constexpr int NCOMP = POT ? 1 : 3;
    using S = Shape<T, L>;
    constexpr int E = S::E, TPP = S::TPP, NB = S::NB;
    __shared__ cpx<T> tw[L];
    __shared__ cpx<T> lds[NB * L];
    const int Kp = d.Kp, Ly = d.Ly, ny = d.ny, nz = d.nz, mz = d.mz, ny1 = ny + 1;
    for (int i = threadIdx.x; i < L; i += S::THREADS) tw[i] = gld(twg + i);
    const int b = threadIdx.x % NB, j = threadIdx.x / NB;
    const int kx = bx * NB + b;
    const bool live = kx < d.Kx;
    const size_t zs = (size_t)Ly * Kp;
    const cpx<T> *Ap = A + (size_t)ky * Kp + (live ? kx : 0);
    cpx<T> p[E], pi[E];
#pragma unroll
    for (int q = 0; q < E; ++q) {
        p[q] = cpx<T>{(T)0, (T)0};
        if (q < E / 2) {
            const int e = j + q * TPP;
            const bool on = live && e < mz;
            const cpx<T> t = gld(Ap + (size_t)(on ? e : 0) * zs);
            p[q] = on ? t : cpx<T>{(T)0, (T)0};
        }
    }
    mix::fft<T, L, E, -1>(p, j, lds + b, NB, tw);
    if constexpr (CATH) {
        // The image -rho(mz - 1 - z) (z < mz, zero-padded) has the spectrum
        // -w_L^((mz-1) k) P[-k]; P[-k] is held by another lane, so the
        // spectrum goes through LDS once instead of a second transform.
        __syncthreads();  // every lane past the transform's last exchange
#pragma unroll
        for (int q = 0; q < E; ++q) lds[b + (j + q * TPP) * NB] = p[q];
        __syncthreads();
#pragma unroll
        for (int q = 0; q < E; ++q) {
            const int k = j + q * TPP;
            const cpx<T> m = lds[b + (k == 0 ? 0 : L - k) * NB];
            const cpx<T> r = c_mul(tw[((mz - 1) * k) % L], m);
            pi[q] = cpx<T>{-r.x, -r.y};
        }
    }
    const bool kyneg = ky > ny;
    const int kyp = kyneg ? Ly - ky : ky;
    const size_t M1 = (size_t)(nz + 1) * ny1 * Kp;
    const size_t MI = (size_t)L * ny1 * Kp;
    const int kxc = live ? kx : 0;  // keep dead lanes' loads in bounds
#pragma unroll
    for (int c = 0; c < NCOMP; ++c) {
        const T sy = (!POT && c == 1 && kyneg) ? (T)-1 : (T)1;
        cpx<T> w[E];
#pragma unroll
        for (int q = 0; q < E; ++q) {
            const int kz = j + q * TPP;
            const bool kzneg = kz > nz;
            const int kzp = kzneg ? L - kz : kz;
            const T sz = (!POT && c == 2 && kzneg) ? (T)-1 : (T)1;
            const T g = sy * sz * gld(Gf + c * M1 + ((size_t)kzp * ny1 + kyp) * Kp + kxc);
            if constexpr (POT)
                w[q] = cpx<T>{p[q].x * g, p[q].y * g};  // rho_hat * g
            else
                w[q] = cpx<T>{-p[q].y * g, p[q].x * g};  // rho_hat * (i g)
            if constexpr (CATH) {
                cpx<T> gi = gld(Gi + c * MI + ((size_t)kz * ny1 + kyp) * Kp + kxc);
                gi.x *= sy;
                gi.y *= sy;
                if (c < 2) gi = cpx<T>{-gi.y, gi.x};
                w[q] = c_add(w[q], c_mul(pi[q], gi));
            }
        }
        mix::fft<T, L, E, +1>(w, j, lds + b, NB, tw);
        if (live) {
            cpx<T> *Bc = B + (size_t)c * mz * zs + (size_t)ky * Kp + kx;
#pragma unroll
            for (int q = 0; q < E / 2; ++q)
                if (j + q * TPP < mz) gst(Bc + (size_t)(j + q * TPP) * zs, w[q]);
        }
    }
}

// Transposed z convolution (see k_zconv_adj in sc_solve.hip): the three g_E
// spectra in Gs are transformed one at a time and their products with
// conj(G_c^) summed in registers; the image sum, reversed in z, is
// subtracted in the spectrum (a phase factor and the mirror bin, through
// LDS), so one backward transform serves both.
template <typename T, int L, bool CATH>
__global__ void __launch_bounds__((Shape<T, L>::THREADS))
__attribute__((amdgpu_waves_per_eu(1)))
k_zconv_adj_m(const cpx<T> *__restrict__ Gs, cpx<T> *__restrict__ out, const T *__restrict__ Gf,
              const cpx<T> *__restrict__ Gi, const cpx<T> *__restrict__ twg, Dims d)
{
    using S = Shape<T, L>;
    constexpr int E = S::E, TPP = S::TPP, NB = S::NB;
    __shared__ cpx<T> tw[L];
    __shared__ cpx<T> lds[NB * L];
    const int Kp = d.Kp, Ly = d.Ly, ny = d.ny, nz = d.nz, mz = d.mz, ny1 = ny + 1;
    for (int i = threadIdx.x; i < L; i += S::THREADS) tw[i] = gld(twg + i);
    const int b = threadIdx.x % NB, j = threadIdx.x / NB;
    // free space: a 1-D grid of div_up(Kx, NB) * Ly workgroups in XCD order;
    // with the cathode image a grid (div_up(Kx, NB), Ly), as in k_zconv_m
    int bx, ky;
    if (CATH) {
        bx = (int)blockIdx.x;
        ky = (int)blockIdx.y;
    } else {
        zconv_pencils(xcd_task((int)blockIdx.x, (int)gridDim.x), (d.Kx + NB - 1) / NB, Ly, bx, ky);
    }
    const int kx = bx * NB + b;
    const bool live = kx < d.Kx;
    const size_t zs = (size_t)Ly * Kp;
    const bool kyneg = ky > ny;
    const int kyp = kyneg ? Ly - ky : ky;
    const size_t M1 = (size_t)(nz + 1) * ny1 * Kp;
    const size_t MI = (size_t)L * ny1 * Kp;
    const int kxc = live ? kx : 0;  // keep dead lanes' loads in bounds
    cpx<T> w[E], wi[E];
#pragma unroll
    for (int q = 0; q < E; ++q) {
        w[q] = cpx<T>{(T)0, (T)0};
        wi[q] = cpx<T>{(T)0, (T)0};
    }
#pragma unroll 1
    for (int c = 0; c < 3; ++c) {
        const cpx<T> *Gp = Gs + (size_t)c * mz * zs + (size_t)ky * Kp + kxc;
        cpx<T> p[E];
#pragma unroll
        for (int q = 0; q < E; ++q) {
            p[q] = cpx<T>{(T)0, (T)0};
            if (q < E / 2) {
                const int e = j + q * TPP;
                const bool on = live && e < mz;
                const cpx<T> t = gld(Gp + (size_t)(on ? e : 0) * zs);
                p[q] = on ? t : cpx<T>{(T)0, (T)0};
            }
        }
        mix::fft<T, L, E, -1>(p, j, lds + b, NB, tw);
        const T sy = (c == 1 && kyneg) ? (T)-1 : (T)1;
#pragma unroll
        for (int q = 0; q < E; ++q) {
            const int kz = j + q * TPP;
            const bool kzneg = kz > nz;
            const int kzp = kzneg ? L - kz : kz;
            const T sz = (c == 2 && kzneg) ? (T)-1 : (T)1;
            const T g = sy * sz * gld(Gf + c * M1 + ((size_t)kzp * ny1 + kyp) * Kp + kxc);
            w[q] = c_add(w[q], cpx<T>{p[q].y * g, -p[q].x * g});  // p * conj(i g)
            if constexpr (CATH) {
                cpx<T> gi = gld(Gi + c * MI + ((size_t)kz * ny1 + kyp) * Kp + kxc);
                gi.x *= sy;
                gi.y *= sy;
                if (c < 2) gi = cpx<T>{-gi.y, gi.x};
                wi[q] = c_add(wi[q], c_mul(p[q], cpx<T>{gi.x, -gi.y}));
            }
        }
    }
    if constexpr (CATH) {
        // out[z] = IFFT(W)[z] - IFFT(WI)[mz-1-z].  The reversed transform is
        // IFFT(U) with U[k] = WI[-k] w_L^((mz-1) k), so one backward
        // transform of W - U gives both; WI[-k] is held by another lane.
        __syncthreads();  // every lane past the last forward transform's exchange
#pragma unroll
        for (int q = 0; q < E; ++q) lds[b + (j + q * TPP) * NB] = wi[q];
        __syncthreads();
#pragma unroll
        for (int q = 0; q < E; ++q) {
            const int k = j + q * TPP;
            const cpx<T> m = lds[b + (k == 0 ? 0 : L - k) * NB];
            w[q] = c_sub(w[q], c_mul(tw[((mz - 1) * k) % L], m));
        }
    }
    mix::fft<T, L, E, +1>(w, j, lds + b, NB, tw);
    if (live) {
        cpx<T> *o = out + (size_t)ky * Kp + kx;
#pragma unroll
        for (int q = 0; q < E / 2; ++q)
            if (j + q * TPP < mz) gst(o + (size_t)(j + q * TPP) * zs, w[q]);
    }
}

// Backward y pass: pencils (kx, z < nz) of each field spectrum, y < ny kept.
template <typename T, int L>
__global__ void __launch_bounds__((Shape<T, L>::THREADS))
k_inv_y_m(cpx<T> *__restrict__ B, const cpx<T> *__restrict__ twg, Dims d,
          const SBunch *__restrict__ tab, int per)
{
    using S = Shape<T, L>;
    constexpr int E = S::E, TPP = S::TPP, NB = S::NB;
    __shared__ cpx<T> tw[L];
    __shared__ cpx<T> lds[NB * L];
    const SBunch *sb;
    const int bx = group_block(tab, per, sb);
    if (sb) B = static_cast<cpx<T> *>(sb->inv);
    for (int i = threadIdx.x; i < L; i += S::THREADS) tw[i] = gld(twg + i);
    const int b = threadIdx.x % NB, j = threadIdx.x / NB;
    const int kx = bx * NB + b, z = blockIdx.y, c = blockIdx.z;
    const int Kx = d.Kx, Kp = d.Kp;
    const bool live = kx < Kx;
    cpx<T> *Bp = B + ((size_t)c * d.mz + z) * d.Ly * Kp + (live ? kx : 0);
    cpx<T> v[E];
#pragma unroll
    for (int q = 0; q < E; ++q) v[q] = gld(Bp + (size_t)(j + q * TPP) * Kp);
    mix::fft<T, L, E, +1>(v, j, lds + b, NB, tw);
    if (live) {
#pragma unroll
        for (int q = 0; q < E / 2; ++q)
            if (j + q * TPP < d.my) gst(Bp + (size_t)(j + q * TPP) * Kp, v[q]);
    }
}

// Backward x pass (complex to real) with Hermitian completion.
template <typename T, int L>
__global__ void __launch_bounds__((Shape<T, L>::THREADS))
k_inv_x_m(const cpx<T> *__restrict__ B, T *__restrict__ E_, const cpx<T> *__restrict__ twg, Dims d,
          const SBunch *__restrict__ tab, int per)
{
    using S = Shape<T, L>;
    constexpr int E = S::E, TPP = S::TPP, NB = S::NB;
    __shared__ cpx<T> tw[L];
    __shared__ cpx<T> lds[NB * reg::padded<L, E>()];
    const SBunch *sb;
    const int bx = group_block(tab, per, sb);
    if (sb) {
        B = static_cast<const cpx<T> *>(sb->inv);
        E_ = static_cast<T *>(sb->out);
    }
    for (int i = threadIdx.x; i < L; i += S::THREADS) tw[i] = gld(twg + i);
    const int b = threadIdx.x / TPP, j = threadIdx.x % TPP;
    const int r = bx * NB + b, c = blockIdx.y;
    const int nrows = d.my * d.mz, nx = d.nx, mx = d.mx;
    const bool live = r < nrows;
    const int rr = live ? r : 0;
    const int y = rr % d.my, z = rr / d.my;
    const cpx<T> *row = B + (size_t)c * d.mz * d.Ly * d.Kp + ((size_t)z * d.Ly + y) * d.Kp;
    // one unconditional load per element (the Hermitian half reads the
    // mirror), so all of a lane's loads are in flight together
    cpx<T> v[E];
#pragma unroll
    for (int q = 0; q < E; ++q) {
        const int k = j + q * TPP;
        const bool direct = q < E / 2 || k == nx;
        v[q] = gld(row + (direct ? k : L - k));
    }
#pragma unroll
    for (int q = 0; q < E; ++q) {
        const int k = j + q * TPP;
        if (!(q < E / 2 || k == nx)) v[q].y = -v[q].y;
    }
    mix::fft<T, L, E, +1>(v, j, lds + b * reg::padded<L, E>(), 1, tw);
    if (live) {
        T *out = E_ + ((size_t)c * nrows + r) * mx;
#pragma unroll
        for (int q = 0; q < E / 2; ++q)
            if (j + q * TPP < mx) gst(out + j + q * TPP, v[q].x);
    }
}

template <typename T, int L>
void launch_all(Mesh *m, const Dims &d, int axis_kernel, const SolveIO &io)
{
    Workspace &ws = m->ws;
    Ctx *ctx = m->ctx;
    hipStream_t st = ctx->stream;
    using S = Shape<T, L>;
    const cpx<T> *tw = static_cast<const cpx<T> *>(ws.twT[axis_kernel == 0 || axis_kernel == 4 ? 0
                                                           : axis_kernel == 2         ? 2
                                                                                      : 1]);
    cpx<T> *F = static_cast<cpx<T> *>(io.fwd);
    cpx<T> *B = static_cast<cpx<T> *>(io.inv);
    switch (axis_kernel) {
    case 0:
        launch_begin(ctx, K_RHO_FWD_X);
        hipLaunchKernelGGL((k_rho_fwd_x_m<T, L>), dim3(div_up(d.my * d.mz, S::NB), io.nin),
                           dim3(S::THREADS), 0, st, static_cast<const T *>(io.in), F, tw, d,
                           (const SBunch *)nullptr, 0);
        launch_end(ctx, K_RHO_FWD_X);
        break;
    case 1:
        launch_begin(ctx, K_RHO_FWD_Y);
        hipLaunchKernelGGL((k_rho_fwd_y_m<T, L>), dim3(div_up(d.Kx, S::NB), d.mz, io.nin),
                           dim3(S::THREADS), 0, st, F, tw, d, (const SBunch *)nullptr, 0);
        launch_end(ctx, K_RHO_FWD_Y);
        break;
    case 2: {
        launch_begin(ctx, K_ZCONV);
        const int nbx = div_up(d.Kx, S::NB);
        const bool cath_mode = io.mode == kFieldCathode || io.mode == kAdjointCathode;
        const dim3 zgrid = cath_mode ? dim3(nbx, d.Ly) : dim3(nbx * d.Ly);
        const cpx<T> *Fc = F;
        const T *Gf = static_cast<const T *>(ws.Gf);
        const cpx<T> *Gi = static_cast<const cpx<T> *>(ws.Gi);
        switch (io.mode) {
        case kFieldCathode:
            if constexpr (zconv_here<T, L>(kFieldCathode))
                hipLaunchKernelGGL((k_zconv_m<T, L, kFieldCathode>), zgrid, dim3(S::THREADS), 0, st, Fc, B,
                                   Gf, Gi, tw, d, (const SBunch *)nullptr, nbx);
            break;
        case kPotential:
            hipLaunchKernelGGL((k_zconv_m<T, L, kPotential>), zgrid, dim3(S::THREADS), 0, st, Fc, B, Gf, Gi,
                               tw, d, (const SBunch *)nullptr, nbx);
            break;
        case kAdjointFree:
            hipLaunchKernelGGL((k_zconv_adj_m<T, L, false>), zgrid, dim3(S::THREADS), 0, st, Fc, B, Gf, Gi,
                               tw, d);
            break;
        case kAdjointCathode:
            if constexpr (zconv_here<T, L>(kAdjointCathode))
                hipLaunchKernelGGL((k_zconv_adj_m<T, L, true>), zgrid, dim3(S::THREADS), 0, st, Fc, B, Gf,
                                   Gi, tw, d);
            break;
        default:
            hipLaunchKernelGGL((k_zconv_m<T, L, kFieldFree>), zgrid, dim3(S::THREADS), 0, st, Fc, B, Gf, Gi,
                               tw, d, (const SBunch *)nullptr, nbx);
            break;
        }
        launch_end(ctx, K_ZCONV);
        break;
    }
    case 3:
        launch_begin(ctx, K_INV_Y);
        hipLaunchKernelGGL((k_inv_y_m<T, L>), dim3(div_up(d.Kx, S::NB), d.mz, io.nout),
                           dim3(S::THREADS), 0, st, B, tw, d, (const SBunch *)nullptr, 0);
        launch_end(ctx, K_INV_Y);
        break;
    case 4:
        launch_begin(ctx, K_INV_X);
        hipLaunchKernelGGL((k_inv_x_m<T, L>), dim3(div_up(d.my * d.mz, S::NB), io.nout),
                           dim3(S::THREADS), 0, st, (const cpx<T> *)B, static_cast<T *>(io.out), tw, d,
                           (const SBunch *)nullptr, 0);
        launch_end(ctx, K_INV_X);
        break;
    }
}

// Solve kernel `which` of nb same-shape bunches in one launch (x stacked).
template <typename T, int L>
void launch_all_grouped(const Dims &d, const cpx<T> *tw, int nb, const SBunch *tab, int which,
                        int mode, int nin, int nout, hipStream_t st)
{
    using S = Shape<T, L>;
    switch (which) {
    case 0: {
        const int per = div_up(d.my * d.mz, S::NB);
        hipLaunchKernelGGL((k_rho_fwd_x_m<T, L>), dim3(per * nb, nin), dim3(S::THREADS), 0, st,
                           (const T *)nullptr, (cpx<T> *)nullptr, tw, d, tab, per);
        break;
    }
    case 1: {
        const int per = div_up(d.Kx, S::NB);
        hipLaunchKernelGGL((k_rho_fwd_y_m<T, L>), dim3(per * nb, d.mz, nin), dim3(S::THREADS), 0, st,
                           (cpx<T> *)nullptr, tw, d, tab, per);
        break;
    }
    case 2: {
        const int per = div_up(d.Kx, S::NB);
        const dim3 zgrid(per * nb, d.Ly);
        if (mode == kFieldCathode)
            hipLaunchKernelGGL((k_zconv_m<T, L, kFieldCathode>), zgrid, dim3(S::THREADS), 0, st,
                               (const cpx<T> *)nullptr, (cpx<T> *)nullptr, (const T *)nullptr,
                               (const cpx<T> *)nullptr, tw, d, tab, per);
        else
            hipLaunchKernelGGL((k_zconv_m<T, L, kFieldFree>), zgrid, dim3(S::THREADS), 0, st,
                               (const cpx<T> *)nullptr, (cpx<T> *)nullptr, (const T *)nullptr,
                               (const cpx<T> *)nullptr, tw, d, tab, per);
        break;
    }
    case 3: {
        const int per = div_up(d.Kx, S::NB);
        hipLaunchKernelGGL((k_inv_y_m<T, L>), dim3(per * nb, d.mz, nout), dim3(S::THREADS), 0, st,
                           (cpx<T> *)nullptr, tw, d, tab, per);
        break;
    }
    case 4: {
        const int per = div_up(d.my * d.mz, S::NB);
        hipLaunchKernelGGL((k_inv_x_m<T, L>), dim3(per * nb, nout), dim3(S::THREADS), 0, st,
                           (const cpx<T> *)nullptr, (T *)nullptr, tw, d, tab, per);
        break;
    }
    }
}

}  // namespace

// One length: solve kernel `which` of one mesh, or (tab) of nb same-shape
// bunches.  Defined in the part that compiles the length.
template <typename T, int L>
void launch_mix_length(Mesh *m, const Dims &d, int which, const SolveIO &io)
{
    launch_all<T, L>(m, d, which, io);
}
template <typename T, int L>
void launch_mix_length_grouped(const Dims &d, const cpx<T> *tw, int nb, const SBunch *tab, int which,
                           int mode, int nin, int nout, hipStream_t st)
{
    launch_all_grouped<T, L>(d, tw, nb, tab, which, mode, nin, nout, st);
}

#define SC_MIX_INSTANCE(T, L)                                                      \
    template void launch_mix_length<T, L>(Mesh *, const Dims &, int, const SolveIO &);  \
    template void launch_mix_length_grouped<T, L>(const Dims &, const cpx<T> *, int, const SBunch *, \
                                              int, int, int, int, hipStream_t);
#define SC_MIX_EXTERN(T, L) extern SC_MIX_INSTANCE(T, L)

#if SC_MIX_PART == 0
#define X(L) SC_MIX_INSTANCE(float, L)
SC_MIX_SHORT(X)
#undef X
#define X(L) SC_MIX_EXTERN(float, L)
SC_MIX_LONG(X) SC_MIX_POW2(X)
#undef X
#define X(L) SC_MIX_EXTERN(double, L)
SC_MIX_LENGTHS(X)
#undef X
#elif SC_MIX_PART == 1
#define X(L) SC_MIX_INSTANCE(float, L)
SC_MIX_LONG(X) SC_MIX_POW2(X)
#undef X
#elif SC_MIX_PART == 2
#define X(L) SC_MIX_INSTANCE(double, L)
SC_MIX_SHORT(X)
#undef X
#else
#define X(L) SC_MIX_INSTANCE(double, L)
SC_MIX_LONG(X) SC_MIX_POW2(X)
#undef X
#endif

#if SC_MIX_PART == 0

template <typename T>
void launch_mix_grouped(const Mesh *m0, int nb, const SBunch *tab, int which, int mode, int nin,
                         int nout, hipStream_t st)
{
    const Dims d = make_dims(m0);
    const int axis = (which == 0 || which == 4) ? 0 : (which == 2 ? 2 : 1);
    const int L = axis == 0 ? d.Lx : (axis == 2 ? d.Lz : d.Ly);
    const cpx<T> *tw = static_cast<const cpx<T> *>(m0->ws.twT[axis]);
    switch (L) {
#define X(LL)                                                                        \
    case LL:                                                                         \
        launch_mix_length_grouped<T, LL>(d, tw, nb, tab, which, mode, nin, nout, st); \
        break;
        SC_MIX_LENGTHS(X)
#undef X
    default: break;  // the caller groups only supported lengths
    }
}

template void launch_mix_grouped<float>(const Mesh *, int, const SBunch *, int, int, int, int,
                                         hipStream_t);
template void launch_mix_grouped<double>(const Mesh *, int, const SBunch *, int, int, int, int,
                                          hipStream_t);

// Runs one solve kernel (0 rho_fwd_x, 1 rho_fwd_y, 2 zconv, 3 inv_y,
// 4 inv_x) with the register engine if it supports its transform length;
// returns false (nothing launched) otherwise.
template <typename T>
bool launch_mix(Mesh *m, int which, const SolveIO &io)
{
    const Dims d = make_dims(m);
    const int L = (which == 0 || which == 4) ? d.Lx : (which == 2 ? d.Lz : d.Ly);
    switch (L) {
#define X(LL) \
    case LL:                                                                   \
        if (which == 2 && !zconv_here<T, LL>(io.mode)) return false;               \
        launch_mix_length<T, LL>(m, d, which, io);                                 \
        return true;
        SC_MIX_LENGTHS(X)
#undef X
    default: return false;
    }
}

template bool launch_mix<float>(Mesh *, int, const SolveIO &);
template bool launch_mix<double>(Mesh *, int, const SolveIO &);

#endif  // SC_MIX_PART == 0

}  // namespace sc
