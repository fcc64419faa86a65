// sc_fft_mix.h -- register-resident pencil FFT for lengths of factors 2, 3, 5.
//
// The scheme of sc_fft_reg.h (which stays the path of unpadded powers of two)
// with mixed radices: a pencil of length L is held by TPP = L/E lanes, E
// elements each.  Lane j starts with x[j + r*TPP], r < E (the "input
// layout"), runs Stockham passes entirely in registers (radix E first, then
// the largest divisors of E that divide what is left of L), and exchanges
// data through LDS only between passes.  After the last pass lane j holds
// X[j + r*TPP] again, with a compile-time register permutation, so a forward
// transform can feed a backward one without touching memory.
//
// Stockham pass with radix R, NS = product of the earlier radices: butterfly
// b (b < L/R) reads x[b + q*L/R], multiplies element q by w_L^(q*(b mod NS)*
// L/(NS*R)), does an R-point DFT and writes output q to
// (b/NS)*NS*R + (b mod NS) + q*NS.  Lane j owns butterflies j + s*TPP,
// s < E/R.
//
// The lengths (SC_MIX_LENGTHS) are even, at most 512, and split into passes
// whose radices divide one E of at most 20 values; axes of at most 256 nodes
// are transformed at the next of them (transform_half, padding_pays in
// sc_solve_common.h).
// Radix-20 lanes (200 points as 20 x 10) took 20-40% longer than radix-10
// ones (10 x 10 x 2) in every pass of a 100^3 Float32 solve: the shorter
// lanes' third pass costs less than their occupancy gains.
#pragma once

#include <hip/hip_runtime.h>

#include "sc_fft_reg.h"

namespace sc {

constexpr int kMixMaxLength = 512;  // the longest of SC_MIX_LENGTHS

namespace mix {

// X(L) for every supported length: those that only this engine transforms
// (in two parts, compiled apart), and the powers of two that it takes on
// padded meshes (on others they run on sc_fft_reg.h).
#define SC_MIX_SHORT(X) X(16) X(24) X(48) X(72) X(80) X(96) X(100) X(144) X(160)
#define SC_MIX_LONG(X) X(192) X(200) X(288) X(320) X(384) X(400)
#define SC_MIX_POW2(X) X(32) X(64) X(128) X(256) X(512)
#define SC_MIX_LENGTHS(X) SC_MIX_SHORT(X) SC_MIX_LONG(X) SC_MIX_POW2(X)

// Elements per lane: few enough that a pencil and its product stay in
// registers beside the butterfly's temporaries (Float64 takes half as many
// where the length allows it), many enough for two or three passes.
template <typename T, int L>
constexpr int elems()
{
    constexpr bool f32 = sizeof(T) == 4;
    switch (L) {
    case 16: return 4;
    case 32: case 64: return 8;
    case 24: case 48: case 72: case 96: case 144: case 192: case 288: case 384: return 12;
    case 80: case 160: case 320: return 20;
    case 100: case 200: case 400: return 10;
    default: return f32 ? 16 : 8;  // 128, 256, 512
    }
}

// Shape of a workgroup: E values per lane, TPP lanes per pencil, NB pencils.
// NB is 16 (Float32) or 8 (Float64) where TPP alone fills a few waves, so that
// the NB neighbouring pencils of a strided pass read and write whole 128-byte
// lines and few lanes of the last workgroup along kx (Kx = L/2 + 1 columns)
// are idle; more for few lanes per pencil, to make whole waves (4 for the
// longest Float64 pencils, whose slices would not fit).
template <typename T, int L>
struct Shape {
    static constexpr int E = elems<T, L>();
    static constexpr int TPP = L / E;
    static constexpr bool kF32 = sizeof(T) == 4;
    static constexpr int NB = TPP <= 2 || TPP == 6 || (TPP == 10 && kF32) ? 32
                              : TPP >= 64                                ? 4
                              : TPP >= 32 || (!kF32 && (TPP >= 20 || L == 320)) ? 8
                                                                                : 16;
    static constexpr int THREADS = NB * TPP;
};

template <int DIR, typename T>
__device__ __forceinline__ void dft3(cpx<T> *v)
{
    const T h = (T)0.86602540378443864676;  // sin(2 pi / 3)
    const cpx<T> s = c_add(v[1], v[2]), d = c_sub(v[1], v[2]);
    const cpx<T> m{v[0].x - (T)0.5 * s.x, v[0].y - (T)0.5 * s.y};
    const cpx<T> r = reg::rot<DIR>(cpx<T>{h * d.x, h * d.y});
    v[0] = c_add(v[0], s);
    v[1] = c_add(m, r);
    v[2] = c_sub(m, r);
}

template <int DIR, typename T>
__device__ __forceinline__ void dft5(cpx<T> *v)
{
    const T c1 = (T)0.30901699437494742410, c2 = (T)-0.80901699437494742410;  // cos(2 pi k / 5)
    const T s1 = (T)0.95105651629515357212, s2 = (T)0.58778525229247312917;   // sin(2 pi k / 5)
    const cpx<T> a = c_add(v[1], v[4]), b = c_add(v[2], v[3]);
    const cpx<T> c = c_sub(v[1], v[4]), d = c_sub(v[2], v[3]);
    const cpx<T> m1{v[0].x + c1 * a.x + c2 * b.x, v[0].y + c1 * a.y + c2 * b.y};
    const cpx<T> m2{v[0].x + c2 * a.x + c1 * b.x, v[0].y + c2 * a.y + c1 * b.y};
    const cpx<T> n1 = reg::rot<DIR>(cpx<T>{s1 * c.x + s2 * d.x, s1 * c.y + s2 * d.y});
    const cpx<T> n2 = reg::rot<DIR>(cpx<T>{s2 * c.x - s1 * d.x, s2 * c.y - s1 * d.y});
    v[0] = c_add(v[0], c_add(a, b));
    v[1] = c_add(m1, n1);
    v[4] = c_sub(m1, n1);
    v[2] = c_add(m2, n2);
    v[3] = c_sub(m2, n2);
}

template <int R, int DIR, typename T>
__device__ __forceinline__ void dft(cpx<T> *v);

constexpr int inv_mod(int a, int m)  // a^-1 mod m, a and m coprime
{
    for (int i = 1; i < m; ++i)
        if (a * i % m == 1) return i;
    return 0;
}

// A B point DFT, A and B coprime, by the prime-factor index maps
// n = B n1 + A n2, k = B (B^-1 mod A) k1 + A (A^-1 mod B) k2 (mod A B), which
// turn it into B A-point and A B-point DFTs without twiddles between them.
template <int A, int B, int DIR, typename T>
__device__ __forceinline__ void dft_pf(cpx<T> *v)
{
    constexpr int N = A * B, kb = B * inv_mod(B % A, A), ka = A * inv_mod(A % B, B);
    cpx<T> t[B][A];
#pragma unroll
    for (int n2 = 0; n2 < B; ++n2) {
#pragma unroll
        for (int n1 = 0; n1 < A; ++n1) t[n2][n1] = v[(B * n1 + A * n2) % N];
        dft<A, DIR>(t[n2]);
    }
#pragma unroll
    for (int k1 = 0; k1 < A; ++k1) {
        cpx<T> u[B];
#pragma unroll
        for (int n2 = 0; n2 < B; ++n2) u[n2] = t[n2][k1];
        dft<B, DIR>(u);
#pragma unroll
        for (int k2 = 0; k2 < B; ++k2) v[(kb * k1 + ka * k2) % N] = u[k2];
    }
}

template <int R, int DIR, typename T>
__device__ __forceinline__ void dft(cpx<T> *v)
{
    if constexpr (R == 2) reg::dft2<DIR>(v[0], v[1]);
    else if constexpr (R == 3) dft3<DIR>(v);
    else if constexpr (R == 4) reg::dft4<DIR>(v[0], v[1], v[2], v[3]);
    else if constexpr (R == 5) dft5<DIR>(v);
    else if constexpr (R == 6) dft_pf<2, 3, DIR>(v);
    else if constexpr (R == 8) reg::dft8<DIR>(v);
    else if constexpr (R == 10) dft_pf<2, 5, DIR>(v);
    else if constexpr (R == 12) dft_pf<4, 3, DIR>(v);
    else if constexpr (R == 16) reg::dft16<DIR>(v);
    else if constexpr (R == 20) dft_pf<4, 5, DIR>(v);
    else static_assert(R == 2, "no butterfly of this radix");
}

// Radix of a pass with m = L / (earlier radices) left: the largest divisor of
// E that divides m.
constexpr int next_radix(int m, int E)
{
    for (int d = E; d > 1; --d)
        if (E % d == 0 && m % d == 0) return d;
    return m;
}
template <int L, int E>
constexpr int npasses()
{
    int n = 0, m = L;
    while (m > 1) {
        m /= next_radix(m, E);
        ++n;
    }
    return n;
}
template <int L, int E>
constexpr int radix(int p)
{
    int m = L;
    for (int i = 0; i < p; ++i) m /= next_radix(m, E);
    return next_radix(m, E);
}
template <int L, int E>
constexpr int ns_before(int p)
{
    int ns = 1;
    for (int i = 0; i < p; ++i) ns *= radix<L, E>(i);
    return ns;
}

// Work of one pass in registers: twiddles and butterflies.
template <typename T, int L, int E, int P, int DIR>
__device__ __forceinline__ void pass_compute(cpx<T> *v, int j, const cpx<T> *__restrict__ tw)
{
    constexpr int R = radix<L, E>(P), NS = ns_before<L, E>(P);
    constexpr int TPP = L / E, NBF = E / R;
#pragma unroll
    for (int s = 0; s < NBF; ++s) {
        if constexpr (NS > 1) {
            const int k = (j + s * TPP) % NS;
#pragma unroll
            for (int q = 1; q < R; ++q) {
                cpx<T> w = tw[q * k * (L / (NS * R))];
                if constexpr (DIR > 0) w.y = -w.y;
                v[s * R + q] = c_mul(v[s * R + q], w);
            }
        }
        dft<R, DIR>(v + s * R);
    }
}

// LDS exchange after pass P (all lanes of the workgroup participate).
// `lds` is this pencil's slice: element e at lds[reg::slot<E>(e, es)] (a
// contiguous slice, es == 1, holds reg::padded<L, E>() entries).  The elements of
// one butterfly are NS (written) or L/R2 (read) apart; both are multiples of
// E except the first pass's NS = 1, whose E elements share one e / E, so the
// slots are a base and a constant step.
template <typename T, int L, int E, int P>
__device__ __forceinline__ void pass_exchange(cpx<T> *v, int j, cpx<T> *lds, int es)
{
    constexpr int R = radix<L, E>(P), NS = ns_before<L, E>(P);
    constexpr int R2 = radix<L, E>(P + 1);
    constexpr int TPP = L / E, NBF = E / R, NBF2 = E / R2;
    static_assert(NS == 1 ? R == E : NS % E == 0, "one slot step per butterfly");
    static_assert((L / R2) % E == 0, "one slot step per butterfly");
    const int wstep = es == 1 ? NS + NS / E : NS * es;
    const int rstep = es == 1 ? L / R2 + L / R2 / E : (L / R2) * es;
#pragma unroll
    for (int s = 0; s < NBF; ++s) {
        const int b = j + s * TPP;
        cpx<T> *o = lds + reg::slot<E>((b / NS) * NS * R + b % NS, es);
#pragma unroll
        for (int q = 0; q < R; ++q) o[q * wstep] = v[s * R + q];
    }
    __syncthreads();
#pragma unroll
    for (int s = 0; s < NBF2; ++s) {
        const cpx<T> *i = lds + reg::slot<E>(j + s * TPP, es);
#pragma unroll
        for (int q = 0; q < R2; ++q) v[s * R2 + q] = i[q * rstep];
    }
}

// Full transform.  v holds the input layout on entry and the output in the
// input layout on exit (x[j + r*TPP] <-> v[r]).  Every lane of the
// workgroup must call it; it contains (npasses - 1) exchanges, each with a
// barrier, plus one barrier at entry so that `lds` may be reused.
template <typename T, int L, int E, int DIR>
__device__ __forceinline__ void fft(cpx<T> *v, int j, cpx<T> *lds, int es,
                                    const cpx<T> *__restrict__ tw)
{
    constexpr int NP = npasses<L, E>();
    static_assert(L % E == 0 && radix<L, E>(0) == E, "a lane's elements form the first butterfly");
    __syncthreads();
    pass_compute<T, L, E, 0, DIR>(v, j, tw);
    if constexpr (NP > 1) {
        pass_exchange<T, L, E, 0>(v, j, lds, es);
        pass_compute<T, L, E, 1, DIR>(v, j, tw);
    }
    if constexpr (NP > 2) {
        __syncthreads();
        pass_exchange<T, L, E, 1>(v, j, lds, es);
        pass_compute<T, L, E, 2, DIR>(v, j, tw);
    }
    if constexpr (NP > 3) {
        __syncthreads();
        pass_exchange<T, L, E, 2>(v, j, lds, es);
        pass_compute<T, L, E, 3, DIR>(v, j, tw);
    }
    static_assert(NP <= 4, "at most four passes");
    // last pass: butterfly b = j + s*TPP holds X[b + q*L/R] in v[s*R + q];
    // put X[j + r*TPP] into v[r] (r = s + q*NBF)
    constexpr int RL = radix<L, E>(NP - 1);
    constexpr int NBF = E / RL;
    if constexpr (NBF > 1) {
        cpx<T> t[E];
#pragma unroll
        for (int s = 0; s < NBF; ++s)
#pragma unroll
            for (int q = 0; q < RL; ++q) t[s + q * NBF] = v[s * RL + q];
#pragma unroll
        for (int r = 0; r < E; ++r) v[r] = t[r];
    }
}

}  // namespace mix
}  // namespace sc
