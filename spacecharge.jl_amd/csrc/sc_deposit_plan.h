// sc_deposit_plan.h -- how the deposit splits its work, and the scratch that it
// takes.  Host arithmetic only, free of HIP types.
#pragma once

#include <cstdint>

namespace sc {

constexpr int kBinMaxSlices = 2048;  // binning workgroups (columns of the count matrix)
constexpr int64_t kCmatBudget = (int64_t)1 << 22;  // count-matrix entries (slices x tiles)
constexpr int kDepThreads = 512;     // deposit workgroup size

// direct deposit (k_deposit_direct): most tiles, particles per workgroup,
// workgroups aimed at
constexpr int kDirectTiles = 64;
constexpr int kDirectLog2 = 13;
constexpr int kDirectBlocks = 128;

// The binning workgroups split the particles into G contiguous slices of
// `slice` particles; all three binning kernels use the same split.
struct Split {
    int64_t n, slice;
    int G;
};

// At most kBinMaxSlices slices of about 2^slice_log2 particles, and at
// most kCmatBudget / ntiles (the count matrix has a row per tile).
inline Split split_of(int64_t n, int slice_log2, int ntiles)
{
    Split sp;
    sp.n = n;
    const int64_t per = (int64_t)1 << slice_log2;
    int64_t G = (n + per - 1) / per;
    if (G > kBinMaxSlices) G = kBinMaxSlices;
    const int64_t gmax = kCmatBudget / (ntiles > 0 ? ntiles : 1);
    if (G > gmax) G = gmax;
    if (G < 1) G = 1;
    sp.G = (int)G;
    sp.slice = (n + G - 1) / G;
    return sp;
}

// Most particles that the direct deposit takes on a mesh of T tiles (0: none),
// f32 the mesh type, nchan charge channels.  Its cost grows with the particle-tile
// pairs and with the sub-grids, the binned chain's hardly; particles that fill
// the mesh are the binned chain's best case, so the line lies below where those
// break even.  Measured (replayed from a graph, uniform particles, direct / binned,
// us), Float64: 10k on 16^3 7.7 / 37; 8 tiles, 262k (2M pairs) 27.6 / 48.7, 524k 37 /
// 51, 734k 67 / 52; 27 tiles, 155k (4M pairs) 41.5 / 42.9, 217k 49.5 / 48; 64 tiles,
// 33k (2M pairs) 29.6 / 35.7, 46k 36.1 / 36.2, 66k 49.7 / 36.9.  Float32, with one
// launch more and a cheaper chain: 10k on 16^3 13 / 32; 8 tiles, 262k 31 / 41, 524k
// 40 / 45, 734k 60 / 46; 27 tiles, 54k (1.4M pairs) 27.6 / 32, 78k (2M) 38 / 33; 64
// tiles, 23k (1.4M) 31.5 / 32.6, 46k 40 / 33.  One tile has no pairs to spare: there
// only the size of the sub-grids ends the range.  Three channels triple the
// sub-grids and share one binning: 4k on 64 tiles 50 / 39 in Float32, 44.7 / 43.2 in
// Float64, 9k on 27 tiles 35.8 / 33.9 in Float32; Float64 on 4 tiles, 245k (2.8M) 35 /
// 53, 350k 57 / 52.
inline int64_t direct_most(int T, bool f32, int nchan)
{
    constexpr int64_t k = (int64_t)1 << 20;
    const int64_t pairs = T == 1 ? 16 * k : f32 ? (T <= 8 ? 2 * k : 7 * k / 5) : T <= 32 ? 4 * k : 5 * k / 2;
    if (nchan > 1 && T > 1) {
        if (T > (f32 ? 8 : 32)) return 0;
        if (pairs > 3 * k) return 3 * k / ((int64_t)T * nchan);
    }
    return T > kDirectTiles ? 0 : pairs / ((int64_t)T * nchan);
}

// Slices of the direct deposit of n particles, n <= direct_most; it grows with n.
inline int direct_slices(int64_t n, int T)
{
    const int64_t per = (int64_t)1 << kDirectLog2;
    const int64_t least = (n + per - 1) / per;  // slices of at most 2^kDirectLog2
    const int64_t most = (n + kDepThreads - 1) / kDepThreads;
    int64_t G = (T == 1 ? 2 : 1) * kDirectBlocks / T;
    if (G > most) G = most;
    if (G < least) G = least;
    return (int)G;
}

// Scratch entries of a deposit.
struct DepositNeed {
    int64_t chunks;  // chunk table entries, and sub-grids per channel
    int64_t cmat;    // count-matrix entries, or flags of the direct deposit's sub-grids
};

inline DepositNeed binned_need(int64_t n, int T, int chunk_log2, int slice_log2)
{
    // chunks: at most T + n / chunk; sub-grid slots: below 2 T + chunks
    // (slots of the row scan's reservation order, k_bin_rowscan)
    return {2 * (int64_t)T + (n >> chunk_log2) + 1, (int64_t)T * split_of(n, slice_log2, T).G};
}
inline DepositNeed direct_need(int64_t n, int T, int nchan)
{
    const int64_t subs = (int64_t)T * direct_slices(n, T);
    return {subs, subs * nchan};
}

// Scratch that a deposit of n particles reserves: enough for every deposit of at
// most n particles and nchan channels on the same mesh, by either path.  A
// smaller deposit may be direct and take more sub-grids than this one binned, and
// a batched one is binned where a single one is direct; none of them may move
// the buffers, whose addresses a captured graph holds, nor allocate while one is
// being captured.
inline DepositNeed deposit_need(int64_t n, int T, bool f32, int nchan, int chunk_log2, int slice_log2)
{
    DepositNeed r = binned_need(n, T, chunk_log2, slice_log2);
    for (int c = 1; c <= nchan; ++c) {
        const int64_t most = direct_most(T, f32, c);
        if (most == 0) continue;
        const DepositNeed d = direct_need(n < most ? n : most, T, c);
        if (d.chunks > r.chunks) r.chunks = d.chunks;
        if (d.cmat > r.cmat) r.cmat = d.cmat;
    }
    return r;
}

}  // namespace sc
