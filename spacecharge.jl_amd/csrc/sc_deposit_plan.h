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
// pairs and with the sub-grids, the binned chain's hardly; but it is two or three
// launches, the chain six, and a step of so few particles waits for the host as
// often as for the GPU.  Deposit alone (replayed from a graph, uniform particles, the
// chain's best case, direct / binned, us), Float64: 10k on 16^3 7.7 / 37; 8 tiles, 524k 37 /
// 51, 734k 67 / 52; 27 tiles, 217k (5.6M pairs) 49.5 / 48; 64 tiles, 66k (4M) 49.7 / 36.9.
// Float32: 10k on 16^3 13 / 32; 8 tiles, 524k 40 / 45; 27 tiles, 78k (2M) 38 / 33; 64
// tiles, 23k 31.5 / 32.6, 46k 40 / 33.  Steps (uniform, then rms a tenth of the mesh),
// Float64: 64 tiles, 42k 103 / 105 and 101 / 107, 55k (3.4M) 105 / 105 and 102 / 109, 65k
// 111 / 106 and 108 / 110; 48 tiles, 60k 99 / 104 and 97 / 106, 87k (4M) 111 / 104 and 102 /
// 106; 36 tiles, 75k 89 / 95 and 88 / 98.  Float32: 18 tiles, 116k (2M) 76 / 84 and 75 /
// 87; 27 tiles, 77k 87 / 89 and 89 / 97; 64 tiles, 32k 87 / 96 and 87 / 98.  Three
// channels triple the sub-grids and share one binning, so that replayed from a graph
// they lose sooner (Float32, 27 tiles, 13k 44 / 41 and 41 / 48; 64 tiles, 8k 59 / 48 and
// 53 / 46; Float64, 64 tiles, 16k 60 / 57), but the gradient step that they are part
// of gains (Float32, 27 tiles, 26k 179 / 181 and 187 / 194; 64 tiles, 11k 190 / 209; Float64, 64
// tiles, 16k 218 / 229, 22k 234 / 228; 36 tiles, 39k 186 / 206).  One tile has no pairs to
// spare: there only the size of the sub-grids ends the range.
inline int64_t direct_most(int T, bool f32, int nchan)
{
    constexpr int64_t k = (int64_t)1 << 20;
    const int64_t pairs = T == 1 ? 16 * k : f32 ? 2 * k : T <= 32 ? 4 * k : 7 * k / 2;
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
