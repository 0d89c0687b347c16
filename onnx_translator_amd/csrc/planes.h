// planes.h — row tiles of image planes in LDS, for the operators that slide a window
// over single planes (depthwise convolution, MaxPool).
//
// A block stages one tile of rows of a plane (or several small planes) in LDS as f32,
// window padding included, with every load of a thread issued before its first LDS
// store; its threads then work on strips of R output rows of one column.
#pragma once

#include <algorithm>

#include "runtime.h"

namespace tohip {

constexpr int kPlaneThreads = 256;
constexpr int kPlaneTile = 4096;        // floats of LDS tile aimed at: eight blocks or more per CU
constexpr int kPlaneTileMax = 12288;    // and the most that a wide plane's shortest tile may take

struct PlaneTiles {
    int C, H, W, OH, OW, M;             // input planes [N, C], output planes [N, M] (M / C per input plane)
    int KH, KW, pt, pl, sh, sw, dh, dw;
    int planes;          // N * M output planes
    int np;              // planes per block (more than one only when a block holds whole planes)
    int tiles;           // row tiles per plane
    int TR;              // output rows per tile: ns strips
    int ns;              // strips per tile
    int PR, PW;          // LDS rows per plane and their pitch
    int cc;              // column chunks of a row in the staging loop
    int lxl, lxo;        // log2 of the threads along a row: staging, output
    uint32_t xbytes;
    FastDiv fd_tiles, fd_cc, fd_pr, fd_ns, fd_m, fd_mg;

    __device__ __forceinline__ int in_plane(int p) const {
        if (M == C) return p;           // one output plane per input plane
        const int n = (int)fd_m.div((uint32_t)p);
        return n * C + (int)fd_mg.div((uint32_t)(p - n * M));
    }
    __device__ __forceinline__ int channel(int p) const { return p - (int)fd_m.div((uint32_t)p) * M; }
};

// Stages the input rows of tile tl of planes p0 .. p0 + np - 1 (EB bytes per element).
// ld(off) gives the value at byte offset off of X, or the padding's for kOOB.
template <int EB, bool MULTI, class LD>
__device__ __forceinline__ void stage_planes(float* tile, const PlaneTiles& g, int tl, int p0, int np, LD ld) {
    const int lx = (int)threadIdx.x & ((1 << g.lxl) - 1), ly = (int)threadIdx.x >> g.lxl;
    const int step = kPlaneThreads >> g.lxl;
    const int ih0 = tl * g.TR * g.sh - g.pt;
    constexpr int U = 8;
    if constexpr (!MULTI) {
        // one plane: a thread keeps its column; a row on is one addition to the
        // load's and the LDS offset
        const int rows0 = g.in_plane(p0) * g.H, ih_end = max(0, min(g.H, ih0 + g.PR));
        for (int c = lx; c < g.PW; c += 1 << g.lxl) {
            const int iw = c - g.pl;
            const bool col = (unsigned)iw < (unsigned)g.W;
            for (int r0 = ly; r0 < g.PR; r0 += step * U) {
                float v[U];
                uint32_t off = (uint32_t)((rows0 + ih0 + r0) * g.W + iw) * EB;
#pragma unroll
                for (int u = 0; u < U; u++) {
                    const int ih = ih0 + r0 + u * step;
                    v[u] = ld(col && (unsigned)ih < (unsigned)ih_end ? off : kOOB);
                    off += (uint32_t)(step * g.W) * EB;
                }
                float* to = tile + r0 * g.PW + c;
#pragma unroll
                for (int u = 0; u < U; u++) {
                    if (r0 + u * step < g.PR) *to = v[u];
                    to += step * g.PW;
                }
            }
        }
    } else {
        const int items = np * g.PR * g.cc;
        for (int i0 = ly; i0 < items; i0 += step * U) {
            float v[U];
            int at[U];
#pragma unroll
            for (int u = 0; u < U; u++) {
                const int i = i0 + u * step;
                const int rr = g.cc == 1 ? i : (int)g.fd_cc.div((uint32_t)i);
                const int c = ((i - rr * g.cc) << g.lxl) + lx;
                const int q = (int)g.fd_pr.div((uint32_t)rr);
                const int row0 = g.in_plane(min(p0 + q, g.planes - 1)) * g.H;
                const int ih = ih0 + rr - q * g.PR, iw = c - g.pl;
                const bool in = i < items && c < g.PW;
                const bool ok = in && (unsigned)ih < (unsigned)g.H && (unsigned)iw < (unsigned)g.W;
                at[u] = in ? rr * g.PW + c : -1;
                v[u] = ld(ok ? (uint32_t)((row0 + ih) * g.W + iw) * EB : kOOB);
            }
#pragma unroll
            for (int u = 0; u < U; u++)
                if (at[u] >= 0) tile[at[u]] = v[u];
        }
    }
}

// Threads along a row of n elements (log2): the most, up to a wave, that leave at
// most a quarter of them idle against the best of 16, 32 and 64 (8 for rows that
// short): wide rows keep their loads and stores contiguous.
inline int row_threads_log2(int n) {
    if (n <= 8) return 3;
    auto cost = [n](int l) { return (n + (1 << l) - 1) >> l << l; };
    const int best = std::min(cost(4), std::min(cost(5), cost(6)));
    for (int l = 6; l > 4; l--)
        if (4 * cost(l) <= 5 * best) return l;
    return 4;
}

// Fills in the tiles for strips of R output rows (extra: floats of LDS per plane besides
// its rows).  H, W, ..., dw, C, M and planes are set; false when a row is too wide or the
// blocks are more than one launch holds.
inline bool plan_planes(PlaneTiles& p, int R, int extra) {
    const int64_t pw = (int64_t)(p.OW - 1) * p.sw + (int64_t)(p.KW - 1) * p.dw + 1;
    auto rows = [&](int64_t tr) { return (tr - 1) * p.sh + (int64_t)(p.KH - 1) * p.dh + 1; };
    if (pw > kPlaneTileMax || rows(R) * pw > kPlaneTileMax) return false;
    const int all = (p.OH + R - 1) / R;                  // strips of a plane
    // the most strips whose rows fit the tile aimed at
    const int64_t most = ((kPlaneTile / pw - (int64_t)(p.KH - 1) * p.dh - 1) / p.sh + 1) / R;
    const int ns = (int)std::max<int64_t>(1, std::min<int64_t>(all, most));
    p.tiles = (all + ns - 1) / ns;
    p.ns = (all + p.tiles - 1) / p.tiles;                // even tiles
    p.TR = p.ns * R;
    p.PR = (int)rows(p.TR);
    p.PW = (int)pw;
    p.np = 1;
    if (p.tiles == 1) {
        // several small planes per block, as long as two blocks per CU remain
        const int64_t fit = kPlaneTile / ((int64_t)p.PR * p.PW + extra);
        p.np = (int)std::max<int64_t>(1, std::min<int64_t>(fit, p.planes / (2 * num_cus())));
    }
    // the runtime takes fewer than 2^32 work-items per grid dimension
    if ((p.planes + (int64_t)p.np - 1) / p.np * p.tiles * kPlaneThreads >= (int64_t)1 << 32) return false;
    p.lxl = row_threads_log2(p.PW);
    p.lxo = row_threads_log2(p.OW);
    p.cc = (p.PW + (1 << p.lxl) - 1) >> p.lxl;
    p.fd_tiles = make_fastdiv((uint32_t)p.tiles);
    p.fd_cc = make_fastdiv((uint32_t)p.cc);
    p.fd_pr = make_fastdiv((uint32_t)p.PR);
    p.fd_ns = make_fastdiv((uint32_t)p.ns);
    p.fd_m = make_fastdiv((uint32_t)p.M);
    p.fd_mg = make_fastdiv((uint32_t)(p.M / p.C));
    return true;
}

}  // namespace tohip
