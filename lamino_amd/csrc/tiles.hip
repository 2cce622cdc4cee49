// Spreading (type 1) of the three-component projectors on the matrix cores.
//
// A point touches W x W cells of the (z, x) plane with weights wz (x) wx, times the y
// weights of its line.  Every point of a line (projection, detector row) has the same y,
// because the in-plane basis vector u has no y component.  Over the points of one tile and
// one row, spreading is therefore a matrix product,
//   H[(z, c)][(x, i)] = sum_points (wz[z] v_c) (wx[x] d_i),
// c: re, im; i: the component (the value v d_i has rank one), followed by
// F(z, y, x) += wy[y] H for the W planes of the row.  A stamp of 6 x 6 cells fills 216 of
// the 1024 products of a 32 x 32 block, but the sums stay in registers, where the vector
// form walked the points one by one through read-modify-writes of an LDS box and then sent
// every row's plane through memory (5.4 GB written, 6.7 GB read per launch at
// (359, 71, 359) / 615): here only the finished planes go out, 42 instead of 308.
//
// Measured on MI355X, spread of one dataset with its y pass, per launch: (359, 71, 359) /
// 615 x 615 x 360: 6.04 -> 3.39 ms; (179, 43, 179) / 305 x 305 x 180: 0.95 -> 0.58 ms;
// (89, 21, 89) / 89 x 89 x 90: 0.112 -> 0.070 ms; grids whose tilt varies, (127, 31, 127) /
// 181 x 181 x 120: 1.55 -> 0.50 ms.  fp32 matrix instructions and vector instructions share
// the SIMD on gfx950 (measured: a wave of each side by side takes the sum of their times;
// a bf16 one overlaps), so what bounds the kernel is their sum: 2.29e9 + 3.24e9 SIMD cycles
// of the 6.63e9 of a launch at the largest shape.  Hence the 32 x 32 block of all components:
// with one wave per component and 16 x 16 blocks the matrix part is half as much again, and
// the launch took 3.65 ms against 2.9 ms.  Where other forms are the better ones: row_tiles_pay and
// first_cell_tiles_pay below.
#include <algorithm>
#include <cmath>
#include <cstdlib>
#include <cstring>
#include <type_traits>

#include "nufft_point.h"
#include "tiles.h"

namespace lam {

// y weights of a row slot and its first plane (unwrapped); direct plans use iy only
struct RowY {
    float w[12];
    int iy, pad[3];
};

// A projection's geometry as the staging lanes read it: 16 bytes per axis, and float d_i.
struct __attribute__((aligned(16))) TileGeo {
    double uz, vz, ux, vx, vy, pad;
    float d[4];
};

namespace {

typedef float v16f __attribute__((ext_vector_type(16)));

constexpr int kBlock = 16;                 // matrix-core block edge
constexpr int kRec = kBlock * 32;          // complex values of a tile's record of one plane
constexpr unsigned kNoPoint = 0xffffffffu; // padding of a (tile, slot)

// Components per matrix block and the x cells they leave room for: the 32 columns hold 10
// cells of 3 components, or one component's 32 cells for the widest kernels.
constexpr int tile_comps(int W) { return W <= 8 ? 3 : 1; }
template <int NI>
constexpr int kXCells = 32 / NI;

// occupancy hint (waves per SIMD): what the W-plane window leaves room for without spills
constexpr int spread_waves(int W) { return W <= 6 ? 3 : W <= 8 ? 2 : 1; }

// ------------------------------------------------------------------ plan building
// The points of a line cross a tile in one run of consecutive columns, so the points are
// sorted as runs (about 10 points each) and not one by one.

// Launches of a wave per item stride over their items: a dimension of a launch holds fewer than
// 2^32 threads, 2^26 waves, and a plan may have more lines and buckets than that.
constexpr unsigned kMaxWaveBlocks = 1u << 20;
dim3 wave_grid(long long items) { return dim3(grid_for((size_t)items, 4, kMaxWaveBlocks)); }

// Wave per 64 consecutive points of a line: the lanes where a new run starts, with its
// bucket (tile, slot).  PASS 0 counts points and runs per bucket; PASS 1 stores the runs at
// a cursor (their order inside the bucket is settled by k_run_expand).
template <int PASS>
__global__ __launch_bounds__(256) void k_tile_runs(const Geo *__restrict__ geo, long long nwaves, int R, int C,
                                                   PointFrame fr, TileGeom tg, unsigned cpl,
                                                   unsigned long long *__restrict__ count,
                                                   const unsigned *__restrict__ roff, unsigned *__restrict__ cursor,
                                                   uint2 *__restrict__ runs) {
    const int lane = threadIdx.x & 63;
    const long long S = (long long)R * C, H = (S + 1) / 2;
    for (long long wave = blockIdx.x * 4ll + (threadIdx.x >> 6); wave < nwaves; wave += gridDim.x * 4ll) {
        const long long line = wave / cpl;
        const int chunk = (int)(wave - line * cpl);
        const int p = (int)(line / tg.Jn), j = (int)(line - (long long)p * tg.Jn);
        const int k = chunk * 64 + lane;
        const long long idx = (long long)j * C + k;
        const bool ok = k < C && idx < H;
        double tx, ty, tz;
        point_coords(geo[p], fr, j, k, tx, ty, tz);
        int bucket = -1;
        if (ok) {
            const int ix = wrap0(first_cell(tx, tg.nfx, fr.rx, tg.W), tg.nfx);
            const int iz = wrap0(first_cell(tz, tg.nfz, fr.rz, tg.W), tg.nfz);
            const unsigned tile = tg.fTz.div((unsigned)iz) * (unsigned)tg.ntx + tg.fTx.div((unsigned)ix);
            const int slot = tg.direct ? wrap0(first_cell(ty, tg.nfy, fr.ry, tg.W), tg.nfy)
                                       : (tg.dir > 0 ? j : tg.Jn - 1 - j);
            bucket = (int)(tile * (unsigned)tg.nrho + (unsigned)slot);
        }
        const int prev = __shfl_up(bucket, 1);
        const bool start = ok && (lane == 0 || bucket != prev);
        const unsigned long long starts = __ballot(start), valid = __ballot(ok);
        if (!start) continue;
        const unsigned long long after = lane == 63 ? 0ull : starts >> (lane + 1);
        const int end = after ? lane + 1 + __builtin_ctzll(after) : __popcll(valid);
        const unsigned len = (unsigned)(end - lane);
        if constexpr (PASS == 0) {
            atomicAdd(&count[bucket], (1ull << 32) | len);
        } else {
            const unsigned pos = roff[bucket] + atomicAdd(&cursor[bucket], 1u);
            runs[pos] = make_uint2((unsigned)((long long)p * H + idx), len);
        }
    }
}

// Exclusive scans of the low and high words of counts (PAD: the low words rounded up to
// multiples of 4, the buckets' padded point counts).
constexpr int kScanItems = 8, kScanBlock = 256 * kScanItems;

template <bool PAD>
__device__ __forceinline__ uint2 scan_item(const unsigned long long *count, long long i, long long n) {
    if (i >= n) return make_uint2(0u, 0u);
    const unsigned long long c = count[i];
    return make_uint2(PAD ? ((unsigned)c + 3u) & ~3u : (unsigned)c, (unsigned)(c >> 32));
}

// exclusive scan of one value per thread of a 256-thread block; total: the block's sum
__device__ __forceinline__ uint2 block_scan(uint2 v, uint2 &total) {
    __shared__ uint2 part[256];
    const int t = threadIdx.x;
    part[t] = v;
    __syncthreads();
    for (int s = 1; s < 256; s <<= 1) {
        const uint2 o = t >= s ? part[t - s] : make_uint2(0u, 0u);
        __syncthreads();
        part[t].x += o.x;
        part[t].y += o.y;
        __syncthreads();
    }
    total = part[255];
    const uint2 incl = part[t];
    __syncthreads();
    return make_uint2(incl.x - v.x, incl.y - v.y);
}

template <bool PAD>
__global__ __launch_bounds__(256) void k_scan_sums(const unsigned long long *__restrict__ count, long long n,
                                                   uint2 *__restrict__ sums) {
    uint2 v = make_uint2(0u, 0u), total;
    const long long i0 = blockIdx.x * (long long)kScanBlock + threadIdx.x * kScanItems;
    for (int u = 0; u < kScanItems; ++u) {
        const uint2 a = scan_item<PAD>(count, i0 + u, n);
        v.x += a.x;
        v.y += a.y;
    }
    block_scan(v, total);
    if (threadIdx.x == 0) sums[blockIdx.x] = total;
}

// one block: sums -> exclusive offsets, and the grand totals
__global__ __launch_bounds__(256) void k_scan_top(uint2 *__restrict__ sums, int nb, uint2 *__restrict__ grand) {
    uint2 carry = make_uint2(0u, 0u);
    for (int b0 = 0; b0 < nb; b0 += 256) {
        const int b = b0 + threadIdx.x;
        uint2 total;
        const uint2 e = block_scan(b < nb ? sums[b] : make_uint2(0u, 0u), total);
        if (b < nb) sums[b] = make_uint2(carry.x + e.x, carry.y + e.y);
        carry.x += total.x;
        carry.y += total.y;
    }
    if (threadIdx.x == 0) *grand = carry;
}

template <bool PAD>
__global__ __launch_bounds__(256) void k_scan_apply(const unsigned long long *__restrict__ count, long long n,
                                                    const uint2 *__restrict__ sums, unsigned *__restrict__ lo,
                                                    unsigned *__restrict__ hi) {
    uint2 a[kScanItems], v = make_uint2(0u, 0u), total;
    const long long i0 = blockIdx.x * (long long)kScanBlock + threadIdx.x * kScanItems;
    for (int u = 0; u < kScanItems; ++u) {
        a[u] = scan_item<PAD>(count, i0 + u, n);
        v.x += a[u].x;
        v.y += a[u].y;
    }
    uint2 e = block_scan(v, total);
    const uint2 s = sums[blockIdx.x];
    e.x += s.x;
    e.y += s.y;
    for (int u = 0; u < kScanItems; ++u) {
        if (i0 + u > n) break;
        lo[i0 + u] = e.x;   // entry n: the grand total
        hi[i0 + u] = e.y;
        e.x += a[u].x;
        e.y += a[u].y;
    }
}

// A scan of n counts: offsets of the low and high words in lo and hi (n + 1 entries each), the
// grand totals in `grand` (pinned host memory).
struct ScanArgs {
    const unsigned long long *count = nullptr;
    long long n = 0;
    unsigned *lo = nullptr, *hi = nullptr;
    uint2 *grand = nullptr;
};

// Up to kScanOne counts: one workgroup per scan, up to two scans, in one launch.  On the smallest
// grids a plan's time is that of its launches and allocations (see get_tileplan).
constexpr long long kScanOne = 8 * kScanBlock;

template <bool PAD>
__global__ __launch_bounds__(256) void k_scan_one(ScanArgs first, ScanArgs second) {
    const ScanArgs s = blockIdx.x ? second : first;
    uint2 carry = make_uint2(0u, 0u);
    for (long long b0 = 0; b0 <= s.n; b0 += kScanBlock) {
        uint2 a[kScanItems], v = make_uint2(0u, 0u), total;
        const long long i0 = b0 + threadIdx.x * kScanItems;
        for (int u = 0; u < kScanItems; ++u) {
            a[u] = scan_item<PAD>(s.count, i0 + u, s.n);
            v.x += a[u].x;
            v.y += a[u].y;
        }
        uint2 e = block_scan(v, total);
        e.x += carry.x;
        e.y += carry.y;
        for (int u = 0; u < kScanItems; ++u) {
            if (i0 + u > s.n) break;
            s.lo[i0 + u] = e.x;
            s.hi[i0 + u] = e.y;
            e.x += a[u].x;
            e.y += a[u].y;
        }
        carry.x += total.x;
        carry.y += total.y;
    }
    if (threadIdx.x == 0) *s.grand = carry;
}

long long scan_blocks(long long n) { return (n + kScanBlock) / kScanBlock; }   // cover entry n too

template <bool PAD>
void run_scan(Ctx &cx, const ScanArgs &s, uint2 *sums) {
    const int nsb = (int)scan_blocks(s.n);
    hipLaunchKernelGGL(k_scan_sums<PAD>, dim3(nsb), dim3(256), 0, cx.stream, s.count, s.n, sums);
    check_launch();
    hipLaunchKernelGGL(k_scan_top, dim3(1), dim3(256), 0, cx.stream, sums, nsb, s.grand);
    check_launch();
    hipLaunchKernelGGL(k_scan_apply<PAD>, dim3(nsb), dim3(256), 0, cx.stream, s.count, s.n, sums, s.lo, s.hi);
    check_launch();
}

// sums: scan_blocks(n) entries for the longer of the scans; second.n may be 0
template <bool PAD>
void run_scans(Ctx &cx, const ScanArgs &first, const ScanArgs &second, uint2 *sums) {
    if (std::max(first.n, second.n) <= kScanOne) {
        hipLaunchKernelGGL(k_scan_one<PAD>, dim3(second.n ? 2 : 1), dim3(256), 0, cx.stream, first, second);
        check_launch();
        return;
    }
    run_scan<PAD>(cx, first, sums);
    if (second.n) run_scan<PAD>(cx, second, sums);
}

// Wave per bucket: its runs in order of their first point number, written out as point ids.  A
// run's place is found against all others, so buckets of more than kRunsRanked runs (the tiles
// around the origin, where the planes of a scan cross) are left to k_run_order, by a list.
constexpr unsigned kRunsRanked = 256;
__global__ __launch_bounds__(256) void k_run_expand(const unsigned long long *__restrict__ count, long long nb,
                                                    const unsigned *__restrict__ off,
                                                    const unsigned *__restrict__ roff, const uint2 *__restrict__ runs,
                                                    unsigned *__restrict__ ids, unsigned *__restrict__ nlong,
                                                    unsigned *__restrict__ longer) {
    const int lane = threadIdx.x & 63;
    for (long long b = blockIdx.x * 4ll + (threadIdx.x >> 6); b < nb; b += gridDim.x * 4ll) {
        const unsigned long long c = count[b];
        const unsigned n = (unsigned)(c >> 32), npts = (unsigned)c;
        if (n == 0) continue;
        const unsigned base = off[b];
        const unsigned pad = (4u - (npts & 3u)) & 3u;
        if ((unsigned)lane < pad) ids[base + npts + lane] = kNoPoint;
        if (n > kRunsRanked) {
            if (lane == 0) longer[atomicAdd(nlong, 1u)] = (unsigned)b;
            continue;
        }
        const uint2 *rb = runs + roff[b];
        for (unsigned i0 = 0; i0 < n; i0 += 64) {
            const uint2 mine = i0 + lane < n ? rb[i0 + lane] : make_uint2(kNoPoint, 0u);
            unsigned pos = 0;
            for (unsigned j0 = 0; j0 < n; j0 += 64) {
                const uint2 o = j0 + lane < n ? rb[j0 + lane] : make_uint2(kNoPoint, 0u);
                const int m = (int)min(64u, n - j0);
                for (int t = 0; t < m; ++t) {
                    const unsigned kt = (unsigned)__builtin_amdgcn_readlane((int)o.x, t);
                    const unsigned lt = (unsigned)__builtin_amdgcn_readlane((int)o.y, t);
                    pos += kt < mine.x ? lt : 0u;
                }
            }
            if (i0 + lane < n)
                for (unsigned m = 0; m < mine.y; ++m) ids[base + pos + m] = mine.x + m;
        }
    }
}

// Workgroup per listed bucket: its runs grouped in tmp by kRunBins equal ranges of point numbers
// (about a projection each), a run's place then found within its range.  One wave ranking a bucket's
// runs against all others took most of a first adjoint: (127, 31, 127) / 181 x 181 with varying tilt,
// 120 projections 1148 -> 954 us, 720 projections 11.7 -> 3.1 ms; (89, 21, 89) / 89 x 89 x 4000 14.7 ->
// 2.5 ms.
constexpr int kRunBins = 8 * 256;
__global__ __launch_bounds__(256) void k_run_order(const unsigned long long *__restrict__ count,
                                                   const unsigned *__restrict__ off,
                                                   const unsigned *__restrict__ roff, const uint2 *__restrict__ runs,
                                                   uint2 *tmp, unsigned span, unsigned *__restrict__ ids,
                                                   const unsigned *__restrict__ nlong,
                                                   const unsigned *__restrict__ longer) {
    __shared__ unsigned cur[kRunBins], pts[kRunBins];   // runs, and points, before a range
    const unsigned t = threadIdx.x, nl = *nlong;
    for (unsigned i = blockIdx.x; i < nl; i += gridDim.x) {
        const unsigned b = longer[i], n = (unsigned)(count[b] >> 32), base = off[b];
        const uint2 *rb = runs + roff[b];
        uint2 *tb = tmp + roff[b];
        for (unsigned q = t; q < kRunBins; q += 256) cur[q] = pts[q] = 0u;
        __syncthreads();
        for (unsigned r = t; r < n; r += 256) {
            const uint2 run = rb[r];
            atomicAdd(&cur[run.x / span], 1u);
            atomicAdd(&pts[run.x / span], run.y);
        }
        __syncthreads();
        uint2 mine[8], sum = make_uint2(0u, 0u), total;
#pragma unroll
        for (int u = 0; u < 8; ++u) {
            mine[u] = make_uint2(cur[8 * t + u], pts[8 * t + u]);
            sum.x += mine[u].x;
            sum.y += mine[u].y;
        }
        uint2 at = block_scan(sum, total);
#pragma unroll
        for (int u = 0; u < 8; ++u) {
            cur[8 * t + u] = at.x;
            pts[8 * t + u] = at.y;
            at.x += mine[u].x;
            at.y += mine[u].y;
        }
        __syncthreads();
        for (unsigned r = t; r < n; r += 256) {
            const uint2 run = rb[r];
            tb[atomicAdd(&cur[run.x / span], 1u)] = run;
        }
        __syncthreads();   // cur[q] is now the end of range q
        for (unsigned r = t; r < n; r += 256) {
            const uint2 run = tb[r];
            const unsigned q = run.x / span, e = cur[q];
            unsigned pos = base + pts[q];
            for (unsigned o = q ? cur[q - 1] : 0u; o < e; ++o) pos += tb[o].x < run.x ? tb[o].y : 0u;
            for (unsigned m = 0; m < run.y; ++m) ids[pos + m] = run.x + m;
        }
        __syncthreads();
    }
}

// Jobs of one tile: its points, in order, cut into equal parts of at most `most` (a row may be
// cut too).  A tile that would have more than `many` jobs, as in small volumes under many points,
// takes sqrt(n / deep) of them, at least `many`: a cell's sum goes over the tile's jobs one after
// another, which then outweighs a job's own chain (`deep`: a job's time in the sum over a point's
// in a job).  Whole adjoints in us, with jobs of `most` and so: (9, 5, 11) / 200 x 200 x 200 4219
// and 858, (22, 22, 3) / 349 x 9 x 250 at width 10 952 and 392, first-cell slots (5, 32, 32) / 52 x
// 203 x 120 535 and 395; with a quarter and four times `deep` the first takes 1100 and 997.  With
// 24, 12, 8 and 6 for `many` first-cell slots take 0.870, 0.854, 0.848 and 0.847 of the 3-D bins'
// time over 90 small grids.
// emit(i, beg, end, r0, r1): part i holds ids [beg, end) of slots [r0, r1).
constexpr unsigned kDeep = 24, kDeepDirect = 8;
template <class F>
__device__ __forceinline__ void tile_jobs(const unsigned *__restrict__ o, int nrho, unsigned most, unsigned many,
                                          float deep, F emit) {
    const unsigned first = o[0], n = o[nrho] - first;
    if (n == 0) return;
    unsigned parts = (n + most - 1) / most;
    if (parts > many) parts = max(many, min(parts, (unsigned)sqrtf((float)n / deep)));
    const unsigned step = ((n + parts - 1) / parts + 3u) & ~3u;
    auto below = [&](unsigned v) {   // slots whose points start at or before v
        int lo = 0, hi = nrho;
        while (lo < hi) {
            const int m = (lo + hi) / 2;
            if (o[m] <= v) lo = m + 1;
            else hi = m;
        }
        return lo;
    };
    for (unsigned i = 0; i * step < n; ++i) {
        const unsigned beg = first + i * step, end = min(first + n, beg + step);
        emit(i, beg, end, below(beg) - 1, below(end - 1));
    }
}

// Tiles of one interpolation unit, side by side in x: they share a block of 16 cells.
constexpr int kUnitTiles = 2;

// Interpolation jobs: a job takes whole row slots [r0, r1) of a unit, or part `part` of `parts`
// of one slot that alone holds more than a job.  The unit's wave holds 64 slots' sizes in its
// lanes and walks the non-empty ones.
template <class F>
__device__ __forceinline__ void unit_jobs(const unsigned *__restrict__ off, unsigned u, const TileGeom &tg,
                                          unsigned most, F emit) {
    const int ut = kUnitTiles, lane = threadIdx.x & 63;
    const unsigned nux = (unsigned)(tg.ntx + ut - 1) / (unsigned)ut, uz = u / nux, ux = u - uz * nux;
    const unsigned *o = off + (long long)(uz * (unsigned)tg.ntx + (unsigned)ut * ux) * tg.nrho;
    const int tiles = min(ut, tg.ntx - ut * (int)ux);
    int r0 = -1, last = 0;   // last: one past the last slot with points
    unsigned held = 0;
    for (int rb = 0; rb < tg.nrho; rb += 64) {
        unsigned size = 0;
        if (rb + lane < tg.nrho)
            for (int t = 0; t < tiles; ++t) size += o[t * tg.nrho + rb + lane + 1] - o[t * tg.nrho + rb + lane];
        for (unsigned long long mask = __ballot(size > 0); mask; mask &= mask - 1ull) {
            const int i = __builtin_ctzll(mask), r = rb + i;
            const unsigned n = (unsigned)__builtin_amdgcn_readlane((int)size, i);
            if (r0 >= 0 && held + n > most) {
                emit(r0, last, 0u, 1u);
                r0 = -1;
                held = 0;
            }
            if (n > most) {
                const unsigned parts = (n + most - 1) / most;
                for (unsigned k = 0; k < parts; ++k) emit(r, r + 1, k, parts);
                continue;
            }
            if (r0 < 0) r0 = r;
            held += n;
            last = r + 1;
        }
    }
    if (r0 >= 0) emit(r0, last, 0u, 1u);
}

// How a plan's points are shared out.  Workgroups of one wave: the first take 64 tiles' spread
// jobs, a thread each, the others one unit's interpolation jobs (nunits 0: none).
struct ShareArgs {
    const unsigned *off;
    const RowY *rowy;
    unsigned jmost, umost, nunits, many;
    float deep;
};
unsigned tile_blocks(const TileGeom &tg) { return (tg.ntiles + 63) / 64; }

// jcount[tile]: planes its jobs record (low word), jobs (high word); ucount[unit]: its jobs
__global__ __launch_bounds__(64) void k_share_count(ShareArgs A, TileGeom tg, unsigned tblocks,
                                                    unsigned long long *__restrict__ jcount,
                                                    unsigned long long *__restrict__ ucount) {
    if (blockIdx.x >= tblocks) {
        const unsigned u = blockIdx.x - tblocks;
        unsigned jobs = 0;
        unit_jobs(A.off, u, tg, A.umost, [&](int, int, unsigned, unsigned) { ++jobs; });
        if (threadIdx.x == 0) ucount[u] = jobs;
        return;
    }
    const unsigned t = blockIdx.x * 64u + threadIdx.x;
    if (t >= tg.ntiles) return;
    unsigned planes = 0, jobs = 0;
    tile_jobs(A.off + (long long)t * tg.nrho, tg.nrho, A.jmost, A.many, A.deep, [&](unsigned, unsigned, unsigned, int r0, int r1) {
        planes += (unsigned)(A.rowy[r1 - 1].iy + tg.W - A.rowy[r0].iy);
        ++jobs;
    });
    jcount[t] = ((unsigned long long)jobs << 32) | planes;
}

__global__ __launch_bounds__(64) void k_share_emit(ShareArgs A, TileGeom tg, unsigned tblocks,
                                                   const unsigned *__restrict__ plane0,
                                                   const unsigned *__restrict__ job0,
                                                   const unsigned *__restrict__ ujob0, TileJob *__restrict__ jobs,
                                                   UnitJob *__restrict__ ujobs) {
    if (blockIdx.x >= tblocks) {
        const unsigned u = blockIdx.x - tblocks;
        unsigned j = ujob0[u];
        unit_jobs(A.off, u, tg, A.umost, [&](int r0, int r1, unsigned part, unsigned parts) {
            if (threadIdx.x == 0) ujobs[j] = UnitJob{u, r0, r1, part, parts};
            ++j;
        });
        return;
    }
    const unsigned t = blockIdx.x * 64u + threadIdx.x;
    if (t >= tg.ntiles) return;
    unsigned plane = plane0[t];
    tile_jobs(A.off + (long long)t * tg.nrho, tg.nrho, A.jmost, A.many, A.deep,
              [&](unsigned i, unsigned beg, unsigned end, int r0, int r1) {
                  TileJob j;
                  j.tile = t;
                  j.beg = beg;
                  j.end = end;
                  j.r0 = r0;
                  j.r1 = r1;
                  j.y0 = A.rowy[r0].iy;
                  j.np = A.rowy[r1 - 1].iy + tg.W - j.y0;
                  j.plane = plane;
                  j.yw = j.y0 % tg.nfy;
                  if (j.yw < 0) j.yw += tg.nfy;
                  plane += (unsigned)j.np;
                  jobs[job0[t] + i] = j;
              });
}

// ------------------------------------------------------------------ shared by both kernels
// Walk over the non-empty row slots of a job: 64 slots' sizes sit in the lanes.
struct SlotWalk {
    const unsigned *off;   // the tile's first entry
    unsigned beg, end;     // the job's ids
    int next0, r1, base;   // first slot of the next block of 64; end; first slot of this block
    int groups;            // lane: groups of 4 points of slot base + lane
    unsigned long long mask;
    __device__ __forceinline__ void start(const unsigned *tile_off, const TileJob &j) {
        off = tile_off;
        beg = j.beg;
        end = j.end;
        next0 = j.r0;
        r1 = j.r1;
        base = j.r0;
        groups = 0;
        mask = 0ull;
    }
    // the next non-empty slot and its number of groups; there is one
    __device__ __forceinline__ int step(int lane, int &left) {
        while (mask == 0ull && next0 < r1) {
            base = next0;
            next0 += 64;
            const int r = base + lane;
            groups = r < r1 ? (int)((min(off[r + 1], end) - max(off[r], beg)) >> 2) : 0;
            mask = __ballot(groups > 0);
        }
        const int t = mask ? __builtin_ctzll(mask) : 0;
        mask &= mask - 1ull;
        left = __builtin_amdgcn_readlane(groups, t);
        return base + t;
    }
};

// The coordinate of one axis of a point, (qX u + qY v) s, as in point_coords.
__device__ __forceinline__ double axis_coord(double qX, double qY, double u, double v, double s) {
#pragma clang fp contract(off)
    return (qX * u + qY * v) * s;
}
__device__ __forceinline__ double line_coord(double qY, double v, double s) {
#pragma clang fp contract(off)
    return (qY * v) * s;
}
__device__ __forceinline__ double detector_coord(int i, double centre, double step) {
#pragma clang fp contract(off)
    return ((double)i - centre) * step;
}

struct TileArgs {
    long long S;
    float b2;   // beta log2 e
    PointFrame fr;
    FastDiv fH, fC;
};

// Orders a wave's LDS accesses before those that follow, across its lanes: the hardware keeps a
// wave's order by itself, so this costs no instruction, but the compiler must not move them.
__device__ __forceinline__ void wave_lds_order() {
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
}

// ------------------------------------------------------------------ spreading
// One wave per (job, component group).  Batches of 32 points are staged in LDS by
// lane pairs: lane p < 32 evaluates the z weights of point p and writes wz (re v, im v) into
// row p of A (32 entries (z, c), zero outside the stamp), lane p + 32 the x weights and
// writes wx d_i into row p of B (entries (x, i)); the next batch's points are loaded
// meanwhile.  Two points then take one v_mfma_f32_32x32x2_f32, rows (z, c) by columns (x, i).
// After a row's points the block goes into the window of the W planes that later rows can
// still reach, in registers; a plane that no later row reaches is written to the record.
constexpr int kSPts = 32;                       // points per batch
constexpr int kSRow = 34;                       // staged floats per row: 32, padded for the lanes' writes
constexpr int kSHalf = (kSPts + 4) * kSRow;     // A, then B; 4 rows more are read ahead, never used

template <int W, int NI, bool DIRECT>
__global__ __launch_bounds__(64, spread_waves(W)) void k_tile_spread(
    float2 *__restrict__ rec, const float2 *__restrict__ c, const TileGeo *__restrict__ geo,
    const unsigned *__restrict__ off, const unsigned *__restrict__ ids, const RowY *__restrict__ rowy,
    const TileJob *__restrict__ jobs, TileArgs A, TileGeom tg, unsigned plane0, int paired) {
    __shared__ __attribute__((aligned(16))) float st_[2 * kSHalf];
    __shared__ float sy[DIRECT ? (kSPts + 4) * W : 1];   // [point][plane]
    constexpr int kGroups = 3 / NI;
    const unsigned jn = blockIdx.x / kGroups;
    const int grp = (int)(blockIdx.x - jn * kGroups);
    const TileJob job = jobs[jn];
    const unsigned tile = job.tile, beg = job.beg, end = job.end;
    const unsigned *toff = off + (long long)tile * tg.nrho;
    const int lane = threadIdx.x, pt = lane & 31, hi = lane >> 5;
    const bool zl = lane < 32;
    const int npts = (int)(end - beg), nbat = (npts + kSPts - 1) / kSPts;
    const unsigned tz = tg.fntx.div(tile), tx = tile - tz * (unsigned)tg.ntx;
    const int org = zl ? (int)tz * tg.Tz : (int)tx * tg.Tx;      // the axis this lane places points on
    const int nf = zl ? tg.nfz : tg.nfx, lmax = (zl ? kBlock : kXCells<NI>) - W;
    const double sc = zl ? A.fr.sz : A.fr.sx, rnf = zl ? A.fr.rz : A.fr.rx;
    const double dnf = (double)nf;

    struct Pt {
        unsigned gid;
        double u, v, vy;
        float q[4];   // z lanes: c(q), c(-q); x lanes: d_i
    };
    auto load_id = [&](int bat) {
        const int i = bat * kSPts + pt;
        return i < npts ? ids[beg + i] : kNoPoint;
    };
    auto load_pt = [&](unsigned gid, Pt &t) {
        t.gid = gid;
        if (gid == kNoPoint) return;
        const unsigned p = A.fH.div(gid);
        const TileGeo *g = geo + p;
        const double2 uv = *reinterpret_cast<const double2 *>(zl ? &g->uz : &g->ux);
        t.u = uv.x;
        t.v = uv.y;
        if (DIRECT) t.vy = g->vy;
        if (zl) {
            const long long idx = gid - p * A.fH.d, mir = A.S - 1 - idx;
            const float2 *pc = c + (long long)(paired ? p & ~1u : p) * A.S;
            const float2 a = pc[idx], b = pc[mir];
            t.q[0] = a.x;
            t.q[1] = a.y;
            t.q[2] = b.x;
            t.q[3] = b.y;
        } else {
            const float4 d = *reinterpret_cast<const float4 *>(g->d);
            t.q[0] = d.x;
            t.q[1] = d.y;
            t.q[2] = d.z;
        }
    };
    auto stage = [&](const Pt &t) {
        const bool have = t.gid != kNoPoint;
        const unsigned gid = have ? t.gid : 0u;
        const unsigned p = A.fH.div(gid), idx = gid - p * A.fH.d;
        const unsigned j = A.fC.div(idx), k = idx - j * A.fC.d;
        const double qY = detector_coord((int)j, A.fr.j0, A.fr.dY);
        const double qX = detector_coord((int)k, A.fr.k0, A.fr.dX);
        double x = axis_coord(qX, qY, t.u, t.v, sc);
        const int i = first_cell(x, dnf, rnf, W);
        float w[W];
        es_weights2<W>(x, i, A.b2, w);
        // i - org folded into the tile (i is in [-W / 2, nf]).  Inside it by the plan (same
        // arithmetic); the clamp only bounds the LDS index.
        int l = i - org;
        l += l < 0 ? nf : 0;
        l -= l >= nf ? nf : 0;
        l = min(max(l, 0), lmax);
        // the wave clears the batch and then writes the stamps
        wave_lds_order();   // after the last batch's reads
        const float4 z4 = make_float4(0.f, 0.f, 0.f, 0.f);
#pragma unroll
        for (int q = 0; q < (2 * kSHalf + 255) / 256; ++q)
            if (q * 256 + lane * 4 < 2 * kSHalf) *reinterpret_cast<float4 *>(st_ + q * 256 + lane * 4) = z4;
        wave_lds_order();
        if (have) {
            if (zl) {
                const float2 v = half_point_value(make_float2(t.q[0], t.q[1]), make_float2(t.q[2], t.q[3]), p, idx,
                                                  A.S, paired);
                float *row = st_ + pt * kSRow + 2 * l;
#pragma unroll
                for (int m = 0; m < W; ++m)
                    *reinterpret_cast<float2 *>(row + 2 * m) = make_float2(w[m] * v.x, w[m] * v.y);
            } else {
                float *row = st_ + kSHalf + pt * kSRow + NI * l;
                const float d[3] = {NI == 1 ? (grp == 0 ? t.q[0] : grp == 1 ? t.q[1] : t.q[2]) : t.q[0], t.q[1], t.q[2]};
#pragma unroll
                for (int m = 0; m < W; ++m)
#pragma unroll
                    for (int q = 0; q < NI; ++q) row[NI * m + q] = w[m] * d[q];
            }
        }
        if constexpr (DIRECT) {
            double y = line_coord(qY, t.vy, A.fr.sy);
            const int iy = first_cell(y, (double)tg.nfy, A.fr.ry, W);
            float wy[W];
            es_weights2<W>(y, iy, A.b2, wy);
            if (zl) {
#pragma unroll
                for (int m = 0; m < W; ++m) sy[pt * W + m] = have ? wy[m] : 0.f;
            }
        }
        wave_lds_order();   // before other lanes read the stamps
    };

    // block of the open row, and the window of W planes from yb
    struct Plane {
        float f[16];
        __device__ __forceinline__ float &operator[](int r) { return f[r]; }
    };
    std::conditional_t<DIRECT, v16f, Plane> win[W];   // matrix accumulators, or plain sums
    v16f h;
#pragma unroll
    for (int r = 0; r < 16; ++r) {
        h[r] = 0.f;
#pragma unroll
        for (int b = 0; b < W; ++b) win[b][r] = 0.f;
    }
    int yb = job.y0;
    // the window's first plane to the record, the window on by one.  Lane (hi, n) register r
    // holds row 8 (r / 4) + 4 hi + r % 4 = 2 z + c of column n.
    auto flush = [&]() {
        float2 *dst = rec + ((long long)(job.plane - plane0 + (unsigned)(yb - job.y0)) * kGroups + grp) * kRec +
                      2 * hi * 32 + pt;
#pragma unroll
        for (int t = 0; t < 8; ++t) dst[(4 * (t >> 1) + (t & 1)) * 32] = make_float2(win[0][2 * t], win[0][2 * t + 1]);
#pragma unroll
        for (int b = 0; b + 1 < W; ++b) win[b] = win[b + 1];
#pragma unroll
        for (int r = 0; r < 16; ++r) win[W - 1][r] = 0.f;
        ++yb;
    };

    SlotWalk walk;
    walk.start(toff, job);
    // groups of 4 points: of the open row, of the next row, of the rows not found yet
    int left = 0, next_left = 0, todo = npts >> 2;
    RowY ry{}, rn{};   // the next row's y weights are loaded while the open row's points go through
    auto find_row = [&]() {
        const int slot = walk.step(lane, next_left);
        todo -= next_left;
        rn = rowy[slot];
    };
    auto open_row = [&]() {
        if constexpr (DIRECT) {
            const int slot = walk.step(lane, left);
            todo -= left;
            while (yb < slot) flush();
        } else {
            ry = rn;
            left = next_left;
            next_left = 0;
            if (todo > 0) find_row();
        }
    };
    auto close_row = [&]() {
        if constexpr (!DIRECT) {
            while (yb < ry.iy) flush();
#pragma unroll
            for (int b = 0; b < W; ++b)
#pragma unroll
                for (int r = 0; r < 16; ++r) win[b][r] += ry.w[b] * h[r];
#pragma unroll
            for (int r = 0; r < 16; ++r) h[r] = 0.f;
        }
        if (DIRECT ? todo > 0 : next_left > 0) open_row();
    };

    Pt cur{};
    load_pt(load_id(0), cur);
    unsigned id1 = load_id(1);
    if constexpr (!DIRECT) find_row();
    open_row();
    for (int k = 0; k < nbat; ++k) {
        stage(cur);
        load_pt(id1, cur);
        id1 = load_id(k + 2);
        const int ng = min(kSPts / 4, (npts - k * kSPts) >> 2);
        const float *pa = st_ + hi * kSRow + pt, *pb = pa + kSHalf;
        float a0 = pa[0], a1 = pa[2 * kSRow], b0 = pb[0], b1 = pb[2 * kSRow];
        for (int g = 0; g < ng; ++g) {
            pa += 4 * kSRow;
            pb += 4 * kSRow;
            if constexpr (DIRECT) {
                const float ca0 = a0, ca1 = a1, cb0 = b0, cb1 = b1;
                a0 = pa[0];
                a1 = pa[2 * kSRow];
                b0 = pb[0];
                b1 = pb[2 * kSRow];
                const float *wy = sy + (4 * g + hi) * W;
#pragma unroll
                for (int b = 0; b < W; ++b) {
                    win[b] = __builtin_amdgcn_mfma_f32_32x32x2f32(ca0 * wy[b], cb0, win[b], 0, 0, 0);
                    win[b] = __builtin_amdgcn_mfma_f32_32x32x2f32(ca1 * wy[2 * W + b], cb1, win[b], 0, 0, 0);
                }
            } else {
                h = __builtin_amdgcn_mfma_f32_32x32x2f32(a0, b0, h, 0, 0, 0);
                a0 = pa[0];
                b0 = pb[0];
                h = __builtin_amdgcn_mfma_f32_32x32x2f32(a1, b1, h, 0, 0, 0);
                a1 = pa[2 * kSRow];
                b1 = pb[2 * kSRow];
            }
            if (--left == 0) close_row();
        }
    }
    while (yb < job.y0 + job.np) flush();
}

// Adds the jobs' records into the fine grid: every cell takes the blocks that reach it (its
// own tile's and those of the tiles before it along z and x), in the order of the maps and of
// a tile's jobs.  A thread owns one value (z, x, component) of kMergePlanes consecutive
// planes, so that as many loads are in flight for each job it looks up.
constexpr int kMergePlanes = 8;

template <int NI>
__global__ __launch_bounds__(256) void k_tile_merge(float2 *__restrict__ fine, const float2 *__restrict__ rec,
                                                    const TileJob *__restrict__ jobs,
                                                    const unsigned *__restrict__ job0, unsigned jfirst, unsigned jlast,
                                                    unsigned plane0, const int *__restrict__ zmap,
                                                    const int *__restrict__ xmap, TileGeom tg, int ylo, int ly,
                                                    int add) {
    const unsigned nxb = (unsigned)(3 * tg.nfx + 255) / 256u;   // workgroups: [plane chunk][z][x block]
    const unsigned row = blockIdx.x / nxb, chunk = row / (unsigned)tg.nfz;
    const int e = (int)((blockIdx.x - row * nxb) * 256 + threadIdx.x);
    if (e >= 3 * tg.nfx) return;
    const int x = (int)((unsigned)e / 3u), m = e - 3 * x;
    const int z = (int)(row - chunk * (unsigned)tg.nfz);
    const int yl0 = (int)chunk * kMergePlanes;
    int y = ylo + yl0;
    if (y >= tg.nfy) y -= tg.nfy;
    float2 acc[kMergePlanes];
#pragma unroll
    for (int u = 0; u < kMergePlanes; ++u) acc[u] = make_float2(0.f, 0.f);
    const int *ze = zmap + tg.nfz + 1, *xe = xmap + tg.nfx + 1;
    for (int iz = zmap[z]; iz < zmap[z + 1]; ++iz) {
        const unsigned trow = (unsigned)ze[2 * iz] * (unsigned)tg.ntx;
        const int zc = ze[2 * iz + 1] * 32;
        for (int ix = xmap[x]; ix < xmap[x + 1]; ++ix) {
            const unsigned tile = trow + (unsigned)xe[2 * ix];
            const int cell = zc + (NI == 3 ? 3 * xe[2 * ix + 1] + m : m * kRec + xe[2 * ix + 1]);
            const unsigned j1 = min(job0[tile + 1], jlast);
            for (unsigned j = max(job0[tile], jfirst); j < j1; ++j) {
                const int np = jobs[j].np;
                int d = y - jobs[j].yw;   // the job's plane at y, modulo the period
                const float2 *r = rec + (long long)(jobs[j].plane - plane0) * ((3 / NI) * kRec) + cell;
                float2 v[kMergePlanes];
#pragma unroll
                for (int u = 0; u < kMergePlanes; ++u) {
                    if (d < 0) d += tg.nfy;
                    if (d >= tg.nfy) d -= tg.nfy;
                    v[u] = make_float2(0.f, 0.f);
                    if (d < np) v[u] = r[(long long)d * ((3 / NI) * kRec)];
                    if (d + tg.nfy < np) v[u] = cadd(v[u], r[(long long)(d + tg.nfy) * ((3 / NI) * kRec)]);
                    ++d;
                }
#pragma unroll
                for (int u = 0; u < kMergePlanes; ++u) acc[u] = cadd(acc[u], v[u]);
            }
        }
    }
#pragma unroll
    for (int u = 0; u < kMergePlanes; ++u) {
        if (yl0 + u < ly) {
            float2 *dst = fine + ((long long)z * tg.nfy + y) * tg.nfx * 3 + e;
            *dst = add ? cadd(*dst, acc[u]) : acc[u];
        }
        if (++y == tg.nfy) y = 0;
    }
}

// ------------------------------------------------------------------ interpolation
// Type 2 of a shared-tilt grid: G(z, x) = sum_b wy[b] F(z, iy + b, x) for each row, then W^2
// taps per point.  Workgroup per unit job.  A thread owns one cell of the unit's 16 x 16
// block and keeps the W planes around the rows in registers (one more is loaded ahead); G of
// several rows goes to LDS, and then the threads take those rows' points, one each.
// Bound by LDS reads (108 of 8 bytes per point at W = 6; the banks collide 2.6-fold) over
// vector work (1.4 ms of 2.5).  Before, G of all rows went through memory (1.17 ms to write it,
// 2.04 ms to read and interpolate): 3.21 -> 2.46 ms per dataset at (359, 71, 359) / 615,
// (179, 43, 179) / 305 0.45 -> 0.36, (89, 21, 89) / 89 0.047 -> 0.040.  The
// same products on the fp32 matrix unit (16 x 16 blocks, 16 points at a time) took 4.5 ms.
constexpr int kUnitThreads = 256;
constexpr int kUnitRows = 8;                               // most rows staged at a time
// Staged cells per block row.  The points of a line step through cells in every direction, so
// a wave's reads fall on banks at random; measured at (359, 71, 359) / 615, per launch: 16 cells
// (rows on the same banks) 4.18 ms, 17: 2.81, 18: 2.51, 19: 2.41, 21: 2.55.
constexpr int kUnitRow = 19;
constexpr int kUnitCells = kBlock * kUnitRow;              // staged cells per detector row

template <int W>
__global__ __launch_bounds__(kUnitThreads, 4) void k_tile_interp(
    const float2 *__restrict__ fine, float2 *__restrict__ c, const TileGeo *__restrict__ geo,
    const unsigned *__restrict__ off, const unsigned *__restrict__ ids, const RowY *__restrict__ rowy,
    const UnitJob *__restrict__ jobs, TileArgs A, TileGeom tg, int nr) {
    extern __shared__ float2 gs[];   // [nr][kUnitCells][3]
    constexpr int kRowF = (W + 4) / 4 * 4;                         // floats per staged row: w[W], iy
    __shared__ __attribute__((aligned(16))) float rw[2][kUnitRows * kRowF];   // y weights of a step's rows
    constexpr int UT = kUnitTiles;
    const UnitJob job = jobs[blockIdx.x];
    const unsigned nux = (unsigned)(tg.ntx + UT - 1) / (unsigned)UT, uz = job.unit / nux, ux = job.unit - uz * nux;
    const unsigned *o[UT];   // the unit's tiles (a missing one: no points)
    int live[UT];
#pragma unroll
    for (int t = 0; t < UT; ++t) {
        live[t] = UT * (int)ux + t < tg.ntx ? 1 : 0;
        o[t] = off + (long long)(uz * (unsigned)tg.ntx + (unsigned)UT * ux + (live[t] ? t : 0)) * tg.nrho;
    }
    const int oz = (int)uz * tg.Tz, ox = UT * (int)ux * tg.Tx;
    const int tid = threadIdx.x, cz = tid >> 4, cx = tid & 15;

    float2 win[W][3], ahead[3];
    int yb = rowy[job.r0].iy, yw = yb % tg.nfy;   // first plane of the window; the next to load (wrapped)
    if (yw < 0) yw += tg.nfy;
    const float2 *cell;
    {
        int z = oz + cz, x = ox + cx;
        while (z >= tg.nfz) z -= tg.nfz;
        while (x >= tg.nfx) x -= tg.nfx;
        cell = fine + ((long long)z * tg.nfy * tg.nfx + x) * 3;
    }
    auto load_plane = [&](float2 *dst) {
        const float2 *src = cell + (long long)yw * tg.nfx * 3;
#pragma unroll
        for (int m = 0; m < 3; ++m) dst[m] = src[m];
        if (++yw == tg.nfy) yw = 0;
    };
#pragma unroll
    for (int b = 0; b < W; ++b) load_plane(win[b]);
    load_plane(ahead);

    // thread (row, float) of a step's rows
    auto load_row = [&](int r) {
        const int q = tid / kRowF, f = tid - q * kRowF;
        if (q >= nr || r + q >= job.r1) return 0.f;
        const RowY *y = rowy + (r + q);
        return f < W ? y->w[f] : __int_as_float(y->iy);
    };
    if (tid < nr * kRowF) rw[0][tid] = load_row(job.r0);
    __syncthreads();
    const double dnz = (double)tg.nfz, dnx = (double)tg.nfx;
    int buf = 0;
    for (int r = job.r0; r < job.r1; r += nr, buf ^= 1) {
        const int rn = min(r + nr, job.r1);
        unsigned first[UT], upto[UT], n = 0;   // tile t holds numbers [upto[t - 1], upto[t])
#pragma unroll
        for (int t = 0; t < UT; ++t) {
            first[t] = o[t][r] - n;
            n += live[t] ? o[t][rn] - o[t][r] : 0u;
            upto[t] = n;
        }
        const unsigned lo = (unsigned)((unsigned long long)n * job.part / job.parts),
                       hi = (unsigned)((unsigned long long)n * (job.part + 1) / job.parts);
        auto load_id = [&](unsigned i) {
            if (i >= hi) return kNoPoint;
            unsigned f = first[0];
#pragma unroll
            for (int t = 1; t < UT; ++t) f = i >= upto[t - 1] ? first[t] : f;
            return ids[f + i];
        };
        unsigned gid = load_id(lo + tid);
        const float nrow = tid < nr * kRowF ? load_row(r + nr) : 0.f;
        for (int q = n ? r : rn; q < rn; ++q) {
            float w[kRowF];
#pragma unroll
            for (int f = 0; f < kRowF; f += 4)
                *reinterpret_cast<float4 *>(w + f) = *reinterpret_cast<const float4 *>(&rw[buf][(q - r) * kRowF + f]);
            unsigned held = 0;
#pragma unroll
            for (int t = 0; t < UT; ++t) held += live[t] ? o[t][q + 1] - o[t][q] : 0u;
            if (held == 0) continue;
            const int iy = __builtin_amdgcn_readfirstlane(__float_as_int(w[W]));
            while (yb < iy) {
#pragma unroll
                for (int m = 0; m < 3; ++m) {
#pragma unroll
                    for (int b = 0; b + 1 < W; ++b) win[b][m] = win[b + 1][m];
                    win[W - 1][m] = ahead[m];
                }
                ++yb;
                load_plane(ahead);
            }
            float2 *g = gs + (size_t)((q - r) * kUnitCells + cz * kUnitRow + cx) * 3;
#pragma unroll
            for (int m = 0; m < 3; ++m) {
                float2 s = make_float2(0.f, 0.f);
#pragma unroll
                for (int b = 0; b < W; ++b) {
                    s.x += w[b] * win[b][m].x;
                    s.y += w[b] * win[b][m].y;
                }
                g[m] = s;
            }
        }
        if (tid < nr * kRowF) rw[buf ^ 1][tid] = nrow;
        __syncthreads();
        for (unsigned i = lo + tid; i < hi; i += kUnitThreads) {
            if (i >= lo + kUnitThreads) gid = load_id(i);
            if (gid == kNoPoint) continue;
            const unsigned p = A.fH.div(gid), idx = gid - p * A.fH.d;
            const unsigned j = A.fC.div(idx), k = idx - j * A.fC.d;
            const TileGeo *ge = geo + p;
            const double2 gz = *reinterpret_cast<const double2 *>(&ge->uz), gx = *reinterpret_cast<const double2 *>(&ge->ux);
            const float4 d = *reinterpret_cast<const float4 *>(ge->d);
            const double qY = detector_coord((int)j, A.fr.j0, A.fr.dY), qX = detector_coord((int)k, A.fr.k0, A.fr.dX);
            double tz = axis_coord(qX, qY, gz.x, gz.y, A.fr.sz), tx = axis_coord(qX, qY, gx.x, gx.y, A.fr.sx);
            const int iz = first_cell(tz, dnz, A.fr.rz, W), ix = first_cell(tx, dnx, A.fr.rx, W);
            float wz[W], wx[W];
            es_weights2<W>(tz, iz, A.b2, wz);
            es_weights2<W>(tx, ix, A.b2, wx);
            // folded into the unit; inside it by the plan, the clamps only bound the LDS index
            int lz = iz - oz, lx = ix - ox;
            lz += lz < 0 ? tg.nfz : 0;
            lz -= lz >= tg.nfz ? tg.nfz : 0;
            lx += lx < 0 ? tg.nfx : 0;
            lx -= lx >= tg.nfx ? tg.nfx : 0;
            lz = min(max(lz, 0), kBlock - W);
            lx = min(max(lx, 0), kBlock - W);
            const int slot = tg.dir > 0 ? (int)j : tg.Jn - 1 - (int)j;
            const int row = min(max(slot - r, 0), nr - 1);
            const float2 *g = gs + (size_t)(row * kUnitCells + lz * kUnitRow + lx) * 3;
            float2 acc[3];
#pragma unroll
            for (int m = 0; m < 3; ++m) acc[m] = make_float2(0.f, 0.f);
#pragma unroll
            for (int a = 0; a < W; ++a) {
                float2 ra[3];
#pragma unroll
                for (int m = 0; m < 3; ++m) ra[m] = make_float2(0.f, 0.f);
#pragma unroll
                for (int e = 0; e < W; ++e)
#pragma unroll
                    for (int m = 0; m < 3; ++m) {
                        const float2 v = g[(a * kUnitRow + e) * 3 + m];
                        ra[m].x += v.x * wx[e];
                        ra[m].y += v.y * wx[e];
                    }
#pragma unroll
                for (int m = 0; m < 3; ++m) {
                    acc[m].x += ra[m].x * wz[a];
                    acc[m].y += ra[m].y * wz[a];
                }
            }
            float2 s;
            s.x = d.x * acc[0].x + d.y * acc[1].x + d.z * acc[2].x;
            s.y = d.x * acc[0].y + d.y * acc[1].y + d.z * acc[2].y;
            const long long mir = A.S - 1 - (long long)idx;
            if (mir == (long long)idx) s.y = 0.f;   // the transform of a real volume is real at q = 0
            float2 *pc = c + (long long)p * A.S;
            pc[idx] = s;
            if (mir != (long long)idx) pc[mir] = cconj(s);
        }
        __syncthreads();
    }
}

// ------------------------------------------------------------------ host
#define LAM_TILE_WIDTH(w, CALL)                                            \
    switch (w) {                                                           \
        case 4: { constexpr int W = 4; CALL; } break;                      \
        case 6: { constexpr int W = 6; CALL; } break;                      \
        case 8: { constexpr int W = 8; CALL; } break;                      \
        case 10: { constexpr int W = 10; CALL; } break;                    \
        case 12: { constexpr int W = 12; CALL; } break;                    \
        default: throw Error(LAM_ERR_NUFFT, "Error in finufft_makeplan: unsupported kernel width"); \
    }

// Tile edge of an axis of nf cells: a block of `cells` leaves cells + 1 - W first cells.  A
// divisor within a tenth of that gives equal tiles; otherwise the widest tiles, evened out.
int tile_edge(int nf, int W, int cells) {
    const int widest = std::min(cells + 1 - W, nf);
    for (int t = widest; 10 * t >= 9 * widest; --t)
        if (nf % t == 0) return t;
    const int nt = (nf + widest - 1) / widest;
    return (nf + nt - 1) / nt;
}

TileGeom tile_geom(const int nf[3], int W, long long R, long long C, bool direct) {
    TileGeom tg;
    tg.W = W;
    tg.nfz = nf[0];
    tg.nfy = nf[1];
    tg.nfx = nf[2];
    tg.Tz = tile_edge(nf[0], W, kBlock);
    // 10 cells of 3 components, and the tiles of a unit share the interpolation's 16 cells
    tg.Tx = tile_edge(nf[2], W, tile_comps(W) == 1 ? 32 : W <= 6 ? std::min(10, (kBlock + 1 - W) / kUnitTiles + W - 1) : 10);
    tg.ntz = (nf[0] + tg.Tz - 1) / tg.Tz;
    tg.ntx = (nf[2] + tg.Tx - 1) / tg.Tx;
    tg.ntiles = (unsigned)(tg.ntz * tg.ntx);
    const long long H = (R * C + 1) / 2;
    tg.Jn = (int)((H - 1) / C + 1);
    tg.direct = direct ? 1 : 0;
    tg.nrho = direct ? nf[1] : tg.Jn;
    tg.fTz = FastDiv((unsigned)tg.Tz);
    tg.fTx = FastDiv((unsigned)tg.Tx);
    tg.fntx = FastDiv((unsigned)tg.ntx);
    return tg;
}

// Whether the buckets and the padded point list (up to 3 fillers per non-empty bucket) have
// 32-bit numbers.  What the row form and the 3-D bins took always fits: fewer than 2^31 points,
// and at most 2^32 cells per row (or of the fine grid) for tiles of 27 or more.
bool tile_fits(const TileGeom &tg, long long total) {
    const long long nb = (long long)tg.ntiles * tg.nrho;
    return nb < (1ll << 31) - kScanBlock && total + 3 * std::min(nb, total) < (1ll << 32);
}

// Points a job may hold.  Every job records W - 1 planes more than its rows have, and a wave
// takes its points one batch after another, so the jobs are as large as the waves in flight
// allow (3 per SIMD), within a range.  Measured, spread + merge in us: (89, 21, 89) / 89 with
// 128, 256, 512 and 1024 points: 79, 67, 73, 83; (179, 43, 179) / 305 with 684, 1367, 2048:
// 620, 578, 581; (359, 71, 359) / 615 with 4096, 5543, 8192: 3392, 3403, 3516.
//
// First-cell slots take a matrix product per point pair and plane, W times as many, so that a
// job's own chain is longer: there the least is the square root of the points, which weighs that
// chain against the jobs that a cell's sum goes over, from 64.  A whole adjoint in us with 64,
// 96, 128, 192 and 384 points: 4420 points 92, 93, 95, 102, 129; 21,800 132, 119, 113, 115, 138;
// 60,800 194, 159, 142, 131, 140; 192,000 217, 180, 161, 156, 154.
constexpr unsigned kJobMin = 384, kJobMinDirect = 64, kJobMax = 5120, kJobTarget = 6144;

unsigned job_points(long long total, bool direct) {
    const long long least =
        direct ? std::clamp<long long>((long long)std::sqrt((double)total), kJobMinDirect, kJobMin) : kJobMin;
    return (unsigned)std::max<long long>(least, std::min<long long>(kJobMax, total / kJobTarget)) & ~3u;
}

// Points an interpolation job may hold: a job loads W planes of its block before its first
// point, and the launch should be several times the workgroups the chip holds (1280).
// Measured in us, (256..4096 points, 8192 jobs) against (512..8192, 4096): (89, 21, 89) / 89
// 39 and 49, (179, 43, 179) / 305 396 and 416, (359, 71, 359) / 615 2817 and 2959.
unsigned unit_points(long long total) {
    return (unsigned)std::max<long long>(256, std::min<long long>(4096, total / 8192));
}

// Rows staged at a time: about a workgroup's worth of points (256), and LDS for 5 workgroups
// per CU where the rows are dense.  Measured in us with 4 and 8 rows: (89, 21, 89) / 89, 27
// points per unit and row: 39 and 35; 96 x 24 x 100 / 128, W = 8, 13 points: 128 and 108;
// (179, 43, 179) / 305, 42 points: 396 and 429; (359, 71, 359) / 615, 63 points: 2817 and 3113.
int unit_rows(const TilePlan &tp, long long total) {
    return total < 32ll * tp.nunits * tp.tg.nrho ? 8 : 4;
}

// (tile, block cell) pairs of every cell of an axis
std::vector<int> axis_map(int nf, int T, int nt, int W) {
    const auto each = [&](auto f) {
        for (int t = 0; t < nt; ++t)
            for (int i = 0; i < std::min(T, nf - t * T) + W - 1; ++i) f((t * T + i) % nf, t, i);
    };
    std::vector<int> out(nf + 1, 0);
    each([&](int x, int, int) { ++out[x + 1]; });
    for (int x = 0; x < nf; ++x) out[x + 1] += out[x];
    std::vector<int> at(out.begin(), out.end() - 1);
    out.resize(nf + 1 + 2 * (size_t)out[nf]);
    each([&](int x, int t, int i) {
        const int e = nf + 1 + 2 * at[x]++;
        out[e] = t;
        out[e + 1] = i;
    });
    return out;
}

// Places parts of one buffer, 16 bytes aligned.
struct Carve {
    size_t bytes = 0;
    size_t take(size_t n) {
        const size_t at = bytes;
        bytes += (n + 15) & ~(size_t)15;
        return at;
    }
};
template <class T>
T *part(const DevBuf &b, size_t at) {
    return reinterpret_cast<T *>(b.as<char>() + at);
}

// bytes of one recorded plane of a job
size_t record_bytes(const TileGeom &tg) { return (size_t)(3 / tile_comps(tg.W)) * kRec * sizeof(float2); }

// Memory of the plane records of one group of jobs (LAMINO_NUFFT_SLAB_BYTES, default 8 GiB):
// more jobs than it holds are spread and merged group by group.
size_t record_budget() {
    const char *e = std::getenv("LAMINO_NUFFT_SLAB_BYTES");
    if (e && *e) {
        const long long v = std::atoll(e);
        if (v > 0) return (size_t)v;
    }
    return (size_t)8 << 30;
}

// Room made for `need` bytes of records, of at most `bound`: more than asked for, so that the next
// grid of the shape, whose jobs record more or less, finds it large enough.  Twice the need while
// that is small (the records of a few projections vary with their angles), else an eighth more.
size_t record_room(size_t need, size_t bound) {
    return std::max(need, std::min(bound, need <= ((size_t)128 << 20) ? 2 * need : need + need / 8));
}

TileArgs tile_args(const Grid &g, const NufftPlan &pl) {
    TileArgs a;
    a.S = g.R * g.C;
    a.b2 = (float)((double)pl.beta * 1.4426950408889634);
    a.fr = point_frame(g, pl);
    a.fH = FastDiv((unsigned)((a.S + 1) / 2));
    a.fC = FastDiv((unsigned)g.C);
    return a;
}

// y coordinate of detector row j of a shared-tilt grid, and its first plane (unwrapped)
double row_coord(const Grid &g, const NufftPlan &pl, int j) {
    const PointFrame fr = point_frame(g, pl);
    const double qY = ((double)j - fr.j0) * fr.dY;
    return (qY * g.geo_host[0].vy) * fr.sy;
}
int row_first(const Grid &g, const NufftPlan &pl, int j) {
    return (int)std::ceil(row_coord(g, pl, j) - 0.5 * pl.w);
}

// The plan's job groups under the present budget.  The list is kept: as long as the budget
// stays what it was, spreading waits for nothing on the host and can be captured.
const JobGroups &job_groups(Ctx &cx, TilePlan &tp) {
    JobGroups &jg = tp.groups;
    const size_t cap = std::max<size_t>(1, record_budget() / record_bytes(tp.tg));
    if (cap == jg.cap) return jg;
    if (tp.planes > cap && tp.job_plane.empty()) {
        std::vector<TileJob> jobs(tp.njobs);
        LAM_HIP(hipMemcpyAsync(jobs.data(), tp.jobs, sizeof(TileJob) * jobs.size(), hipMemcpyDeviceToHost,
                               cx.stream));
        LAM_HIP(hipStreamSynchronize(cx.stream));
        tp.job_plane.reserve(jobs.size());
        for (const TileJob &j : jobs) tp.job_plane.push_back(j.plane);
    }
    jg.first.assign(1, {0u, 0u});
    jg.most = tp.planes;
    if (tp.planes > cap) {
        jg.most = 0;
        for (unsigned j = 0; j < tp.njobs; ++j) {
            const unsigned end = j + 1 < tp.njobs ? tp.job_plane[j + 1] : tp.planes;   // jobs' planes follow each other
            if (j > jg.first.back().first && end - jg.first.back().second > cap)
                jg.first.emplace_back(j, tp.job_plane[j]);
            jg.most = std::max<size_t>(jg.most, end - jg.first.back().second);
        }
    }
    jg.cap = cap;
    return jg;
}

}  // namespace

void row_window(const Grid &g, const NufftPlan &pl, int &ylo, int &ly) {
    const long long H = (g.R * g.C + 1) / 2;
    const int a = row_first(g, pl, 0), b = row_first(g, pl, (int)((H - 1) / g.C));
    const int lo = std::min(a, b), len = std::max(a, b) + pl.w - lo;
    ylo = ly = 0;
    if (len < pl.nf[1]) {
        ylo = ((lo % pl.nf[1]) + pl.nf[1]) % pl.nf[1];
        ly = len;
    }
}

// A tile records the planes between its first row and its last, 4 KB each however few points are
// on them, where the row form moves a slab per row; the tiles are cheaper per point (about 40 ps
// against 67).  Where the rows are few against the planes they span, or the points few on both,
// the records outweigh that: whole adjoints by tiles and by rows took 359 and 203 us at (33, 166,
// 166) / 79 x 16 x 67, width 8; 640 and 440 at (130, 130, 130) / 34 x 167 x 68; 149 and 203 at
// (89, 21, 89) / 89 x 89 x 90, whose records exceed the slabs by 30 bytes a point.  Of 250 laminography
// scans (tilts of 25 to 40 degrees, thin volumes of 40 to 260) the line at 160 bytes a point and 60 MB
// sends 4 by rows, all at width 8 and none of them faster by tiles, and leaves 2 by tiles that rows
// would take 3 to 6 % less for.  Over 1000 arbitrary grids it halves those that tiles are more than a
// tenth slower for, from 137; most of the rest are volumes of a few cells.
bool row_tiles_pay(const Grid &g, const NufftPlan &pl) {
    const TileGeom tg = tile_geom(pl.nf, pl.w, g.R, g.C, false);
    const double span = std::min<double>(tg.nfy, std::floor(tg.Jn * std::fabs(g.geo_host[0].vy) * tg.nfy / (double)g.R) + pl.w);
    const double tiles = (double)tg.ntiles * span * (double)record_bytes(tg);
    const double slabs = (double)tg.Jn * tg.nfz * tg.nfx * 3 * sizeof(float2);
    return tiles - slabs <= 160.0 * (double)(g.P * ((g.R * g.C + 1) / 2)) + 6e7;
}

// The 3-D bins' spreader, which the forward of such grids shares its plan with, is the better one
// where the tiles' fixed costs show (fewer than 2048 points; a whole adjoint at 98 to 1976 points
// takes 52 to 113 us with it and 0.76 to 1.61 of that by tiles, 1.13 at the median), and where all
// points crowd into a few tiles: (4, 4, 4) / 236 x 31 x 44 299 us against 422, (15, 7, 3) / 209 x
// 352 x 68 at width 10 1451 against 3173, (14, 14, 14) / 207 x 297 x 58 at width 8 775 and 1158; above width 8 the line lies at fewer points, since three
// waves then stage each ((4, 4, 4) / 281 x 27 x 2 at width 10 104 and 195).  Elsewhere the tiles
// are: (60, 15, 60) / 200 x 200 x 200 1141 and 850, (11, 3, 11) / 80 x 28 x 21 at width 8 213 and 173.
bool first_cell_tiles_pay(const Grid &g, const NufftPlan &pl) {
    const TileGeom tg = tile_geom(pl.nf, pl.w, g.R, g.C, true);
    const long long total = g.P * ((g.R * g.C + 1) / 2);
    const bool crowded = (tg.ntiles < 64 && total > 32768ll * tg.ntiles) || (tile_comps(pl.w) == 1 && tg.ntiles < 6);
    return total >= 2048 && !crowded;
}

TileBytes tile_bytes(const NufftPlan &pl, long long P, long long R, long long C, bool direct) {
    const size_t total = (size_t)P * (size_t)((R * C + 1) / 2);
    const TileGeom tg = tile_geom(pl.nf, pl.w, R, C, direct);
    const size_t nb = (size_t)tg.ntiles * tg.nrho, ids = total + 3 * std::min(nb, total);
    const size_t jobs = tg.ntiles + ids / job_points((long long)total, direct) + 1;
    // an interpolation job and the next one of its unit hold more points than one may
    const size_t ujobs = tg.ntiles + 4 * (ids / unit_points((long long)total)) + 1;
    // a job's planes: its rows' first planes and W - 1 more; the half set spans at most half
    // the period
    const size_t planes = (size_t)tg.ntiles * (size_t)(direct ? tg.nfy : tg.nfy / 2 + 2) + jobs * (size_t)pl.w;
    const size_t largest = record_bytes(tg) * ((size_t)tg.nfy + pl.w);   // of one job
    TileBytes b;
    b.kept = 4 * (ids + nb + tg.ntiles) + sizeof(TileJob) * jobs + sizeof(UnitJob) * ujobs +
             sizeof(TileGeo) * (size_t)P + sizeof(RowY) * tg.nrho + 64 * (size_t)(tg.nfz + tg.nfx) + 4096;
    b.setup = 17 * total + 4096;   // the runs, twice, and the list of long buckets
    // counts, run offsets and cursors per bucket and scan sums, in the record buffer
    b.records = std::max(17 * nb + 64 * (size_t)tg.ntiles + 65536,
                         std::min(record_bytes(tg) * planes, std::max(record_budget(), largest)));
    return b;
}

// A plan takes few launches, allocations and waits: on small grids the first pass on a new grid is
// made of them.  With an array per allocation, three launches per scan and a thread per unit,
// the first adjoint of (9, 5, 11) / 13 x 15 x 12 took 338 us, now 154; (89, 21, 89) / 89 x 89 x 90
// 470, now 276; (179, 43, 179) / 305 x 305 x 180 1594, now 1251; the headline grid 8776, now 8114.
TilePlan &get_tileplan(Ctx &cx, Grid &g, NufftPlan &pl, bool direct) {
    std::vector<long long> key = {pl.nf[0], pl.nf[1], pl.nf[2], pl.w, direct ? 1 : 0};
    auto it = g.tileplans.find(key);
    if (it != g.tileplans.end()) return *it->second;
    TimedScope ts(cx, "bin_points");
    const long long S = g.R * g.C, H = (S + 1) / 2, total = g.P * H;
    LAM_REQUIRE(total < (1ll << 31), LAM_ERR_ARG, "too many points in one polar grid for 32-bit bins");
    auto tp = std::make_unique<TilePlan>();
    TileGeom &tg = tp->tg;
    tg = tile_geom(pl.nf, pl.w, g.R, g.C, direct);
    const int W = pl.w, Jn = tg.Jn;
    const long long nb = (long long)tg.ntiles * tg.nrho;
    LAM_REQUIRE(tile_fits(tg, total), LAM_ERR_ARG, "fine grid too large for 32-bit point bins");
    const PointFrame fr = point_frame(g, pl);

    // Row slots: first planes, and for a shared tilt the y weights, from the same coordinate
    // expression as the kernels (ty = (qY vy) sy), in double.  Unwrapped, the first plane of
    // a detector row is linear in the row and so monotonic.
    std::vector<RowY> rows(tg.nrho, RowY{});
    if (direct) {
        for (int r = 0; r < tg.nrho; ++r) rows[r].iy = r;
    } else {
        tg.dir = row_first(g, pl, Jn - 1) >= row_first(g, pl, 0) ? 1 : -1;
        for (int r = 0; r < Jn; ++r) {
            const int j = tg.dir > 0 ? r : Jn - 1 - r;
            const double ty = row_coord(g, pl, j);
            RowY &y = rows[r];
            y.iy = row_first(g, pl, j);
            for (int m = 0; m < W; ++m) {
                const double z = ((double)(y.iy + m) - ty) * (2.0 / W);
                const double rr = 1.0 - z * z;
                y.w[m] = rr > 0 ? (float)std::exp((double)pl.beta * (std::sqrt(rr) - 1.0)) : 0.f;
            }
            LAM_REQUIRE(r == 0 || y.iy >= rows[r - 1].iy, LAM_ERR_STATE, "row first cells are not monotonic");
        }
        row_window(g, pl, tp->ylo, tp->ly);
    }
    // what the host works out, in one upload
    {
        const std::vector<int> zmap = axis_map(tg.nfz, tg.Tz, tg.ntz, W), xmap = axis_map(tg.nfx, tg.Tx, tg.ntx, W);
        Carve c;
        const size_t og = c.take(sizeof(TileGeo) * g.P), orow = c.take(sizeof(RowY) * rows.size()),
                     oz = c.take(sizeof(int) * zmap.size()), ox = c.take(sizeof(int) * xmap.size());
        std::vector<char> host(c.bytes);
        for (long long p = 0; p < g.P; ++p) {
            const Geo &e = g.geo_host[p];
            const TileGeo t{e.uz, e.vz, e.ux, e.vx, e.vy, 0.0, {(float)e.d0, (float)e.d1, (float)e.d2, 0.f}};
            std::memcpy(host.data() + og + sizeof(TileGeo) * p, &t, sizeof(t));
        }
        std::memcpy(host.data() + orow, rows.data(), sizeof(RowY) * rows.size());
        std::memcpy(host.data() + oz, zmap.data(), sizeof(int) * zmap.size());
        std::memcpy(host.data() + ox, xmap.data(), sizeof(int) * xmap.size());
        tp->fixed.alloc(c.bytes);
        upload_now(cx, tp->fixed.ptr, host.data(), c.bytes);
        tp->geo = part<TileGeo>(tp->fixed, og);
        tp->rowy = part<RowY>(tp->fixed, orow);
        tp->zmap = part<int>(tp->fixed, oz);
        tp->xmap = part<int>(tp->fixed, ox);
    }
    tp->nunits = tile_interp_fits(pl.w) && !direct
                     ? (unsigned)tg.ntz * (unsigned)((tg.ntx + kUnitTiles - 1) / kUnitTiles)
                     : 0u;
    Carve ci;
    const size_t ooff = ci.take(sizeof(unsigned) * (nb + 1)), ojob0 = ci.take(sizeof(unsigned) * (tg.ntiles + 1ull));
    tp->index.alloc(ci.bytes);
    unsigned *off = part<unsigned>(tp->index, ooff), *job0 = part<unsigned>(tp->index, ojob0);
    tp->off = off;
    tp->job0 = job0;
    // The temporaries sit in the record buffer, which the spread needs anyway.
    Carve cs;
    const size_t ocount = cs.take(sizeof(unsigned long long) * nb), ocursor = cs.take(sizeof(unsigned) * nb),
                 onlong = cs.take(sizeof(unsigned)), zeroed = cs.bytes, oroff = cs.take(sizeof(unsigned) * (nb + 1)),
                 osums = cs.take(sizeof(uint2) * scan_blocks(std::max<long long>(nb, std::max(tg.ntiles, tp->nunits)))),
                 ojcount = cs.take(sizeof(unsigned long long) * tg.ntiles),
                 ojplane = cs.take(sizeof(unsigned) * (tg.ntiles + 1ull)),
                 oucount = cs.take(sizeof(unsigned long long) * tp->nunits),
                 oujob0 = cs.take(sizeof(unsigned) * (tp->nunits + 1ull)),
                 ouhigh = cs.take(sizeof(unsigned) * (tp->nunits + 1ull));
    if (pl.rec.bytes < cs.bytes)
        pl.rec.ensure(record_room(cs.bytes, tile_bytes(pl, g.P, g.R, g.C, direct).records));
    const DevBuf &tmp = pl.rec;
    auto *count = part<unsigned long long>(tmp, ocount);
    unsigned *cursor = part<unsigned>(tmp, ocursor), *roff = part<unsigned>(tmp, oroff);
    uint2 *sums = part<uint2>(tmp, osums), *grand = reinterpret_cast<uint2 *>(cx.sums.get());

    // points: runs counted per bucket, scanned, stored, ordered and written out
    LAM_HIP(hipMemsetAsync(tmp.ptr, 0, zeroed, cx.stream));
    const unsigned cpl = (unsigned)((g.C + 63) / 64);
    const long long nwaves = g.P * Jn * (long long)cpl;
    const dim3 rgrid = wave_grid(nwaves);
    hipLaunchKernelGGL(k_tile_runs<0>, rgrid, dim3(256), 0, cx.stream, g.geo.as<Geo>(), nwaves, (int)g.R, (int)g.C, fr,
                       tg, cpl, count, (const unsigned *)nullptr, (unsigned *)nullptr, (uint2 *)nullptr);
    check_launch();
    run_scans<true>(cx, ScanArgs{count, nb, off, roff, grand}, ScanArgs{}, sums);
    LAM_HIP(hipStreamSynchronize(cx.stream));
    const uint2 points = grand[0];
    LAM_REQUIRE((long long)points.x >= total && (long long)points.y <= total, LAM_ERR_STATE,
                "bin counts do not add up to the point count");
    DevBuf own;   // the runs and their regrouping, where the record buffer has no room left for them
    const bool order = points.y > kRunsRanked;   // else no bucket has that many
    Carve cr;
    const size_t orun = cr.take(sizeof(uint2) * points.y), otmp = cr.take(order ? sizeof(uint2) * points.y : 0),
                 olong = cr.take(order ? sizeof(unsigned) * (points.y / kRunsRanked + 1) : 0);
    if (cs.bytes + cr.bytes > tmp.bytes) own.alloc(cr.bytes);
    char *rest = own.ptr ? own.as<char>() : part<char>(tmp, cs.bytes);
    uint2 *runs = reinterpret_cast<uint2 *>(rest + orun);
    unsigned *nlong = part<unsigned>(tmp, onlong), *longer = reinterpret_cast<unsigned *>(rest + olong);
    tp->ids.alloc(sizeof(unsigned) * std::max<size_t>(points.x, 1));
    unsigned *ids = tp->ids.as<unsigned>();
    hipLaunchKernelGGL(k_tile_runs<1>, rgrid, dim3(256), 0, cx.stream, g.geo.as<Geo>(), nwaves, (int)g.R, (int)g.C, fr,
                       tg, cpl, (unsigned long long *)nullptr, roff, cursor, runs);
    check_launch();
    hipLaunchKernelGGL(k_run_expand, wave_grid(nb), dim3(256), 0, cx.stream, count, nb, off, roff, runs, ids, nlong,
                       longer);
    check_launch();
    if (order) {
        hipLaunchKernelGGL(k_run_order, dim3(grid_for(points.y / kRunsRanked, 1, 2048)), dim3(256), 0, cx.stream, count,
                           off, roff, runs, reinterpret_cast<uint2 *>(rest + otmp),
                           (unsigned)((total + kRunBins - 1) / kRunBins), ids, nlong, longer);
        check_launch();
    }
    // shares: counted per tile and unit, scanned, written out
    const ShareArgs sa{off, tp->rowy, job_points(total, direct), unit_points(total), tp->nunits, direct ? kDeepDirect : kDeep,
                       direct ? 160.f / W : 96.f};
    const unsigned tblocks = tile_blocks(tg);
    const dim3 sgrid(tblocks + tp->nunits);
    auto *jcount = part<unsigned long long>(tmp, ojcount), *ucount = part<unsigned long long>(tmp, oucount);
    unsigned *jplane = part<unsigned>(tmp, ojplane), *ujob0 = part<unsigned>(tmp, oujob0);
    hipLaunchKernelGGL(k_share_count, sgrid, dim3(64), 0, cx.stream, sa, tg, tblocks, jcount, ucount);
    check_launch();
    run_scans<false>(cx, ScanArgs{jcount, tg.ntiles, jplane, job0, grand + 1},
                     ScanArgs{ucount, tp->nunits, ujob0, part<unsigned>(tmp, ouhigh), grand + 2}, sums);
    LAM_HIP(hipStreamSynchronize(cx.stream));
    tp->planes = grand[1].x;
    tp->njobs = grand[1].y;
    tp->nujobs = tp->nunits ? grand[2].x : 0u;
    Carve cw;
    const size_t ojobs = cw.take(sizeof(TileJob) * tp->njobs), oujobs = cw.take(sizeof(UnitJob) * tp->nujobs);
    tp->shares.alloc(std::max<size_t>(cw.bytes, 16));
    tp->jobs = part<TileJob>(tp->shares, ojobs);
    tp->ujobs = part<UnitJob>(tp->shares, oujobs);
    hipLaunchKernelGGL(k_share_emit, sgrid, dim3(64), 0, cx.stream, sa, tg, tblocks, jplane, job0, ujob0,
                       part<TileJob>(tp->shares, ojobs), part<UnitJob>(tp->shares, oujobs));
    check_launch();
    if (own.ptr) LAM_HIP(hipStreamSynchronize(cx.stream));   // it goes
    TilePlan &ref = *tp;
    g.tileplans.emplace(std::move(key), std::move(tp));
    return ref;
}

void tile_spread(Ctx &cx, Grid &g, NufftPlan &pl, TilePlan &tp, const float2 *c, bool paired, bool add) {
    const TileGeom &tg = tp.tg;
    const size_t per_plane = record_bytes(tg);
    const JobGroups &jg = job_groups(cx, tp);
    const auto &groups = jg.first;
    if (pl.rec.bytes < per_plane * jg.most)
        pl.rec.ensure(record_room(per_plane * jg.most, tile_bytes(pl, g.P, g.R, g.C, tg.direct != 0).records));
    const TileArgs a = tile_args(g, pl);
    const int ly = tp.ly > 0 ? tp.ly : tg.nfy, ylo = tp.ly > 0 ? tp.ylo : 0;
    for (size_t k = 0; k < groups.size(); ++k) {
        const unsigned j0 = groups[k].first, j1 = k + 1 < groups.size() ? groups[k + 1].first : tp.njobs;
        if (j1 > j0) {
            TimedScope ts(cx, "tile_spread");
            const dim3 grid((j1 - j0) * (unsigned)(3 / tile_comps(pl.w)));
#define LAM_TILE_SPREAD(DIRECT)                                                                                  \
    LAM_TILE_WIDTH(pl.w, hipLaunchKernelGGL((k_tile_spread<W, tile_comps(W), DIRECT>), grid, dim3(64), 0, cx.stream, \
                                            pl.rec.as<float2>(), c, tp.geo, tp.off, \
                                            tp.ids.as<unsigned>(), tp.rowy,                           \
                                            tp.jobs + j0, a, tg, groups[k].second, paired ? 1 : 0))
            if (tg.direct) {
                LAM_TILE_SPREAD(true);
            } else {
                LAM_TILE_SPREAD(false);
            }
#undef LAM_TILE_SPREAD
            check_launch();
        }
        TimedScope ts(cx, "tile_merge");
        const dim3 mgrid((unsigned)((3 * tg.nfx + 255) / 256) * (unsigned)tg.nfz *
                         (unsigned)((ly + kMergePlanes - 1) / kMergePlanes));
        LAM_TILE_WIDTH(pl.w, hipLaunchKernelGGL((k_tile_merge<tile_comps(W)>), mgrid, dim3(256), 0, cx.stream,
                                                pl.fine.as<float2>(), pl.rec.as<float2>(), tp.jobs,
                                                tp.job0, j0, j1, groups[k].second, tp.zmap,
                                                tp.xmap, tg, ylo, ly, add || k > 0 ? 1 : 0));
        check_launch();
    }
}

// Wider kernels leave a unit few first cells (9 x 6 at W = 8), so that forming G costs more
// than the points: 0.10 ms against the row slabs' 0.076 at (100, 24, 96) / 120 x 128, W = 8.
bool tile_interp_fits(int w) { return w <= 6; }

void tile_interp(Ctx &cx, Grid &g, NufftPlan &pl, TilePlan &tp, float2 *c) {
    const TileGeom &tg = tp.tg;
    const TileArgs a = tile_args(g, pl);
    TimedScope ts(cx, "tile_interp");
    const int nr = unit_rows(tp, g.P * ((g.R * g.C + 1) / 2));
    static_assert(sizeof(float2) * 3 * kUnitRows * kUnitCells <= 64 * 1024, "no larger LDS limit to ask for");
    const size_t lds = (size_t)nr * kUnitCells * 3 * sizeof(float2);
#define LAM_TILE_INTERP(WW)                                                                                         \
    hipLaunchKernelGGL((k_tile_interp<WW>), dim3(tp.nujobs), dim3(kUnitThreads), lds, cx.stream, pl.fine.as<float2>(), \
                       c, tp.geo, tp.off, tp.ids.as<unsigned>(), tp.rowy,   \
                       tp.ujobs, a, tg, nr)
    if (pl.w == 4) LAM_TILE_INTERP(4);
    else LAM_TILE_INTERP(6);
#undef LAM_TILE_INTERP
    check_launch();
}

}  // namespace lam
