// Matrix-core spreading of the three-component projectors over (z, x) tiles of the fine grid
// (tiles.hip).
#pragma once
#include "nufft.h"

namespace lam {

struct TileGeo;   // tiles.hip
struct RowY;

// Cutting of the (z, x) plane into tiles of Tz x Tx first cells.  Tile (tz, tx) owns the points
// whose first kernel cell lies in [tz Tz, (tz + 1) Tz) x [tx Tx, (tx + 1) Tx).  With its halo a
// tile fits one 32 x 32 matrix-core block of (z, re/im) rows and (x, component) columns: 16 z
// cells (Tz + W - 1 <= 16), and in x 10 cells of three components or, for widths above 8, 32
// cells of one.
struct TileGeom {
    int W = 0;
    int Tz = 0, Tx = 0, ntz = 0, ntx = 0;
    unsigned ntiles = 0;
    int nfz = 0, nfy = 0, nfx = 0;
    int Jn = 0;      // rows of the half point set
    int nrho = 0;    // row slots: detector rows (shared tilt) or first y cells (direct)
    int dir = 1;     // slot of row j: j (+1) or Jn - 1 - j (-1), so that first y cells never fall
    int direct = 0;  // the slot is the point's wrapped first y cell
    FastDiv fTz, fTx, fntx;
};

// A share of one tile's points for one wave: ids [beg, end), of the row slots [r0, r1), which
// reach the planes [y0, y0 + np) (unwrapped; yw = y0 modulo the period), recorded from plane
// record `plane`.
struct TileJob {
    unsigned tile, beg, end;
    int r0, r1, y0, np, yw;
    unsigned plane;
};

// A share of one unit's rows for one interpolating workgroup (a unit: a few tiles side by
// side in x): the row slots [r0, r1), or part `part` of `parts` of one slot's points.
struct UnitJob {
    unsigned unit;
    int r0, r1;
    unsigned part, parts;
};

// Groups of consecutive jobs whose records fit a budget of `cap` planes, one job at least:
// (first job, its first plane) of each, and the planes of the largest.
struct JobGroups {
    size_t cap = 0, most = 0;
    std::vector<std::pair<unsigned, unsigned>> first;
};

// Points of one grid ordered by (tile, row slot, point number), each (tile, slot) padded to
// a multiple of 4 with kNoPoint.
struct TilePlan {
    TileGeom tg;
    int ylo = 0, ly = 0;           // the y planes touched: [ylo, ylo + ly) mod nfy (ly 0: all)
    unsigned njobs = 0, planes = 0;   // planes: recorded by all jobs
    unsigned nunits = 0, nujobs = 0;
    DevBuf fixed, index, ids, shares;   // what the pointers below point into
    const TileGeo *geo = nullptr;       // [P]
    const RowY *rowy = nullptr;         // [nrho]
    // cells of each axis as (tile, cell of its block) pairs: starts [nf + 1], then pairs
    const int *zmap = nullptr, *xmap = nullptr;
    const unsigned *off = nullptr;      // [ntiles * nrho + 1] first id of each (tile, slot)
    const unsigned *job0 = nullptr;     // [ntiles + 1] first job of each tile
    const TileJob *jobs = nullptr;      // [njobs], tile by tile
    const UnitJob *ujobs = nullptr;     // [nujobs]
    std::vector<unsigned> job_plane;  // host: first plane of each job, once a budget needed groups
    JobGroups groups;                 // of the budget last used
};

// The y planes [ylo, ylo + ly) (mod nfy) that the rows of a shared-tilt grid touch (ly 0: all).
void row_window(const Grid &g, const NufftPlan &pl, int &ylo, int &ly);

// Whether the spread of a shared-tilt grid goes by tiles (row slots) or by the row form.
bool row_tiles_pay(const Grid &g, const NufftPlan &pl);

// Whether the spread of a grid without row slots goes by tiles (first-cell slots) or by 3-D bins.
bool first_cell_tiles_pay(const Grid &g, const NufftPlan &pl);

TilePlan &get_tileplan(Ctx &cx, Grid &g, NufftPlan &pl, bool direct);

// fine (+)= the type-1 spread of the half point set.  add = false writes every plane of the
// plan's window (every plane when ly is 0).
void tile_spread(Ctx &cx, Grid &g, NufftPlan &pl, TilePlan &tp, const float2 *c, bool paired, bool add);

// c = the type-2 gather of the half point set and its mirror, for shared-tilt grids and the
// kernel widths tile_interp_fits() names.
bool tile_interp_fits(int w);
void tile_interp(Ctx &cx, Grid &g, NufftPlan &pl, TilePlan &tp, float2 *c);

// Upper bounds of the device bytes of a plan (kept, and temporaries while it is built) and
// of the plane records of its spread.
struct TileBytes {
    size_t kept = 0, setup = 0, records = 0;
};
TileBytes tile_bytes(const NufftPlan &pl, long long P, long long R, long long C, bool direct);   // pl: w and nf

}  // namespace lam
