// The harmonic scattered field on fewer points than pixels.
//
// Outside r = l/k, l the highest order whose radial function a threshold rule
// cuts visibly (Nl, or where a batch's own coefficients are known the order
// past which |B_l| times the largest cut value, 0.0145, is below 1e-8 of the
// field), a sphere's field is an analytic function with local wavenumbers of
// at most k but for its decaying part.  On a tile of T x T pixels whose half
// edge is h, such a field is its interpolant at q x q Chebyshev nodes,
// q = kh + 6 (kh)^(1/3) + 2.5, to 3e-8 of its size there (the tile no nearer
// to the centre than 4/k and 1.3 h either, where the field of a small sphere
// is steep; measured on spheres of ka from 0.2 to 40); a tile of 64 pixels at
// a tenth of a wavelength each takes 40 x 40 nodes, and finer pixels fewer.
// So each instance's slice is cut into tiles of 128 or 64 pixels, those a
// sphere is too near to into tiles of half the edge down to 16 for it, and a
// sphere's sum is evaluated at the nodes of the coarsest tiles that are far
// from it and at the pixels of the 16 x 16 tiles that none is.
// harm_expand_kernel then forms every pixel: E V E^T per tile of each size,
// plus the near tiles' own values.
//
// The harmonic kernel is bound by the instructions of a (point, sphere), so
// the points are what it costs: on a 64-image sweep (512 x 512, 20 spheres)
// its launches take 3.6 ms for 9.5 ms, on one image of 1024 x 1024 and 50
// spheres 0.39 for 1.2 ms, with 0.42 and 0.03 ms for the expansions.
// A wave holds nodes of one tile only (its last wave partly filled), so that
// the spheres it skips are the wave's own.  A plan takes the nodes of an
// instance where the points it then evaluates cost less than the pixels
// would (node_plan_instance); otherwise its pixels
// are evaluated as they are.
#pragma once

#include <cstdint>
#include <map>
#include <vector>

#include "us_series.h"

namespace bimsim {

constexpr int kNodeLevels = 4;
constexpr int kNodeTile[kNodeLevels] = {128, 64, 32, 16};
constexpr int kNearTile = 16;       // a near tile is a block's 256 pixels
// Nodes per edge: at most 3/4 of the tile's pixels, and 64 (the expansion's
// LDS).
constexpr int kNodeMaxQ = 64;
// Costs are in units of one order of one planar sphere at one point (some
// 0.7e-6 us where the chip is full).
// An instance's pixels below which they are evaluated as they are (64 images a
// batch, one sphere, us by pixels and by nodes: 192 x 192, 39 orders, 2.9e6, 322
// and 339, 21 orders, 2.2e6, 242 and 241 or on a wide slice 281 and 267; above
// it 256 x 256, 12 orders, 3.4e6, 345 and 264, 21, 4e6, 362 and 297; 320 x 320,
// 21, 6.2e6, 633 and 503; 384 x 384, 12, 7.7e6, 752 and 537).
constexpr double kNodeMinWork = 3.0e6;
// What a plan's time is but for its points' work: the longest chain of spheres
// at a point (whatever the number of points), and for nodes the expansion's
// launch and its phases for each size of tiles.  Fitted to 760 images of 128^2
// to 1024^2 pixels and 1 to 20 spheres of 13 to 39 orders, planar or not,
// timed by pixels and by nodes: 15 of them are slower than their pixels by
// more than 3 per cent (1.2 times at most), and the mean is 2.0 per cent from
// the better of the two.  (Thresholds on the pixels' work and chain alone: 73,
// 1.38 times and 6.2 per cent.)  On either side of the line, us by pixels and
// by nodes: planar spheres of 39 orders, 512 x 512, three 94 and 111, six 155
// and 135; 256 x 256, six 105 and 120, twenty 288 and 230; of 18 orders, two on
// 512 x 512 49 and 50, on 768 x 768 78 and 57; off the plane, 256 x 256, one of
// 39 102 and 118, six of 28 214 and 167.
constexpr double kNodeChain = 2.0e5;
constexpr double kNodeLaunch = 1.5e7;
constexpr double kNodeLevel = 4.0e6;

struct NodeCost {
    double work = 0.0, chain = 0.0;
    int levels = 0;
    double total() const {
        return work + kNodeChain * chain + (levels > 0 ? kNodeLaunch + kNodeLevel * levels : 0.0);
    }
    void add(const NodeCost& c) {
        work += c.work;
        chain = chain > c.chain ? chain : c.chain;
        levels = levels > c.levels ? levels : c.levels;
    }
};

// Host tables of a plan's nodes, uploaded by series_plan_create.
struct NodeTables {
    std::vector<NodeInst> inst;
    std::vector<int2> tiles;              // first pixel (column, row) of each tile
    std::vector<unsigned long long> mask; // spheres evaluated at each tile, by bit
    std::vector<int> idx;                 // tile of each cell of a level's grid, or -1
    std::vector<float> E;                 // interpolation matrices [node][pixel]
    std::vector<double> X;                // node positions, in pixels from the tile's first
    std::vector<int4> blocks;             // 64 x 64 pixel blocks (instance, column, row)
    long long n_v = 0, n_w = 0;
    std::map<std::pair<int, int>, std::pair<int, int>> mats;   // (T, q) -> offsets in E, X
};

// The instance evaluated at its pixels.  planar: every sphere of the plan is
// (one that is not puts its order bucket on the general sums).
NodeCost node_pixel_cost(const SeriesInst& I, const SeriesSph* sph, bool planar);

// Adds instance i's nodes to the tables when they cost less than its pixels
// (else its entry has n_lev = 0); returns what the instance then costs.  sph:
// its spheres in plan order.
NodeCost node_plan_instance(const SeriesInst& I, const SeriesSph* sph, bool planar, NodeTables* t);

// Whether the tile's mask (words 64-bit words at m) has a sphere of
// [begin, begin + n).
bool node_mask_any(const unsigned long long* m, int begin, int n);

// The bound SeriesSph::reach of a sphere at wavenumber k from its own B_l
// (interleaved re, im).
int node_reach(const SphereDev& S, double k, const double* B);

// Every pixel of the instances with nodes from V and W into U.
int node_expand_launch(bimsim_ctx* ctx, const SeriesPlan& P, float2* U);

}  // namespace bimsim
