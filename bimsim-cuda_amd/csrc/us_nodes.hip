// Planning of the harmonic form's nodes and the kernel that forms the pixels
// from them (us_nodes.h).
#include "us_nodes.h"

#include <algorithm>
#include <cmath>

#include "internal.h"

namespace bimsim {
namespace {

// The expansion's block: 64 x 64 pixels, a wave to four rows of them.
constexpr int kBlock = 64;
constexpr int kThreads = 1024;
constexpr int kRows = kBlock * kBlock / kThreads;   // per thread
// Rows of nodes expanded at a time (3/4 of 64 pixels' worth: one round for
// every size but 128), and the node values they hold.
constexpr int kRound = 48;
constexpr int kRoundNodes = kRound * kRound;
static_assert(kNodeMaxQ / 2 * kNodeMaxQ <= kRoundNodes, "a round of the largest tile's nodes");

// Nodes per edge for a tile of half edge h at wavenumber k: the smallest q
// whose interpolant of exp(i k x) on [-h, h] is within 3e-8, rounded up
// (found for kh from 0.1 to 40).
int node_count(double kh) { return (int)std::ceil(kh + 6.0 * std::cbrt(kh) + 2.5); }

// One point and a sphere of n = Nl + 1 orders (the planar sums' products on the
// matrix cores hardly show beside the radial steps).
double point_cost(int n, bool planar) { return planar ? n : 0.155 * n * n + 27.0; }
// A point's position and its result, whatever its spheres.
constexpr double kPointCost = 40.0;
// An FMA of the expansion.
constexpr double kExpandCost = 0.04;

// Interpolation matrix and node positions of (T, q): offsets in E and X.
std::pair<int, int> matrix(NodeTables* t, int T, int q) {
    auto it = t->mats.find({T, q});
    if (it != t->mats.end()) return it->second;
    const std::pair<int, int> at{(int)t->E.size(), (int)t->X.size()};
    std::vector<double> x(q), w(q);
    for (int a = 0; a < q; ++a) {
        const double th = M_PI * (a + 0.5) / q;
        x[a] = std::cos(th);
        w[a] = ((a & 1) ? -1.0 : 1.0) * std::sin(th);
        t->X.push_back(0.5 * (T - 1) * (1.0 + x[a]));
    }
    std::vector<double> row(q);
    t->E.resize(t->E.size() + (size_t)q * T);
    for (int i = 0; i < T; ++i) {
        const double y = -1.0 + 2.0 * i / (T - 1);
        double sum = 0.0;
        int hit = -1;
        for (int a = 0; a < q; ++a) {
            const double d = y - x[a];
            if (std::fabs(d) < 1e-14) hit = a;
            row[a] = w[a] / d;
            sum += row[a];
        }
        for (int a = 0; a < q; ++a)
            t->E[at.first + (size_t)a * T + i] =
                hit >= 0 ? (a == hit ? 1.f : 0.f) : (float)(row[a] / sum);
    }
    t->mats[{T, q}] = at;
    return at;
}

// The tiles of one instance, before they are added to the tables, the
// largest of size kNodeTile[top].
struct Tiling {
    const SeriesInst& I;
    const SeriesSph* sph;
    int words;
    bool active[kNodeLevels];
    int q[kNodeLevels];
    double h[kNodeLevels];
    // the slice's geometry: pixel pitch, and for an orthogonal slice each
    // centre in pixels and its squared distance from the plane
    double px, py;
    bool ortho;
    std::vector<double> cu, cv, cz2, reach, one;        // one: its cost at a point
    std::vector<unsigned long long> cell[kNodeLevels];   // masks of the cell being cut
    std::vector<int2> tiles[kNodeLevels + 1];   // the last: near tiles
    std::vector<unsigned long long> mask[kNodeLevels + 1];
    NodeCost cost;

    Tiling(const SeriesInst& inst, const SeriesSph* s, bool planar, int top) : I(inst), sph(s) {
        words = (I.ns + 63) / 64;
        const double lx = len(I.q.X), ly = len(I.q.Y);
        px = lx / I.uR;
        py = ly / I.vR;
        ortho = std::fabs(dot(I.q.X, I.q.Y)) <= 1e-9 * lx * ly;
        for (int l = 0; l < kNodeLevels; ++l) {
            h[l] = 0.5 * (kNodeTile[l] - 1) * std::max(px, py);
            q[l] = node_count(I.kmag * h[l]);
            active[l] = l >= top && q[l] <= std::min(kNodeMaxQ, 3 * kNodeTile[l] / 4);
        }
        for (int t = 0; t < I.ns; ++t) {
            const SphereDev& S = sph[t].s;
            const d3 c = sub(mk(S.p), I.q.A);
            const double a = dot(c, I.q.X) / lx, b = dot(c, I.q.Y) / ly;
            cu.push_back(a / px);
            cv.push_back(b / py);
            cz2.push_back(std::max(0.0, dot(c, c) - a * a - b * b));
            const int order = std::max(sph[t].reach > 0 ? sph[t].reach : S.Nl, 4);
            reach.push_back(std::max(order / I.kmag, S.a) * (1.0 + 1e-9));
            one.push_back(point_cost(S.Nl + 1, planar));
        }
        for (auto& c : cell) c.resize(2 * (size_t)words);
    }
    // whether sphere t is far from the tile of level l at pixel (i0, j0): no
    // point of it within reach of the centre, nor within 1.3 half edges
    bool far(int t, int l, int i0, int j0) const {
        const int T = kNodeTile[l];
        const double need = std::max(reach[t], 1.3 * h[l]);
        if (ortho) {
            const double du = std::max({i0 - cu[t], cu[t] - (i0 + T - 1), 0.0}) * px;
            const double dv = std::max({j0 - cv[t], cv[t] - (j0 + T - 1), 0.0}) * py;
            return du * du + dv * dv + cz2[t] >= need * need;
        }
        const double m = 0.5 * (T - 1);
        const d3 p = quad_at(I.q, (i0 + m) / I.uR, (j0 + m) / I.vR);
        return len(sub(p, mk(sph[t].s.p))) - m * (px + py) >= need;
    }
    // f(sphere) for each of the mask's
    template <class F>
    void each(const unsigned long long* m, F&& f) const {
        for (int w = 0; w < words; ++w)
            for (unsigned long long b = m[w]; b; b &= b - 1) f(64 * w + __builtin_ctzll(b));
    }
    void add(int l, int i0, int j0, const unsigned long long* m, int points) {
        tiles[l].push_back(make_int2(i0, j0));
        mask[l].insert(mask[l].end(), m, m + words);
        double sum = 0.0;
        each(m, [&](int t) { sum += one[t]; });
        cost.work += points * (sum + kPointCost);
        cost.chain = std::max(cost.chain, sum);
    }
    // (left and m of a size of tiles are free again once its cell is cut)
    void cut(int l, int i0, int j0, const unsigned long long* parent) {
        unsigned long long* const left = cell[l].data();
        unsigned long long* const m = left + words;
        std::copy(parent, parent + words, left);
        if (active[l]) {
            std::fill(m, m + words, 0);
            bool any = false;
            each(left, [&](int t) {
                if (!far(t, l, i0, j0)) return;
                m[t >> 6] |= 1ull << (t & 63);
                any = true;
            });
            if (any) add(l, i0, j0, m, (q[l] * q[l] + 63) / 64 * 64);
            for (int w = 0; w < words; ++w) left[w] &= ~m[w];
        }
        if (std::all_of(left, left + words, [](unsigned long long w) { return w == 0; })) return;
        if (l == kNodeLevels - 1) {
            add(kNodeLevels, i0, j0, left, kNearTile * kNearTile);
            return;
        }
        const int T = kNodeTile[l + 1];
        for (int b = 0; b < 2; ++b)
            for (int a = 0; a < 2; ++a)
                if (i0 + a * T < I.uR && j0 + b * T < I.vR) cut(l + 1, i0 + a * T, j0 + b * T, left);
    }
    // the whole slice, and what expanding its pixels costs: 2 q FMAs a pixel
    // for the rows, and the columns' share
    void run() {
        const std::vector<unsigned long long> all = [&] {
            std::vector<unsigned long long> m(words, 0);
            for (int t = 0; t < I.ns; ++t) m[t >> 6] |= 1ull << (t & 63);
            return m;
        }();
        const int T0 = kNodeTile[0];
        for (int j0 = 0; j0 < I.vR; j0 += T0)
            for (int i0 = 0; i0 < I.uR; i0 += T0) cut(0, i0, j0, all.data());
        double fma = 30.0 * I.uR * I.vR;
        for (int l = 0; l < kNodeLevels; ++l) {
            fma += (double)tiles[l].size() * kNodeTile[l] * kNodeTile[l] *
                   (2.0 * q[l] + 2.0 * q[l] * q[l] / std::min(64, kNodeTile[l]));
            cost.levels += !tiles[l].empty();
        }
        cost.work += kExpandCost * fma;
    }
};

}  // namespace

int node_reach(const SphereDev& S, double k, const double* B) {
    double scale = 0.0;
    for (int l = 0; l <= S.Nl; ++l)
        scale += (B[2 * l] * B[2 * l] + B[2 * l + 1] * B[2 * l + 1]) / (2 * l + 1);
    const double most = 1e-8 * std::sqrt(scale);
    double tail = 0.0;
    for (int l = S.Nl; l > 0; --l) {
        tail += kJMin * std::max(1.0, k * S.a) * std::hypot(B[2 * l], B[2 * l + 1]);
        if (!(tail < most)) return l;
    }
    return 1;
}

bool node_mask_any(const unsigned long long* m, int begin, int n) {
    for (int t = begin; t < begin + n; ++t)
        if ((m[t >> 6] >> (t & 63)) & 1) return true;
    return false;
}

NodeCost node_pixel_cost(const SeriesInst& I, const SeriesSph* sph, bool planar) {
    NodeCost c;
    for (int s = 0; s < I.ns; ++s) c.chain += point_cost(sph[s].s.Nl + 1, planar);
    c.work = (c.chain + kPointCost) * I.uR * I.vR;
    return c;
}

NodeCost node_plan_instance(const SeriesInst& I, const SeriesSph* sph, bool planar, NodeTables* t) {
    const int at = (int)t->inst.size();
    t->inst.push_back(NodeInst{});
    const NodeCost pixels = node_pixel_cost(I, sph, planar);
    if (I.ns == 0 || pixels.work < kNodeMinWork) return pixels;
    Tiling wide(I, sph, planar, 0), narrow(I, sph, planar, 1);
    if (narrow.active[1] || narrow.active[2] || narrow.active[3]) narrow.run();
    else return pixels;
    if (wide.active[0]) wide.run();
    Tiling& g = wide.active[0] && wide.cost.work < narrow.cost.work ? wide : narrow;
    if (g.cost.levels == 0 || g.cost.work > 0.8 * pixels.work) return pixels;
    NodeInst& N = t->inst[at];
    N.words = g.words;
    N.tile_first = (int)t->tiles.size();
    N.mask0 = (long long)t->mask.size();
    N.v0 = t->n_v;
    N.w0 = t->n_w;
    auto grid = [&](const std::vector<int2>& tiles, int T, int* gw) {
        const long long o = (long long)t->idx.size();
        *gw = (I.uR + T - 1) / T;
        const int gh = (I.vR + T - 1) / T;
        t->idx.resize(t->idx.size() + (size_t)*gw * gh, -1);
        for (size_t k = 0; k < tiles.size(); ++k)
            t->idx[o + (long long)(tiles[k].y / T) * *gw + tiles[k].x / T] = (int)k;
        return o;
    };
    for (int l = 0; l < kNodeLevels; ++l) {
        if (g.tiles[l].empty()) continue;
        NodeLevel& L = N.lev[N.n_lev++];
        L.T = kNodeTile[l];
        L.q = g.q[l];
        L.tile0 = (int)t->tiles.size();
        L.n_tiles = (int)g.tiles[l].size();
        L.node0 = N.n_nodes;
        N.n_nodes += L.n_tiles * L.q * L.q;
        L.wave0 = N.n_waves;
        L.wpt = (L.q * L.q + 63) / 64;
        N.n_waves += L.n_tiles * L.wpt;
        L.idx0 = grid(g.tiles[l], L.T, &L.gw);
        const auto m = matrix(t, L.T, L.q);
        L.e0 = m.first;
        L.x0 = m.second;
        t->tiles.insert(t->tiles.end(), g.tiles[l].begin(), g.tiles[l].end());
        t->mask.insert(t->mask.end(), g.mask[l].begin(), g.mask[l].end());
    }
    N.near0 = (int)t->tiles.size();
    N.n_near = (int)g.tiles[kNodeLevels].size();
    N.near_idx0 = grid(g.tiles[kNodeLevels], kNearTile, &N.near_gw);
    t->tiles.insert(t->tiles.end(), g.tiles[kNodeLevels].begin(), g.tiles[kNodeLevels].end());
    t->mask.insert(t->mask.end(), g.mask[kNodeLevels].begin(), g.mask[kNodeLevels].end());
    t->n_v += N.n_nodes;
    t->n_w += (long long)N.n_near * kNearTile * kNearTile;
    for (int y = 0; y < (I.vR + kBlock - 1) / kBlock; ++y)
        for (int x = 0; x < (I.uR + kBlock - 1) / kBlock; ++x)
            t->blocks.push_back(make_int4(at, x, y, 0));
    return g.cost;
}

namespace {

// One size of a block's tiles into its pixels (harm_expand_kernel): nb x nb
// tiles of P pixels (P = 64, 32 or 16), their numbers at tiles, or (kBig) the
// quarter (ci, cj) of one of 128.  A round of node rows at a time: their
// values into LDS, V's columns expanded, W[row][i] = sum_a E[a][i] V[row][a],
// then the rows, whose E values every lane of a wave shares.
struct ExpandLds {
    float E[kNodeMaxQ * kBlock];   // [a][column of the block's part]
    float F[kRound * kBlock];      // a tile of 128: [b][row of its part]
    float2 V[kRoundNodes];         // [tile][row][a]
    float2 W[kRound * kBlock];     // [band and row][column]
};

template <int P, bool kBig>
__device__ __forceinline__ void expand_size(ExpandLds& S, const HarmNodes& nodes,
                                            const float2* __restrict__ V, const NodeLevel& L,
                                            const int* tiles, int ci, int cj, float* ar,
                                            float* ai) {
    constexpr int nb = kBig ? 1 : kBlock / P, kWaves = kThreads / 64;
    const int lane = (int)threadIdx.x & 63, g = (int)threadIdx.x >> 6;
    const int q = L.q;
    const int rounds = (nb * q + kRound - 1) / kRound, rows = (q + rounds - 1) / rounds;
    const int il = lane & (P - 1), col = lane / P;
    const float* __restrict__ gE = nodes.E + L.e0;
    constexpr int T = kBig ? 2 * kBlock : P;
    for (int b0 = 0; b0 < q; b0 += rows) {
        const int nr = min(rows, q - b0), per = nr * q;
        __syncthreads();   // the previous round's tables are consumed
        if (b0 == 0)
            for (int t = threadIdx.x; t < q * P; t += kThreads)
                S.E[t] = gE[(t / P) * T + ci + (t & (P - 1))];
        if constexpr (kBig)
            for (int t = threadIdx.x; t < nr * kBlock; t += kThreads)
                S.F[t] = gE[(b0 + t / kBlock) * T + cj + (t & (kBlock - 1))];
        // kWaves / nb^2 waves to a tile, whose rows of the round are one run
        constexpr int share = kThreads / (nb * nb);
        const int mine = (int)threadIdx.x / share;
        const int tile = tiles[mine];
        if (tile >= 0) {
            const float2* __restrict__ v = V + ((long long)tile * q + b0) * q;
            for (int e = (int)threadIdx.x % share; e < per; e += share) S.V[mine * per + e] = v[e];
        }
        __syncthreads();
        for (int r = g; r < nb * nr; r += kWaves) {
            const int band = nb == 1 ? 0 : r / nr, b = r - band * nr;
            const float2* v = S.V + (band * nb + col) * per + b * q;
            float wr = 0.f, wi = 0.f;
            if (nb == 1 || tiles[band * nb + col] >= 0) {
#pragma unroll 4
                for (int a = 0; a < q; ++a) {
                    const float e = S.E[a * P + il];
                    const float2 x = v[a];
                    wr = fmaf(e, x.x, wr);
                    wi = fmaf(e, x.y, wi);
                }
            }
            S.W[r * kBlock + lane] = make_float2(wr, wi);
        }
        __syncthreads();
        const int band = kRows * g / P, j0 = kRows * g - band * P;
        const float2* W = S.W + band * nr * kBlock + lane;
        const float* E = (kBig ? S.F : S.E + b0 * P) + j0;
#pragma unroll 4
        for (int b = 0; b < nr; ++b) {
            const float2 w = W[b * kBlock];
#pragma unroll
            for (int j = 0; j < kRows; ++j) {
                const float e = E[b * P + j];
                ar[j] = fmaf(e, w.x, ar[j]);
                ai[j] = fmaf(e, w.y, ai[j]);
            }
        }
    }
}

// One block of 64 x 64 pixels: E V E^T of its tiles of each size added up,
// then the near tiles.  Lane i of wave g holds pixels (i, 4 g .. 4 g + 3).
// Some 100 to 200 FMAs a pixel; bound by the latency of its phases (global
// loads, two expansions and their barriers, per size) on one image, whose
// blocks are few, and by LDS reads and FMA issue on many.
// Measured: 25 us on a 512 x 512 image, 28 on 1024 x 1024, 0.42 ms on 64 of
// 512 x 512 (tile numbers looked up and divided out per element: 32, 33 and
// 0.51; blocks of 256 lanes, without tiles of 128: 42 on one image).
__global__ __launch_bounds__(kThreads) void harm_expand_kernel(
    const SeriesInst* __restrict__ insts, HarmNodes nodes, const int4* __restrict__ blocks,
    float2* __restrict__ U) {
    __shared__ ExpandLds S;
    __shared__ int s_tile[kNodeLevels][16];   // the block's tiles of each size, or -1
    const int4 B = blocks[blockIdx.x];
    const SeriesInst& I = insts[B.x];
    const NodeInst& N = nodes.inst[B.x];
    const int lane = (int)threadIdx.x & 63, g = (int)threadIdx.x >> 6;
    if (g < N.n_lev && lane < 16) {
        const NodeLevel& L = N.lev[g];
        const int T = L.T, nb = T > kBlock ? 1 : kBlock / T;
        int tile = -1;
        if (lane < nb * nb) {
            const int x = T > kBlock ? B.y >> 1 : B.y * nb + lane % nb;
            const int y = T > kBlock ? B.z >> 1 : B.z * nb + lane / nb;
            if (x < L.gw && y < (I.vR + T - 1) / T)
                tile = nodes.idx[L.idx0 + (long long)y * L.gw + x];
        }
        s_tile[g][lane] = tile;
    }
    float ar[kRows], ai[kRows];
#pragma unroll
    for (int j = 0; j < kRows; ++j) ar[j] = ai[j] = 0.f;
    __syncthreads();
    for (int l = 0; l < N.n_lev; ++l) {
        const NodeLevel& L = N.lev[l];
        const int* tiles = s_tile[l];
        // (every wave asks for the same tiles, so the skip is the block's)
        if (__ballot(lane < 16 && tiles[lane & 15] >= 0) == 0) continue;
        const float2* V = nodes.V + N.v0 + L.node0;
        if (L.T > kBlock)
            expand_size<kBlock, true>(S, nodes, V, L, tiles, (B.y & 1) * kBlock,
                                      (B.z & 1) * kBlock, ar, ai);
        else if (L.T == 64)
            expand_size<64, false>(S, nodes, V, L, tiles, 0, 0, ar, ai);
        else if (L.T == 32)
            expand_size<32, false>(S, nodes, V, L, tiles, 0, 0, ar, ai);
        else
            expand_size<16, false>(S, nodes, V, L, tiles, 0, 0, ar, ai);
    }
    const int iu = kBlock * B.y + lane, j0 = kBlock * B.z + kRows * g;
    if (iu >= I.uR) return;
    if (j0 < I.vR) {
        const int t = nodes.idx[N.near_idx0 + (long long)(j0 / kNearTile) * N.near_gw + iu / kNearTile];
        if (t >= 0) {
            const float2* w = nodes.W + N.w0 + (long long)t * (kNearTile * kNearTile) +
                              (j0 & (kNearTile - 1)) * kNearTile + (lane & (kNearTile - 1));
#pragma unroll
            for (int j = 0; j < kRows; ++j) {
                const float2 x = w[j * kNearTile];
                ar[j] += x.x;
                ai[j] += x.y;
            }
        }
    }
    float2* o = U + I.u_off + (long long)j0 * I.uR + iu;
#pragma unroll
    for (int j = 0; j < kRows; ++j) {
        if (j0 + j < I.vR) {
            float2 v = make_float2(0.f, 0.f);
            if (I.accumulate) v = o[(long long)j * I.uR];
            o[(long long)j * I.uR] = make_float2(v.x + ar[j], v.y + ai[j]);
        }
    }
}

}  // namespace

int node_expand_launch(bimsim_ctx* ctx, const SeriesPlan& P, float2* U) {
    if (P.n_xblocks == 0) return BIMSIM_OK;
    hipLaunchKernelGGL(harm_expand_kernel, dim3((unsigned)P.n_xblocks), dim3(kThreads), 0,
                       ctx->stream, P.d_inst, P.nodes, P.d_xblocks, U);
    BIMSIM_HIP_CHECK(ctx, hipGetLastError());
    return BIMSIM_OK;
}

}  // namespace bimsim
