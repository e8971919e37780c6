// ttsh_layout.h -- which K_rhs tile a droplet runs, and z-depths of the step
// kernels' work items over the active droplets of a batch, by predicted time.
// Host code without HIP; the tile counts of the kernels are passed in.
#pragma once
#include <algorithm>
#include <cmath>
#include <vector>

namespace ttsh {

// K_rhs variants, as callers and tuning tables number them 0 .. 6.  There are
// three kernels, named here by the largest tile they run; 0, 2, 4 and 6 are
// further numbers of the second.
enum RhsVariant { RHS_60x16 = 1, RHS_60x8 = 3, RHS_32x26 = 5, RHS_NVARIANTS = 7 };

// By number: the smallest box that it is taken for (every kernel runs every
// size; a number keeps the bound that callers know it by), and the waves and
// records per tile row of its kernel.
struct RhsVar {
    int least, nw, w;
};
constexpr RhsVar kRhsVars[RHS_NVARIANTS] = {
    {34, 8, 64}, {18, 16, 64}, {66, 8, 64}, {18, 8, 64}, {34, 8, 64}, {34, 16, 36}, {66, 8, 64},
};
inline bool rhs_fits(int variant, int N)
{
    return variant >= 0 && variant < RHS_NVARIANTS && N >= kRhsVars[variant].least;
}

// K_rhs variant of a new droplet of size N: the one it asks for, or the tuning
// table's where that fits, or 60 x 16, which is taken for every size (-1: none).
// own: for the droplet by itself; engine: for droplets that share launches with
// one that asks, `engine` before; -1: it asks for one that does not fit.
struct RhsChoice {
    int own, engine;
};
inline RhsChoice choose_rhs(int N, int asked, int tuned, int engine)
{
    const int own = asked >= 0 ? asked : rhs_fits(tuned, N) ? tuned : (int)RHS_60x16;
    const int v = engine < 0 ? own : engine;
    if (rhs_fits(v, N)) return {own, v};
    return {own, asked >= 0 ? -1 : (int)RHS_60x16};
}

// Active droplets of one size and one depth of reduction blocks.  The
// predictions below run over these and not over the slots: at many depths each,
// for a batch of 4,096 slots they took 1 to 1.5 ms of a table rebuild that way.
struct SizeCount {
    int N, proj_tz, n;
};

inline void count_size(std::vector<SizeCount>& sizes, int N, int proj_tz)
{
    for (SizeCount& s : sizes)
        if (s.N == N && s.proj_tz == proj_tz) {
            ++s.n;
            return;
        }
    sizes.push_back(SizeCount{N, proj_tz, 1});
}

// z is split into ceil(N/d) chunks of near-equal depth.
inline int z_chunks(int N, int d) { return (N + d - 1) / d; }

// Depths 1 .. most that split some size differently from the depth before.
inline std::vector<int> chunk_depths(const std::vector<SizeCount>& sizes, int most)
{
    std::vector<int> out;
    for (int d = 1; d <= most; ++d) {
        bool differs = d == 1;
        for (const SizeCount& s : sizes) differs = differs || z_chunks(s.N, d) != z_chunks(s.N, d - 1);
        if (differs) out.push_back(d);
    }
    return out;
}

// Predicted time of z-chunks of depth d, in plane iterations of one
// work-group: `over` iterations of a chunk (planes beyond its own, loading,
// launch) come on top of d, `at_once` groups run together, and a last round
// that is partly empty counts whole while there are few rounds.
template <typename Tiles>
double chunk_time(const std::vector<SizeCount>& sizes, int d, double over, double at_once, Tiles&& tiles)
{
    double items = 0.0, deepest = 0.0;
    for (const SizeCount& s : sizes) {
        const int nz = z_chunks(s.N, d);
        items += (double)tiles(s.N) * nz * s.n;
        deepest = std::max(deepest, (double)((s.N + nz - 1) / nz));
    }
    const double rounds = items / at_once;
    return (rounds < 3.0 ? std::ceil(rounds) : rounds + 0.5) * (deepest + over);
}

// The first of the depths with the least predicted time.
struct Depth {
    int d;
    double time;
};
template <typename Tiles>
Depth least_depth(const std::vector<SizeCount>& sizes, const std::vector<int>& depths, double over, double at_once,
                  Tiles&& tiles)
{
    Depth best{0, 0.0};
    for (int d : depths) {
        const double t = chunk_time(sizes, d, over, at_once, tiles);
        if (!best.d || t < best.time) best = Depth{d, t};
    }
    return best;
}

// Reduction blocks of a divergence item: items of about d planes, and at most
// eight blocks, since a block's sums cost about half a plane and droplets with
// blocks of one plane would hold up the launch.
inline int div_blocks(int N, int proj_tz, int d)
{
    const int nzp = z_chunks(N, proj_tz);
    return std::max(1, std::min({nzp, 8, d * nzp / N}));
}

// Depth (at most `most`) of K_div's items with the least predicted time: all
// items over two groups per CU, and half of the longest item for the end.
template <typename Tiles>
int div_depth(const std::vector<SizeCount>& sizes, int most, int cus, Tiles&& tiles)
{
    int depth = 1;
    double best = 0.0;
    for (int d = 1; d <= most; ++d) {
        double all = 0.0, longest = 0.0;
        for (const SizeCount& s : sizes) {
            const int nzp = z_chunks(s.N, s.proj_tz), g = div_blocks(s.N, s.proj_tz, d);
            const double c = (double)s.N * g / nzp + 3.0 + 0.5 * g;
            all += c * tiles(s.N) * ((nzp + g - 1) / g) * s.n;
            longest = std::max(longest, c);
        }
        const double rounds = all / (2.0 * cus * longest);
        const double t = rounds < 1.0 ? longest : all / (2.0 * cus) + 0.5 * longest;
        if (d > 1 && t >= best) continue;
        best = t;
        depth = d;
    }
    return depth;
}

}  // namespace ttsh
