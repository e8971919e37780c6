// ttsh_dev.h -- device-side data layout shared by the TTSH3D step kernels.
//
// One droplet lives in HBM as unpadded FP32 structure-of-arrays, x fastest and
// z slowest: idx = (z*N + y)*N + x, the interior ordering of the reference's
// padded fields (TTSH3D.cu:477 without the Nb halo).  Periodic boundaries are
// index wraps inside the tile loaders; there are no halo arrays and no halo
// kernels (the reference's BounPeriU, TTSH3D.cu:1422-1607, has no counterpart).
//
// Buffers per droplet (N^3 each unless stated):
//   phi[2]           phase field, ping-pong (K_rhs reads one, writes the other)
//   P[3], v[3]       polarization and flow (updated in place by K_corr)
//   vs[2][3],ps[2][3] predictors v*, P*, ping-pong by step parity; the other
//                    parity holds the previous step's v*, P*, which the
//                    divergence reads across the periodic boundary exactly as
//                    the reference's stale halo does (TTSH3D.cu:366-371,405-407,665-667)
//   c                complex FP32 N^3: (div v* + i div P*)/dt0, transformed in place;
//                    the first forward pass scales the imaginary part by 1/sigma
//
// All kernels take a device table of droplet descriptors and a work table of
// (droplet, tile...) entries, so one launch serves one droplet or a batch of
// droplets of different sizes.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <type_traits>

namespace ttsh {

constexpr int kMaxStages = 8;
constexpr int kMaxN = 256;

// FP32 coefficients of one droplet, computed in FP64 on the host.
struct Coef {
    float d1;         // 1/(2h): first-derivative prefactor (TTSH3D.cu:3287)
    float sw0, sw1;   // transverse smoothing S=[sw1,sw0,sw1] = [1,4,1]/6
    float lc;         // 1/(12 h^2): scale of the whole-number Laplacian (1, 8, -56; TTSH3D.cu:3331-3343)
    float Dt;         // dt0 (Dt never changes in the reference, TTSH3D.cu:759)
    float s;          // 1/(72 h): scale of the whole-number first-derivative stencils
    float inv_dt0;    // 1/dt0, the getStream type-0 divisor (TTSH3D.cu:665)
    float mu, cA, alpha, beta, eta, La2, lambda0, aPhi2, kPhi, gamma, A;
    float pk0;        // -1/(k2s N^3), k2 = k2s*(mx^2+my^2+mz^2), k2s = (2 pi/(N h))^2 (TTSH3D.cu:1094-1114)
    float inv_n3;     // 1/N^3, the type-2 divisor (TTSH3D.cu:687)
    int   anchoring;  // A != 0: evaluate the anchoring term
};

constexpr int kPartSums = 6;

struct Drop {
    int N;
    int nst;                 // FFT stages
    int rad[kMaxStages];     // radices (4, 2 or 3), product N
    const float2* tw;        // exp(-2 pi i q/N), q in [0,N)
    float* phi[2];
    float* P[3];
    float* v[3];
    float* vs[2][3];
    float* ps[2][3];
    float2* c;
    // transposed copy of c, [x][z][y], of sizes up to kMaxPlane: the memory of
    // P and v, whose values are not used between K_rhs and K_corr
    float2* ct;
    // FP64 sums per reduction block, kPartSums each: s.x, s.y, s.x^2, s.y^2
    // over the block's cells and |v*|^2, |P*|^2 over the same cells.  A block
    // is one divergence tile over one of nzp z-ranges (the droplet's tuned
    // z-chunks); npart = tiles * nzp, ordered by z-range, then tile.  A
    // divergence work item covers one or more whole blocks of one tile.
    double* part;
    int npart;
    int nzp;
    // Per step, from the sums of all items (k_proj_stats): stat[0..1] the
    // k = 0 coefficient of s/sigma (FP64); sigma the power-of-two scale of
    // the imaginary part.  The packed transform carries div v* and div P*/
    // sigma, and K_corr multiplies p_p back by sigma: with sigma chosen so
    // that the FP32 rounding of either half disturbs the other by the same
    // relative amount in the corrected v and P, a droplet whose div P* is
    // orders of magnitude above its div v* keeps the accuracy of v.
    double* stat;
    float* sigma;
    // x = 0 and x = N-1 columns of v*, P* per parity slot, laid out with a
    // field's z-stride: plane z holds at ((slot*6 + f)*2 + side)*N + y the
    // value of field f (vx..vz, Px..Pz) at x = side ? N-1 : 0, row y.  The
    // stale-halo divergence reads the previous step's columns here instead
    // of fetching a whole cache line of the previous predictor per row end.
    // eslot[p] is the slot of the predictors in vs[p], ps[p].
    float* edge;
    int eslot[2];
    int faithful;            // 1: stale-halo divergence (the reference's semantics)
    int nsteps;              // steps this droplet takes in the current launch sequence
    Coef co;
};

// Work item: droplet index and up to three tile coordinates.  Kernels skip an
// item whose droplet has nsteps <= kstep (the step index within a launch
// sequence), so droplets with different step budgets share one sequence.
struct Work {
    int d, a, b, c;
};

// K_rhs's tiles for a box of N.  A tile row has at most W records, four of
// which are apron; the box's rows are cut into equal parts.  A tile has one
// row per wave (W = 64), or as many as fit the waves' 60 positions each.
__host__ __device__ constexpr int rhs_tiles_x(int N, int W) { return (N + W - 5) / (W - 4); }
__host__ __device__ constexpr int rhs_tile_width(int N, int W) { return (N + rhs_tiles_x(N, W) - 1) / rhs_tiles_x(N, W); }
__host__ __device__ constexpr int rhs_tile_rows(int NW, int W) { return W == 64 ? NW : NW * 60 / W; }

// Tiles of the divergence: a wave is a row whose 64 lanes
// include one apron cell on each side, a work-group 16 rows of which the
// first and last are apron.
constexpr int kProjWaves = 16;
constexpr int kProjRows = kProjWaves - 2;
constexpr int kProjMaxTX = 62;
__host__ __device__ constexpr int proj_tiles_x(int N) { return (N + kProjMaxTX - 1) / kProjMaxTX; }
__host__ __device__ constexpr int proj_tile_width(int N) { return (N + proj_tiles_x(N) - 1) / proj_tiles_x(N); }
__host__ __device__ constexpr int proj_tiles(int N) { return proj_tiles_x(N) * ((N + kProjRows - 1) / kProjRows); }

// Work-groups are dispatched round-robin over the 8 XCDs, each with its own
// L2.  Visit v of the grid-stride loop maps to work item
//   (v mod 8) * chunk + v / 8,   chunk = ceil(nwork / 8),
// so each XCD processes one contiguous, spatially ordered block of the work
// table and tiles that share halo cache lines share an L2.  The loop runs v
// over [0, 8*chunk) and skips items >= nwork.
constexpr int kXcds = 8;
__device__ __forceinline__ int xcd_span(int nwork) { return kXcds * ((nwork + kXcds - 1) / kXcds); }
__device__ __forceinline__ int xcd_item(int v, int nwork)
{
    const int chunk = (nwork + kXcds - 1) / kXcds;
    return (v % kXcds) * chunk + v / kXcds;
}

// Global-memory views of the descriptor's pointers.  Pointers read from a
// table in memory are generic to the compiler, which then emits flat loads and
// stores; those count against the LDS wait counter too, so the first LDS wait
// after a prefetch would also wait for the prefetch's HBM loads.  A cast to
// the global address space gives global loads, tracked by the vector-memory
// counter alone.
template <typename T>
using gptr = __attribute__((address_space(1))) T*;
template <typename T>
__device__ __forceinline__ gptr<T> glb(T* p)
{
    return (gptr<T>)p;
}

// float2 elements of global memory go through a plain two-float vector: the
// HIP float2 class has no assignment operators for an address-space-qualified
// object.
typedef float fvec2 __attribute__((ext_vector_type(2)));
typedef float fvec4 __attribute__((ext_vector_type(4)));
__device__ __forceinline__ float2 ld2(gptr<const float2> p, size_t i)
{
    const fvec2 t = *(gptr<const fvec2>)(p + i);
    return make_float2(t.x, t.y);
}
__device__ __forceinline__ void st2(gptr<float2> p, size_t i, float2 v)
{
    fvec2 t;
    t.x = v.x;
    t.y = v.y;
    *(gptr<fvec2>)(p + i) = t;
}

// Byte-offset access to a plane: a uniform base plus a 32-bit per-lane byte
// offset, the form of a global load or store with a scalar base address.
__device__ __forceinline__ float ldb(gptr<const float> base, unsigned boff)
{
    return *(gptr<const float>)((gptr<const char>)base + boff);
}
__device__ __forceinline__ void stb(gptr<float> base, unsigned boff, float v)
{
    *(gptr<float>)((gptr<char>)base + boff) = v;
}

// A value that the compiler cannot derive, so that a global access keeps its
// scalar base and 32-bit lane offset instead of a hoisted 64-bit address.
__device__ __forceinline__ unsigned opaque(unsigned a)
{
    asm volatile("" : "+v"(a));
    return a;
}

__device__ __forceinline__ float fma_(float a, float b, float c) { return __builtin_fmaf(a, b, c); }

// The value of the lane at x-1 / x+1 of a wave that is a row of cells (DPP
// wave_shr:1, wave_shl:1; 0 past the ends of the wave, whose lanes are apron).
__device__ __forceinline__ float from_left(float a)
{
    return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(a), 0x138, 0xf, 0xf, true));
}
__device__ __forceinline__ float from_right(float a)
{
    return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(a), 0x130, 0xf, 0xf, true));
}
__device__ __forceinline__ float xpair(float a) { return from_left(a) + from_right(a); }
__device__ __forceinline__ float xdiff(float a) { return from_right(a) - from_left(a); }

// Adds to each value the one that DPP control CTRL brings, 0 where none comes.
template <int CTRL, int N>
__device__ __forceinline__ void dpp_add(double (&e)[N])
{
#pragma unroll
    for (int k = 0; k < N; ++k) {
        const unsigned long long b = __double_as_longlong(e[k]);
        const unsigned lo = __builtin_amdgcn_update_dpp(0, (int)(unsigned)b, CTRL, 0xf, 0xf, false);
        const unsigned hi = __builtin_amdgcn_update_dpp(0, (int)(unsigned)(b >> 32), CTRL, 0xf, 0xf, false);
        e[k] += __longlong_as_double((long long)(((unsigned long long)hi << 32) | lo));
    }
}

// Sums over a wave, complete in lane 63: row_shr 1, 2, 4, 8 and the two row
// broadcasts.  Shuffles through LDS would take 72 ds_bpermute, 3 us for the 16
// waves of a work-group; this takes 0.7.
template <int N>
__device__ __forceinline__ void wave_sum(double (&e)[N])
{
    dpp_add<0x111>(e);
    dpp_add<0x112>(e);
    dpp_add<0x114>(e);
    dpp_add<0x118>(e);
    dpp_add<0x142>(e);
    dpp_add<0x143>(e);
}

// log2 x for x >= 0 (-inf at 0, +inf at inf): exponent plus the FP32 log2 of
// the mantissa, enough for a rounded power of two
__device__ __forceinline__ double log2_coarse(double x)
{
    if (!(x > 0.0)) return -INFINITY;
    if (x == INFINITY) return INFINITY;
    int ex;
    const double m = frexp(x, &ex);
    return (double)ex + (double)log2f((float)m);
}

// log2 of this step's sigma from the projection's sums (derivation in
// k_proj.hip).  log2 of 0 is -inf, of inf +inf; -inf + inf is NaN.
__device__ __forceinline__ int proj_sigma_log2(const double (&t)[kPartSums])
{
    const double l = 0.25 * ((log2_coarse(t[3]) + log2_coarse(t[5])) - (log2_coarse(t[2]) + log2_coarse(t[4])));
    return t[3] > 0.0 && l == l ? (int)rint(fmin(fmax(l, -30.0), 30.0)) : 0;
}
__device__ __forceinline__ void put_proj_stats(const Drop& D, const double (&t)[kPartSums], int e)
{
    glb(D.sigma)[0] = ldexpf(1.f, e);
    glb(D.stat)[0] = t[0];
    glb(D.stat)[1] = ldexp(t[1], -e);
}

// The projection's sums of a droplet of at most kFoldedParts reduction blocks,
// by one wave: lane l adds the blocks l, l + 64, ..., then the lanes are added;
// t is complete in lane 63.  In a forward x pass of few work-groups every one
// does this while its lines are on their way (FFT_MODE_FWD_FOLD), which saves
// the launch of k_proj_stats: steps of 36.1 -> 34.8 us at 32^3, 51.4 -> 49.5 at
// 64^3, 130 -> 128 at 128^3.  With many groups the repeated sums cost more
// than the launch (the 20-droplet sweep: x pass 58 -> 87 us).  The order does
// not depend on the work-group or the kernel, so all get the same sigma.
constexpr int kFoldedParts = 512;
__device__ __forceinline__ void fold_proj_stats(const Drop& D, int lane, double (&t)[kPartSums])
{
    const gptr<const double> pt = glb<const double>(D.part);
    const int np = D.npart;
#pragma unroll
    for (int k = 0; k < kPartSums; ++k) t[k] = 0.0;
#pragma unroll 4
    for (int j = lane; j < np; j += 64) {
#pragma unroll
        for (int k = 0; k < kPartSums; ++k) t[k] += pt[(size_t)kPartSums * j + k];
    }
    wave_sum(t);
}

// Compile-time phase of an unrolled z-march (register slot rotation).
template <int K>
using Ph = std::integral_constant<int, K>;

// Waits for every outstanding vector-memory load (s_waitcnt vmcnt(0), the
// export and LDS counters left at their maxima).  Issued at the end of a
// prologue whose loads fill a loop's rolling registers, so the compiler's
// wait analysis enters the loop with no load pending and does not fence the
// loop's own prefetch of the next plane behind later LDS traffic.
__device__ __forceinline__ void wait_vmem() { __builtin_amdgcn_s_waitcnt(0x0F70); }

__device__ __forceinline__ int wrapi(int i, int N)
{
    i += (i < 0) ? N : 0;
    i -= (i >= N) ? N : 0;
    return i;
}

__device__ __forceinline__ size_t gidx(int N, int x, int y, int z)
{
    return ((size_t)z * (size_t)N + (size_t)y) * (size_t)N + (size_t)x;
}

}  // namespace ttsh
