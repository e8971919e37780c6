// k_proj.hip -- divergence (K_div) and corrector (K_corr) stencils of the
// projection, and the FP64 reductions.
//
// Reference: getStream type 0 (TTSH3D.cu:654-669), getVNew (TTSH3D.cu:494-516).
// The reference projects v* and P* with two complex transforms each; since
// -1/k^2 is real and even, packing div v* into the real part and div P* into
// the imaginary part of one complex field gives IFFT(-FFT(a + i b)/k^2) =
// p_v + i p_p exactly, so K_div writes s = (D.v* + i D.P*)/dt0 and K_corr
// reads p_v + i p_p after the inverse transforms (k_fft.hip).
//
// In FP32 the rounding of the larger half of s leaks into the smaller one.
// An aster's div P* can exceed div v* by 10^2 and its P by 10^3 its v; left
// unscaled, v then loses three digits in the first step.  k_proj_stats
// picks a power of two sigma per droplet and step; the first forward pass
// divides the imaginary part by it and K_corr multiplies p_p back (both
// exact).  Cross-talk into v scales with |div P*|/(sigma |div v*|) relative
// to |P|/|v|, into P with the inverse, so
//   sigma^4 = (sum (div P*)^2 sum |P*|^2) / (sum (div v*)^2 sum |v*|^2)
// gives both corrected fields the same relative share, rounded to 2^e,
// |e| <= 30 (e = 0 when s has no imaginary part or a sum is undefined).
//
// K_div applies the stencils one axis at a time, like K_rhs (k_rhs.hip): a wave
// is a row of cells, marching in z with three planes of every value in
// registers.  With S = [1,4,1], d = [-1,0,1] and s = 1/(72 h),
// D_x = s d_x S_y S_z, D_y = s S_x d_y S_z, D_z = s S_x S_y d_z
// (TTSH3D.cu:3280-3328):
//   z  a = S_z f, b = d_z f
//   x  X = d_x a, A = S_x a, B = S_x b, by DPP wave shifts
//   y  4 X + Xm + Xp, Ap - Am, 4 B + Bm + Bp with the rows at y-1 (m) and y+1
//      (p), whose values come through LDS
// so a plane costs one barrier (two LDS buffers) and no 2D neighbourhood is
// read from LDS.  K_corr is a z-marching 2D tile.
//
// K_div reproduces the reference's stale halo: an apron or wrapped-plane
// position, i.e. any position outside the box that the reference reads from
// its halo, is taken from the previous step's v*, P* (TTSH3D.cu:366-371,
// 405-407: the halo was filled before getVStar overwrote the interior).
#include "ttsh_dev.h"
#include "ttsh_kernels.h"

namespace ttsh {

// K_div.  The divergence needs X of the x field, A of the y field and B of the
// z field; a row's part of its neighbours' sum is U = X + A + B for the row
// below and W = X - A + B for the row above, so each of the two divergences
// exchanges two values.
//
// Bound by HBM when the device is full.  The 32x8 tile it replaces read 3x3
// neighbourhoods of six fields from LDS behind two barriers per plane and
// fetched a 33% ring; here the apron is 64*16/(62*14), 18%.  Waves hold 64
// VGPRs, so that two work-groups share a CU and one loads while the other
// waits at its barrier.  Measured with the 4.7 us of k_proj_stats, which lone
// droplets up to 128^3 do without: 96^3 19.5 -> 15.8 us, 128^3 26.1 -> 23.1,
// 180^3 70 -> 55, 256^3 166 -> 142; k_div alone moves 604 MB in 137 us at 256^3,
// 4.4 TB/s.
__global__ __launch_bounds__(64 * kProjWaves, 8) void k_div(const Drop* __restrict__ drops,
                                                            const Work* __restrict__ work,
                                                            const int* __restrict__ nwork_p, int parity, int kstep)
{
    // every fused multiply-add is written out, so that a cell's result does not
    // depend on how the loop was compiled
#pragma clang fp contract(off)
    __shared__ float4 rec[2][kProjWaves * 64];  // U_v, W_v, U_p, W_p of a row
    __shared__ double red[2][kPartSums * kProjWaves];
    const int lane = threadIdx.x & 63;
    const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int nwork = *nwork_p;
    for (int vi = blockIdx.x; vi < xcd_span(nwork); vi += gridDim.x) {
        const int w = xcd_item(vi, nwork);
        if (w >= nwork) continue;
        const Work wk = work[w];
        const Drop& D = drops[wk.d];
        if (kstep >= D.nsteps) continue;
        const int N = D.N;
        const int nbx = proj_tiles_x(N), TX = proj_tile_width(N);
        const int x0 = (wk.a % nbx) * TX, y0 = (wk.a / nbx) * kProjRows;
        const int zb = wk.b & 0xffff, ze = wk.b >> 16;
        const int pp = D.faithful ? (parity ^ 1) : parity;
        const unsigned NN = (unsigned)N * (unsigned)N;  // 4 N^3 bytes of a field fit 32 bits
        // Own cell: lanes 1 .. TX of waves 1 .. 14.  Lanes and rows past the
        // tile load some cell of the box (x0 + 62 and y0 + 14 are below 2 N).
        const int gx = x0 + lane - 1, gy = y0 + wv - 1;
        const bool own = lane >= 1 && lane <= TX && gx < N && wv >= 1 && wv <= kProjRows && gy < N;
        const bool outside = gx < 0 || gx >= N || gy < 0 || gy >= N;
        const unsigned o = 4u * ((unsigned)wrapi(gy, N) * (unsigned)N + (unsigned)wrapi(gx, N));
        // Per field, the current and the previous step's buffer are addressed
        // from the lower of the two (scalar base) with a per-lane byte offset
        // that adds the distance to reach the higher one; the buffers of a
        // droplet share one allocation, so the distance fits 32 bits.  In the
        // stale-halo mode, lanes outside the box in x read the previous step's
        // x = 0 / x = N-1 columns from the edge buffer (same z-stride as a
        // field, so the same scalar base serves; K_corr writes each step's
        // columns).  A plane outside the box in z is read wholly from the
        // previous step's buffers.
        gptr<const float> lo[6], prv[6];
        unsigned off[6];
        const bool xedge = D.faithful != 0 && (gx < 0 || gx >= N);
        const unsigned col = 4u * (unsigned)((D.eslot[pp] * 12 + (gx < 0 ? 1 : 0)) * N + wrapi(gy, N));
#pragma unroll
        for (int f = 0; f < 6; ++f) {
            const gptr<const float> c = glb<const float>(f < 3 ? D.vs[parity][f] : D.ps[parity][f - 3]);
            prv[f] = glb<const float>(f < 3 ? D.vs[pp][f] : D.ps[pp][f - 3]);
            const bool hi = prv[f] > c;
            lo[f] = hi ? c : prv[f];
            const unsigned dist = 4u * (unsigned)(hi ? prv[f] - c : c - prv[f]);
            off[f] = xedge ? 4u * (unsigned)(glb<const float>(D.edge) - lo[f]) + col + 8u * (unsigned)(f * N)
                           : o + (outside == hi ? dist : 0u);
        }
        float q[6][3];
        auto fetch = [&](int slot, int z) {
            const unsigned zo = (unsigned)wrapi(z, N) * NN;
            if (z >= 0 && z < N) {
#pragma unroll
                for (int f = 0; f < 6; ++f) q[f][slot] = ldb(lo[f] + zo, opaque(off[f]));
            } else {
                const unsigned oo = opaque(o);
#pragma unroll
                for (int f = 0; f < 6; ++f) q[f][slot] = ldb(prv[f] + zo, oo);
            }
        };
        // sums over this item's cells (see Drop::part): s in FP64 (the k = 0
        // coefficient), the squares, which only set sigma, per thread in FP32
        double d0 = 0.0, d1 = 0.0;
        float q2 = 0.f, q3 = 0.f, q4 = 0.f, q5 = 0.f;
        // The sums are written per reduction block (see Drop::part): the item
        // starts at block wk.c, and at the last plane of each block every wave
        // reduces its sums and starts the next.  The sums of a block are then
        // the same whichever item covers it.  The waves' sums are added, in
        // order, behind the next plane's barrier (or the one after the last
        // plane), so that a block costs no barrier of its own; two buffers
        // keep them until then.
        const int ntile = proj_tiles(N);
        int ordb = wk.c;
        int zend = (wk.c / ntile + 1) * N / D.nzp;
        bool pending = false;  // uniform across the work-group, as is rb
        int rb = 0;
        auto flush = [&]() {
            double e[kPartSums] = {d0, d1, q2, q3, q4, q5};
            wave_sum(e);
            if (lane == 63) {
#pragma unroll
                for (int k = 0; k < kPartSums; ++k) red[rb][kPartSums * wv + k] = e[k];
            }
            d0 = d1 = 0.0;
            q2 = q3 = q4 = q5 = 0.f;
            pending = true;
        };
        auto finish = [&]() {
            if (threadIdx.x < kPartSums) {
                double a = 0.0;
#pragma unroll
                for (int i = 0; i < kProjWaves; ++i) a += red[rb][kPartSums * i + threadIdx.x];
                glb(D.part)[(size_t)kPartSums * ordb + threadIdx.x] = a;
            }
            pending = false;
            rb ^= 1;
            ordb += ntile;
            zend = (ordb / ntile + 1) * N / D.nzp;
        };
        // D.v*/dt0 and D.P*/dt0 of a cell
        // (s/dt0 rounded once from FP64 is nearer on the whole, but at dt0 = 0.01
        // and h = 1 it is low, as the transform's constants are, and a step at
        // 32^3 is then off by 9.8e-8 instead of 9.4e-8)
        const float scale = D.co.s * D.co.inv_dt0;
        const unsigned oc = 2u * o;
        int buf = 0;
        const int own_i = wv * 64 + lane;
        const int below = max(wv - 1, 0) * 64 + lane, above = min(wv + 1, kProjWaves - 1) * 64 + lane;
        auto body = [&](auto ph, int zm) {
            constexpr int S0 = decltype(ph)::value, S1 = (S0 + 1) % 3, S2 = (S0 + 2) % 3;
            float xb[2], u[2], v[2];
#pragma unroll
            for (int F = 0; F < 2; ++F) {
                const float* fx = q[3 * F];
                const float* fy = q[3 * F + 1];
                const float* fz = q[3 * F + 2];
                const float ax = fma_(4.f, fx[S1], fx[S0] + fx[S2]);
                const float ay = fma_(4.f, fy[S1], fy[S0] + fy[S2]);
                const float b = fz[S2] - fz[S0];
                const float A = fma_(4.f, ay, xpair(ay));
                xb[F] = xdiff(ax) + fma_(4.f, b, xpair(b));
                u[F] = xb[F] + A;
                v[F] = xb[F] - A;
            }
            rec[buf][own_i] = make_float4(u[0], v[0], u[1], v[1]);
            if (own) {
                q4 = fma_(q[0][S1], q[0][S1], fma_(q[1][S1], q[1][S1], fma_(q[2][S1], q[2][S1], q4)));
                q5 = fma_(q[3][S1], q[3][S1], fma_(q[4][S1], q[4][S1], fma_(q[5][S1], q[5][S1], q5)));
            }
            fetch(S0, min(zm + 2, ze));  // past ze: a redundant reload of plane ze
            __syncthreads();
            const float4 m = rec[buf][below], p = rec[buf][above];
            buf ^= 1;
            if (pending) finish();
            if (own) {
                fvec2 sv;
                sv.x = scale * fma_(4.f, xb[0], m.y + p.x);
                sv.y = scale * fma_(4.f, xb[1], m.w + p.z);
                *(gptr<fvec2>)((gptr<char>)(D.c + (unsigned)zm * NN) + opaque(oc)) = sv;
                d0 += (double)sv.x;
                d1 += (double)sv.y;
                q2 = fma_(sv.x, sv.x, q2);
                q3 = fma_(sv.y, sv.y, q3);
            }
            if (zm == zend - 1) flush();  // uniform across the work-group
        };
        fetch(0, zb - 1);
        fetch(1, zb);
        fetch(2, zb + 1);
        wait_vmem();
        __syncthreads();  // the previous item has read both buffers
        for (int zm = zb;;) {
            body(Ph<0>{}, zm);
            if (++zm >= ze) break;
            body(Ph<1>{}, zm);
            if (++zm >= ze) break;
            body(Ph<2>{}, zm);
            if (++zm >= ze) break;
        }
        // the item ends at a block end
        __syncthreads();
        if (pending) finish();
    }
}

// One work-group per droplet (work item (d, -, -)): the sums of its reduction
// blocks, then the k = 0 coefficient of s/sigma and this step's sigma
// (derivation at the top of this file).  Up to kFoldedParts blocks one wave
// adds them as the forward x pass would (fold_proj_stats), so that the result
// is the same where that does it.
constexpr int kStatsThreads = 256;

__global__ __launch_bounds__(kStatsThreads) void k_proj_stats(const Drop* __restrict__ drops,
                                                              const Work* __restrict__ work,
                                                              const int* __restrict__ nwork_p, int kstep)
{
    constexpr int NW = kStatsThreads / 64;
    __shared__ double red[kPartSums * NW];
    __shared__ double tot[kPartSums];
    const int tid = threadIdx.x;
    const int nwork = *nwork_p;
    for (int w = blockIdx.x; w < nwork; w += gridDim.x) {
        const Drop& D = drops[work[w].d];
        if (kstep >= D.nsteps) continue;
        const int np = D.npart;
        if (np <= kFoldedParts) {
            if (tid < 64) {
                double t[kPartSums];
                fold_proj_stats(D, tid, t);
                if (tid == 63) put_proj_stats(D, t, proj_sigma_log2(t));
            }
            continue;
        }
        const gptr<const double> pt = glb<const double>(D.part);
        double q[kPartSums] = {0.0, 0.0, 0.0, 0.0, 0.0, 0.0};
#pragma unroll 4
        for (int j = tid; j < np; j += kStatsThreads) {
#pragma unroll
            for (int e = 0; e < kPartSums; ++e) q[e] += pt[(size_t)kPartSums * j + e];
        }
#pragma unroll
        for (int off = 32; off > 0; off >>= 1) {
#pragma unroll
            for (int e = 0; e < kPartSums; ++e) q[e] += __shfl_down(q[e], off, 64);
        }
        __syncthreads();
        if ((tid & 63) == 0) {
#pragma unroll
            for (int e = 0; e < kPartSums; ++e) red[kPartSums * (tid >> 6) + e] = q[e];
        }
        __syncthreads();
        if (tid < kPartSums) {
            double a = 0.0;
#pragma unroll
            for (int i = 0; i < NW; ++i) a += red[kPartSums * i + tid];
            tot[tid] = a;
        }
        __syncthreads();
        if (tid == 0) {
            double t[kPartSums];
#pragma unroll
            for (int e = 0; e < kPartSums; ++e) t[e] = tot[e];
            put_proj_stats(D, t, proj_sigma_log2(t));
        }
    }
}

template <int TX, int TY>
__global__ __launch_bounds__(TX * TY) void k_corr(const Drop* __restrict__ drops, const Work* __restrict__ work,
                                                  const int* __restrict__ nwork_p, int parity, int kstep)
{
    constexpr int NT = TX * TY, W1 = TX + 2, A1 = W1 * (TY + 2);
    __shared__ float2 sp[A1];
    const int tid = threadIdx.x, tx = tid % TX, ty = tid / TX;
    const int nwork = *nwork_p;
    for (int v = blockIdx.x; v < xcd_span(nwork); v += gridDim.x) {
        const int w = xcd_item(v, nwork);
        if (w >= nwork) continue;
        const Work wk = work[w];
        const Drop& D = drops[wk.d];
        if (kstep >= D.nsteps) continue;
        const int N = D.N;
        const Coef co = D.co;
        const int nbx = (N + TX - 1) / TX;
        const int x0 = (wk.a % nbx) * TX, y0 = (wk.a / nbx) * TY;
        const int zb = wk.b & 0xffff, ze = wk.b >> 16;
        const gptr<const float2> c = glb<const float2>(D.c);
        // p_p = sigma * Im(p): the power-of-two scale folded into Dt
        const float dts = co.Dt * glb(D.sigma)[0];
        gptr<const float> src[6];
        gptr<float> dst[6];
#pragma unroll
        for (int f = 0; f < 3; ++f) {
            src[f] = glb<const float>(D.vs[parity][f]);
            src[3 + f] = glb<const float>(D.ps[parity][f]);
            dst[f] = glb(D.v[f]);
            dst[3 + f] = glb(D.P[f]);
        }
        const int gx = x0 + tx, gy = y0 + ty;
        const bool own = gx < N && gy < N;
        // accumulators of D_x p, D_y p, D_z p (complex) for planes zi-1, zi, zi+1
        float2 xm = {0.f, 0.f}, xc = {0.f, 0.f}, xp = {0.f, 0.f};
        float2 ym = {0.f, 0.f}, yc = {0.f, 0.f}, yp = {0.f, 0.f};
        float2 zmv = {0.f, 0.f}, zcv = {0.f, 0.f}, zpv = {0.f, 0.f};
        // planes of p are loaded two ahead into two register slots, with the
        // v*, P* of the own cell at the plane finished by the slot's
        // iteration; loads are unconditional (clamped positions and planes)
        // so no register needs a merge copy
        // slot 0: the own cell (whole aligned rows per wave); slot 1: the
        // one-cell ring around the tile, clamped so every thread loads it
        static_assert(A1 - NT == 2 * W1 + 2 * TY, "slot 1 holds the ring");
        constexpr int MAXP = 2;
        unsigned off[MAXP];
        int lds_i[MAXP];  // the position's LDS index (-1: nothing to store)
#pragma unroll
        for (int k = 0; k < MAXP; ++k) {
            int i;
            if (k == 0) {
                i = (ty + 1) * W1 + (tx + 1);
                lds_i[k] = i;
            } else {
                const int r = min(tid, 2 * W1 + 2 * TY - 1);
                if (r < W1) i = r;                                      // row y0-1
                else if (r < 2 * W1) i = (TY + 1) * W1 + (r - W1);      // row y0+TY
                else if (r < 2 * W1 + TY) i = (r - 2 * W1 + 1) * W1;    // column x0-1
                else i = (r - 2 * W1 - TY + 1) * W1 + (W1 - 1);         // column x0+TX
                lds_i[k] = tid < 2 * W1 + 2 * TY ? i : -1;
            }
            off[k] = (unsigned)wrapi(y0 - 1 + i / W1, N) * (unsigned)N + (unsigned)wrapi(x0 - 1 + i % W1, N);
        }
        const unsigned own_off = 4u * ((unsigned)min(gy, N - 1) * (unsigned)N + (unsigned)min(gx, N - 1));
        const size_t NN = (size_t)N * N;
        // In the stale-halo mode the cells at x = 0 and x = N-1 also store
        // this step's v*, P* in the edge buffer: the next step's divergence
        // reads them there (the layout of Drop::edge).
        const bool ewr = D.faithful != 0 && own && (gx == 0 || gx == N - 1);
        const unsigned ewo = 4u * (unsigned)(((D.eslot[parity] * 6) * 2 + (gx == 0 ? 0 : 1)) * N + min(gy, N - 1));
        float2 pre[2][MAXP];
        float sv[2][6];
        auto fetch = [&](int slot, int zi) {
            const gptr<const float2> cz = c + (size_t)wrapi(zi, N) * NN;
#pragma unroll
            for (int k = 0; k < MAXP; ++k) pre[slot][k] = ld2(cz, off[k]);
            // own-cell predictors of plane zi-1, the output of iteration zi
            const size_t zo = (size_t)wrapi(max(zi - 1, zb), N) * NN;
#pragma unroll
            for (int f = 0; f < 6; ++f) sv[slot][f] = ldb(src[f] + zo, own_off);
        };
        auto body = [&](auto ph, int zi) {
            constexpr int S = decltype(ph)::value;
            __syncthreads();
#pragma unroll
            for (int k = 0; k < MAXP; ++k) {
                const int i = lds_i[k];
                if (i >= 0) sp[i] = pre[S][k];
            }
            // this iteration's own-cell predictors, before the slot is reused
            float svc[6];
#pragma unroll
            for (int f = 0; f < 6; ++f) svc[f] = sv[S][f];
            fetch(S, min(zi + 2, ze));  // past ze: a redundant reload of plane ze
            __syncthreads();
            const int o = (ty + 1) * W1 + (tx + 1);
            float2 ax, ay, bz;
#define SPX(k) sp[k].x
#define SPY(k) sp[k].y
            ax.x = co.sw0 * (SPX(o + 1) - SPX(o - 1)) + co.sw1 * ((SPX(o - W1 + 1) - SPX(o - W1 - 1)) + (SPX(o + W1 + 1) - SPX(o + W1 - 1)));
            ax.y = co.sw0 * (SPY(o + 1) - SPY(o - 1)) + co.sw1 * ((SPY(o - W1 + 1) - SPY(o - W1 - 1)) + (SPY(o + W1 + 1) - SPY(o + W1 - 1)));
            ay.x = co.sw0 * (SPX(o + W1) - SPX(o - W1)) + co.sw1 * ((SPX(o + W1 - 1) - SPX(o - W1 - 1)) + (SPX(o + W1 + 1) - SPX(o - W1 + 1)));
            ay.y = co.sw0 * (SPY(o + W1) - SPY(o - W1)) + co.sw1 * ((SPY(o + W1 - 1) - SPY(o - W1 - 1)) + (SPY(o + W1 + 1) - SPY(o - W1 + 1)));
            {
                const float r0x = co.sw0 * SPX(o) + co.sw1 * (SPX(o - 1) + SPX(o + 1));
                const float rmx = co.sw0 * SPX(o - W1) + co.sw1 * (SPX(o - W1 - 1) + SPX(o - W1 + 1));
                const float rpx = co.sw0 * SPX(o + W1) + co.sw1 * (SPX(o + W1 - 1) + SPX(o + W1 + 1));
                const float r0y = co.sw0 * SPY(o) + co.sw1 * (SPY(o - 1) + SPY(o + 1));
                const float rmy = co.sw0 * SPY(o - W1) + co.sw1 * (SPY(o - W1 - 1) + SPY(o - W1 + 1));
                const float rpy = co.sw0 * SPY(o + W1) + co.sw1 * (SPY(o + W1 - 1) + SPY(o + W1 + 1));
                bz.x = co.d1 * (co.sw0 * r0x + co.sw1 * (rmx + rpx));
                bz.y = co.d1 * (co.sw0 * r0y + co.sw1 * (rmy + rpy));
            }
#undef SPX
#undef SPY
            ax.x *= co.d1; ax.y *= co.d1; ay.x *= co.d1; ay.y *= co.d1;
            xm.x += co.sw1 * ax.x; xm.y += co.sw1 * ax.y;
            xc.x += co.sw0 * ax.x; xc.y += co.sw0 * ax.y;
            xp.x += co.sw1 * ax.x; xp.y += co.sw1 * ax.y;
            ym.x += co.sw1 * ay.x; ym.y += co.sw1 * ay.y;
            yc.x += co.sw0 * ay.x; yc.y += co.sw0 * ay.y;
            yp.x += co.sw1 * ay.x; yp.y += co.sw1 * ay.y;
            zmv.x += bz.x; zmv.y += bz.y;  // plane zi is the z+1 plane of output zi-1
            zpv.x -= bz.x; zpv.y -= bz.y;  // and the z-1 plane of output zi+1
            const int zo = zi - 1;
            if (zo >= zb && own) {
                const size_t g = gidx(N, gx, gy, zo);
                dst[0][g] = svc[0] - co.Dt * xm.x;
                dst[1][g] = svc[1] - co.Dt * ym.x;
                dst[2][g] = svc[2] - co.Dt * zmv.x;
                dst[3][g] = svc[3] - dts * xm.y;
                dst[4][g] = svc[4] - dts * ym.y;
                dst[5][g] = svc[5] - dts * zmv.y;
                if (ewr) {
                    const gptr<float> e = glb(D.edge) + (size_t)zo * NN;
#pragma unroll
                    for (int f = 0; f < 6; ++f) stb(e, ewo + 4u * (unsigned)(f * 2 * N), svc[f]);
                }
            }
            xm = xc; xc = xp; xp = make_float2(0.f, 0.f);
            ym = yc; yc = yp; yp = make_float2(0.f, 0.f);
            zmv = zcv; zcv = zpv; zpv = make_float2(0.f, 0.f);
        };
        fetch(0, zb - 1);
        fetch(1, zb);
        wait_vmem();
        for (int zi = zb - 1;;) {
            body(Ph<0>{}, zi);
            if (++zi > ze) break;
            body(Ph<1>{}, zi);
            if (++zi > ze) break;
        }
    }
}

// ===========================================================================
// FP64 reductions
// ===========================================================================
__global__ __launch_bounds__(256) void k_reduce_part(const Drop* __restrict__ drops, int parity, double* part, int nblk)
{
    __shared__ double red[3 * 4];
    const int d = blockIdx.y;
    const Drop& D = drops[d];
    const unsigned n = (unsigned)D.N * (unsigned)D.N * (unsigned)D.N;
    const gptr<const float> phi = glb<const float>(D.phi[parity]);
    gptr<const float> P[3], v[3];
#pragma unroll
    for (int a = 0; a < 3; ++a) {
        P[a] = glb<const float>(D.P[a]);
        v[a] = glb<const float>(D.v[a]);
    }
    double m = 0.0, pm = 0.0, ke = 0.0;
    // Latency bound: four cells' loads in flight (through global pointers and
    // 32-bit indices); the sums stay in cell order.  A read of a 96^3 droplet's
    // reductions takes 33 us where it took 83
#pragma unroll 4
    for (unsigned i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (unsigned)nblk * blockDim.x) {
        const double px = P[0][i], py = P[1][i], pz = P[2][i];
        const double vx = v[0][i], vy = v[1][i], vz = v[2][i];
        m += (double)phi[i];
        pm += sqrt(px * px + py * py + pz * pz);
        ke += vx * vx + vy * vy + vz * vz;
    }
    const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) {
        m += __shfl_down(m, off, 64);
        pm += __shfl_down(pm, off, 64);
        ke += __shfl_down(ke, off, 64);
    }
    if (lane == 0) { red[3 * wid] = m; red[3 * wid + 1] = pm; red[3 * wid + 2] = ke; }
    __syncthreads();
    if (threadIdx.x == 0) {
        double a = 0, b = 0, c = 0;
        for (int w = 0; w < 4; ++w) { a += red[3 * w]; b += red[3 * w + 1]; c += red[3 * w + 2]; }
        double* o = part + 3 * ((size_t)d * nblk + blockIdx.x);
        o[0] = a; o[1] = b; o[2] = c;
    }
}

__global__ __launch_bounds__(256) void k_reduce_final(const double* part, int nblk, double* out)
{
    __shared__ double red[3 * 4];
    const int d = blockIdx.x;
    double m = 0.0, pm = 0.0, ke = 0.0;
    for (int j = threadIdx.x; j < nblk; j += blockDim.x) {
        const double* p = part + 3 * ((size_t)d * nblk + j);
        m += p[0]; pm += p[1]; ke += p[2];
    }
    const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) {
        m += __shfl_down(m, off, 64);
        pm += __shfl_down(pm, off, 64);
        ke += __shfl_down(ke, off, 64);
    }
    if (lane == 0) { red[3 * wid] = m; red[3 * wid + 1] = pm; red[3 * wid + 2] = ke; }
    __syncthreads();
    if (threadIdx.x == 0) {
        double a = 0, b = 0, c = 0;
        for (int w = 0; w < 4; ++w) { a += red[3 * w]; b += red[3 * w + 1]; c += red[3 * w + 2]; }
        out[3 * d] = a; out[3 * d + 1] = b; out[3 * d + 2] = c;
    }
}

// ===========================================================================
// launchers
// ===========================================================================
hipError_t launch_div(const Drop* drops, const Work* work, const int* nwork_p, int parity, int kstep, int grid,
                      hipStream_t st)
{
    if (grid <= 0) return hipSuccess;
    return launch_kernel(k_div, dim3(grid), dim3(64 * kProjWaves), st, drops, work, nwork_p, parity, kstep);
}

hipError_t launch_proj_stats(const Drop* drops, const Work* work, const int* nwork_p, int kstep, int grid,
                             hipStream_t st)
{
    if (grid <= 0) return hipSuccess;
    return launch_kernel(k_proj_stats, dim3(grid), dim3(kStatsThreads), st, drops, work, nwork_p, kstep);
}

// One thread per (z, y): the two end columns of the six predictor fields.
__global__ __launch_bounds__(256) void k_fill_edges(const float* __restrict__ v0, const float* __restrict__ v1,
                                                    const float* __restrict__ v2, const float* __restrict__ p0,
                                                    const float* __restrict__ p1, const float* __restrict__ p2,
                                                    float* __restrict__ edge, int slot, int N)
{
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= N * N) return;
    const int y = i % N, z = i / N;
    const size_t row = ((size_t)z * N + y) * N, NN = (size_t)N * N;
    const float* src[6] = {v0, v1, v2, p0, p1, p2};
    const gptr<float> e = glb(edge) + (size_t)z * NN;
#pragma unroll
    for (int f = 0; f < 6; ++f) {
        e[((slot * 6 + f) * 2 + 0) * N + y] = glb(src[f])[row];
        e[((slot * 6 + f) * 2 + 1) * N + y] = glb(src[f])[row + N - 1];
    }
}

hipError_t launch_fill_edges(const float* const vs[3], const float* const ps[3], float* edge, int slot, int N,
                             hipStream_t st)
{
    hipLaunchKernelGGL(k_fill_edges, dim3((N * N + 255) / 256), dim3(256), 0, st, vs[0], vs[1], vs[2], ps[0], ps[1],
                       ps[2], edge, slot, N);
    return hipGetLastError();
}

// Field blockIdx.y of a list, n elements each (floats, or groups of four where
// every address is a multiple of 16 bytes), in memory that the device reaches,
// no destination overlapping another.  One launch for the 13 fields of a
// state: 13 copies of the runtime cost a call of one 32^3 step 70 us on each
// side of the step, this 5.
template <typename T>
__global__ __launch_bounds__(256) void k_copy_fields(FieldList f, unsigned n)
{
    const gptr<const T> src = glb((const T*)f.src[blockIdx.y]);
    const gptr<T> dst = glb((T*)f.dst[blockIdx.y]);
    for (unsigned i = blockIdx.x * 256 + threadIdx.x; i < n; i += gridDim.x * 256) dst[i] = src[i];
}

hipError_t launch_copy_fields(const FieldList& f, size_t n, hipStream_t st)
{
    if (f.count <= 0 || n == 0) return hipSuccess;
    size_t bits = n * sizeof(float);
    for (int k = 0; k < f.count; ++k) bits |= (size_t)f.src[k] | (size_t)f.dst[k];
    const bool wide = bits % 16 == 0;
    const unsigned m = (unsigned)(wide ? n / 4 : n);
    const dim3 grid(std::min((m + 255) / 256, 64u), f.count);
    if (wide) hipLaunchKernelGGL(k_copy_fields<fvec4>, grid, dim3(256), 0, st, f, m);
    else hipLaunchKernelGGL(k_copy_fields<float>, grid, dim3(256), 0, st, f, m);
    return hipGetLastError();
}

// Fill n 32-bit words with a value (vector stores; grid-stride).
__global__ __launch_bounds__(256) void k_fill_u32(uint32_t* __restrict__ p, uint32_t value, size_t n)
{
    const size_t stride = (size_t)gridDim.x * blockDim.x;
    for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += stride) glb(p)[i] = value;
}

hipError_t launch_fill_u32(void* p, uint32_t value, size_t n, hipStream_t st)
{
    if (n == 0) return hipSuccess;
    const size_t blocks = std::min<size_t>((n + 255) / 256, 4096);
    hipLaunchKernelGGL(k_fill_u32, dim3((unsigned)blocks), dim3(256), 0, st, static_cast<uint32_t*>(p), value, n);
    return hipGetLastError();
}

hipError_t launch_corr(const Drop* drops, const Work* work, const int* nwork_p, int parity, int kstep, int grid,
                       hipStream_t st)
{
    if (grid <= 0) return hipSuccess;
    return launch_kernel(k_corr<kCorrTX, kCorrTY>, dim3(grid), dim3(kCorrTX * kCorrTY), st, drops, work, nwork_p,
                         parity, kstep);
}

hipError_t launch_reduce(const Drop* drops, int ndrops, int parity, double* part, int nblk, double* out,
                         hipStream_t st)
{
    hipLaunchKernelGGL(k_reduce_part, dim3(nblk, ndrops), dim3(256), 0, st, drops, parity, part, nblk);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
    hipLaunchKernelGGL(k_reduce_final, dim3(ndrops), dim3(256), 0, st, part, nblk, out);
    return hipGetLastError();
}

}  // namespace ttsh
