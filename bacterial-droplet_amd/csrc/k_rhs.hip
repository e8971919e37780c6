// k_rhs.hip -- K_rhs: the fused right-hand side and predictor of one step.
//
// Replaces the reference's getRHS (TTSH3D.cu:363-468: 94 halo fills plus
// getTempVari_1 :537-558, getTempVari_2 :561-605, getDtF :608-632) and
// getVStar (:471-491) with one pass that reads phi, P, v once and writes
// phi^{n+1}, v*, P*:
//
//   G_ab  = D_a P_b                    mu0 = 2 aPhi (phi - 3phi^2 + 2phi^3) - kPhi L phi
//   mu_b  = phi P_b + La^2 L P_b       Sig_ab = phi G_ab
//   dtv_b = -v.D v_b + mu L v_b + mu0 D_b phi + cA sum_a D_a Sig_ab
//   dtP_b = -v.D P_b - alpha phi P_b - beta |P|^2 P_b + eta L mu_b - lambda0 P.D P_b
//           - A (|D phi|^2 |P|^2 P_b + |P| sum_c D_b phi D_c phi P_c)
//   dtphi = -v.D phi + gamma L mu0
//   v* = v + Dt dtv,  P* = P + Dt dtP,  phi^{n+1} = phi + Dt dtphi   (getVNew :513)
//
// The reference's integer-division zeros (TTSH3D.cu:579-602: DP = OP = 0, the
// 1/28 correction of Sigma and the 1/3 trace of A) are terms that are exactly
// zero for finite fields, so they are not evaluated; kappa therefore has no
// effect, as in the reference.
//
// Stencils (TTSH3D.cu:3280-3343).  With S = [1,4,1], d = [-1,0,1] and
// s = 1/(72 h), lc = 1/(12 h^2),
//   D_x = s d_x S_y S_z,  D_y = s S_x d_y S_z,  D_z = s S_x S_y d_z
//   L f = lc (sum of the 8 corners + 8 sum of the 6 faces - 56 f)
// is applied one axis at a time, each axis where its neighbours are cheapest:
//   z  three planes of a value in registers, rotating with the z-march:
//        t = f(z-1)+f(z+1), b = f(z+1)-f(z-1), a = S_z f = 4 f + t
//   x  lanes of a wave are consecutive x; neighbours come by DPP wave shifts:
//        X = d_x a, A = S_x a, B = S_x b, E = t(x-1)+t(x+1) + 8 f,
//        O = t + f(x-1)+f(x+1) - 7 f
//   y  a wave is one row; X, A, B, E of a row go to LDS as one 16-byte record
//        and the rows at y-1 (m) and y+1 (p) are read back:
//        D_x/s = 4 X + Xm + Xp, D_y/s = Ap - Am, D_z/s = 4 B + Bm + Bp,
//        L/lc = 8 O + Em + Ep
// The scales s and lc are folded into the pointwise factors.  The
// intermediates (Sig, mu, mu0) take the same x and y stages, and their z
// stage is an accumulation into the three output planes that a plane touches.
//
// What bounds it: VALU issue.  The kernel that this one replaced kept whole
// z-prepared tiles in LDS and read every 2D stencil from there: 226 LDS and
// 704 VALU instructions per plane and wave, LDS 57-74% busy at about 120
// bytes per clock and CU, the rate of 4- and 8-byte reads.  16-byte reads run
// at 230.  A record per row and field needs one 16-byte write and two 16-byte
// reads per field where the 2D stencils took 22 values, and each one-axis sum
// is made once instead of by every neighbour: 44 LDS and 430 VALU
// instructions per plane and wave.  Measured, 16-row tiles against the best of
// the former tiles, each at its best depth: 64^3 37 -> 17 us (in z-chunks of two
// planes instead of eight), 128^3 75 -> 58 (46 with the flattened tile),
// 180^3 216 -> 98, 240^3 463 -> 207, 256^3 498 -> 282.
//
// Tiles.  W = 64: one wave per row of TX <= 60 cells, whose 64 lanes include
// the 2-cell x apron; 8 or 16 rows per work-group.  N is cut into ceil(N/60)
// tiles of equal width.  W = 36: TX <= 32 cells and 26 rows, the tile's rows
// one after another over 16 waves, each of which holds 60 positions of them
// and two of its neighbours' on either side.  A wave of a 60-wide tile is
// idle in part where 60 does not divide N well (64^3, 128^3: a third to a
// half), a wave of the flattened tile only at its ends.  At 128^3 that makes
// 20 tiles of 24 and 46 us of 58; where the counts are equal the flattened
// tile is 3% (96^3) to 12% (256^3, its rows end inside cache lines more often)
// slower, so the tuning table chooses per size.  Two rows per wave (213
// VGPRs, two waves per SIMD) measured 4% slower at 128^3 and equal at 240^3
// and 256^3.  The rows above and below the tile are staged by all waves, one
// or two (row, field) pairs each, and the first eight waves compute the
// intermediates of the two rows next to the tile.
//
// 16 waves (128 VGPRs, 160 KB of LDS: one group per CU, four waves per SIMD)
// have the smaller share of apron rows and are faster wherever the device is
// full: 240^3 207 against 316 us.  8 waves (98 KB) take 2.1 us per plane
// instead of 3.2 when a CU holds one group, which wins for small boxes.  All
// do the same arithmetic in the same order (no contraction in this file), so a
// droplet's result does not depend on the tile.
#include <type_traits>

#include "ttsh_dev.h"
#include "ttsh_kernels.h"

#pragma clang fp contract(off)

namespace ttsh {

// Keeps the compiler from sinking a value's computation past this point: sunk
// past a barrier, all its inputs would stay live instead of the one value.
__device__ __forceinline__ void pin(float& a) { asm volatile("" : "+v"(a)); }

// A row of one field after its z and x stages; X, A, B, E are the record that
// the neighbouring rows read.
struct XRow {
    float X, A, B, E, O;
    __device__ __forceinline__ fvec4 record() const { return fvec4{X, A, B, E}; }
};
__device__ __forceinline__ XRow xrow(float fm, float f, float fp)
{
    XRow r;
    const float t = fm + fp;
    const float b = fp - fm;
    const float a = fma_(4.f, f, t);
    const float pt = xpair(t), pf = xpair(f);
    r.X = xdiff(a);
    r.A = fma_(4.f, a, fma_(4.f, pf, pt));
    r.B = fma_(4.f, b, xpair(b));
    r.E = fma_(8.f, f, pt);
    r.O = fma_(-7.f, f, t + pf);
    return r;
}

// D_x/s, D_y/s, D_z/s, L/lc of a row from its own stage and the records of
// the rows below (m) and above (p).
struct Der {
    float dx, dy, dz, l;
};
__device__ __forceinline__ Der yder(const XRow& r, const fvec4& m, const fvec4& p)
{
    Der d;
    d.dx = fma_(4.f, r.X, m.x + p.x);
    d.dy = p.y - m.y;
    d.dz = fma_(4.f, r.B, m.z + p.z);
    d.l = fma_(8.f, r.O, m.w + p.w);
    return d;
}

// The intermediates of one P component after their x stage.  With
// X = d_x Sig_xb and A = S_x Sig_yb, the row's part of S_y d_x Sig_x +
// d_y S_x Sig_y is 4 X for itself, U = X + A for the row below it and
// W = X - A for the row above; B = S_x Sig_zb; pm = mu(x-1)+mu(x+1).
struct IRow {
    float X, U, W, B, pm, m;
};
__device__ __forceinline__ IRow irow(float sx, float sy, float sz, float m)
{
    IRow o;
    o.X = xdiff(sx);
    const float A = fma_(4.f, sy, xpair(sy));
    o.U = o.X + A;
    o.W = o.X - A;
    o.B = fma_(4.f, sz, xpair(sz));
    o.pm = xpair(m);
    o.m = m;
    return o;
}

// mu0 of a cell: -kPhi lc, the raw Laplacian, 2 aPhi
__device__ __forceinline__ float mu0_of(float ph, float l, float kl, float a2)
{
    const float ph2 = ph * ph;
    return fma_(-kl, l, a2 * fma_(2.f * ph2, ph, fma_(-3.f, ph2, ph)));
}

// NW waves, W records per tile row.  W = 64: a wave is a row.  W < 64: the
// tile's rows lie one after another and wave w holds the positions 60 w - 2 ..
// 60 w + 61 of that sequence; the two positions at each end are also those of
// its neighbours, which store them.
template <int NW, int W>
__global__ __launch_bounds__(64 * NW, NW / 4) void k_rhs(const Drop* __restrict__ drops, const Work* __restrict__ work,
                                                         const int* __restrict__ nwork_p, int parity, int kstep)
{
    constexpr int TY = rhs_tile_rows(NW, W);
    // Records of a field: rows -2 .. TY+1 of phi and P; rows -1 .. TY of v and
    // of the intermediates; with W < 64, 64 more that take what lanes without
    // a position of their own would store.
    constexpr int FP = (TY + 4) * W + (W < 64 ? 64 : 0), FV = (TY + 2) * W + (W < 64 ? W + 64 : 0);
    // Two buffers of BUF records.  A plane uses them as: phi, P -> X; the
    // intermediates -> Y; v -> X; then X and Y swap.  Each exchange then
    // writes the buffer whose readers passed the previous barrier.
    // Intermediates: per component (U, W, B, pm), then (m_0, m_1, m_2, mu0),
    // then mu0's pm.
    constexpr int IM = 3 * FV, IP = 4 * FV;
    constexpr int BUF = W == 64 ? 4 * FP : IP + (FV + 3) / 4;
    static_assert(4 * FP <= BUF && IP + (FV + 3) / 4 <= BUF && 32 * BUF <= 160 * 1024, "buffers");
    // apron rows of phi, P staged per wave: (field, inner row) and (field,
    // outer row) for 8 waves, one of them for 16
    constexpr int NT = NW == 8 ? 2 : 1;
    static_assert(NW == 8 || NW == 16, "apron rows are dealt to 8 or 16 waves");
    __shared__ fvec4 lds[2 * BUF];

    const int lane = threadIdx.x & 63;
    const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int nwork = *nwork_p;

    for (int vi = blockIdx.x; vi < xcd_span(nwork); vi += gridDim.x) {
        const int w = xcd_item(vi, nwork);
        if (w >= nwork) continue;
        const Work wk = work[w];
        const Drop& D = drops[wk.d];
        if (kstep >= D.nsteps) continue;
        const Coef co = D.co;
        const int N = D.N;
        const unsigned NN = (unsigned)N * (unsigned)N;
        const int TX = rhs_tile_width(N, W);
        const int x0 = wk.a * TX, y0 = wk.b * TY;
        const int zb = wk.c & 0xffff;
        const int ze = wk.c >> 16;
        const gptr<const float> gin[4] = {glb<const float>(D.phi[parity]), glb<const float>(D.P[0]),
                                          glb<const float>(D.P[1]), glb<const float>(D.P[2])};
        const gptr<const float> gv[3] = {glb<const float>(D.v[0]), glb<const float>(D.v[1]),
                                         glb<const float>(D.v[2])};
        const gptr<float> ophi = glb(D.phi[parity ^ 1]);
        const gptr<float> ovs[3] = {glb(D.vs[parity][0]), glb(D.vs[parity][1]), glb(D.vs[parity][2])};
        const gptr<float> ops[3] = {glb(D.ps[parity][0]), glb(D.ps[parity][1]), glb(D.ps[parity][2])};

        // own cell: columns 2 .. TX+1 of a row; the other columns are apron
        // (or, past it, any cell: x0 + 61 < 2 N since N >= 32)
        int row = wv, col = lane;
        bool mine = true;
        if constexpr (W < 64) {
            const int q = wv * 60 + lane - 2;
            mine = lane >= 2 && lane < 62 && q < TY * W;
            row = min(max(q, 0), TY * W - 1) / W;
            col = min(max(q, 0), TY * W - 1) % W;
        }
        const int gx = x0 + col - 2, gy = y0 + row;
        const int cx = wrapi(gx, N);
        const bool own = mine && col >= 2 && col < 2 + TX && gx < N && gy < N;
        auto row_off = [&](int y, int c) { return 4u * ((unsigned)wrapi(y, N) * (unsigned)N + (unsigned)c); };
        const unsigned off = row_off(gy, cx);
        // Apron rows: field `part` (phi, P_x, P_y, P_z) at the row next to the
        // tile (inner: -1 or TY) or beyond it (-2 or TY+1), side 0 below and 1
        // above.  Waves 0..7 stage an inner row and compute its intermediates;
        // the outer rows go to the same waves (8 rows) or to waves 8..15, and
        // with them v_x, v_y, v_z of the inner rows.
        const int part = (wv & 7) >> 1, side = wv & 1;
        const bool inner = wv < 8;
        const bool vrow = part < 3 && (NW == 8 || !inner);
        const int ri = side ? TY : -1, ro = side ? TY + 1 : -2;
        const int r0 = inner ? ri : ro;  // first staged row; the second is ro
        const int ac = W == 64 ? cx : wrapi(x0 + min(lane, W - 1) - 2, N);
        const unsigned off0 = row_off(y0 + r0, ac), off1 = row_off(y0 + ro, ac), offv = row_off(y0 + ri, ac);
        const gptr<const float> gp = part == 0 ? gin[0] : part == 1 ? gin[1] : part == 2 ? gin[2] : gin[3];
        const gptr<const float> gpv = part == 0 ? gv[0] : part == 1 ? gv[1] : gv[2];

        // record indices: column c of row q of a field at (q - first row) W + c.
        // lp, lv: the own cell's, which the rows above and below are read from;
        // wp, wv_: where its records go
        constexpr int LP = (TY + 4) * W;  // the first record of no position, of phi and P
        const int lp = (row + 2) * W + col, lv = lp - W;
        const int wp = mine ? lp : LP + lane, wv_ = wp - W;
        const int la = W == 64 || lane < W ? lane : -1;
        const int l0 = part * FP + (la < 0 ? LP + lane : (r0 + 2) * W + la);
        const int l1 = part * FP + (la < 0 ? LP + lane : (ro + 2) * W + la);
        const int lvr = part * FV + (la < 0 ? LP - W + lane : (ri + 1) * W + la);
        const int lir = la < 0 ? LP - W + lane : (ri + 1) * W + la;
        const int lri = part * FP + (r0 + 2) * W + min(lane, W - 1);  // the staged inner row, to read beside it

        auto put_i = [&](fvec4* y, int b, int i, const IRow& o) {
            y[b * FV + i] = fvec4{o.U, o.W, o.B, o.pm};
            ((float*)(y + IM + i))[b] = o.m;
        };
        auto put_m = [&](fvec4* y, int i, float pm, float m) {
            ((float*)(y + IM + i))[3] = m;
            ((float*)(y + IP))[i] = pm;
        };

        // three z-planes per value, in slots rotating with the z-march: in
        // phase K the slots K, K+1, K+2 (mod 3) hold planes zm-1, zm, zm+1
        float f[4][3], vf[3][3], tf[NT][3], tv[3];
        auto load_p = [&](int slot, int z) {
            const size_t zo = (size_t)wrapi(z, N) * NN;
            const unsigned o = opaque(off);
#pragma unroll
            for (int k = 0; k < 4; ++k) f[k][slot] = ldb(gin[k] + zo, o);
            tf[0][slot] = ldb(gp + zo, opaque(off0));
            if constexpr (NT == 2) tf[1][slot] = ldb(gp + zo, opaque(off1));
        };
        auto load_v = [&](int slot, int z) {
            const size_t zo = (size_t)wrapi(z, N) * NN;
            const unsigned o = opaque(off);
#pragma unroll
            for (int b = 0; b < 3; ++b) vf[b][slot] = ldb(gv[b] + zo, o);
            tv[slot] = ldb(gpv + zo, opaque(offv));
        };
#pragma unroll
        for (int k = 0; k < 3; ++k) {
            load_p(k, zb - 2 + k);
            load_v(k, zb - 2 + k);
        }
        wait_vmem();

        // per output plane (same rotation): sums of D.Sig/s, L mu/lc, L mu0/lc,
        // and the rest of the update
        //   [b]   v_b + Dt (-v.D v_b + mu L v_b + mu0 D_b phi)
        //   [3+b] P_b + Dt (-v.D P_b - alpha phi P_b - beta |P|^2 P_b - lambda0 P.D P_b - anchoring_b)
        //   [6]   phi + Dt (-v.D phi)
        float aS[3][3], aL[3][3], aL0[3], nx[3][7];
        XRow xv[3];  // v of the plane staged last
#pragma unroll
        for (int b = 0; b < 3; ++b) {
            aL0[b] = 0.f;
            xv[b] = XRow{0.f, 0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int q = 0; q < 3; ++q) { aS[q][b] = 0.f; aL[q][b] = 0.f; }
        }
#pragma unroll
        for (int j = 0; j < 7; ++j) nx[0][j] = 0.f;
        fvec4 *bx = lds, *by = lds + BUF;
        const float s = co.s, lc = co.lc;

        __syncthreads();  // the previous item has read both buffers
        auto body = [&](auto ph_, int zm) {
            constexpr int S0 = decltype(ph_)::value, S1 = (S0 + 1) % 3, S2 = (S0 + 2) % 3;
            // ---- a: y stage of v of plane zm-1 (records in Y), which ends its
            // update terms; z and x stages of phi, P of plane zm.  The 8-wave
            // kernel, whose chunks are shallow, leaves v out where the plane
            // is not stored (32^3 10.9 -> 10.4 us); with 16 waves the branch
            // costs 16 spilled registers.
            if (NW == 16 || zm > zb) {
                const float mulc = co.mu * lc;
                const float vx = vf[0][S0] * s, vy = vf[1][S0] * s, vz = vf[2][S0] * s;
#pragma unroll
                for (int b = 0; b < 3; ++b) {
                    const fvec4* q = by + b * FV + lv;
                    const Der d = yder(xv[b], q[-W], q[W]);
                    const float adv = fma_(vx, d.dx, fma_(vy, d.dy, vz * d.dz));
                    nx[S0][b] = fma_(co.Dt, fma_(mulc, d.l, nx[S0][b]) - adv, vf[b][S0]);
                    pin(nx[S0][b]);
                    __builtin_amdgcn_sched_barrier(0);
                }
            }
            // phi of the inner apron row, for its intermediates
            const float phr = ldb(gin[0] + (size_t)wrapi(zm, N) * NN, opaque(offv));
            XRow xp[4];
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                xp[k] = xrow(f[k][S0], f[k][S1], f[k][S2]);
                pin(xp[k].O);
                bx[k * FP + wp] = xp[k].record();
                __builtin_amdgcn_sched_barrier(0);
            }
            XRow xi = xrow(tf[0][S0], tf[0][S1], tf[0][S2]);
            pin(xi.O);
            bx[l0] = xi.record();
            if constexpr (NT == 2) {
                __builtin_amdgcn_sched_barrier(0);
                bx[l1] = xrow(tf[1][S0], tf[1][S1], tf[1][S2]).record();
            }
            __builtin_amdgcn_sched_barrier(0);
            load_p(S0, min(zm + 2, ze + 1));
            __syncthreads();

            // ---- b: y stage of phi, P; pointwise terms; x stage of the
            // intermediates of plane zm
            IRow im[3];
            float m0, pm0;
            {
                const float ph = f[0][S1];
                float w0, w1, w2, q1, an[3] = {0.f, 0.f, 0.f};
                {
                    const fvec4* q = bx + lp;
                    const Der d = yder(xp[0], q[-W], q[W]);
                    m0 = mu0_of(ph, d.l, co.kPhi * lc, co.aPhi2);
                    pm0 = xpair(m0);
                    put_m(by, wv_, pm0, m0);
                    const float P0 = f[1][S1], P1 = f[2][S1], P2 = f[3][S1];
                    const float v0 = vf[0][S1], v1 = vf[1][S1], v2 = vf[2][S1];
                    const float pp = fma_(P0, P0, fma_(P1, P1, P2 * P2));
                    q1 = fma_(co.alpha, ph, co.beta * pp);
                    // v + lambda0 P: the two advections of P are one
                    w0 = s * fma_(co.lambda0, P0, v0);
                    w1 = s * fma_(co.lambda0, P1, v1);
                    w2 = s * fma_(co.lambda0, P2, v2);
                    const float adv = s * fma_(v0, d.dx, fma_(v1, d.dy, v2 * d.dz));
                    nx[S1][6] = fma_(-co.Dt, adv, ph);
                    const float ms = m0 * s;
                    nx[S1][0] = ms * d.dx;
                    nx[S1][1] = ms * d.dy;
                    nx[S1][2] = ms * d.dz;
#pragma unroll
                    for (int b = 0; b < 3; ++b) pin(nx[S1][b]);
                    pin(nx[S1][6]);
                    if (co.anchoring) {
                        const float dx = d.dx * s, dy = d.dy * s, dz = d.dz * s;
                        const float dd = fma_(dx, dx, fma_(dy, dy, dz * dz)) * pp;
                        const float sp = sqrtf(pp) * fma_(dx, P0, fma_(dy, P1, dz * P2));
                        an[0] = co.A * fma_(dd, P0, sp * dx);
                        an[1] = co.A * fma_(dd, P1, sp * dy);
                        an[2] = co.A * fma_(dd, P2, sp * dz);
                    }
                }
                __builtin_amdgcn_sched_barrier(0);
                const float phs = ph * s, la = co.La2 * lc;
#pragma unroll
                for (int b = 0; b < 3; ++b) {
                    const fvec4* q = bx + (1 + b) * FP + lp;
                    const Der d = yder(xp[1 + b], q[-W], q[W]);
                    const float Pb = f[1 + b][S1];
                    const float dt = fma_(q1, Pb, fma_(w0, d.dx, fma_(w1, d.dy, w2 * d.dz))) + an[b];
                    nx[S1][3 + b] = fma_(-co.Dt, dt, Pb);
                    pin(nx[S1][3 + b]);
                    im[b] = irow(phs * d.dx, phs * d.dy, phs * d.dz, fma_(la, d.l, ph * Pb));
                    put_i(by, b, wv_, im[b]);
                    __builtin_amdgcn_sched_barrier(0);
                }
            }
            if (NW == 8 || inner) {
                const Der d = yder(xi, bx[lri - W], bx[lri + W]);
                if (part == 0) {
                    const float m = mu0_of(phr, d.l, co.kPhi * lc, co.aPhi2);
                    put_m(by, lir, xpair(m), m);
                } else {
                    const float ps = phr * s;
                    put_i(by, part - 1, lir,
                          irow(ps * d.dx, ps * d.dy, ps * d.dz, fma_(co.La2 * lc, d.l, phr * tf[0][S1])));
                }
            }
            __syncthreads();

            // ---- c: y stage of the intermediates, added to planes zm-1, zm,
            // zm+1; store plane zm-1; z and x stages of v of plane zm
            __builtin_amdgcn_sched_barrier(0);
            {
                const fvec4 mm = by[IM + lv - W], mp = by[IM + lv + W];
#pragma unroll
                for (int b = 0; b < 3; ++b) {
                    const fvec4* q = by + b * FV + lv;
                    const fvec4 im_ = q[-W], ip_ = q[W];
                    const IRow& o = im[b];
                    const float A = fma_(4.f, o.X, ip_.x + im_.y);
                    const float B = fma_(4.f, o.B, im_.z + ip_.z);
                    const float E = fma_(8.f, o.m, im_.w + ip_.w);
                    const float F = fma_(-7.f, o.m, (mm[b] + mp[b]) + o.pm);
                    aS[S0][b] += A + B;
                    aS[S1][b] = fma_(4.f, A, aS[S1][b]);
                    aS[S2][b] = A - B;
                    aL[S0][b] += E;
                    aL[S1][b] = fma_(8.f, F, aL[S1][b]);
                    aL[S2][b] = E;
#pragma unroll
                    for (int q3 = 0; q3 < 3; ++q3) { pin(aS[q3][b]); pin(aL[q3][b]); }
                    __builtin_amdgcn_sched_barrier(0);
                }
                const float* const q = (const float*)(by + IP) + lv;
                const float E = fma_(8.f, m0, q[-W] + q[W]);
                const float F = fma_(-7.f, m0, (mm.w + mp.w) + pm0);
                aL0[S0] += E;
                aL0[S1] = fma_(8.f, F, aL0[S1]);
                aL0[S2] = E;
#pragma unroll
                for (int q3 = 0; q3 < 3; ++q3) pin(aL0[q3]);
            }
            if (zm - 1 >= zb && own) {
                const size_t pz = (size_t)(zm - 1) * NN;
                const float ka = co.Dt * co.cA * s, ke = co.Dt * co.eta * lc, kg = co.Dt * co.gamma * lc;
                const unsigned o = opaque(off);
                stb(ophi + pz, o, fma_(kg, aL0[S0], nx[S0][6]));
#pragma unroll
                for (int b = 0; b < 3; ++b) {
                    stb(ovs[b] + pz, o, fma_(ka, aS[S0][b], nx[S0][b]));
                    stb(ops[b] + pz, o, fma_(ke, aL[S0][b], nx[S0][3 + b]));
                }
            }
            __builtin_amdgcn_sched_barrier(0);
            if (NW == 16 || (zm >= zb && zm < ze)) {
#pragma unroll
                for (int b = 0; b < 3; ++b) {
                    xv[b] = xrow(vf[b][S0], vf[b][S1], vf[b][S2]);
                    pin(xv[b].O);
                    bx[b * FV + wv_] = xv[b].record();
                    __builtin_amdgcn_sched_barrier(0);
                }
                if (vrow) bx[lvr] = xrow(tv[S0], tv[S1], tv[S2]).record();
            }
            load_v(S0, min(zm + 2, ze));
            __syncthreads();
            fvec4* const t = bx;
            bx = by;
            by = t;
        };
        // planes zb-1 .. ze; plane zm-1 is stored in the iteration of zm
        for (int zm = zb - 1;;) {
            body(Ph<0>{}, zm);
            if (++zm > ze) break;
            body(Ph<1>{}, zm);
            if (++zm > ze) break;
            body(Ph<2>{}, zm);
            if (++zm > ze) break;
        }
    }
}

hipError_t launch_rhs(int variant, const Drop* drops, const Work* work, const int* nwork_p, int parity, int kstep,
                      int grid, hipStream_t st)
{
    if (grid <= 0) return hipSuccess;
    if (variant < 0 || variant >= RHS_NVARIANTS) return hipErrorInvalidValue;
    const RhsVar& v = kRhsVars[variant];
    if (v.nw == 8)
        return launch_kernel(k_rhs<8, 64>, dim3(grid), dim3(512), st, drops, work, nwork_p, parity, kstep);
    if (v.w == 36)
        return launch_kernel(k_rhs<16, 36>, dim3(grid), dim3(1024), st, drops, work, nwork_p, parity, kstep);
    return launch_kernel(k_rhs<16, 64>, dim3(grid), dim3(1024), st, drops, work, nwork_p, parity, kstep);
}

int rhs_rows(int variant)
{
    return variant >= 0 && variant < RHS_NVARIANTS ? rhs_tile_rows(kRhsVars[variant].nw, kRhsVars[variant].w) : 0;
}

int rhs_cols(int variant, int N)
{
    return variant >= 0 && variant < RHS_NVARIANTS ? rhs_tiles_x(N, kRhsVars[variant].w) : 0;
}

}  // namespace ttsh
