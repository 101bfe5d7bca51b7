// The fused MPDATA step of the standard antidiffusive variant: donor-cell
// upwind, the standard pseudo-velocities, the non-oscillatory limiter on the
// donor fluxes of the pseudo-velocities, the sign-aware limited velocities
// and the flux-form update of the reference's two-step GPUBC path
// (advection/src_algorithms/upwind3d-gpubc.f90:101-198,
// antidiff3d-standard-gpubc.f90:72-459) in one kernel that reads x, u1, u2,
// u3, h, rhr once and writes the new x once.  The limiter can be off
// (NONOS = false: the pass uses the pseudo-velocities as they are) and any
// direction can be periodic (PER: the clean period-n wrap of the per-stage
// kernels).  Built exactly rounded (mpdata_fused_std.hip: -ffp-contract=off,
// IEEE division; FAST = false) the results are bit-identical to the per-stage
// kernels; the fast build (mpdata_fused_fast.hip: FMA contraction, FAST =
// true, every division a product with a Newton-refined reciprocal) stays
// within 1e-12 of it.
//
// The k-march, work items, tile roles and register queues are those of the
// gauge kernel (mpdata_fused_impl.hpp).  Per plane K the workgroup
//   A  computes xant on plane K over the tile plus a 2-cell ring, and
//      xant/rhr (the ratio every standard flux donates),
//   F  the limited x/y face fluxes of plane Q=K-2,
//   B  the pseudo-velocities V1,V2 on plane P=K-1 and V3 on face K, with the
//      donor fluxes of the pseudo-velocities that the limiter bounds,
//   C  the limiter ratios cp,cn on plane P,
//   D  the new x on plane Q.
// A position's own V1, V2 (in LDS slots of its own) and V3 are used by itself
// for the flux through its left, lower and bottom faces; the limiter's donor
// flux through the right face comes from the lane to the right, the one
// through the upper y-face through LDS.  The inputs of V1 from column i-1
// come from the lane to the left, those of V2 from column j-1 through LDS.
//
// What bounds it is the chain of a plane, as in the gauge kernel, with more of
// it in the divisions (seventeen a cell).  The same means and the tiling rule
// of std_step took 384x320x192 from 760 to 642 us (fast build), 190x147x83 in
// place from 149 to 111 us (exact) and ten steps of a periodic 64x64x32 from
// 323 to 234 us.
#pragma once

#include "mpdata_fused_impl.hpp"

namespace mpdata {

namespace {

// The value held by lane l+1 of the wave (DPP wave_shl:1; lane 63 gets 0).
// Convergent: called with every lane of the wave active.
__device__ __forceinline__ double from_right_lane(double v) {
    const unsigned long long b = (unsigned long long)__double_as_longlong(v);
    const int lo = __builtin_amdgcn_mov_dpp((int)(unsigned)b, 0x130, 0xf, 0xf, true);
    const int hi = __builtin_amdgcn_mov_dpp((int)(unsigned)(b >> 32), 0x130, 0xf, 0xf, true);
    return __longlong_as_double((long long)(((unsigned long long)(unsigned)hi << 32) | (unsigned)lo));
}
__device__ __forceinline__ float from_right_lane(float v) {
    return __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), 0x130, 0xf, 0xf, true));
}

// |v| in the precision of v (the generic lambda below would otherwise see
// only the double overload of fabs at its definition)
__device__ __forceinline__ double abs_(double v) { return __builtin_fabs(v); }
__device__ __forceinline__ float abs_(float v) { return __builtin_fabsf(v); }

// vdyfa and vcorra (mpdata_common.hpp) with the build's division: the same
// operations in the same order when FAST is false
template <bool FAST, typename T>
__device__ __forceinline__ T vdyfa_(T x1, T x2, T a, T rinv) {
    return div_<FAST>((fabs(a) - a * a * rinv) * (fabs(x2) - fabs(x1)),
                      fabs(x2) + fabs(x1) + Eps<T>::v);
}
template <bool FAST, typename T>
__device__ __forceinline__ T vcorra_(T a, T b, T y1, T y2, T rinv) {
    return -div_<FAST>(T(0.125) * a * b * y1 * rinv, y2);
}

// LDS of one workgroup of the standard kernel.
template <typename T, int RX, int RY>
struct StdLds {
    T sx[2][RY + 2][RX + 2];  // x on planes K and K+1 with a 3-cell ring
    T sxa[3][RY][RX];         // xant, planes K-2 .. K
    T src[3][RY][RX];         // xant/rhr, planes K-2 .. K
    T sf1[RY][RX];            // flux through the left x-face, plane Q
    T sf2[RY][RX];            // flux through the lower y-face, plane Q
    T sw2[RY][RX];            // donor flux of V2 through the lower y-face, plane P
    T scp[RY][RX];            // cp, cn: plane K-1 from C on, K-2 until then
    T scn[RY][RX];
    // a thread's own V1, V2 of plane P until the next step's F
    T sv1[RY][RX], sv2[RY][RX];
    // h, u1 (face i), u3 (faces P, P+1) of each source column on plane P,
    // read by the position above for V2
    T e_h[RY][RX], e_u1[RY][RX], e_u3a[RY][RX], e_u3b[RY][RX];
};
static_assert(sizeof(StdLds<double, 32, 32>) <= 160 * 1024, "LDS of one CU");

// The standard variant's limited velocity (antidiff3d-standard-gpubc.f90:
// 372-383): pp(v)*(a1*pp(SIGN(1,xm)) + a2*pp(SIGN(1,-xm))) - pn(v)*(a2*pp(
// SIGN(1,xc)) + a1*pp(SIGN(1,-xc))).  One of each pair of pp(SIGN) factors is
// 1 and the other 0, a1, a2 are in [0,1] (never -0), so each bracket is
// a*1 + (+0) = a exactly: the factor of the sign of xm (xc) selects a1 or a2.
template <typename T>
__device__ __forceinline__ T slim(T v, T a1, T a2, T xm, T xc) {
    return hw::pp(v) * (signbit(xm) ? a2 : a1) - hw::pn(v) * (signbit(xc) ? a1 : a2);
}

// One work item (see fused_item in mpdata_fused_impl.hpp for the k-march).
// PER: any of g.px, g.py, g.pz may be set (otherwise they are taken as 0).
// TAPE (limiter on, open boundaries, ih = 1): the step also writes the
// intermediates the adjoint step reads to tp, as the per-stage recording
// leaves them: x with inflow values / edge copies on the wall halo, xant
// with its mirrored x/y halo ring, V on every face of the domain (zero on
// the x/y walls, mirrored on the lids), cp and cn.  Each cell and face is
// written by the one position that owns it.
template <typename T, int RX, int RY, bool NONOS, bool PER, bool TAPE = false, bool FAST = false>
__device__ __forceinline__ void fused_std_item(const Geo& g, const Off& o, int ntx, int tile,
                                               int k0, int k1, const T* __restrict__ x,
                                               const T* __restrict__ u1, const T* __restrict__ u2,
                                               const T* __restrict__ u3,
                                               const T* __restrict__ rhr,
                                               const T* __restrict__ h,
                                               const T* __restrict__ bcx,
                                               const T* __restrict__ bcy, T* __restrict__ xo,
                                               StdLds<T, RX, RY>& L,
                                               const StdTape<T>* tp = nullptr) {
    static_assert(!TAPE || (NONOS && !PER), "the tape covers the limited step with open walls");
    static_assert(!(TAPE && FAST), "the tape is recorded by the exactly rounded build");
    constexpr int NT = RX * RY, TX = RX - 4, TY = RY - 4;
    constexpr int SW = RX + 2, SH = RY + 2, NRING = 2 * SW + 2 * (SH - 2);
    static_assert((64 % RX == 0 || RX % 64 == 0) && NT % 64 == 0, "row layout of the waves");
    static_assert(NRING <= NT, "x ring must fit one extra slot per thread");
    auto& sx = L.sx;
    const int np = g.np, mp = g.mp, lp = g.lp;
    const bool px = PER && g.px, py = PER && g.py, pz = PER && g.pz;
    const int t = threadIdx.x;
    const int pi = t % RX, pj = t / RX;  // region index
    const int li = pi - 2, lj = pj - 2;  // tile-local position
    const T ep = Eps<T>::v;
    using hw::donor; using hw::max2; using hw::min2; using hw::min3; using hw::pp; using hw::pn;
    const int SXY = o.sxy, FXY = o.fxy, YXY = o.yxy;

    int rsi = 0, rsj = 0;
    if (t < SW) { rsi = t; rsj = 0; }
    else if (t < 2 * SW) { rsi = t - SW; rsj = SH - 1; }
    else if (t < NRING) { const int r = t - 2 * SW; rsj = 1 + r / 2; rsi = (r & 1) ? SW - 1 : 0; }

    // planes of cells and of z-faces: clamped into the domain on open lids,
    // wrapped with a periodic z (face lp+1 is face 1)
    auto kc = [&](int k) { return pz ? wrap(k, lp) : (k < 1 ? 1 : (k > lp ? lp : k)); };
    auto fc = [&](int k) { return pz ? wrap(k, lp) : (k < 1 ? 1 : (k > lp + 1 ? lp + 1 : k)); };
    // where the x value of region cell (gi, gj) comes from: x (wrapped in
    // periodic directions), the inflow arrays on open walls, else nothing
    auto xsrc = [&](int gi, int gj) -> XSrc<T> {
        if (px) gi = wrap(gi, np);
        if (py) gj = wrap(gj, mp);
        const bool ii = gi >= 1 && gi <= np, jj = gj >= 1 && gj <= mp;
        if (ii && jj) return {x, o.s(gi, gj, 0), SXY};
        if (jj && gi == 0) return {bcx, (gj - 1) - mp, mp};
        if (jj && gi == np + 1) return {bcx, (gj - 1) + mp * lp - mp, mp};
        if (ii && gj == 0) return {bcy, (gi - 1) - np, np};
        if (ii && gj == mp + 1) return {bcy, (gi - 1) + np * lp - np, np};
        return {nullptr, 0, 0};
    };
    auto ld = [&](const XSrc<T>& s, int k) -> T { return s.p ? s.p[s.base + s.stride * kc(k)] : T(0); };

    const int i0 = 1 + (tile % ntx) * TX, j0 = 1 + (tile / ntx) * TY;
    const int gi = i0 + li, gj = j0 + lj;
    const bool in_dom = gi >= 1 && gi <= np && gj >= 1 && gj <= mp;
    // a position in a periodic direction stands for the wrapped cell
    const bool valid = (px || (gi >= 1 && gi <= np)) && (py || (gj >= 1 && gj <= mp));
    const bool do_v1 = valid && (px || gi >= 2) && li >= -1 && lj >= -1 && lj <= TY;
    const bool do_v2 = valid && (py || gj >= 2) && li >= -1 && li <= TX && lj >= -1;
    const bool do_c = valid && li >= -1 && li <= TX && lj >= -1 && lj <= TY;
    const bool do_d = in_dom && li >= 0 && li < TX && lj >= 0 && lj < TY;
    // open wall faces, where the per-stage path sets the flux to zero
    // (flux_x_bcd / flux_y_bcd): the left x-face / lower y-face of this
    // position is face gi / gj of the domain
    const bool wall1 = !px && (gi <= 1 || gi > np), wall2 = !py && (gj <= 1 || gj > mp);
    // source column: the cell itself, wrapped in periodic directions; on
    // open walls the mirror image on the one-cell ring, clamped beyond
    const int ai = px ? wrap(gi, np) : clampi(mirror(gi, np), 1, np);
    const int aj = py ? wrap(gj, mp) : clampi(mirror(gj, mp), 1, mp);
    // the source column's sx coordinates (a periodic position computes the
    // upwind at its own place, where sx holds the wrapped neighbours)
    const int sai = px ? pi + 1 : ai - i0 + 3, saj = py ? pj + 1 : aj - j0 + 3;
    const XSrc<T> own = valid ? XSrc<T>{x, o.s(ai, aj, 0), SXY} : xsrc(gi, gj);
    const uint32_t so = uint32_t(o.s(ai, aj, 1 - o.ih)) * uint32_t(sizeof(T));
    const uint32_t fo = uint32_t(o.f1(ai, aj, 1 - o.ih)) * uint32_t(sizeof(T));
    // faces i+1 and j+1 of the source column (wrapped in periodic directions)
    uint32_t fob = 0, sob = 0;
    if constexpr (PER) {
        const int ib = (px && ai == np) ? 1 : ai + 1;
        const int jb = (py && aj == mp) ? 1 : aj + 1;
        fob = uint32_t(o.f1(ib, aj, 1 - o.ih)) * uint32_t(sizeof(T));
        sob = uint32_t(o.f2(ai, jb, 1 - o.ih)) * uint32_t(sizeof(T));
    }
    // past an open x's last column a position holds a mirrored column's u1:
    // its element of e_u1 is the last column's face n+1 instead
    const bool wall_e = !px && gi == np + 1, last_e = !px && gi == np && pi < RX - 1;
    // tape ownership: x/y halo cells of xant and the wall faces n+1 belong to
    // the tile whose output range touches them
    bool own_fx = false, own_fy = false, own_s = false;
    uint32_t tso = 0, tfo = 0;
    if constexpr (TAPE) {
        const bool ci = li >= 0 && li < TX && gi >= 1 && gi <= np;
        const bool cj = lj >= 0 && lj < TY && gj >= 1 && gj <= mp;
        const bool hi = (gi == 0 && li == -1) || (gi == np + 1 && li >= 0 && li <= TX);
        const bool hj = (gj == 0 && lj == -1) || (gj == mp + 1 && lj >= 0 && lj <= TY);
        own_fx = (ci || (gi == np + 1 && li >= 0 && li <= TX)) && cj;
        own_fy = (cj || (gj == mp + 1 && lj >= 0 && lj <= TY)) && ci;
        own_s = (ci || hi) && (cj || hj);
        if (own_s || own_fx || own_fy) {
            tso = uint32_t(o.s(gi, gj, 1 - o.ih)) * uint32_t(sizeof(T));
            tfo = uint32_t(o.f1(gi, gj, 1 - o.ih)) * uint32_t(sizeof(T));
        }
    }
    const int ihm = o.ih - 1;
    auto pl = [&](auto* a, int stride, int k) { return a + (long long)stride * (k + ihm); };
    // loads of the source column's faces i+1 / j+1 on the plane at p
    auto ld_u1b = [&](const T* p) -> T {
        if constexpr (PER) return ldo(p, fob);
        else return ldo(p + 1, fo);
    };
    auto ld_u2b = [&](const T* p) -> T {
        if constexpr (PER) return ldo(p, sob);
        else return ldo(p + o.yx, so);
    };
    const XSrc<T> ring = t < NRING ? xsrc(i0 + rsi - 3, j0 + rsj - 3) : XSrc<T>{nullptr, 0, 0};
    // x-neighbour availability for the in-plane max/min (edge copies on open
    // walls duplicate the centre and do not change it)
    const bool nxm = px || gi > 1, nxp = px || gi < np, nym = py || gj > 1, nyp = py || gj < mp;

    const int Ks = pz ? k0 - 2 : max(1, k0 - 2), Ke = k1 + 2;
    const int Alast = pz ? k1 + 2 : min(lp, k1 + 2);
    const int Plo = pz ? k0 - 1 : max(1, k0 - 1), Phi = pz ? k1 + 1 : min(lp, k1 + 1);
    // register queues of the source column (as in the gauge kernel) and of
    // the position's own V3 and its donor flux on face K-1
    T xq[3], u1a[2], u1b[2], u2a[2], u2b[2], u3q[3], hq[2];
    xq[0] = ldo(pl(x, SXY, kc(Ks - 1)), so); xq[1] = ldo(pl(x, SXY, kc(Ks)), so);
    xq[2] = ldo(pl(x, SXY, kc(Ks + 1)), so);
    u1a[0] = ldo(pl(u1, FXY, kc(Ks - 1)), fo); u1a[1] = ldo(pl(u1, FXY, kc(Ks)), fo);
    u1b[0] = ld_u1b(pl(u1, FXY, kc(Ks - 1))); u1b[1] = ld_u1b(pl(u1, FXY, kc(Ks)));
    u2a[0] = ldo(pl(u2, YXY, kc(Ks - 1)), so); u2a[1] = ldo(pl(u2, YXY, kc(Ks)), so);
    u2b[0] = ld_u2b(pl(u2, YXY, kc(Ks - 1))); u2b[1] = ld_u2b(pl(u2, YXY, kc(Ks)));
    u3q[0] = ldo(pl(u3, SXY, fc(Ks - 1)), so); u3q[1] = ldo(pl(u3, SXY, fc(Ks)), so);
    u3q[2] = ldo(pl(u3, SXY, fc(Ks + 1)), so);
    hq[0] = ldo(pl(h, SXY, kc(Ks - 1)), so); hq[1] = ldo(pl(h, SXY, kc(Ks)), so);
    T rq2 = ldo(pl(rhr, SXY, kc(Ks)), so);
    T v3 = T(0), w3 = T(0);
    T v3q1 = T(0);  // V3 on face K-2, for the tape
    T xmx[2] = {T(0), T(0)}, xmn[2] = {T(0), T(0)};
    T f3c = T(0);  // flux through the upper z-face of the last output plane

    sx[0][pj + 1][pi + 1] = valid ? xq[1] : ld(own, Ks);
    if (t < NRING) sx[0][rsj][rsi] = ld(ring, Ks);
    // x of plane K+1 for the LDS: ring cell, and the own cell where it is
    // not in the queue; loaded a step ahead (a null source keeps the zero)
    T xr = T(0), xown = T(0);
    const bool ring_on = t < NRING && ring.p, own_on = !valid && own.p;
    const uint32_t rstr = uint32_t(ring.stride) * uint32_t(sizeof(T)),
                   ostr = uint32_t(own.stride) * uint32_t(sizeof(T));
    const char* rp = ring_on ? (const char*)(ring.p + ring.base) : nullptr;
    const char* op = own_on ? (const char*)(own.p + own.base) : nullptr;
    if constexpr (!PER) {
        rp += (uint64_t)rstr * (uint32_t)Ks;
        op += (uint64_t)ostr * (uint32_t)Ks;
    }
    auto ld_halo = [&](int k) __attribute__((always_inline)) {
        if constexpr (PER) {
            if (ring_on) xr = ldo((const T*)(rp + (uint64_t)rstr * (uint32_t)kc(k)), 0);
            if (own_on) xown = ldo((const T*)(op + (uint64_t)ostr * (uint32_t)kc(k)), 0);
        } else {
            rp += rstr;
            op += ostr;
            if (ring_on) xr = ldo((const T*)rp, 0);
            if (own_on) xown = ldo((const T*)op, 0);
        }
    };
    if (Ks + 1 <= Alast) ld_halo(Ks + 1);
    __syncthreads();

    uint32_t so_k = so, fo_k = fo;
    // x of the source column's 3x3 neighbourhood, from one opaque address
    using LT = StdLds<T, RX, RY>;
    constexpr int SZ = (int)sizeof(T);
    // and the position's own elements of the tile arrays, from three (the
    // arrays lie beyond the reach of one immediate offset, and without this
    // the compiler keeps a dozen address registers through the loop)
    constexpr int PLN = RY * RX * SZ;  // one plane of a tile array
    constexpr int MID = (int)offsetof(LT, sf1);
    constexpr int HI = (int)offsetof(LT, e_h) - RX * SZ;  // read one row back
    uint32_t lsx = uint32_t(offsetof(LT, sx) + ((saj - 1) * SW + (sai - 1)) * SZ);
    uint32_t llo = uint32_t(t * SZ);
    asm volatile("" : "+v"(lsx), "+v"(llo));
// the other two, formed anew where a stage uses them (an add instead of a
// register through the loop)
#define LMID_BASE                   \
    uint32_t lmid = llo + MID;      \
    asm volatile("" : "+v"(lmid));
#define LHI_BASE                    \
    uint32_t lhi = llo + HI;        \
    asm volatile("" : "+v"(lhi));
    char* const lds0 = reinterpret_cast<char*>(&L);
#define LSX(s, db, da) \
    (*reinterpret_cast<T*>(lds0 + lsx + ((s) * (SW * SH) + (db) * SW + (da)) * SZ))
// array `arr` at ring slot s, offset (db rows, da columns) from the position
#define LLO(arr, s, db, da) \
    (*reinterpret_cast<T*>(lds0 + llo + ((int)offsetof(LT, arr) + (s) * PLN + ((db) * RX + (da)) * SZ)))
#define LMID(arr, db, da) \
    (*reinterpret_cast<T*>(lds0 + lmid + ((int)offsetof(LT, arr) - MID + ((db) * RX + (da)) * SZ)))
#define LHI(arr, r) (*reinterpret_cast<T*>(lds0 + lhi + ((int)offsetof(LT, arr) - HI + (r) * SZ)))
    // Plane pointers of the loads of a step (in scalar registers): moved by a
    // plane until the last one on open lids, formed anew with a periodic z.
    // a limiter factor: min(1, a, b), where cp and cn are held as min(1, .)
    // (the tape holds them as they are)
    auto lmin = [](T a, T b) {
        if constexpr (TAPE) return min3(T(1), a, b);
        else return min2(a, b);
    };
    const uint32_t SB8 = plane_bytes<T>(SXY), FB8 = plane_bytes<T>(FXY), YB8 = plane_bytes<T>(YXY);
    const T* qx = uniform(pl(x, SXY, kc(Ks + 1)));
    const T* qu1 = uniform(pl(u1, FXY, kc(Ks)));
    const T* qu2 = uniform(pl(u2, YXY, kc(Ks)));
    const T* qu3 = uniform(pl(u3, SXY, fc(Ks + 1)));
    const T* qh = uniform(pl(h, SXY, kc(Ks)));
    const T* qr = uniform(pl(rhr, SXY, kc(Ks)));
    auto adv = [](auto* p, uint32_t d) { return (decltype(p))((uintptr_t)uniform(p) + d); };
    T* qxo = uniform(pl(xo, SXY, Ks - 4));  // plane K-3 during step K
    T xst = T(0);                           // the new x of that plane
    const bool edge_d = do_d && ((!px && (gi == 1 || gi == np)) || (!py && (gj == 1 || gj == mp)));
    // TAPE: what the last steps left for the tape, stored with it (as the new
    // x): V1, V2 of plane K-2; V3, cp and cn of plane K-3; x of plane K with
    // the inflow values on the wall halo (the upwind's input) and with edge
    // copies there (the limiter's bounds)
    T tv1 = T(0), tv2 = T(0), tv3 = T(0), tcp = T(0), tcn = T(0), tx = T(0);
    auto store_tape = [&](int K) __attribute__((always_inline)) {
        if (K - 2 >= k0 && K - 2 <= k1) {
            if (own_fx) sto(pl(tp->v[0], FXY, K - 2), tfo, tv1);
            if (own_fy) sto(pl(tp->v[1], YXY, K - 2), tso, tv2);
        }
        if (do_d && K - 3 >= k0 && K - 3 <= k1) {
            const int Q = K - 3;
            T* const tv = pl(tp->v[2], SXY, Q);
            sto(tv, so, tv3);
            if (Q == lp) sto(tv + SXY, so, -tv3);
            sto(pl(tp->cp, SXY, Q), so, tcp);
            sto(pl(tp->cn, SXY, Q), so, tcn);
        }
        if (do_d && K >= k0 && K <= k1) {
            T* const tb = pl(tp->xb, SXY, K);
            T* const t0 = pl(tp->x0, SXY, K);
            sto(tb, so, tx);
            sto(t0, so, tx);
            if (gi == 1) { sto(tb - 1, so, bcx[(gj - 1) + mp * (K - 1)]); sto(t0 - 1, so, tx); }
            if (gi == np) { sto(tb + 1, so, bcx[(gj - 1) + mp * ((K - 1) + lp)]); sto(t0 + 1, so, tx); }
            if (gj == 1) { sto(tb - o.sx, so, bcy[(gi - 1) + np * (K - 1)]); sto(t0 - o.sx, so, tx); }
            if (gj == mp) { sto(tb + o.sx, so, bcy[(gi - 1) + np * ((K - 1) + lp)]); sto(t0 + o.sx, so, tx); }
        }
    };
    auto step = [&](auto phase, int K) __attribute__((always_inline)) {
        constexpr int PH = decltype(phase)::value;
        asm volatile("" : "+s"(K));
        constexpr int Q3a = PH % 3, Q3b = (PH + 1) % 3, Q3c = (PH + 2) % 3;
        constexpr int Q2a = PH % 2, Q2b = (PH + 1) % 2;
        constexpr int R0 = Q3a, R1 = Q3c, R2 = Q3b, E0 = Q2a, E1 = Q2b;
        T& xq1 = xq[Q3a]; T& xq2 = xq[Q3b]; T& xq3 = xq[Q3c];
        T& u1a0 = u1a[Q2a]; T& u1a1 = u1a[Q2b]; T& u1b0 = u1b[Q2a]; T& u1b1 = u1b[Q2b];
        T& u2a0 = u2a[Q2a]; T& u2a1 = u2a[Q2b]; T& u2b0 = u2b[Q2a]; T& u2b1 = u2b[Q2b];
        T& u3q0 = u3q[Q3a]; T& u3q1 = u3q[Q3b]; T& u3q2 = u3q[Q3c];
        T& hq1 = hq[Q2a]; T& hq2 = hq[Q2b];
        T& xmx0 = xmx[Q2a]; T& xmn0 = xmn[Q2a]; T& xmx1 = xmx[Q2b]; T& xmn1 = xmn[Q2b];
        asm volatile("" : "+v"(so_k), "+v"(fo_k));
        const uint32_t so = so_k, fo = fo_k;
        const bool A_on = K <= Alast;
        // the one wait for the loads of the step, then the store of the last
        // output plane and the edge copies (as in the gauge kernel)
        __builtin_amdgcn_s_waitcnt(0x0f70);  // vmcnt(0)
        qxo = adv(qxo, SB8);
        if (do_d && K - 3 >= k0 && K - 3 <= k1) sto(qxo, so, xst);
        if constexpr (TAPE) {
            tx = xq2;
            store_tape(K);
        }
        if (edge_d && K >= k0 && K <= k1) {
            T* const xok = pl(xo, SXY, K);
            if (!px && gi == 1) sto(xok - 1, so, xq2);
            if (!px && gi == np) sto(xok + 1, so, xq2);
            if (!py && gj == 1) sto(xok - o.sx, so, xq2);
            if (!py && gj == mp) sto(xok + o.sx, so, xq2);
        }
        if (K + 1 <= Alast) {
            sx[E1][pj + 1][pi + 1] = valid ? xq3 : xown;
            if (t < NRING) {
                // the slot's address formed anew (kept, it was spilled)
                uint32_t q = llo;
                asm volatile("" : "+v"(q));
                q /= (uint32_t)SZ;
                const uint32_t r = q - 2 * SW;
                const uint32_t c = q < SW ? q
                                   : q < 2 * SW ? q + (SH - 2) * SW
                                                : (1 + r / 2) * SW + ((r & 1) ? SW - 1 : 0);
                *reinterpret_cast<T*>(lds0 + ((int)offsetof(LT, sx) + E1 * (SW * SH) * SZ) + c * SZ) = xr;
            }
        }
        // V1's inputs from column i-1: the source column of the lane to the
        // left wherever V1 is formed (gi >= 2, or a periodic x)
        const T hx = from_left_lane(hq1) + hq1;
        const T s2x = from_left_lane(u2a0 + u2b0) + u2b0 + u2a0;
        const T s3x = from_left_lane(u3q0 + u3q1) + u3q1 + u3q0;
        const int P = K - 1;
        const bool BC_on = P >= Plo && P <= Phi;
        // the source column's inputs of V2 at the position above (its
        // column j-1)
        if (BC_on) {
            LHI_BASE
            LHI(e_h, 0) = hq1;
            if (!wall_e) LHI(e_u1, 0) = u1a0;
            if (last_e) LHI(e_u1, 1) = u1b0;
            LHI(e_u3a, 0) = u3q0;
            LHI(e_u3b, 0) = u3q1;
        }

        // ---- A: xant and xant/rhr on plane K ------------------------------
        T xa_new;
        auto stage_a = [&](auto edge) __attribute__((always_inline)) {
            constexpr bool EDGE = decltype(edge)::value;
            const bool gnd = EDGE && !pz && K == 1, sky = EDGE && !pz && K == lp;
            const T xc = xq2;
            const T xw = LSX(E0, 1, 0), xe = LSX(E0, 1, 2), xs = LSX(E0, 0, 1), xn = LSX(E0, 2, 1);
            const T hinv = rcp_<FAST>(hq2);
            const T f1p = donor(xc, xe, u1b1);
            const T f1 = donor(xw, xc, u1a1);
            const T f2p = donor(xc, xn, u2b1);
            const T f2 = donor(xs, xc, u2a1);
            T f3p, f3;
            if (gnd) {
                f3p = donor(xc, xq3, u3q2);
                f3 = -f3p;
            } else if (sky) {
                f3 = donor(xq1, xc, u3q1);
                f3p = -f3;
            } else {
                f3p = donor(xc, xq3, u3q2);
                f3 = donor(xq1, xc, u3q1);
            }
            xa_new = rq2 * (xc - (f1p - f1 + f2p - f2 + f3p - f3) * hinv);
            LLO(sxa, R0, 0, 0) = xa_new;
            if constexpr (TAPE)
                if (own_s && K >= k0 && K <= k1) sto(pl(tp->psi, SXY, K), tso, xa_new);
            LLO(src, R0, 0, 0) = div_<FAST>(xa_new, rq2);
            if constexpr (NONOS) {
                T m = xc, n = xc;
                { const T v = nxm ? xw : xc; m = max2(m, v); n = min2(n, v); }
                { const T v = nxp ? xe : xc; m = max2(m, v); n = min2(n, v); }
                { const T v = nym ? xs : xc; m = max2(m, v); n = min2(n, v); }
                { const T v = nyp ? xn : xc; m = max2(m, v); n = min2(n, v); }
                if (!gnd) { m = max2(m, xq1); n = min2(n, xq1); }
                if (!sky) { m = max2(m, xq3); n = min2(n, xq3); }
                xmx1 = m;
                xmn1 = n;
            }
        };
        if (A_on) {
            if (!pz && (K == 1 || K == lp)) stage_a(std::true_type{});
            else stage_a(std::false_type{});
        }
        // the ring of plane K+2, whose registers are free already
        if constexpr (!PER)
            if (K + 2 <= Alast) ld_halo(K + 2);
        __syncthreads();
// xant, xant/rhr of plane K-d at tile position (a, b)
#define XA(d, a, b) LLO(sxa, (d) == 0 ? R0 : ((d) == 1 ? R1 : R2), (b) - lj, (a) - li)
#define RC(d, a, b) LLO(src, (d) == 0 ? R0 : ((d) == 1 ? R1 : R2), (b) - lj, (a) - li)
// cp, cn of plane Q until C
#define CP(a, b) LMID(scp, (b) - lj, (a) - li)
#define CN(a, b) LMID(scn, (b) - lj, (a) - li)
        const int Q = K - 2;
        const bool Dq = Q >= k0 && Q <= k1;
        // ---- limited fluxes through the left x-face and lower y-face of this
        //      position on plane Q (antidiff3d-standard-gpubc.f90:372-407):
        //      V of Q from the previous step, cp/cn of Q and Q-1; formed
        //      before B so that V of Q is dead before V of P is formed ------
        if (Dq) {
            LMID_BASE
            T vl = LMID(sv1, 0, 0), vb = LMID(sv2, 0, 0);
            if constexpr (NONOS) {
                const T c0 = CP(li, lj), n0 = CN(li, lj);
                vl = slim(vl, lmin(c0, CN(li - 1, lj)), lmin(CP(li - 1, lj), n0), XA(2, li - 1, lj),
                          XA(2, li, lj));
                vb = slim(vb, lmin(c0, CN(li, lj - 1)), lmin(CP(li, lj - 1), n0), XA(2, li, lj - 1),
                          XA(2, li, lj));
            }
            const T F1 = donor(RC(2, li - 1, lj), RC(2, li, lj), vl);
            const T F2 = donor(RC(2, li, lj - 1), RC(2, li, lj), vb);
            LMID(sf1, 0, 0) = wall1 ? T(0) : F1;
            LMID(sf2, 0, 0) = wall2 ? T(0) : F2;
        }
        // ---- B: V3 on face K, V1/V2 on plane P (antidiff3d-standard-
        //      gpubc.f90:72-202), their donor fluxes for the limiter -------
        // Straight-line on the interior planes (see the gauge kernel).
        T v3n = T(0), w3n = T(0);
        T w1 = T(0), w2 = T(0);  // donor fluxes of V1/V2 (left, lower faces of P)
        T up, dn;  // (bound - xant) h on plane P, for C
#define SB __builtin_amdgcn_sched_barrier(0);
        auto stage_b = [&](auto edge) __attribute__((always_inline)) {
            constexpr bool EDGE = decltype(edge)::value;
            const bool gnd = EDGE && !pz && P == 1, sky = EDGE && !pz && P == lp;
            const T xc = XA(1, li, lj), xw = XA(1, li - 1, lj), xe = XA(1, li + 1, lj),
                    xs = XA(1, li, lj - 1), xn = XA(1, li, lj + 1);
            T kw, ks, ke, kn;  // plane K
            if (!EDGE || A_on) {
                kw = XA(0, li - 1, lj); ks = XA(0, li, lj - 1);
                ke = XA(0, li + 1, lj); kn = XA(0, li, lj + 1);
            }
            if (!EDGE || (A_on && (pz || K >= 2) && K >= k0 - 1)) {
                const T hmz = rcp_<FAST>(T(0.5) * (hq1 + hq2));
                const T s1 = u1a0 + u1a1 + u1b1 + u1b0;
                const T s2 = u2a0 + u2b0 + u2b1 + u2a1;
                const T a = u3q1;
                v3n = vdyfa_<FAST>(xc, xa_new, a, hmz) +
                      vcorra_<FAST>(a, s1, (abs_(xe) + abs_(ke)) - (abs_(xw) + abs_(kw)),
                                    abs_(xe) + abs_(ke) + abs_(xw) + abs_(kw) + ep, hmz) +
                      vcorra_<FAST>(a, s2, (abs_(xn) + abs_(kn)) - (abs_(xs) + abs_(ks)),
                                    abs_(xn) + abs_(kn) + abs_(xs) + abs_(ks) + ep, hmz);
                if constexpr (NONOS) w3n = donor(xc, xa_new, v3n);
            }
            SB
            if (!EDGE || BC_on) {
                const T xsw = XA(1, li - 1, lj - 1), xnw = XA(1, li - 1, lj + 1),
                        xse = XA(1, li + 1, lj - 1);
                const T bc = XA(2, li, lj);
                T val1, val2;
                {
                    const T hmx = rcp_<FAST>(T(0.5) * hx);
                    const T a = u1a0;
                    val1 = vdyfa_<FAST>(xw, xc, a, hmx) +
                           vcorra_<FAST>(a, s2x, (abs_(xnw) + abs_(xn)) - (abs_(xsw) + abs_(xs)),
                                         abs_(xnw) + abs_(xn) + abs_(xsw) + abs_(xs) + ep, hmx);
                    if (!gnd && !sky) {
                        const T bw = XA(2, li - 1, lj);
                        val1 = val1 + vcorra_<FAST>(a, s3x,
                                                    (abs_(kw) + abs_(xa_new)) - (abs_(bw) + abs_(bc)),
                                                    abs_(kw) + abs_(xa_new) + abs_(bw) + abs_(bc) + ep,
                                                    hmx);
                    }
                }
                SB
                {
                    // column j-1: the source column of the position below
                    LHI_BASE
                    const T nv2_h = LHI(e_h, -RX), nv2_u1a = LHI(e_u1, -RX),
                            nv2_u1b = LHI(e_u1, -RX + 1), nv2_u3a = LHI(e_u3a, -RX),
                            nv2_u3b = LHI(e_u3b, -RX);
                    const T hmy = rcp_<FAST>(T(0.5) * (nv2_h + hq1));
                    const T s1 = nv2_u1a + u1a0 + u1b0 + nv2_u1b;
                    const T a = u2a0;
                    val2 = vdyfa_<FAST>(xs, xc, a, hmy) +
                           vcorra_<FAST>(a, s1, (abs_(xse) + abs_(xe)) - (abs_(xsw) + abs_(xw)),
                                         abs_(xse) + abs_(xe) + abs_(xsw) + abs_(xw) + ep, hmy);
                    if (!gnd && !sky) {
                        const T s3 = nv2_u3a + u3q0 + u3q1 + nv2_u3b;
                        const T bs = XA(2, li, lj - 1);
                        val2 = val2 + vcorra_<FAST>(a, s3,
                                                    (abs_(ks) + abs_(xa_new)) - (abs_(bs) + abs_(bc)),
                                                    abs_(ks) + abs_(xa_new) + abs_(bs) + abs_(bc) + ep,
                                                    hmy);
                    }
                }
                const T v1 = do_v1 ? val1 : T(0), v2 = do_v2 ? val2 : T(0);
                LMID_BASE
                LMID(sv1, 0, 0) = v1;
                LMID(sv2, 0, 0) = v2;
                if constexpr (NONOS) {
                    w1 = donor(xw, xc, val1);
                    w2 = donor(xs, xc, val2);
                    w1 = do_v1 ? w1 : T(0);
                    w2 = do_v2 ? w2 : T(0);
                    LMID(sw2, 0, 0) = w2;
                    T mx = xw, mn = xw;
#define ACC(v, lo, hi) { T t_ = (v); lo = min2(lo, t_); hi = max2(hi, t_); }
                    ACC(xc, mn, mx) ACC(xe, mn, mx) ACC(xs, mn, mx) ACC(xn, mn, mx)
                    if (!gnd) ACC(bc, mn, mx)
                    if (!sky) ACC(xa_new, mn, mx)
#undef ACC
                    mx = max2(mx, xmx0);
                    mn = min2(mn, xmn0);
                    up = (mx - xc) * hq1;
                    dn = (xc - mn) * hq1;
                }
                if constexpr (TAPE) tv1 = v1, tv2 = v2;
            }
        };
        if (BC_on && (pz || (P != 1 && P != lp))) stage_b(std::false_type{});
        else stage_b(std::true_type{});
        // h and rhr of the output plane K-2, for D: first of the loads, so
        // that the wait for them leaves the others in flight (two planes of
        // registers or LDS would keep them, and there are none)
        const T hD = ldo(pl(h, SXY, kc(Q)), so), rD = ldo(pl(rhr, SXY, kc(Q)), so);
        // the oldest slot of each queue becomes the newest of step K+1
        {
            const int Kn = K + 1;
            if (PER && pz) {
                qx = pl(x, SXY, kc(Kn + 1)); qr = pl(rhr, SXY, kc(Kn));
                qu1 = pl(u1, FXY, kc(Kn)); qu2 = pl(u2, YXY, kc(Kn)); qu3 = pl(u3, SXY, fc(Kn + 1));
                qh = pl(h, SXY, kc(Kn));
            } else {
                const bool more = Kn <= lp;
                const uint32_t dS = more ? SB8 : 0, dF = more ? FB8 : 0, dY = more ? YB8 : 0;
                qu1 = adv(qu1, dF); qu2 = adv(qu2, dY); qu3 = adv(qu3, dS);
                qh = adv(qh, dS);
                qx = adv(qx, Kn < lp ? SB8 : 0); qr = adv(qr, dS);
            }
            if constexpr (PER)
                if (Kn + 1 <= Alast) ld_halo(Kn + 1);
            xq1 = ldo(qx, so);
            rq2 = ldo(qr, so);
            u1a0 = ldo(qu1, fo);
            u1b0 = ld_u1b(qu1);
            u2a0 = ldo(qu2, so);
            u2b0 = ld_u2b(qu2);
            u3q0 = ldo(qu3, so);
            hq1 = ldo(qh, so);
        }
        // donor flux of V1 through the right x-face of P: the left face of
        // the position to the right (the lane to the right, in the same row
        // wherever the limiter runs)
        const T w1p = NONOS ? from_right_lane(w1) : T(0);
        __syncthreads();
        // ---- C: cp, cn on plane P (antidiff3d-standard-gpubc.f90:260-347) --
        LMID_BASE
        T cpP, cnP, cpQ, cnQ;  // of the own column on planes P (formed here) and Q
        if constexpr (NONOS) {
            auto stage_c = [&](auto edge) __attribute__((always_inline)) {
                constexpr bool EDGE = decltype(edge)::value;
                const bool gnd = EDGE && !pz && P == 1, sky = EDGE && !pz && P == lp;
                const T a1p = w1p, a1 = w1;
                const T a2p = LMID(sw2, 1, 0), a2 = LMID(sw2, 0, 0);
                T a3p, a3;
                if (gnd) { a3p = w3n; a3 = -a3p; }
                else if (sky) { a3 = w3; a3p = -a3; }
                else { a3p = w3n; a3 = w3; }
                T rp = div_<FAST>(up,
                                  pn(a1p) + pp(a1) + pn(a2p) + pp(a2) + pn(a3p) + pp(a3) + ep);
                T rn = div_<FAST>(dn,
                                  pp(a1p) + pn(a1) + pp(a2p) + pn(a2) + pp(a3p) + pn(a3) + ep);
                if constexpr (!TAPE) {
                    rp = min2(T(1), rp);
                    rn = min2(T(1), rn);
                }
                cpQ = CP(li, lj);
                cnQ = CN(li, lj);
                CP(li, lj) = cpP = do_c ? rp : T(0);
                CN(li, lj) = cnP = do_c ? rn : T(0);
            };
            if (BC_on) {
                if (!pz && (P == 1 || P == lp)) stage_c(std::true_type{});
                else stage_c(std::false_type{});
            } else if constexpr (TAPE) {
                cpQ = CP(li, lj);
                cnQ = CN(li, lj);
            }
        }
        // limited flux through face Q+1 of the own column; the first output
        // plane's lower one is formed on the step before its own
        T F3p = T(0);
        if (BC_on && !(!pz && Q == lp)) {
            T vl = v3;
            if constexpr (NONOS)
                vl = slim(vl, lmin(cpP, cnQ), lmin(cpQ, cnP), XA(2, li, lj), XA(1, li, lj));
            F3p = donor(RC(2, li, lj), RC(1, li, lj), vl);
        }
        const T F3 = f3c;
        f3c = F3p;
        // ---- D: the new x on plane Q (antidiff3d-standard-gpubc.f90:431-459)
        if (Dq) {
            const bool gnd = !pz && Q == 1, sky = !pz && Q == lp;
            const T F1 = LMID(sf1, 0, 0), F1p = LMID(sf1, 0, 1);
            const T F2 = LMID(sf2, 0, 0), F2p = LMID(sf2, 1, 0);
            T sum = F1p - F1 + F2p - F2;
            if (gnd) sum = sum + F3p + F3p;
            else if (sky) sum = sum - F3 - F3;
            else sum = sum + F3p - F3;
            if constexpr (TAPE) {
                // V3 on the lower face Q of the cell (face 1 = -face 2 on the ground)
                // and, above the sky plane, on face lp+1 = -face lp
                tv3 = gnd ? -v3 : v3q1;
                tcp = cpQ;
                tcn = cnQ;
            }
            const T hinv = rcp_<FAST>(hD);
            xst = rD * (RC(2, li, lj) - sum * hinv);
        }
#undef XA
#undef RC
#undef CP
#undef CN
        if constexpr (TAPE) v3q1 = v3;
        v3 = v3n;
        w3 = w3n;
    };
#undef LSX
#undef LLO
#undef LMID
#undef LHI
#undef LMID_BASE
#undef LHI_BASE
#undef SB
    for (int K = Ks;;) {
        step(std::integral_constant<int, 0>{}, K);
        if (++K > Ke) break;
        step(std::integral_constant<int, 1>{}, K);
        if (++K > Ke) break;
        step(std::integral_constant<int, 2>{}, K);
        if (++K > Ke) break;
        step(std::integral_constant<int, 3>{}, K);
        if (++K > Ke) break;
        step(std::integral_constant<int, 4>{}, K);
        if (++K > Ke) break;
        step(std::integral_constant<int, 5>{}, K);
        if (++K > Ke) break;
    }
    if (do_d) sto(pl(xo, SXY, k1), so, xst);
    if constexpr (TAPE) store_tape(k1 + 3);
}

template <typename T, int RX, int RY, int MINB, bool NONOS, bool PER, bool TAPE = false,
          bool FAST = false>
__global__ void __launch_bounds__(RX * RY, MINB)
k_fused_std(Geo g, Off o, March m, const T* __restrict__ x, const T* __restrict__ u1,
            const T* __restrict__ u2, const T* __restrict__ u3, const T* __restrict__ rhr,
            const T* __restrict__ h, const T* __restrict__ bcx, const T* __restrict__ bcy,
            T* __restrict__ xo, StdTape<T> tp) {
    __shared__ StdLds<T, RX, RY> L;
    if (blockIdx.x >= (unsigned)m.nwg) {
        copy_untouched_halo<T>(g, x, xo, blockIdx.x - m.nwg, gridDim.x - m.nwg);
        return;
    }
    march_items(m, g.lp, [&](int tile, int k0, int k1) {
        fused_std_item<T, RX, RY, NONOS, PER, TAPE, FAST>(g, o, m.ntx, tile, k0, k1, x, u1, u2, u3,
                                                          rhr, h, bcx, bcy, xo, L, &tp);
    });
}

template <typename T, int RX, int RY, int MINB, bool NONOS, bool PER, bool TAPE = false,
          bool FAST = false>
hipError_t launch_std(const Geo& g, const Off& o, const Tiling& tl, const T* x, T* xout,
                      const T* u1, const T* u2, const T* u3, const T* rhr, const T* h,
                      const T* bcx, const T* bcy, hipStream_t s,
                      const StdTape<T>& tp = StdTape<T>{}) {
    long long slots = 0;
    const hipError_t e = resident(k_fused_std<T, RX, RY, MINB, NONOS, PER, TAPE, FAST>, RX * RY,
                                  tl.per_cu, slots);
    if (e != hipSuccess) return e;
    const March m = plan_march<RX, RY>(g, slots, tl.chunk);
    // a recorded step leaves the halo of its output alone
    const int hb = TAPE ? 0 : halo_blocks(halo_cells(g), RX * RY);
    k_fused_std<T, RX, RY, MINB, NONOS, PER, TAPE, FAST><<<m.nwg + hb, RX * RY, 0, s>>>(
        g, o, m, x, u1, u2, u3, rhr, h, bcx, bcy, xout, tp);
    return hipGetLastError();
}

template <typename T, int RX, int RY, int MINB, bool FAST = false>
hipError_t launch_std_any(const Geo& g, const Off& o, const Tiling& tl, int nonos, const T* x, T* xout,
                          const T* u1, const T* u2, const T* u3, const T* rhr, const T* h,
                          const T* bcx, const T* bcy, hipStream_t s) {
    const bool per = g.px || g.py || g.pz;
    if (nonos) {
        if (per) return launch_std<T, RX, RY, MINB, true, true, false, FAST>(g, o, tl, x, xout, u1, u2, u3, rhr, h, bcx, bcy, s);
        return launch_std<T, RX, RY, MINB, true, false, false, FAST>(g, o, tl, x, xout, u1, u2, u3, rhr, h, bcx, bcy, s);
    }
    if (per) return launch_std<T, RX, RY, MINB, false, true, false, FAST>(g, o, tl, x, xout, u1, u2, u3, rhr, h, bcx, bcy, s);
    return launch_std<T, RX, RY, MINB, false, false, false, FAST>(g, o, tl, x, xout, u1, u2, u3, rhr, h, bcx, bcy, s);
}

// One step of the standard variant on the build FAST selects, with the tiling
// rule of the gauge kernel (384x320x192, fast build: 638 us with the 32x32
// tiles it picks, 687 with 32x16; 64x64x32 takes 32x16, 23.5 against 30 us).
template <typename T, bool FAST>
hipError_t std_step(const Geo& g, int nonos, const T* x, T* xout, const T* u1, const T* u2,
                    const T* u3, const T* rhr, const T* h, const T* bcx, const T* bcy,
                    hipStream_t s) {
    const Off o = make_off(g);
    const Tiling tl = choose_tiling<T>(g);
    return tl.cfg == 0
               ? launch_std_any<T, 32, 32, 4, FAST>(g, o, tl, nonos, x, xout, u1, u2, u3, rhr, h, bcx, bcy, s)
               : launch_std_any<T, 32, 16, 4, FAST>(g, o, tl, nonos, x, xout, u1, u2, u3, rhr, h, bcx, bcy, s);
}

}  // namespace

}  // namespace mpdata
