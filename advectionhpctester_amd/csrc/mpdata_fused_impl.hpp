// Kernel templates of the fused single-pass MPDATA step, shared by the
// exactly rounded build (mpdata_fused.hip, -ffp-contract=off, IEEE division)
// and the fast one (mpdata_fused_fast.hip, FMA contraction and
// Newton-refined reciprocals, FAST = true).
//
// Fused single-pass MPDATA step for gfx950: donor-cell upwind, infinite-gauge
// pseudo-velocities, non-oscillatory limiter and the limited corrective update
// of the reference's two-step GPUBC path (advection/src_algorithms/
// upwind3d-gpubc.f90:101-198 and antidiff3d-gauge-gpubc.f90:71-430) in one
// kernel that reads x, u1, u2, u3, h, rhr once and writes the new x once.
// The fixed-position kernel also has a density mode (DensIO) for the step of
// mpdata3d-rho-gauge-gpubc.f90:107-622.
//
// Decomposition: one workgroup per TX x TY column tile of the (i,j) plane,
// marching k from the ground to the sky (2.5-D).  Per plane K the workgroup
//   A  computes xant on plane K over the tile plus a 2-cell ring,
//   B  the pseudo-velocities V1,V2 on plane K-1 (tile + 1-face ring) and V3
//      on face K (between planes K-1 and K),
//   C  the limiter ratios cp,cn on plane K-1 (tile + 1-cell ring),
//   D  the new x on plane K-2 (the tile),
// keeping the last three xant planes in an LDS ring, one plane each of V1, V2,
// cp and cn in LDS (plane K-2 until stage B or C replaces it by K-1) and the V3
// faces and the column's inputs in register queues.  Halo values follow the
// reference's boundary semantics directly (inflow values for the upwind,
// mirrored xant, zero wall velocities, edge-copied x for the limiter, zero
// cp/cn halo), so no halo-fill kernels run.  Expressions are those of the
// per-stage kernels, operand for operand, so the fused result is bit-identical
// to them.
#pragma once
#include "mpdata_fused.hpp"

#include <algorithm>
#include <type_traits>
#include <cstdlib>
#include <cstddef>

namespace mpdata {

namespace {

// Offsets with 32-bit arithmetic (the host checks every array fits).
struct Off {
    int sx, sxy;      // scalar strides
    int fx, fxy;      // x-face strides
    int yx, yxy;      // y-face strides
    int ih;
    __device__ int s(int i, int j, int k) const { return (i + ih - 1) + sx * (j + ih - 1) + sxy * (k + ih - 1); }
    __device__ int f1(int i, int j, int k) const { return (i + ih - 1) + fx * (j + ih - 1) + fxy * (k + ih - 1); }
    __device__ int f2(int i, int j, int k) const { return (i + ih - 1) + yx * (j + ih - 1) + yxy * (k + ih - 1); }
    __device__ int f3(int i, int j, int k) const { return s(i, j, k); }  // z-faces share the scalar x/y strides
};

__device__ __forceinline__ int mirror(int i, int n) { return i == 0 ? 2 : (i == n + 1 ? n - 1 : i); }

// Element at byte offset `off` from `p`, where p is uniform over the
// workgroup (an array's plane) and off a per-lane 32-bit offset: the
// global_load/store saddr form (scalar base + 32-bit vector offset), with no
// per-lane 64-bit address arithmetic.
template <typename T>
__device__ __forceinline__ T ldo(const T* p, uint32_t off) {
    typedef const __attribute__((address_space(1))) char* G;
    return *(const __attribute__((address_space(1))) T*)((G)p + off);
}
template <typename T>
__device__ __forceinline__ void sto(T* p, uint32_t off, T v) {
    typedef __attribute__((address_space(1))) char* G;
    *(__attribute__((address_space(1))) T*)((G)p + off) = v;
}

// Bytes of a plane of n elements.  Planes are below 4 GiB (Fused::supports):
// from 2 GiB on the product does not fit an int.
template <typename T>
__host__ __device__ constexpr uint32_t plane_bytes(int n) {
    return uint32_t(n) * uint32_t(sizeof(T));
}
// (evaluated at compile time, where a signed overflow is an error)
static_assert(plane_bytes<double>(1 << 28) == 0x80000000u && plane_bytes<float>(1 << 29) == 0x80000000u);

// A value that is the same in every lane, in scalar registers: the compiler
// cannot tell where it comes from memory that the kernel might write.
template <typename S>
__device__ __forceinline__ S uniform(const S& s) {
    static_assert(sizeof(S) % 4 == 0, "copied by words");
    struct W { int w[sizeof(S) / 4]; } b = __builtin_bit_cast(W, s);
#pragma unroll
    for (int i = 0; i < (int)(sizeof(S) / 4); i++) b.w[i] = __builtin_amdgcn_readfirstlane(b.w[i]);
    return __builtin_bit_cast(S, b);
}

// The value held by lane l-1 of the wave (DPP wave_shr:1; lane 0, which has
// no source lane, gets 0 through bound_ctrl, so no old value has to be set).
// Convergent: called with every lane of the wave active.
__device__ __forceinline__ double from_left_lane(double v) {
    const unsigned long long b = (unsigned long long)__double_as_longlong(v);
    const int lo = __builtin_amdgcn_mov_dpp((int)(unsigned)b, 0x138, 0xf, 0xf, true);
    const int hi = __builtin_amdgcn_mov_dpp((int)(unsigned)(b >> 32), 0x138, 0xf, 0xf, true);
    return __longlong_as_double((long long)(((unsigned long long)(unsigned)hi << 32) | (unsigned)lo));
}
__device__ __forceinline__ float from_left_lane(float v) {
    return __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), 0x138, 0xf, 0xf, true));
}
__device__ __forceinline__ int clampi(int i, int lo, int hi) { return i < lo ? lo : (i > hi ? hi : i); }

// Reciprocal and quotient of the fast build (FAST = true): the hardware
// reciprocal (v_rcp) refined by one Newton step e = 1 - b*r, r += e*r, and
// the quotient a*r: a few ulps from the IEEE quotient, in four
// instructions instead of the ten of the IEEE expansion with its scale and
// fix-up steps.  The 50-step difference from the exact build at
// 512x512x256 is 1.2e-14 (6.6e-15 with a second Newton step and a
// correction of the quotient, 1.9 % slower), against the 1e-12 tolerance.  The operands are positive and of order one (h, rhr and the
// limiter denominators, which include eps), far from the ends of the
// exponent range.  FAST = false is the reference's IEEE division.
__device__ __forceinline__ double rcp_nr(double b) {
    const double r = __builtin_amdgcn_rcp(b);
    return __builtin_fma(__builtin_fma(-b, r, 1.0), r, r);
}
__device__ __forceinline__ float rcp_nr(float b) {
    const float r = __builtin_amdgcn_rcpf(b);
    return __builtin_fmaf(__builtin_fmaf(-b, r, 1.0f), r, r);
}
__device__ __forceinline__ double fma_(double a, double b, double c) { return __builtin_fma(a, b, c); }
__device__ __forceinline__ float fma_(float a, float b, float c) { return __builtin_fmaf(a, b, c); }
template <bool FAST, typename T>
__device__ __forceinline__ T rcp_(T b) {
    if constexpr (FAST) return rcp_nr(b);
    else return T(1) / b;
}
template <bool FAST, typename T>
__device__ __forceinline__ T div_(T a, T b) {
    if constexpr (FAST) {
        return a * rcp_nr(b);
    } else {
        return a / b;
    }
}

// ---------------------------------------------------------------------------
// The fused kernel: fixed per-thread column positions.
//
// A workgroup of RX*RY threads covers an RX x RY region of (i,j) columns:
// the TX x TY output tile (TX=RX-4, TY=RY-4) plus a 2-cell ring.  Thread t
// owns region position (t % RX, t / RX) for the whole k-march, so every value
// a position needs only at its own column (x, u, h, rhr of the planes around
// K, its xant, V3) lives in a register queue, and values read by in-plane
// neighbours go through LDS:
//   sx   x on planes K and K+1 with a 3-cell ring (inflow halo values)
//   sxa  xant, planes K-2 .. K
//   sv1, sv2   V1 and V2: plane K-1 from B on, K-2 until then
//   scp, scn   cp and cn: plane K-1 from C on, K-2 until then
//   sf1, sf2   limited x/y face fluxes of plane K-2
//   e_*  h, u1, u3 of each column on plane K-1
//   rr, hh  a thread's own r and h until the update two planes on
// The z cross terms of V1 and V2 use pair sums:
// rat4(xa(i-1,k-1), xa(i,k-1), xa(i-1,k+1), xa(i,k+1)) =
//   ((xa(i,k+1)+xa(i-1,k+1)) - (xa(i,k-1)+xa(i-1,k-1)))*0.25,
// the same operations in the same order as the reference.
//
// Two barriers per plane: stage A reads the x plane that the previous step
// wrote and writes the next one; B reads the xant A wrote; C/D read the V
// that B wrote.  A slot is rewritten only after a barrier that every other
// thread's reads of its previous plane precede; a thread's own later reads of
// it come before its write in program order.
//
// The grid is persistent: workgroups loop over (tile, k-range) work items, a
// range of output planes [k0,k1] recomputing xant from k0-2 and cp,cn,V from
// k0-1.  Inputs of plane K+1 are loaded while plane K is computed.
//
// What bounds it: not HBM (512x512x256 moves 4.4 GB in 1.26 ms) but the chain of
// a plane.  Four waves per SIMD, all of one workgroup and so in the same
// stage, hide little of a wait, and the registers (128) leave no room for
// more.  So nothing waits inside a step but the two barriers: all loads of a
// step are issued together after B and waited for once, before A; the store
// of a plane is issued right after that wait (not so the extra outputs of PASS
// 1 and of the density mode, and the latter's extra inputs, which stage D
// still stores and loads: the next step's wait exposes them); h and rhr of the
// plane being updated are kept, not loaded again; V, the bounds and cp/cn are
// formed straight-line by every lane, so that their LDS reads go out together.
// Together with the scalar plane pointers and the equal runs of March,
// 512x512x256 went from 1.66 to 1.26 ms (fast build) and 256x256x128 from 294
// to 232 us (exact build).
// ---------------------------------------------------------------------------
template <typename T>
struct XSrc {  // where one sx cell comes from: x, bcx, bcy or nothing
    const T* p;
    int base, stride;
};

// LDS of one workgroup of the fixed-position kernel.
template <typename T, int RX, int RY>
struct FusedLds {
    T sx[2][RY + 2][RX + 2];
    T sxa[3][RY][RX];
    T sv1[RY][RX];
    T sv2[RY][RX];
    T scp[RY][RX];
    T scn[RY][RX];
    T sf1[RY][RX];  // limited flux through the left x-face, plane K-2
    T sf2[RY][RX];  // limited flux through the lower y-face, plane K-2
    // h, u1 (face i), u3 (faces P, P+1) of each source column on plane P
    T e_h[RY * RX], e_u1[RY * RX], e_u3a[RY * RX], e_u3b[RY * RX];
    // r (FAST: r/h) of planes K-2..K and h of plane K-2 of the own column, for
    // the update (a thread's own values, kept here for want of registers)
    T rr[3][RY][RX];
    T hh[RY][RX];
};
static_assert(sizeof(FusedLds<double, 32, 32>) <= 160 * 1024, "LDS of one CU");

// One work item: output tile `tile` (ntx tiles per row) over the output
// planes [k0, k1].  Every argument is uniform over the workgroup, so all
// threads pass the same barriers.
// DENS: the density step (DensIO) -- the upwind divides by h without the
// rhr factor, the update has no rhr, and the output plane also writes
// x_incomp, pexr1, pexr2, rhoadv, rhr and the total mass fluxes
// (mpdata3d-rho-gauge-gpubc.f90:123-192, 377-593).
// FAST: the fast build's division (rcp_, div_); the file that instantiates it
// is compiled with FMA contraction.
// PASS: 0 the two-pass step; 1 the same, also writing the limited
// velocities of the corrective pass (the fluxes F of the infinite gauge) to
// pio->ul1..3 on faces 1..n+1, as the reference's stage returns them for a
// further pass; 2 a further corrective pass (antidiff3d-gauge-gpubc.f90:81-
// 83): stage A reads the previous pass's result pio->xa (at the mirrored
// source column) instead of computing the upwind, u1..u3 are that pass's
// limited velocities and x is the field at time level n (limiter bounds).
// TAPE (the two-pass step with open walls, ih = 1): the step also writes the
// intermediates the adjoint step reads to tp, as the per-stage recording
// leaves them: x with inflow values / edge copies on the wall halo, xant
// with its mirrored x/y halo ring, V on every face of the domain (zero on
// the x/y walls, mirrored on the lids), cp and cn.  Each cell and face is
// written by the one position that owns it.
// EARLY: x and r of the next plane are loaded before the first barrier.  Not
// on the batch's tilings bounded at 2 waves per SIMD: their registers then go
// past 128 and a CU holds one workgroup instead of the two that its LDS fits
// (32 members of 32..256 cells a side, fast build, 64x8 tiles: 3.72 ms a step
// with it, 2.92 without; 32x16: 2.64 and 2.17).
template <typename T, int RX, int RY, bool DENS = false, bool FAST = false, int PASS = 0,
          bool TAPE = false, bool EARLY = FAST>
__device__ __forceinline__ void fused_item(const Geo& g, const Off& o, int ntx, int tile, int k0,
                                           int k1, const T* __restrict__ x, const T* __restrict__ u1,
                                           const T* __restrict__ u2, const T* __restrict__ u3,
                                           const T* __restrict__ rhr, const T* __restrict__ h,
                                           const T* __restrict__ bcx, const T* __restrict__ bcy,
                                           T* __restrict__ xo,
                                           FusedLds<T, RX, RY>& L,
                                           const DensIO<T>* dio = nullptr,
                                           const PassIO<T>* pio = nullptr,
                                           const StdTape<T>* tp = nullptr) {
    static_assert(!TAPE || (!DENS && !FAST && PASS == 0), "the tape covers the two-pass step");
    constexpr int NT = RX * RY, TX = RX - 4, TY = RY - 4;
    constexpr int SW = RX + 2, SH = RY + 2, NRING = 2 * SW + 2 * (SH - 2);
    // lane t-1 holds region position (pi-1, pj) for every pi >= 1, in the
    // same wave, and the workgroup is whole waves
    static_assert((64 % RX == 0 || RX % 64 == 0) && NT % 64 == 0, "row layout of the waves");
    static_assert(NRING <= NT, "x ring must fit one extra slot per thread");
    auto& sx = L.sx;
    auto& sxa = L.sxa;
    auto& sv1 = L.sv1;
    const int np = g.np, mp = g.mp, lp = g.lp;
    const int t = threadIdx.x;
    const int pi = t % RX, pj = t / RX;  // region index
    const int li = pi - 2, lj = pj - 2;  // tile-local position
    const T ep = Eps<T>::v;
    using hw::donor; using hw::gflux; using hw::max2; using hw::min2; using hw::pp; using hw::pn;
    const int SXY = o.sxy, FXY = o.fxy, YXY = o.yxy;

    // ring slot of the sx plane handled by this thread (if t < NRING)
    int rsi = 0, rsj = 0;
    if (t < SW) { rsi = t; rsj = 0; }
    else if (t < 2 * SW) { rsi = t - SW; rsj = SH - 1; }
    else if (t < NRING) { const int r = t - 2 * SW; rsj = 1 + r / 2; rsi = (r & 1) ? SW - 1 : 0; }

    auto xsrc = [&](int gi, int gj) -> XSrc<T> {
        const bool ii = gi >= 1 && gi <= np, jj = gj >= 1 && gj <= mp;
        if (ii && jj) return {x, o.s(gi, gj, 0), SXY};
        if (jj && gi == 0) return {bcx, (gj - 1) - mp, mp};
        if (jj && gi == np + 1) return {bcx, (gj - 1) + mp * lp - mp, mp};
        if (ii && gj == 0) return {bcy, (gi - 1) - np, np};
        if (ii && gj == mp + 1) return {bcy, (gi - 1) + np * lp - np, np};
        return {nullptr, 0, 0};
    };
    auto ld = [](const XSrc<T>& s, int k) -> T { return s.p ? s.p[s.base + s.stride * k] : T(0); };
    auto kc = [&](int k) { return k < 1 ? 1 : (k > lp ? lp : k); };        // cell planes
    auto fc = [&](int k) { return k < 1 ? 1 : (k > lp + 1 ? lp + 1 : k); };  // z-face planes


    const int i0 = 1 + (tile % ntx) * TX, j0 = 1 + (tile / ntx) * TY;
    const int gi = i0 + li, gj = j0 + lj;
    const bool in_dom = gi >= 1 && gi <= np && gj >= 1 && gj <= mp;
    // roles of this position
    const bool do_v1 = in_dom && gi >= 2 && li >= -1 && lj >= -1 && lj <= TY;
    const bool do_v2 = in_dom && gj >= 2 && li >= -1 && li <= TX && lj >= -1;
    const bool do_c = in_dom && li >= -1 && li <= TX && lj >= -1 && lj <= TY;
    const bool do_d = in_dom && li >= 0 && li < TX && lj >= 0 && lj < TY;
    // upwind source cell: itself in the domain, the mirror image on the
    // one-cell halo ring (cp_scnd_last_to_halo_xy_fulld), clamped beyond
    const int ai = clampi(mirror(gi, np), 1, np), aj = clampi(mirror(gj, mp), 1, mp);
    const int sai = ai - i0 + 3, saj = aj - j0 + 3;  // its sx coordinates
    const int bs = o.s(ai, aj, 0);
    const XSrc<T> own = in_dom ? XSrc<T>{x, bs, SXY} : xsrc(gi, gj);
    // byte offsets of the source column inside a plane: so for cell arrays,
    // z-faces and y-faces (whose in-plane strides equal the cell ones),
    // fo for x-faces; planes are addressed by uniform pointers
    const uint32_t so = uint32_t(o.s(ai, aj, 1 - o.ih)) * uint32_t(sizeof(T));
    const uint32_t fo = uint32_t(o.f1(ai, aj, 1 - o.ih)) * uint32_t(sizeof(T));
    const int ihm = o.ih - 1;
    auto pl = [&](auto* a, int stride, int k) { return a + (long long)stride * (k + ihm); };
    const XSrc<T> ring = t < NRING ? xsrc(i0 + rsi - 3, j0 + rsj - 3) : XSrc<T>{nullptr, 0, 0};
    // x-neighbour availability for the in-plane max/min (edge copies
    // duplicate the centre and do not change it)
    const bool nxm = gi > 1, nxp = gi < np, nym = gj > 1, nyp = gj < mp;
    // the position past the last column holds a mirrored column's u1: its
    // element of e_u1 is the last column's face n+1 instead
    const bool wall_e = gi == np + 1, last_e = gi == np && pi < RX - 1;
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

    const int Ks = max(1, k0 - 2), Ke = k1 + 2;
    const int Alast = min(lp, k1 + 2);
    // register queues of the source column; during step K they hold
    //   xq1..3 = x(K-1..K+1), u1a0/1 = u1(i,K-1..K), u1b0/1 = u1(i+1,K-1..K),
    //   u2a/u2b likewise at j and j+1, u3q0..2 = faces K-1..K+1,
    //   hq1..2 = h(K-1..K), rq2 = rhr(K),
    //   xmx0/xmn0 = bounds of x for the limiter on plane K-1 (xmx1/xmn1:
    //   plane K, formed in A).
    // The column's own xant of planes K-2..K comes from sxa: the slot of
    // an own position is rewritten only by this thread, later in program
    // order.
    // The k loop is unrolled six-fold: step PH of a round handles a plane
    // K with K - Ks = PH (mod 6), so every ring slot (K - Ks mod 2 or 3) is
    // a compile-time constant, which makes the LDS offsets immediates, and
    // the queues are arrays whose roles rotate with PH instead of being
    // copied: a new plane is loaded into the slot of the oldest one.
    T xq[3], u1a[2], u1b[2], u2a[2], u2b[2], u3q[3], hq[2];
    xq[0] = ldo(pl(x, SXY, kc(Ks - 1)), so); xq[1] = ldo(pl(x, SXY, kc(Ks)), so);
    xq[2] = ldo(pl(x, SXY, kc(Ks + 1)), so);
    u1a[0] = ldo(pl(u1, FXY, kc(Ks - 1)), fo); u1a[1] = ldo(pl(u1, FXY, kc(Ks)), fo);
    u1b[0] = ldo(pl(u1, FXY, kc(Ks - 1)) + 1, fo); u1b[1] = ldo(pl(u1, FXY, kc(Ks)) + 1, fo);
    u2a[0] = ldo(pl(u2, YXY, kc(Ks - 1)), so); u2a[1] = ldo(pl(u2, YXY, kc(Ks)), so);
    u2b[0] = ldo(pl(u2, YXY, kc(Ks - 1)) + o.yx, so); u2b[1] = ldo(pl(u2, YXY, kc(Ks)) + o.yx, so);
    u3q[0] = ldo(pl(u3, SXY, fc(Ks - 1)), so); u3q[1] = ldo(pl(u3, SXY, fc(Ks)), so);
    u3q[2] = ldo(pl(u3, SXY, fc(Ks + 1)), so);
    hq[0] = ldo(pl(h, SXY, kc(Ks - 1)), so); hq[1] = ldo(pl(h, SXY, kc(Ks)), so);
    T rq2 = T(0);
    if constexpr (!DENS) rq2 = ldo(pl(rhr, SXY, kc(Ks)), so);
    // PASS 2: the previous pass's result on plane K (stage A's xant)
    T xaq = T(0);
    if constexpr (PASS == 2) xaq = ldo(pl(pio->xa, SXY, kc(Ks)), so);
    // V3 of face K-1 during step K; face lp stays past the top (stage B forms
    // no face there), and the tape takes face K-2 too
    T v3q2 = T(0), v3q1 = T(0);
    T xmx[2] = {T(0), T(0)}, xmn[2] = {T(0), T(0)};
    T f3c = T(0);  // limited flux through the upper z-face of the last output plane

    // x of the first plane into LDS; the barrier also orders this item
    // after every LDS read of the previous one
    sx[0][pj + 1][pi + 1] = in_dom ? xq[1] : ld(own, Ks);
    if (t < NRING) sx[0][rsj][rsi] = ld(ring, Ks);
    // x of plane K+1 for the LDS: ring cell, and the own cell where it is
    // not in the queue (positions outside the domain); loaded a step ahead
    // (a null source keeps the zero)
    T xr = T(0), xown = T(0);
    const bool ring_on = t < NRING && ring.p, own_on = !in_dom && own.p;
    const uint32_t rstr = uint32_t(ring.stride) * uint32_t(sizeof(T)),
                   ostr = uint32_t(own.stride) * uint32_t(sizeof(T));
    const char* rp = ring_on ? (const char*)(ring.p + ring.base) + (uint64_t)rstr * (uint32_t)Ks : nullptr;
    const char* op = own_on ? (const char*)(own.p + own.base) + (uint64_t)ostr * (uint32_t)Ks : nullptr;
    auto ld_halo = [&](int k) __attribute__((always_inline)) {  // k >= 1
        rp += rstr; op += ostr;
        if (ring_on) xr = ldo((const T*)rp, 0);
        if (own_on) xown = ldo((const T*)op, 0);
    };
    if (Ks + 1 <= Alast) ld_halo(Ks + 1);
    __syncthreads();

    // The tile arrays from sv2 on lie beyond the 64 KiB that a ds
    // instruction's immediate offset reaches from the lane's position.  They
    // are addressed from two per-lane byte offsets made opaque here, so that
    // every access is one of them plus an immediate; otherwise the compiler
    // keeps one address register per array and ring slot through the loop.
    using LT = FusedLds<T, RX, RY>;
    constexpr int SZ = (int)sizeof(T), PLN = RY * RX * SZ;  // one plane of a tile array
    constexpr int MID = (int)offsetof(LT, sv2);
    constexpr int HI = (int)offsetof(LT, e_h) - RX * SZ;  // e arrays are read one row back
    uint32_t lmid = uint32_t(MID + t * SZ);
    uint32_t lsx = uint32_t(offsetof(LT, sx) + ((saj - 1) * SW + (sai - 1)) * SZ);
    asm volatile("" : "+v"(lmid), "+v"(lsx));
    char* const lds0 = reinterpret_cast<char*>(&L);
    // array `arr` at ring slot s, offset (db rows, da columns) from the lane
#define LMID(arr, s, db, da) \
    (*reinterpret_cast<T*>(lds0 + lmid + ((int)offsetof(LT, arr) - MID + (s) * PLN + ((db) * RX + (da)) * SZ)))
// x of the plane in ring slot s, row db and column da of the 3x3 neighbourhood
// of the source column; for a position in the domain its own
#define LSX(s, db, da) \
    (*reinterpret_cast<T*>(lds0 + lsx + ((s) * (SW * SH) + (db) * SW + (da)) * SZ))
// the second offset, formed anew where a stage uses it (one add instead of a
// register through the loop)
#define LHI_BASE                           \
    uint32_t lhi = lmid + (HI - MID);      \
    asm volatile("" : "+v"(lhi));
#define LHI(arr, r) (*reinterpret_cast<T*>(lds0 + lhi + ((int)offsetof(LT, arr) - HI + (r) * SZ)))

    auto dif4 = [](T z0, T z1, T z2, T z3) { return (z3 + z2) - (z1 + z0); };
    // Pseudo-velocity of a face between x1 and x2 with advector a and h of
    // the two cells summed to h2: s1, s2 the sums of the cross advectors and
    // d1, d2 the cross differences of x (both times 4; one pair at the lids).
    // FAST: the powers of two folded, and every contraction written out, so
    // that all tilings round alike.
    auto vface = [](T x1, T x2, T a, T h2, T s1, T d1, auto... s2d2) __attribute__((always_inline)) {
        if constexpr (FAST) {
            T cr = s1 * d1;
            if constexpr (sizeof...(s2d2) == 2) {
                const T q2[2] = {s2d2...};
                cr = fma_(q2[0], q2[1], cr);
            }
            const T q = a * rcp_nr(h2);
            return fma_(q * cr, T(-0.0625), (x2 - x1) * fma_(-q, a, T(0.5) * T(fabs(a))));
        } else {
            const T hm = T(1) / (T(0.5) * h2);
            T cr = s1 * (d1 * T(0.25));
            if constexpr (sizeof...(s2d2) == 2) {
                const T q2[2] = {s2d2...};
                cr = cr + q2[0] * (q2[1] * T(0.25));
            }
            return vdyf(x1, x2, a, hm) - T(0.125) * a * hm * (cr);
        }
    };
    auto lflux = [](T v, T c_c, T n_m, T c_m, T n_c) {
        if constexpr (TAPE) return gflux(v, c_c, n_m, c_m, n_c);
        else return pp(v) * min2(c_c, n_m) - pn(v) * min2(c_m, n_c);  // capped in C
    };
    uint32_t so_k = so, fo_k = fo;
    // planes of the newest queue slots, and the planes' sizes in bytes
    const uint32_t SB8 = plane_bytes<T>(SXY), FB8 = plane_bytes<T>(FXY), YB8 = plane_bytes<T>(YXY);
    const T* qx = uniform(pl(x, SXY, kc(Ks + 1)));
    const T* qu1 = uniform(pl(u1, FXY, kc(Ks)));
    const T* qu2 = uniform(pl(u2, YXY, kc(Ks)));
    const T* qu3 = uniform(pl(u3, SXY, fc(Ks + 1)));
    const T* qh = uniform(pl(h, SXY, kc(Ks)));
    const T* qr = DENS ? nullptr : uniform(pl(rhr, SXY, kc(Ks)));
    const T* qxa = PASS == 2 ? uniform(pl(pio->xa, SXY, kc(Ks))) : nullptr;
    auto adv = [](auto* p, uint32_t d) {
        // uniform() also keeps it one pointer, not an induction per unrolled step
        return (decltype(p))((uintptr_t)uniform(p) + d);
    };
    T* qxo = uniform(pl(xo, SXY, Ks - 4));  // plane K-3 during step K
    T xst = T(0);                           // the new x of that plane
    const bool edge_d = do_d && (gi == 1 || gi == np || gj == 1 || gj == mp);
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
        // K opaque: every plane-dependent quantity is formed within the
        // step, rather than as one induction variable per unrolled step
        // held in registers through the loop
        asm volatile("" : "+s"(K));
        // queue slots: oldest, middle, newest of a three-plane queue; older,
        // newer of a two-plane one
        constexpr int Q3a = PH % 3, Q3b = (PH + 1) % 3, Q3c = (PH + 2) % 3;
        constexpr int Q2a = PH % 2, Q2b = (PH + 1) % 2;
        // LDS ring slots of plane K-d: mod 3 (R0, R1, R2 for d = 0, 1, 2) and
        // mod 2 (E0 for even d, E1 for odd d)
        constexpr int R0 = Q3a, R1 = Q3c, R2 = Q3b, E0 = Q2a, E1 = Q2b;
        T& xq1 = xq[Q3a]; T& xq2 = xq[Q3b]; T& xq3 = xq[Q3c];
        T& u1a0 = u1a[Q2a]; T& u1a1 = u1a[Q2b]; T& u1b0 = u1b[Q2a]; T& u1b1 = u1b[Q2b];
        T& u2a0 = u2a[Q2a]; T& u2a1 = u2a[Q2b]; T& u2b0 = u2b[Q2a]; T& u2b1 = u2b[Q2b];
        T& u3q0 = u3q[Q3a]; T& u3q1 = u3q[Q3b]; T& u3q2 = u3q[Q3c];
        T& hq1 = hq[Q2a]; T& hq2 = hq[Q2b];
        T& xmx0 = xmx[Q2a]; T& xmn0 = xmn[Q2a]; T& xmx1 = xmx[Q2b]; T& xmn1 = xmn[Q2b];
        // the column offsets are opaque to the optimiser at each plane, so
        // loads keep the saddr form (plane pointer + offset) instead of
        // becoming per-lane 64-bit pointer inductions
        asm volatile("" : "+v"(so_k), "+v"(fo_k));
        const uint32_t so = so_k, fo = fo_k;
        const bool A_on = K <= Alast;
        // Everything loaded for this step is needed now; waited for here, so
        // that the stores below are not waited for before the next step does
        // the same (loads and stores share one in-order counter: a store in
        // stage D, with the wait for the loads right after it, exposed its
        // whole latency on every plane).
        __builtin_amdgcn_s_waitcnt(0x0f70);  // vmcnt(0)
        // x of the last output plane, K-3, and the edge copies of x at level
        // n around plane K
        qxo = adv(qxo, SB8);
        if (do_d && K - 3 >= k0 && K - 3 <= k1) sto(qxo, so, xst);
        if constexpr (TAPE) {
            tx = xq2;
            store_tape(K);
        }
        if (edge_d && K >= k0 && K <= k1) {
            T* const xok = pl(xo, SXY, K);
            if (gi == 1) sto(xok - 1, so, xq2);
            if (gi == np) sto(xok + 1, so, xq2);
            if (gj == 1) sto(xok - o.sx, so, xq2);
            if (gj == mp) sto(xok + o.sx, so, xq2);
        }
        // plane K+1 into the LDS slot that stage A of plane K-1 read
        if (K + 1 <= Alast) {
            sx[E1][pj + 1][pi + 1] = in_dom ? xq3 : xown;
            if (t < NRING) sx[E1][rsj][rsi] = xr;
        }
        auto load_xr = [&](int K) __attribute__((always_inline)) {
            qx = adv(qx, K + 1 < lp ? SB8 : 0);
            if constexpr (!DENS) qr = adv(qr, K < lp ? SB8 : 0);
            if constexpr (PASS == 2) qxa = adv(qxa, K < lp ? SB8 : 0);
            xq1 = ldo(qx, so);
            if constexpr (!DENS) rq2 = ldo(qr, so);
            if constexpr (PASS == 2) xaq = ldo(qxa, so);
        };
        // Temporaries of a step that are read only under the condition
        // that sets them are left unset rather than zeroed: a default value
        // would cost a register move per step on every path.
        // neighbour-column inputs of V1/V2 on plane P=K-1.  Column
        // (gi-1, gj) is the source column of the lane to the left wherever
        // V1 is formed (gi >= 2 in the domain, so the left position is in
        // the domain too), and its queues hold h, u2 and u3 of plane P:
        // taken across lanes.  Column (gi, gj-1) is likewise the source
        // column of the position below wherever V2 is formed (gj >= 2): its
        // h, u1 and u3 go through LDS (written here, read in B).
        const int P = K - 1;
        const bool BC_on = P >= max(1, k0 - 1) && P <= min(lp, k1 + 1);
        const T hx = from_left_lane(hq1) + hq1;
        const T s2x = from_left_lane(u2a0 + u2b0) + u2b0 + u2a0;
        const T s3x = from_left_lane(u3q0 + u3q1) + u3q1 + u3q0;
        if (BC_on) {
            LHI_BASE
            LHI(e_h, 0) = hq1;  // element e = t
            if (!wall_e) LHI(e_u1, 0) = u1a0;
            if (last_e) LHI(e_u1, 1) = u1b0;
            LHI(e_u3a, 0) = u3q0;
            LHI(e_u3b, 0) = u3q1;
        }

        // ---- A: xant on plane K ------------------------------------------
        T xa_new;  // read under A_on, or in C where P < lp implies it
        // A and C are instantiated twice: for the ground and sky planes, and
        // for the interior planes, where the boundary cases compile away
        // (a uniform branch picks one; otherwise both sides of each
        // boundary case would be computed and selected on every plane)
        auto stage_a = [&](auto edge) __attribute__((always_inline)) {
            constexpr bool EDGE = decltype(edge)::value;
            const bool gnd = EDGE && K == 1, sky = EDGE && K == lp;
            T xc = xq2;
            // the source column's neighbours
            const T xw = LSX(E0, 1, 0), xe = LSX(E0, 1, 2), xs = LSX(E0, 0, 1), xn = LSX(E0, 2, 1);
            T hinv;
            if constexpr (PASS != 2 || FAST) hinv = rcp_<FAST>(hq2);
            if constexpr (PASS == 2) {
                xa_new = xaq;
            } else {
            T f1p = donor(xc, xe, u1b1);
            T f1 = donor(xw, xc, u1a1);
            T f2p = donor(xc, xn, u2b1);
            T f2 = donor(xs, xc, u2a1);
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
            if constexpr (DENS) xa_new = (xc - div_<FAST>(f1p - f1 + f2p - f2 + f3p - f3, hq2));
            else xa_new = rq2 * (xc - (f1p - f1 + f2p - f2 + f3p - f3) * hinv);
            }
            sxa[R0][pj][pi] = xa_new;
            if constexpr (TAPE)
                if (own_s && K >= k0 && K <= k1) sto(pl(tp->psi, SXY, K), tso, xa_new);
            // FAST: r*(xant/r - s/h) = xant - (r/h)*s, to rounding
            if constexpr (!DENS) {
                LHI_BASE
                LHI(rr, R0 * RY * RX) = FAST ? rq2 * hinv : rq2;
            }
            // bounds of x for the limiter on plane K: the 7-point stencil,
            // where out-of-domain neighbours are edge copies of the centre
            // (cp_last_to_halo_xy) and leave max/min unchanged
            T m = xc, n = xc;
            { const T v = nxm ? xw : xc; m = max2(m, v); n = min2(n, v); }
            { const T v = nxp ? xe : xc; m = max2(m, v); n = min2(n, v); }
            { const T v = nym ? xs : xc; m = max2(m, v); n = min2(n, v); }
            { const T v = nyp ? xn : xc; m = max2(m, v); n = min2(n, v); }
            if (!gnd) { m = max2(m, xq1); n = min2(n, xq1); }
            if (!sky) { m = max2(m, xq3); n = min2(n, xq3); }
            xmx1 = m;
            xmn1 = n;
        };
        if (A_on) {
            if (K == 1 || K == lp) stage_a(std::true_type{});
            else stage_a(std::false_type{});
        }
        // the ring of plane K+2, x of it and r of plane K+1: their registers are
        // free already, and the loads have a stage more to arrive in (fast
        // build, 512x512x256: 1.35 -> 1.27 ms; the exactly rounded build spills
        // with x and r here and loses 2 % on small domains)
        if (K + 2 <= Alast) ld_halo(K + 2);
        if constexpr (EARLY) load_xr(K);
        __syncthreads();
// xant of plane K-d at tile position (a, b)
#define XA(d, a, b) sxa[(d) == 0 ? R0 : ((d) == 1 ? R1 : R2)][(b) + 2][(a) + 2]
        const int Q = K - 2;
        const bool Dq = Q >= k0 && Q <= k1;
        // ---- limited fluxes through the left x-face and lower y-face of this
        //      position on plane Q: V and cp/cn of Q are from the previous
        //      step and are replaced below; stage D reads them for both faces
        //      a cell shares, so each face flux is formed once
        if (Dq) {
            const T c0 = LMID(scp, 0, 0, 0), n0 = LMID(scn, 0, 0, 0);
            LMID(sf1, 0, 0, 0) = lflux(sv1[pj][pi], c0, LMID(scn, 0, 0, -1), LMID(scp, 0, 0, -1), n0);
            LMID(sf2, 0, 0, 0) =
                lflux(LMID(sv2, 0, 0, 0), c0, LMID(scn, 0, -1, 0), LMID(scp, 0, -1, 0), n0);
        }
        // ---- B: V1/V2 on plane P=K-1, V3 on face K, the limiter's bounds on P
        // Straight-line on the interior planes: every lane forms every
        // quantity and the lanes that do not own it drop it (a select, or a
        // reader that does not look), so that the LDS reads of all of them
        // go out together instead of one exec region after the other.
        T v3n = T(0);
        T up, dn;  // (bound - xant) h on plane P, for C
#define SB __builtin_amdgcn_sched_barrier(0);
        auto stage_b = [&](auto edge) __attribute__((always_inline)) {
            constexpr bool EDGE = decltype(edge)::value;
            const bool gnd = EDGE && P == 1, sky = EDGE && P == lp;
            const T xc = XA(1, li, lj), xw = XA(1, li - 1, lj), xe = XA(1, li + 1, lj),
                    xs = XA(1, li, lj - 1), xn = XA(1, li, lj + 1);
            T kw, ks, ke, kn;  // plane K
            if (!EDGE || A_on) {
                kw = XA(0, li - 1, lj); ks = XA(0, li, lj - 1);
                ke = XA(0, li + 1, lj); kn = XA(0, li, lj + 1);
            }
            if (!EDGE || (A_on && K >= 2 && K >= k0 - 1)) {
                T s1 = u1a0 + u1a1 + u1b1 + u1b0;
                T s2 = u2a0 + u2b0 + u2b1 + u2a1;
                v3n = vface(xc, xa_new, u3q1, hq1 + hq2, s1, dif4(xw, kw, xe, ke), s2,
                            dif4(xs, ks, xn, kn));
            }
            SB
            if (!EDGE || BC_on) {
                const T xsw = XA(1, li - 1, lj - 1), xnw = XA(1, li - 1, lj + 1),
                        xse = XA(1, li + 1, lj - 1);
                const T bc = XA(2, li, lj);
                T val1, val2;
                if (!gnd && !sky)
                    val1 = vface(xw, xc, u1a0, hx, s2x, dif4(xsw, xs, xnw, xn), s3x,
                                 (xa_new + kw) - (bc + XA(2, li - 1, lj)));
                else
                    val1 = vface(xw, xc, u1a0, hx, s2x, dif4(xsw, xs, xnw, xn));
                SB
                {
                    // column (gi, gj-1): element e = t - RX
                    LHI_BASE
                    const T nv2_h = LHI(e_h, -RX), nv2_u1a = LHI(e_u1, -RX),
                            nv2_u1b = LHI(e_u1, -RX + 1), nv2_u3a = LHI(e_u3a, -RX),
                            nv2_u3b = LHI(e_u3b, -RX);
                    const T hy = nv2_h + hq1, s1 = nv2_u1a + u1a0 + u1b0 + nv2_u1b,
                            s3 = nv2_u3a + u3q0 + u3q1 + nv2_u3b;
                    if (!gnd && !sky)
                        val2 = vface(xs, xc, u2a0, hy, s1, dif4(xsw, xw, xse, xe), s3,
                                     (xa_new + ks) - (bc + XA(2, li, lj - 1)));
                    else
                        val2 = vface(xs, xc, u2a0, hy, s1, dif4(xsw, xw, xse, xe));
                }
                val1 = do_v1 ? val1 : T(0);
                val2 = do_v2 ? val2 : T(0);
                sv1[pj][pi] = val1;
                LMID(sv2, 0, 0, 0) = val2;
                if constexpr (TAPE) tv1 = val1, tv2 = val2;
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
        };
        if (BC_on && P != 1 && P != lp) stage_b(std::false_type{});
        else stage_b(std::true_type{});
        T hP;
        // The loaded source-column queues are not read after this point:
        // the oldest slot of each is loaded with the plane step K+1 needs;
        // the latency is covered by C, D and the next step's barrier.
        {
            // the oldest slot of each queue becomes the newest of step K+1;
            // the plane pointers move by one plane until they reach the last
            // (kept in scalar registers: formed anew from K they cost twice
            // the scalar instructions)
            const int Kn = K + 1;
            const uint32_t dS = Kn <= lp ? SB8 : 0, dF = Kn <= lp ? FB8 : 0, dY = Kn <= lp ? YB8 : 0;
            if constexpr (!EARLY) load_xr(K);
            qu1 = adv(qu1, dF); qu2 = adv(qu2, dY); qu3 = adv(qu3, dS); qh = adv(qh, dS);
            u1a0 = ldo(qu1, fo);
            u1b0 = ldo(qu1 + 1, fo);
            u2a0 = ldo(qu2, so);
            u2b0 = ldo(qu2 + o.yx, so);
            u3q0 = ldo(qu3, so);
            if constexpr (!FAST || DENS) hP = hq1;
            hq1 = ldo(qh, so);
        }
        __syncthreads();
        // ---- C: cp, cn on plane P ------------------------------------------
        // cp, cn of the own column on planes P (formed here) and P-1
        T cpP, cnP, cpQ, cnQ;
        auto stage_c = [&](auto edge) __attribute__((always_inline)) {
            constexpr bool EDGE = decltype(edge)::value;
            const bool gnd = EDGE && P == 1, sky = EDGE && P == lp;
            T rp, rn;
            {
                T a1p = sv1[pj][pi + 1], a1 = sv1[pj][pi];
                T a2p = LMID(sv2, 0, 1, 0), a2 = LMID(sv2, 0, 0, 0);
                T a3p, a3;
                if (gnd) { a3p = v3n; a3 = -a3p; }
                else if (sky) { a3 = v3q2; a3p = -a3; }
                else { a3p = v3n; a3 = v3q2; }
                rp = div_<FAST>(up,
                                (pn(a1p) + pp(a1) + pn(a2p) + pp(a2) + pn(a3p) + pp(a3) + ep));
                rn = div_<FAST>(dn,
                                (pp(a1p) + pn(a1) + pp(a2p) + pn(a2) + pp(a3p) + pn(a3) + ep));
            }
            // capped here: every reader takes min(1, .) (the tape holds them
            // as they are)
            if constexpr (!TAPE) {
                rp = min2(T(1), rp);
                rn = min2(T(1), rn);
            }
            cpQ = LMID(scp, 0, 0, 0);
            cnQ = LMID(scn, 0, 0, 0);
            LMID(scp, 0, 0, 0) = cpP = do_c ? rp : T(0);
            LMID(scn, 0, 0, 0) = cnP = do_c ? rn : T(0);
        };
        // limited flux through the upper z-face of plane Q; the first output
        // plane's lower one is formed on the step before its own
        T F3p;
        if (BC_on) {
            if (P == 1 || P == lp) stage_c(std::true_type{});
            else stage_c(std::false_type{});
            F3p = lflux(v3q2, cpP, cnQ, cpQ, cnP);
        } else if constexpr (TAPE) {
            cpQ = LMID(scp, 0, 0, 0);
            cnQ = LMID(scn, 0, 0, 0);
        }
        // ---- D: the new x on plane Q=K-2 -----------------------------------
        const bool gnd = Q == 1, sky = Q == lp;
        T F3 = f3c;
        // the lid's flux is that of the face next to it, reversed
        if (sky) F3p = T(0) - f3c;
        if (gnd) F3 = T(0) - F3p;
        f3c = F3p;
        LHI_BASE
        if (Dq) {
            const T F1 = LMID(sf1, 0, 0, 0), F1p = LMID(sf1, 0, 0, 1);
            const T F2 = LMID(sf2, 0, 0, 0), F2p = LMID(sf2, 0, 1, 0);
            T hQ;
            if constexpr (!FAST || DENS) hQ = LHI(hh, 0);
            if constexpr (DENS) {
                const T xnew = (XA(2, li, lj) - div_<FAST>(F1p - F1 + F2p - F2 + F3p - F3, hQ));
                xst = xnew;
                const T xi = xnew * hQ;
                if (do_d) {
                T* const xincq = pl(dio->xinc, SXY, Q);
                const T rho_n = ldo(xincq, so);
                sto(xincq, so, xi);
                sto(pl(dio->pexr1, SXY, Q), so, xi * ldo(pl(dio->pexe, SXY, Q), so));
                sto(pl(dio->pexr2, SXY, Q), so, xi);
                sto(pl(dio->rhoadv, SXY, Q), so, rho_n);
                sto(pl(dio->rhr, SXY, Q), so, div_<FAST>(rho_n, xi));
                }
            } else {
                const T r = LHI(rr, R2 * RY * RX);
                const T sum = F1p - F1 + F2p - F2 + F3p - F3;
                if constexpr (FAST) xst = XA(2, li, lj) - r * sum;
                else xst = r * (div_<FAST>(XA(2, li, lj), r) - div_<FAST>(sum, hQ));
                if constexpr (PASS == 1) if (do_d) {
                    // the limited velocities through the low faces of the
                    // cell, and through the wall faces n+1 at the last cells
                    T* const q1 = pl(pio->ul1, FXY, Q);
                    T* const q2 = pl(pio->ul2, YXY, Q);
                    sto(q1, fo, F1);
                    sto(q2, so, F2);
                    sto(pl(pio->ul3, SXY, Q), so, F3);
                    if (gi == np) sto(q1 + 1, fo, F1p);
                    if (gj == mp) sto(q2 + o.yx, so, F2p);
                    if (sky) sto(pl(pio->ul3, SXY, Q + 1), so, F3p);
                }
                if constexpr (TAPE) {
                    // V3 on the lower face Q of the cell (face 1 = -face 2 on the ground)
                    // and, above the sky plane, on face lp+1 = -face lp
                    tv3 = gnd ? -v3q2 : v3q1;
                    tcp = cpQ;
                    tcn = cnQ;
                }
            }
            if constexpr (DENS) if (do_d) {
                // total mass fluxes through the low faces of the cell: the
                // upwind's donor fluxes of plane Q (x of level n, inflow
                // values at the walls) plus the limited fluxes; the wall
                // faces as (donor + inflow part) - outflow part.  These reach
                // the outputs, so the compare-and-select operators of the
                // reference are used (signed zeros as the reference's).
                const T* const xq = pl(x, SXY, Q);
                const T xc = ldo(xq, so);
                const T xl = gi == 1 ? bcx[(gj - 1) + mp * (Q - 1)] : ldo(xq - 1, so);
                const T xb = gj == 1 ? bcy[(gi - 1) + np * (Q - 1)] : ldo(xq - o.sx, so);
                const T* const u1q = pl(u1, FXY, Q);
                const T* const u2q = pl(u2, YXY, Q);
                const T f1ns = mpdata::donor(xl, xc, ldo(u1q, fo));
                const T f2ns = mpdata::donor(xb, xc, ldo(u2q, so));
                T f3ns;
                if (gnd) f3ns = -mpdata::donor(xc, ldo(pl(x, SXY, Q + 1), so), ldo(pl(u3, SXY, Q + 1), so));
                else f3ns = mpdata::donor(ldo(pl(x, SXY, Q - 1), so), xc, ldo(pl(u3, SXY, Q), so));
                sto(pl(dio->m1, FXY, Q), fo, f1ns + F1);
                sto(pl(dio->m2, YXY, Q), so, f2ns + F2);
                sto(pl(dio->m3, SXY, Q), so, f3ns + F3);
                if (gi == np) {
                    const T w = mpdata::donor(xc, bcx[(gj - 1) + mp * ((Q - 1) + lp)], ldo(u1q + 1, fo));
                    sto(pl(dio->m1, FXY, Q) + 1, fo, w + T(0));
                }
                if (gj == mp) {
                    const T w = mpdata::donor(xc, bcy[(gi - 1) + np * ((Q - 1) + lp)], ldo(u2q + o.yx, so));
                    sto(pl(dio->m2, YXY, Q) + o.yx, so, w + T(0));
                }
                if (sky) {
                    const T w = -f3ns;
                    sto(pl(dio->m3, SXY, Q + 1), so, w + F3p);
                }
            }
        }
#undef XA
        // ---- the computed queues move to plane K+1 by the slot rotation; V3
        //      of face K goes into the slot of face K-2 ------------------------
        if constexpr (!FAST || DENS) LHI(hh, 0) = hP;
        if constexpr (TAPE) v3q1 = v3q2;
        if (K <= lp) v3q2 = v3n;
    };
#undef LMID
#undef LHI
#undef LHI_BASE
#undef LSX
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

// Work of a persistent launch: which (tile, k-range) items each workgroup
// marches, one after the other.  While there are as many tiles left as
// workgroups, every workgroup takes a whole one (nfull of them each).  The
// tiles that remain are laid end to end, each as `ext` = lp + lead units, of
// which the first `lead` stand for the planes an item marches besides its
// output (two of xant and one of V/cp/cn recomputed below a cut, two above
// the item, and its set-up) and the others for its lp planes; this line is
// cut into equal runs, one a workgroup, so that all of them finish together
// whatever the numbers of tiles and planes.  Chunks of one length for all
// tiles, in rounds, left the last round part-empty: at 256x256x128 100 tiles
// x 2 chunks for 256 CUs, at 384x320x192 504 chunks of 64 planes.  Where they
// fit, and with the tuning override, `run` is such a chunk all the same: then
// lead is 0, ext the next multiple of it, and a workgroup may take several.
// Each XCD gets an equal share of the runs.
struct March {
    int nwg;            // workgroups that take items, a multiple of NXCD from NXCD on
    int ntx, ntile;
    int nfull;          // whole tiles per workgroup
    int run, lead, ext; // see above
    int grp;            // tiles that are cut together
    int share;          // runs of an XCD, neighbouring ones
};

// Calls item(tile, k0, k1) for this workgroup's items (one call site: the
// item is inlined once).  Workgroups are dealt to the XCDs round-robin
// (blockIdx % NXCD), each with its own L2: those of one XCD take neighbouring
// tiles, and in the whole-tile rounds they march them through the same planes.
template <typename F>
__device__ __forceinline__ void march_items(const March& m, int lp, F&& item) {
    const int nxcd = m.nwg >= NXCD ? NXCD : 1;
    const int per_xcd = m.nwg / nxcd;
    const int xcd = blockIdx.x % nxcd, slot = blockIdx.x / nxcd;
    const int ngrp = per_xcd / m.grp, in_grp = slot % m.grp;
    const int base = m.nwg * m.nfull;  // first of the tiles cut into runs
    const long long total = (long long)((m.ntile - base + m.grp - 1) / m.grp) * m.ext;
    // runs slot/grp, slot/grp + ngrp, ... of this XCD's share
    int i = slot / m.grp;
    long long pos = (long long)(xcd * m.share + i) * m.run, end = min(pos + m.run, total);
    if (i >= m.share) end = 0;
    for (int f = 0;;) {
        int tile, k0, k1;
        if (f < m.nfull) {
            tile = (xcd * m.nfull + f++) * per_xcd + slot;
            k0 = 1;
            k1 = lp;
        } else {
            if (pos >= end) {
                if ((i += ngrp) >= m.share) break;
                pos = (long long)(xcd * m.share + i) * m.run;
                end = min(pos + m.run, total);
                if (pos >= end) break;
            }
            const int tt = (int)(pos / m.ext);
            const long long t0 = (long long)tt * m.ext, stop = min(end, t0 + m.ext);
            tile = base + tt * m.grp + in_grp;
            k0 = max((int)(pos - t0) - m.lead, 0) + 1;
            k1 = min((int)(stop - t0) - m.lead, lp);
            pos = stop;
            if (k1 < k0 || tile >= m.ntile) continue;
        }
        item(tile, k0, k1);
    }
}

// What marching alone costs a workgroup over marching beside its x
// neighbours, as a share of a plane's time (any value from 0.06 to 0.25 gives
// the same plans; without it 256x256x128 takes 252 us instead of 233).
constexpr double kAlone = 0.12;
constexpr int kLead = 4;  // as measured: 3 to 5 the same, 2 and 7 take 59^3 from 23.1 to 25.2 us
// By how much chunks have to be the better plan (below 1.07 the model is no
// longer right about which is: 1000x16x16 and 182x10x3 lose 2 to 11 % with
// chunks that it puts 1 to 5 % ahead).
constexpr double kChunks = 1.07;
// The plan for `slots` resident workgroups (chunk > 0: runs of that length) of
// least modelled time, which goes to *time: the planes the busiest workgroup
// marches, dearer the fewer neighbours share their halo columns in L2.  The
// tiles that remain after the whole-tile rounds are cut, in groups of any size,
// either into equal runs of the line of tiles or each into q equal chunks.  A
// run crosses from one tile into the next, so that its length can be anything,
// but pays the lead planes on top; a chunk does not, and a whole tile (q = 1)
// on open lids marches two planes less than that.  On shallow domains this
// decides: 57x872x6, standard, 219 tiles of 32x16 for 256 CUs: 39.2 us in
// equal runs, 25.7 with a whole tile each.
template <int RX, int RY>
March plan_march(const Geo& g, long long slots, int chunk, double* time = nullptr) {
    March m{};
    m.ntx = (g.np + RX - 5) / (RX - 4);
    m.ntile = m.ntx * ((g.mp + RY - 5) / (RY - 4));
    m.grp = 1;
    if (slots >= NXCD) slots = slots / NXCD * NXCD;
    if (chunk > 0) {
        m.run = std::min(chunk, g.lp);
        m.ext = (g.lp + m.run - 1) / m.run * m.run;
        const long long need = (long long)m.ntile * (m.ext / m.run);
        m.nwg = (int)std::min(slots, need);
        if (m.nwg > NXCD) m.nwg = (m.nwg + NXCD - 1) / NXCD * NXCD;
        m.share = (int)(m.nwg >= NXCD ? (need + NXCD - 1) / NXCD : need);
        return m;
    }
    const int nslots = (int)slots, lp = g.lp;
    m.nfull = m.ntile / nslots;
    const int rest = m.ntile - m.nfull * nslots;
    March best{};
    double best_time = 0;
    for (int grp = 1; grp <= 64; grp *= 2) {
        if (grp > 1 && (grp > rest || nslots % (NXCD * grp))) break;
        const int groups = (rest + grp - 1) / grp, ngrp = nslots / grp;
        m.grp = grp;
        for (int q = 0; q <= std::min(8, lp); q++) {  // q chunks a tile; 0: equal runs
            if (q == 1 && grp > 1) continue;  // whole tiles lie side by side in any case
            double t = m.nfull * (double)(lp + kLead);
            if (q == 0) {
                m.lead = kLead;
                m.ext = lp + kLead;
                m.run = (int)std::max(1LL, ((long long)groups * m.ext + ngrp - 1) / ngrp);
                t = (t + (rest ? m.run + kLead : 0)) * (1 + kAlone / grp);
            } else {
                m.lead = 0;
                m.run = (lp + q - 1) / q;
                m.ext = m.run * q;
                const int rounds = (groups * q + ngrp - 1) / ngrp;
                t += (double)rounds * (m.run + (q == 1 && !g.pz ? 2 : kLead));
                t *= kChunks * (1 + kAlone / (q == 1 ? std::max(rest, 1) : grp));
            }
            if (best.grp && t >= best_time) continue;
            best = m;
            best_time = t;
        }
    }
    m = best;
    const long long runs = ((long long)(rest + m.grp - 1) / m.grp * m.ext + m.run - 1) / m.run;
    long long nwg = slots;
    if (m.nfull == 0) {  // no more workgroups than runs, whole groups on every XCD
        const long long need = runs * m.grp, per = (long long)NXCD * m.grp;
        if (m.grp > 1 || need > NXCD) nwg = std::min(slots, (need + per - 1) / per * per);
        else nwg = need;
    }
    m.nwg = (int)nwg;
    m.share = (int)(nwg >= NXCD ? (runs + NXCD - 1) / NXCD : runs);
    if (time) *time = best_time;
    return m;
}

// Halo cells of x_out that the step does not define keep their x_in values:
// the z-halo planes and the x/y halo cells outside the edge copies (all x/y
// halo cells of a periodic direction, which the step leaves alone).  Cell q
// of the three halo slabs -> its offset, or -1 for an edge copy (written by
// the step itself).  32-bit: the arrays have below 2^31 elements.
__device__ __forceinline__ int untouched_halo_cell(const Geo& g, uint32_t q, uint32_t nz_slab,
                                                   uint32_t ny_slab) {
    const uint32_t ih = g.ih, nx = g.np + 2 * ih, ny = g.mp + 2 * ih;
    int i, j, k;
    bool copy = true;
    if (q < nz_slab) {
        const uint32_t layer = q / (nx * ny), r = q - layer * (nx * ny), row = r / nx;
        k = layer < ih ? 1 - (int)ih + (int)layer : g.lp + 1 + (int)(layer - ih);
        i = (int)(r - row * nx) + 1 - (int)ih;
        j = (int)row + 1 - (int)ih;
    } else if (q < nz_slab + ny_slab) {
        const uint32_t r = q - nz_slab, tt = r / nx, row = tt % (2 * ih);
        i = (int)(r - tt * nx) + 1 - (int)ih;
        k = (int)(tt / (2 * ih)) + 1;
        j = row < ih ? 1 - (int)ih + (int)row : g.mp + 1 + (int)(row - ih);
        copy = g.py || !((j == 0 || j == g.mp + 1) && i >= 1 && i <= g.np);
    } else {
        const uint32_t r = q - nz_slab - ny_slab, tt = r / (2 * ih), col = r - tt * (2 * ih);
        k = (int)(tt / (uint32_t)g.mp) + 1;
        j = (int)(tt - (uint32_t)(k - 1) * (uint32_t)g.mp) + 1;
        i = col < ih ? 1 - (int)ih + (int)col : g.np + 1 + (int)(col - ih);
        copy = g.px || !(i == 0 || i == g.np + 1);
    }
    return copy ? (int)off_raw<SCAL>(g, i, j, k) : -1;
}

// Block b of nb copies its share of them.  The step kernels are launched with
// a few blocks more than they have places for work items (halo_blocks), which
// do this and nothing else: they run on what the items leave idle, where a
// kernel of its own came after them (2.7 of 29.8 us at 59^3, 13 us of 1.66 ms
// at 512x512x256).
template <typename T>
__device__ __forceinline__ void copy_untouched_halo(const Geo& g, const T* __restrict__ x,
                                                    T* __restrict__ xo, uint32_t b, uint32_t nb) {
    const uint32_t ih = g.ih, nx = g.np + 2 * ih, ny = g.mp + 2 * ih;
    const uint32_t nz_slab = 2 * ih * nx * ny;        // k outside 1..lp
    const uint32_t ny_slab = 2 * ih * nx * g.lp;      // k in 1..lp, j outside 1..mp
    const uint32_t nx_slab = 2 * ih * g.mp * g.lp;    // k, j inside, i outside 1..np
    const uint32_t total = nz_slab + ny_slab + nx_slab;
    for (uint32_t q = b * blockDim.x + threadIdx.x; q < total; q += nb * blockDim.x) {
        const int c = untouched_halo_cell(g, q, nz_slab, ny_slab);
        if (c >= 0) xo[c] = x[c];
    }
}
inline long long halo_cells(const Geo& g) {
    const long long ih = g.ih, nx = g.np + 2 * ih, ny = g.mp + 2 * ih;
    return 2 * ih * (nx * ny + nx * g.lp + (long long)g.mp * g.lp);
}
// shares of four cells a thread for blocks of nt threads
inline long long halo_shares(long long cells, int nt) {
    return std::max(1LL, (cells + 4LL * nt - 1) / (4LL * nt));
}
// blocks of nt threads for `cells` halo cells: a share each, at most a quarter
// of the chip's CUs
inline int halo_blocks(long long cells, int nt) {
    return (int)std::min(64LL, halo_shares(cells, nt));
}

template <typename T, int RX, int RY, int MINB, bool FAST = false, int PASS = 0>
__global__ void __launch_bounds__(RX * RY, MINB)
k_fused_gauge2(Geo g, Off o, March m, const T* __restrict__ x, const T* __restrict__ u1,
               const T* __restrict__ u2, const T* __restrict__ u3, const T* __restrict__ rhr,
               const T* __restrict__ h, const T* __restrict__ bcx, const T* __restrict__ bcy,
               T* __restrict__ xo, PassIO<T> pio) {
    __shared__ FusedLds<T, RX, RY> L;
    if (blockIdx.x >= (unsigned)m.nwg) {
        copy_untouched_halo<T>(g, x, xo, blockIdx.x - m.nwg, gridDim.x - m.nwg);
        return;
    }
    march_items(m, g.lp, [&](int tile, int k0, int k1) {
        fused_item<T, RX, RY, false, FAST, PASS>(g, o, m.ntx, tile, k0, k1, x, u1, u2, u3, rhr, h,
                                                 bcx, bcy, xo, L, nullptr, &pio);
    });
}

// The two-pass step that also records the adjoint's tape (fused_item's
// TAPE), with the work-item order of k_fused_gauge2.
template <typename T, int RX, int RY, int MINB>
__global__ void __launch_bounds__(RX * RY, MINB)
k_fused_gauge_rec(Geo g, Off o, March m, const T* __restrict__ x, const T* __restrict__ u1,
                  const T* __restrict__ u2, const T* __restrict__ u3, const T* __restrict__ rhr,
                  const T* __restrict__ h, const T* __restrict__ bcx, const T* __restrict__ bcy,
                  T* __restrict__ xo, StdTape<T> tp) {
    __shared__ FusedLds<T, RX, RY> L;
    march_items(m, g.lp, [&](int tile, int k0, int k1) {
        fused_item<T, RX, RY, false, false, 0, true>(g, o, m.ntx, tile, k0, k1, x, u1, u2, u3, rhr,
                                                     h, bcx, bcy, xo, L, nullptr, nullptr, &tp);
    });
}

// Tile configuration (0 = 32x32 lanes at 4 waves per SIMD, the fastest at
// 512x512x256; 1-4 the alternatives in the switch below) and k-chunk
// length; MPDATA_FUSED_CFG / _CHUNK override them for tuning runs (-1: not
// set).
int fused_config() {
    const char* e = getenv("MPDATA_FUSED_CFG");
    return e ? atoi(e) : -1;
}
int fused_chunk_env() {
    const char* e = getenv("MPDATA_FUSED_CHUNK");
    const int c = e ? atoi(e) : -1;
    return c >= 1 ? c : -1;
}

// Workgroups of a batched launch.  The kernel deals workgroups to the
// NXCD XCDs round-robin and gives XCD x the items of its contiguous share
// (items_per_xcd of them), so the grid is a multiple of NXCD with no more
// workgroups per XCD than that share has items (a smaller share would
// leave slots idle while items of the XCD wait for a second round); fewer
// than NXCD items run without the split.
[[maybe_unused]] int persistent_grid(long long nitem, long long items_per_xcd, int ncu, int per_cu) {
    if (nitem < NXCD) return (int)std::max(1LL, nitem);
    const long long slots = (long long)ncu * std::max(per_cu, 1);
    const long long per_xcd = std::max(1LL, std::min(items_per_xcd, slots / NXCD));
    return (int)(per_xcd * NXCD);
}

template <int RX, int RY>
long long items_of(const Geo& g, int clen) {
    const long long ntx = (g.np + RX - 5) / (RX - 4), nty = (g.mp + RY - 5) / (RY - 4);
    return ntx * nty * ((g.lp + clen - 1) / clen);
}

// Workgroups of `kernel` that the device holds at once, at most `want` per CU
// (0: as many as fit).
template <typename K>
hipError_t resident(K kernel, int nt, int want, long long& slots) {
    int dev = 0, ncu = 0, per_cu = 0;
    hipError_t e = hipGetDevice(&dev);
    if (e == hipSuccess) e = hipDeviceGetAttribute(&ncu, hipDeviceAttributeMultiprocessorCount, dev);
    if (e == hipSuccess) e = hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, kernel, nt, 0);
    if (e != hipSuccess) return e;
    per_cu = std::max(per_cu, 1);
    if (want > 0) per_cu = std::min(per_cu, want);
    slots = (long long)std::max(ncu, 1) * per_cu;
    return e;
}

// How a step is tiled: the tile configuration, the workgroups per CU (0: as
// many as fit) and the k-chunk if it is prescribed (0: the runs of March).
struct Tiling {
    int cfg = 0, per_cu = 0, chunk = 0;
};

// Modelled time of a step on RX x RY tiles with per_cu workgroups on each of
// ncu CUs: the planes the busiest workgroup marches, times the time of a
// plane, which a CU's march of 1024 cells sets (4.1 us in FP64) until there
// are too few waves to hide the latency of the chain of a plane: 512 cells
// take no less than 0.69 of it (any value from 0.62 to 0.75 gives the same
// plans; 0.55 takes 190x147x83 standard from 113 to 130 us, 0.9 ten periodic
// steps of 64x64x32 from 235 to 313 us).
template <int RX, int RY>
double tiling_time(const Geo& g, int ncu, int per_cu) {
    double time = 0;
    plan_march<RX, RY>(g, (long long)ncu * per_cu, 0, &time);
    return time * std::max(0.69, RX * RY * per_cu / 1024.0);
}

// Tiling of a single-domain step, the one of least modelled time.  32x32
// tiles recompute the fewest ring cells (23 % of the lanes against 34 % with
// 32x16) but are one workgroup a CU and cut a domain more coarsely; 32x16
// tiles run two to a CU, or alone on it, where a domain is so small that
// halving the planes of each workgroup no longer pays for halving its speed.
template <typename T>
Tiling choose_tiling(const Geo& g) {
    Tiling tl;
    const int env_cfg = fused_config(), env_chunk = fused_chunk_env();
    if (env_chunk > 0) tl.chunk = env_chunk;
    if (env_cfg >= 0) {
        tl.cfg = env_cfg;
        return tl;
    }
    int dev = 0, ncu = 0;
    if (hipGetDevice(&dev) != hipSuccess ||
        hipDeviceGetAttribute(&ncu, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess ||
        ncu < 1)
        ncu = 256;
    const double t32 = tiling_time<32, 32>(g, ncu, 1), t16x2 = tiling_time<32, 16>(g, ncu, 2),
                 t16 = tiling_time<32, 16>(g, ncu, 1);
    if (t32 <= t16x2 && t32 <= t16) return tl;
    tl.cfg = 1;
    tl.per_cu = t16 < t16x2 ? 1 : 2;
    return tl;
}

// Persistent launch of the fixed-position kernel: as many workgroups as fit
// on the device at once, each looping over its items.
template <typename T, int RX, int RY, int MINB, bool FAST = false, int PASS = 0>
hipError_t launch2(const Geo& g, const Off& o, const Tiling& tl, const T* x, T* xout, const T* u1,
                   const T* u2, const T* u3, const T* rhr, const T* h, const T* bcx, const T* bcy,
                   hipStream_t s, const PassIO<T>& pio = PassIO<T>{}) {
    long long slots = 0;
    const hipError_t e =
        resident(k_fused_gauge2<T, RX, RY, MINB, FAST, PASS>, RX * RY, tl.per_cu, slots);
    if (e != hipSuccess) return e;
    const March m = plan_march<RX, RY>(g, slots, tl.chunk);
    // PASS 1 writes an intermediate, whose halo nothing reads
    const int hb = PASS == 1 ? 0 : halo_blocks(halo_cells(g), RX * RY);
    k_fused_gauge2<T, RX, RY, MINB, FAST, PASS><<<m.nwg + hb, RX * RY, 0, s>>>(
        g, o, m, x, u1, u2, u3, rhr, h, bcx, bcy, xout, pio);
    return hipGetLastError();
}

// Three iterations (upwind + two corrective passes) as two launches: the
// two-pass kernel writes its result to sc.x2 and its limited velocities to
// sc.ul, then the pass kernel advances x2 with them into xout, with the
// limiter bounds from x (time level n).  Tilings 32x32 and 32x16 lanes.
template <typename T, bool FAST>
hipError_t launch_three(const Geo& g, const Off& o, const Tiling& tl, const T* x, T* xout,
                        const T* u1, const T* u2, const T* u3, const T* rhr, const T* h,
                        const T* bcx, const T* bcy, const FusedScratch<T>& sc, hipStream_t s) {
    PassIO<T> p1{sc.ul[0], sc.ul[1], sc.ul[2], nullptr};
    PassIO<T> p2{nullptr, nullptr, nullptr, sc.x2};
    hipError_t e;
    if (tl.cfg == 0) {
        e = launch2<T, 32, 32, 4, FAST, 1>(g, o, tl, x, sc.x2, u1, u2, u3, rhr, h, bcx, bcy, s, p1);
        if (e == hipSuccess)
            e = launch2<T, 32, 32, 4, FAST, 2>(g, o, tl, x, xout, sc.ul[0], sc.ul[1], sc.ul[2],
                                               rhr, h, bcx, bcy, s, p2);
    } else {
        e = launch2<T, 32, 16, 4, FAST, 1>(g, o, tl, x, sc.x2, u1, u2, u3, rhr, h, bcx, bcy, s, p1);
        if (e == hipSuccess)
            e = launch2<T, 32, 16, 4, FAST, 2>(g, o, tl, x, xout, sc.ul[0], sc.ul[1], sc.ul[2],
                                               rhr, h, bcx, bcy, s, p2);
    }
    return e;
}

// The density mode of the fixed-position kernel (DensIO), with the work-item
// order of k_fused_gauge2.
template <typename T, int RX, int RY, int MINB, bool FAST = false>
__global__ void __launch_bounds__(RX * RY, MINB)
k_fused_dens(Geo g, Off o, March m, const T* __restrict__ x, const T* __restrict__ u1,
             const T* __restrict__ u2, const T* __restrict__ u3, const T* __restrict__ h,
             const T* __restrict__ bcx, const T* __restrict__ bcy, T* __restrict__ xo,
             DensIO<T> dio) {
    __shared__ FusedLds<T, RX, RY> L;
    march_items(m, g.lp, [&](int tile, int k0, int k1) {
        fused_item<T, RX, RY, true, FAST>(g, o, m.ntx, tile, k0, k1, x, u1, u2, u3, nullptr, h,
                                          bcx, bcy, xo, L, &dio);
    });
}

template <typename T, int RX, int RY, int MINB, bool FAST = false>
hipError_t launch_dens(const Geo& g, const Off& o, const Tiling& tl, const T* x, T* xout,
                       const T* u1, const T* u2, const T* u3, const T* h, const T* bcx,
                       const T* bcy, const DensIO<T>& d, hipStream_t s) {
    long long slots = 0;
    const hipError_t e = resident(k_fused_dens<T, RX, RY, MINB, FAST>, RX * RY, tl.per_cu, slots);
    if (e != hipSuccess) return e;
    const March m = plan_march<RX, RY>(g, slots, tl.chunk);
    k_fused_dens<T, RX, RY, MINB, FAST><<<m.nwg, RX * RY, 0, s>>>(g, o, m, x, u1, u2, u3, h, bcx,
                                                                  bcy, xout, d);
    return hipGetLastError();
}

// ---------------------------------------------------------------------------
// Batched step: many domains (ensemble members, tracers) of different shapes
// in one persistent launch.  The work items of all members form one list
// (member by member, each chunk-major over its tiles); the items of a
// contiguous run of that list go to the workgroups of one XCD.
// ---------------------------------------------------------------------------
template <typename T>
struct Member {  // device descriptor of one member
    Geo g;
    Off o;
    int ntx, ntile, clen, item0;
    int halo0;  // first of its shares of the halo copy
    const T *x, *u1, *u2, *u3, *rhr, *h, *bcx, *bcy;
    T* xo;
};

// Scheduling state of a batched step, after the member descriptors in the
// packed table: the run of the work-item list each XCD takes (items
// bnd[x] .. bnd[x+1]-1, split by modelled cost), and per XCD the counter
// from which its workgroups take their next item and the count of its
// workgroups that have finished.  The last workgroup of an XCD to finish
// resets both, so the next launch (or graph replay) starts from zero with
// no memset.
struct BatchSched {
    int bnd[NXCD + 1];
    int next[NXCD];
    int done[NXCD];
    int nhalo;  // shares of the members' halo copies
};
template <typename T>
size_t sched_offset(int n) {
    return (sizeof(Member<T>) * (size_t)n + 63) & ~size_t(63);
}

// Work items are taken dynamically within each XCD's run (items differ in
// cost: members have different depths, so chunks march different numbers
// of planes), in list order, so the workgroups of an XCD still march
// neighbouring tiles together.  The items left after the run's whole
// rounds (one item per workgroup of the XCD) are each split into up to four
// k-ranges, so that the last round occupies the workgroups; a k-range of a
// chunk gives the same planes as the whole chunk (8 fields of 256x256x128 on
// one grid: 2.02 -> 1.85 ms per step when it was introduced).  The
// single-domain kernels cut their tiles by March instead.
template <typename T, int RX, int RY, int MINB, bool FAST = false>
__global__ void __launch_bounds__(RX * RY, MINB)
k_fused_gauge2_batch(const Member<T>* __restrict__ mem, int nmem, int nitem, int shared,
                     BatchSched* __restrict__ sc, int nitemwg) {
    __shared__ FusedLds<T, RX, RY> L;
    __shared__ int s_w;
    if (blockIdx.x >= (unsigned)nitemwg) {
        // an equal run of the shares of all members' halos
        const int total = sc->nhalo, nb = gridDim.x - nitemwg, b = blockIdx.x - nitemwg;
        const int w1 = (int)((long long)total * (b + 1) / nb);
        int w = (int)((long long)total * b / nb);
        if (w >= w1) return;
        int q = 0;  // last member with halo0 <= w
        for (int hi = nmem - 1; q < hi;) {
            const int mid = (q + hi + 1) >> 1;
            if (mem[mid].halo0 <= w) q = mid;
            else hi = mid - 1;
        }
        for (; w < w1; q++) {
            const Member<T>& m = mem[q];
            const int end = q + 1 < nmem ? mem[q + 1].halo0 : total;
            for (const int h0 = m.halo0; w < min(w1, end); w++)
                copy_untouched_halo<T>(m.g, m.x, m.xo, w - h0, end - h0);
        }
        return;
    }
    const int nxcd = nitemwg >= NXCD ? NXCD : 1;
    const int per_xcd = nitemwg / nxcd;
    const int xcd = blockIdx.x % nxcd;
    if ((int)blockIdx.x >= per_xcd * nxcd) return;
    int w0, w1;  // this XCD's run
    if (nxcd == 1) {
        w0 = 0;
        w1 = nitem;
    } else if (shared) {
        // members on one grid: equal shares (the items of one (tile, chunk)
        // for all members are consecutive and cost the same)
        const int per = (nitem + NXCD - 1) / NXCD;
        w0 = min(nitem, xcd * per);
        w1 = min(nitem, w0 + per);
    } else {
        w0 = __builtin_amdgcn_readfirstlane(sc->bnd[xcd]);
        w1 = __builtin_amdgcn_readfirstlane(sc->bnd[xcd + 1]);
    }
    const int nrun = w1 - w0, full = nrun / per_xcd * per_xcd, rem = nrun - full;
    const int split = rem > 0 ? max(1, min(4, per_xcd / rem)) : 1;
    const int ntake = full + rem * split;
    for (;;) {
        if (threadIdx.x == 0) s_w = atomicAdd(&sc->next[xcd], 1);
        __syncthreads();
        const int i = __builtin_amdgcn_readfirstlane(s_w);
        __syncthreads();  // every thread has read s_w before thread 0 writes it again
        if (i >= ntake) break;
        int w = w0 + i, part = 0, nparts = 1;
        if (i >= full) {
            w = w0 + full + (i - full) / split;
            part = (i - full) % split;
            nparts = split;
        }
        int q, l;
        if (shared) {
            // members on one grid (fields sharing the velocity): the items
            // of one (tile, chunk) for all members are consecutive, so one
            // XCD marches them together and reads u, h, rhr once into its L2
            q = w % nmem;
            l = w / nmem;
        } else {
            int lo = 0, hi = nmem - 1;  // last member with item0 <= w
            while (lo < hi) {
                const int mid = (lo + hi + 1) >> 1;
                if (__builtin_amdgcn_readfirstlane(mem[mid].item0) <= w) lo = mid;
                else hi = mid - 1;
            }
            q = lo;
            l = w - __builtin_amdgcn_readfirstlane(mem[q].item0);
        }
        const Member<T> m = uniform(mem[q]);
        const int chunk = l / m.ntile, tile = l - chunk * m.ntile;
        const int c0 = 1 + chunk * m.clen, c1 = min(m.g.lp, c0 + m.clen - 1);
        const int len = c1 - c0 + 1;
        const int k0 = uniform(c0 + len * part / nparts),
                  k1 = uniform(c0 + len * (part + 1) / nparts - 1);
        if (k0 > k1) continue;  // a chunk shorter than the split (uniform: every thread)
        fused_item<T, RX, RY, false, FAST, 0, false, FAST && MINB >= 4>(
            m.g, m.o, m.ntx, uniform(tile), k0, k1, m.x, m.u1, m.u2, m.u3, m.rhr, m.h, m.bcx, m.bcy,
            m.xo, L);
    }
    if (threadIdx.x == 0 && atomicAdd(&sc->done[xcd], 1) == per_xcd - 1) {
        atomicExch(&sc->next[xcd], 0);
        atomicExch(&sc->done[xcd], 0);
    }
}

Off make_off(const Geo& g) {
    Off o;
    o.ih = g.ih;
    o.sx = g.np + 2 * g.ih;
    o.sxy = o.sx * (g.mp + 2 * g.ih);
    o.fx = g.np + 1 + 2 * g.ih;
    o.fxy = o.fx * (g.mp + 2 * g.ih);
    o.yx = g.np + 2 * g.ih;
    o.yxy = o.yx * (g.mp + 1 + 2 * g.ih);
    return o;
}

// The density step on the build FAST selects, with the tiling of the plain step.
template <typename T, bool FAST>
hipError_t dens_step(const Geo& g, const T* x, T* xout, const T* u1, const T* u2, const T* u3,
                     const T* h, const T* bcx, const T* bcy, const DensIO<T>& d, hipStream_t s) {
    const Off o = make_off(g);
    const Tiling tl = choose_tiling<T>(g);
    if (tl.cfg == 0)
        return launch_dens<T, 32, 32, 4, FAST>(g, o, tl, x, xout, u1, u2, u3, h, bcx, bcy, d, s);
    return launch_dens<T, 32, 16, 4, FAST>(g, o, tl, x, xout, u1, u2, u3, h, bcx, bcy, d, s);
}

template <int RX, int RY>
void tiles_of(const Geo& g, int& ntx, int& nty) {
    ntx = (g.np + RX - 5) / (RX - 4);
    nty = (g.mp + RY - 5) / (RY - 4);
}

template <typename T, int RX, int RY>
int pack_members(const BatchMember<T>* bm, int n, int clen, Member<T>* out) {
    long long item = 0, share = 0;
    for (int q = 0; q < n; q++) {
        Member<T>& m = out[q];
        m.g = bm[q].g;
        m.o = make_off(m.g);
        int ntx, nty;
        tiles_of<RX, RY>(m.g, ntx, nty);
        m.ntx = ntx;
        m.ntile = ntx * nty;
        m.clen = clen < m.g.lp ? clen : m.g.lp;
        m.item0 = (int)item;
        m.halo0 = (int)share;
        share += halo_shares(halo_cells(m.g), RX * RY);
        m.x = bm[q].x; m.u1 = bm[q].u1; m.u2 = bm[q].u2; m.u3 = bm[q].u3;
        m.rhr = bm[q].rhr; m.h = bm[q].h; m.bcx = bm[q].bcx; m.bcy = bm[q].bcy;
        m.xo = bm[q].xo;
        item += (long long)m.ntile * ((m.g.lp + m.clen - 1) / m.clen);
        if (item > (1ll << 30) || share > (1ll << 30)) return -1;
    }
    // XCD runs of equal modelled cost: an item marches its chunk's planes
    // plus the two recomputed below and above it (fewer at the lids)
    BatchSched* sc = reinterpret_cast<BatchSched*>(reinterpret_cast<char*>(out) +
                                                   sched_offset<T>(n));
    auto cost = [](const Member<T>& m, int chunk) -> long long {
        const int k0 = 1 + chunk * m.clen, k1 = std::min(m.g.lp, k0 + m.clen - 1);
        return (long long)(std::min(m.g.lp, k1 + 2) - std::max(1, k0 - 2) + 1);
    };
    long long total = 0;
    for (int q = 0; q < n; q++) {
        const Member<T>& m = out[q];
        for (int c = 0; c * m.clen < m.g.lp; c++) total += cost(m, c) * m.ntile;
    }
    long long cum = 0;
    int x = 1;
    sc->bnd[0] = 0;
    for (int q = 0; q < n && x < NXCD; q++) {
        const Member<T>& m = out[q];
        for (int c = 0; c * m.clen < m.g.lp && x < NXCD; c++) {
            const long long ci = cost(m, c);
            for (int t = 0; t < m.ntile && x < NXCD; t++) {
                cum += ci;
                while (x < NXCD && cum * NXCD >= total * x)
                    sc->bnd[x++] = m.item0 + c * m.ntile + t + 1;
            }
        }
    }
    for (; x <= NXCD; x++) sc->bnd[x] = (int)item;
    for (int d = 0; d < NXCD; d++) sc->next[d] = sc->done[d] = 0;
    sc->nhalo = (int)share;
    return (int)item;
}

// Tile configurations of the batched kernel: (id, RX, RY, waves per SIMD),
// shared by the exact and the fast build.
#define MPDATA_BATCH_CONFIGS(X) \
    X(0, 32, 16, 2)             \
    X(1, 32, 16, 4)             \
    X(2, 64, 16, 4)             \
    X(3, 16, 32, 2)             \
    X(4, 64, 8, 2)              \
    X(5, 32, 32, 4)

template <typename T, int RX, int RY, int MINB, bool FAST = false>
hipError_t launch_batch(const void* table, int n, int nitem, int shared, long long max_halo,
                        hipStream_t s) {
    int dev = 0, ncu = 0, per_cu = 0;
    hipError_t e = hipGetDevice(&dev);
    if (e == hipSuccess) e = hipDeviceGetAttribute(&ncu, hipDeviceAttributeMultiprocessorCount, dev);
    if (e == hipSuccess)
        e = hipOccupancyMaxActiveBlocksPerMultiprocessor(
            &per_cu, k_fused_gauge2_batch<T, RX, RY, MINB, FAST>, RX * RY, 0);
    if (e != hipSuccess) return e;
    const int grid = persistent_grid(nitem, ((long long)nitem + NXCD - 1) / NXCD, ncu, per_cu);
    BatchSched* sc = reinterpret_cast<BatchSched*>(
        reinterpret_cast<char*>(const_cast<void*>(table)) + sched_offset<T>(n));
    // Blocks for the halo shares (pack_members), at most one a CU.  (Every block
    // walking all members took 1000 members of 20x20x10 from 207 to 1190 us a
    // step: their halos were copied one after the other by the few blocks that
    // one halo fills.)
    const int hb = (int)std::min<long long>(std::max(ncu, 1), n * halo_shares(max_halo, RX * RY));
    k_fused_gauge2_batch<T, RX, RY, MINB, FAST><<<grid + hb, RX * RY, 0, s>>>(
        (const Member<T>*)table, n, nitem, shared, sc, grid);
    return hipGetLastError();
}

}  // namespace

}  // namespace mpdata
