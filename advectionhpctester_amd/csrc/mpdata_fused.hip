// The fused MPDATA step, exactly rounded: every operation of the reference in
// its order, rounded once (-ffp-contract=off, IEEE division), so the results
// are bit-identical to the per-stage kernels and the reference.  The kernel
// templates are in mpdata_fused_impl.hpp.
#include "mpdata_fused_impl.hpp"

namespace mpdata {

template <typename T>
bool Fused<T>::supports(const Geo& g, int variant, int iters, int nonos) {
    if (variant == 2) {
        // the standard kernel (mpdata_fused_std.hip): 2 iterations, limiter
        // on or off, any boundaries
        if (iters != 2 || (nonos != 0 && nonos != 1)) return false;
    } else {
        if (variant != 1 || (iters != 2 && iters != 3) || nonos != 1) return false;
        if (g.px || g.py || g.pz) return false;
    }
    // 32-bit element offsets inside the kernel, and 32-bit byte offsets
    // inside one plane of every array
    const long long biggest = len_of<FACEX>(g) > len_of<FACEY>(g) ? len_of<FACEX>(g) : len_of<FACEY>(g);
    const long long plane =
        std::max(nx_of<FACEX>(g) * ny_of<FACEX>(g), nx_of<FACEY>(g) * ny_of<FACEY>(g));
    return biggest < (1ll << 31) - 1 && len_of<FACEZ>(g) < (1ll << 31) - 1 &&
           plane * (long long)sizeof(T) < (1ll << 32);
}

template <typename T>
hipError_t FusedDens<T>::step(const Geo& g, const T* x, T* xout, const T* u1, const T* u2,
                              const T* u3, const T* h, const T* bcx, const T* bcy,
                              const DensIO<T>& d, hipStream_t s) {
    return dens_step<T, false>(g, x, xout, u1, u2, u3, h, bcx, bcy, d, s);
}

template <typename T>
const char* Fused<T>::scope() {
    return "the gauge variant with 2 or 3 iterations, the limiter on and open boundaries, "
           "and the standard variant with 2 iterations";
}

template <typename T>
hipError_t Fused<T>::step(const Geo& g, const T* x, T* xout, const T* u1, const T* u2,
                          const T* u3, const T* rhr, const T* h, const T* bcx, const T* bcy,
                          hipStream_t s, int iters, const FusedScratch<T>* sc) {
    const Off o = make_off(g);
    const Tiling tl = choose_tiling<T>(g);
    if (iters == 3) {
        if (!sc || !sc->x2 || !sc->ul[0] || !sc->ul[1] || !sc->ul[2]) return hipErrorInvalidValue;
        return launch_three<T, false>(g, o, tl, x, xout, u1, u2, u3, rhr, h, bcx, bcy, *sc, s);
    }
    switch (tl.cfg) {
        case 1: return launch2<T, 32, 16, 4>(g, o, tl, x, xout, u1, u2, u3, rhr, h, bcx, bcy, s);
        case 2: return launch2<T, 32, 16, 2>(g, o, tl, x, xout, u1, u2, u3, rhr, h, bcx, bcy, s);
        case 3: return launch2<T, 64, 16, 4>(g, o, tl, x, xout, u1, u2, u3, rhr, h, bcx, bcy, s);
        case 4: return launch2<T, 16, 32, 2>(g, o, tl, x, xout, u1, u2, u3, rhr, h, bcx, bcy, s);
        default: return launch2<T, 32, 32, 4>(g, o, tl, x, xout, u1, u2, u3, rhr, h, bcx, bcy, s);
    }
}

// 32x16 tiles at 2 waves per SIMD (158 VGPRs, no spill), one workgroup per
// CU, cut by the launch plan (March).  At 4 waves per SIMD it spills, and the
// adjoint's backward runs it beside the reverse kernels on another stream,
// where the lighter occupancy leaves them room (128x128x64, 50 steps, when the
// tape was added: forward + backward 16.3-16.5 against 16.7-16.9 ms).
template <typename T>
hipError_t Fused<T>::record(const Geo& g, const T* x, T* xout, const T* u1, const T* u2,
                            const T* u3, const T* rhr, const T* h, const T* bcx, const T* bcy,
                            const StdTape<T>& tp, hipStream_t s) {
    constexpr int RX = 32, RY = 16, MINB = 2;
    if (g.px || g.py || g.pz || g.ih != 1) return hipErrorInvalidValue;
    const Off o = make_off(g);
    long long slots = 0;
    const hipError_t e = resident(k_fused_gauge_rec<T, RX, RY, MINB>, RX * RY, 0, slots);
    if (e != hipSuccess) return e;
    const March m = plan_march<RX, RY>(g, slots, fused_chunk_env());
    // xout: the interior and the edge copies; the other halo cells are left
    // alone (the recorded step defines only the interior)
    k_fused_gauge_rec<T, RX, RY, MINB><<<m.nwg, RX * RY, 0, s>>>(g, o, m, x, u1, u2, u3, rhr, h,
                                                                  bcx, bcy, xout, tp);
    return hipGetLastError();
}

template struct Fused<double>;
template struct Fused<float>;
template struct FusedDens<double>;
template struct FusedDens<float>;

// ---- batched step ------------------------------------------------------------
// (tile configurations: MPDATA_BATCH_CONFIGS in mpdata_fused_impl.hpp)

template <typename T>
int FusedBatch<T>::nconfigs() {
    return 6;
}

template <typename T>
const char* FusedBatch<T>::config_name(int cfg) {
    switch (cfg) {
#define NAME(c, rx, ry, mb) \
    case c: return #rx "x" #ry " threads, " #mb " waves/SIMD";
        MPDATA_BATCH_CONFIGS(NAME)
#undef NAME
    }
    return "?";
}

template <typename T>
size_t FusedBatch<T>::table_bytes(int n) {
    return sched_offset<T>(n) + sizeof(BatchSched);
}

template <typename T>
int FusedBatch<T>::pack(const BatchMember<T>* m, int n, int cfg, int clen, void* table) {
    if (clen < 1) return -1;
    for (int q = 0; q < n; q++)
        if (!Fused<T>::supports(m[q].g, 1, 2, 1)) return -1;
    switch (cfg) {
#define PACK(c, rx, ry, mb) \
    case c: return pack_members<T, rx, ry>(m, n, clen, (Member<T>*)table);
        MPDATA_BATCH_CONFIGS(PACK)
#undef PACK
    }
    return -1;
}

template <typename T>
hipError_t FusedBatch<T>::step(const void* table, int n, int nitem, int cfg, long long max_halo,
                               hipStream_t s, int shared) {
    hipError_t e = hipErrorInvalidValue;
    switch (cfg) {
#define LAUNCH(c, rx, ry, mb) \
    case c: e = launch_batch<T, rx, ry, mb>(table, n, nitem, shared, max_halo, s); break;
        MPDATA_BATCH_CONFIGS(LAUNCH)
#undef LAUNCH
    }
    return e;
}

// Batch tiling for n members on one grid (configuration numbers of
// MPDATA_BATCH_CONFIGS): 32x32 tiles with chunks of 64 planes where they give
// every CU two items, else 32x16 tiles with the longest chunk of 64, 32 or 16
// planes that gives every workgroup slot two.  The batch takes its items
// dynamically, so March's equal runs do not apply to it.
template <typename T>
void FusedBatch<T>::choose_shared(const Geo& g, int n, int& cfg, int& clen) {
    int dev = 0, ncu = 0;
    if (hipGetDevice(&dev) != hipSuccess ||
        hipDeviceGetAttribute(&ncu, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess ||
        ncu < 1)
        ncu = 256;
    if (n * items_of<32, 32>(g, 64) >= 2LL * ncu) {
        cfg = 5;  // 32x32, 4 waves per SIMD
        clen = 64;
    } else {
        cfg = 1;  // 32x16, 4 waves per SIMD
        clen = 16;
        for (int c : {64, 32}) {
            if (n * items_of<32, 16>(g, c) >= 4LL * ncu) { clen = c; break; }
        }
    }
    if (clen > g.lp) clen = g.lp;
}

template struct FusedBatch<double>;
template struct FusedBatch<float>;

}  // namespace mpdata
