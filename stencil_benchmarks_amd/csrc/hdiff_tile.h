// Horizontal diffusion tile worker shared by the plain kernel (hdiff.hip)
// and the batched persistent kernel (batch.hip).  See hdiff.hip for the
// arithmetic and the tile schedule.
#pragma once

#include "sb_internal.h"

namespace sb {
namespace {

// Pointer into device global memory.  The tile worker takes its fields as
// such, so its loads and stores compile to global (not flat) instructions
// whatever the caller's pointers were read from.
template <typename T>
using global_ptr = __attribute__((address_space(1))) T *;

template <typename T>
__device__ __forceinline__ global_ptr<T> as_global(T *p) {
    return (global_ptr<T>)p;
}

struct HdiffGeom {
    int64_t nx, ny, nz, si, sj, sk;
};

// Whether the tile worker's 32-bit plane offsets cover a field: positive i
// and j strides, and point (nx + 1, ny + 1) counted from (-2, -2) below
// 4 GiB.
inline bool hdiff_tile_fits(int64_t nx, int64_t ny, int64_t si, int64_t sj, size_t itemsize) {
    if (si <= 0 || sj <= 0) return false;
    const double span = (double(nx + 3) * double(si) + double(ny + 3) * double(sj)) * double(itemsize);
    return span < 4294967296.0;
}

// Byte offset of point (gi, gj) within a k-plane of field element type T.
template <typename T>
__device__ __forceinline__ uint32_t plane_offset_t(int64_t gi, int64_t gj, const HdiffGeom &a) {
    return uint32_t((gi * a.si + gj * a.sj) * int64_t(sizeof(T)));
}

// `base` advanced by a non-negative byte offset.
template <typename P>
__device__ __forceinline__ P at(P base, uint32_t byte_offset) {
    using B = __attribute__((address_space(1))) const char *;
    return (P)((B)base + byte_offset);
}

template <typename C>
__device__ __forceinline__ C limited(C flux, C gradient) {
    return flux * gradient > C(0) ? C(0) : flux;
}

// `v` of the lane to the left, `first` in lane 0 of the wave.
__device__ __forceinline__ double from_left_lane(double v, double first) {
    constexpr int kWaveShr1 = 0x138;
    const int lo = __builtin_amdgcn_update_dpp(__double2loint(first), __double2loint(v), kWaveShr1,
                                               0xf, 0xf, false);
    const int hi = __builtin_amdgcn_update_dpp(__double2hiint(first), __double2hiint(v), kWaveShr1,
                                               0xf, 0xf, false);
    return __hiloint2double(hi, lo);
}

template <bool NT, typename T>
__device__ __forceinline__ T ld_nt(global_ptr<const T> p) {
    if constexpr (NT)
        return __builtin_nontemporal_load(p);
    else
        return *p;
}

// The tile worker's default hook: nothing.
struct NoTileHook {
    __device__ void operator()() const {}
};

template <bool NT, typename T>
__device__ __forceinline__ void st_nt(global_ptr<T> p, T v) {
    if constexpr (NT)
        __builtin_nontemporal_store(v, p);
    else
        *p = v;
}

// Tile worker: the calling workgroup (64 x TY/RPT threads) computes the
// 64 x TY output tile at (i0, j0) for planes [k_begin, k_end).  Staging:
// each of the NW waves loads rows w, w+NW, ... of the tile's 64 main
// columns (one coalesced 64-element row segment per load), and threads
// 0..4*LH-1 load the four halo columns; out-of-range indices are clamped
// into the 2-point halo, so every load is in bounds and the clamped
// duplicates only feed outputs outside the domain, which are not stored.
// The loads for plane k+1 are issued into registers before plane k is
// computed and written to the other half of the double-buffered LDS tile
// afterwards.  FLAGS bit 0: non-temporal out stores; bit 1: non-temporal
// coeff loads (neither is re-read; inp is, by the neighbouring halos).
// `hook` runs once per call, in every thread, right after the first plane
// is staged (its loads have been waited on), before any barrier.
template <typename T, typename C, int TY, int RPT, int FLAGS>
struct HdiffTile {
    static constexpr int TX = 64;
    static constexpr int NW = TY / RPT;   // waves per workgroup
    static constexpr int LW = TX + 4;     // staged columns: tile i = -2 .. TX+1
    static constexpr int LH = TY + 4;     // staged rows:    tile j = -2 .. TY+1
    static constexpr int PW = TX + 2;     // published Laplacian columns: -1 .. TX
    static constexpr int MAIN = (LH + NW - 1) / NW;
    static constexpr int IN_ELEMS = 2 * LH * LW;  // double-buffered input tile
    static constexpr int LAP_ELEMS = TY * PW;

    // Laplacian, limited fluxes and update of the calling thread's RPT output
    // points (column tx, rows ty*RPT ..) from one staged plane `sin` (SW
    // elements of type S per row, rows -2 .. TY+1, columns from -LEFT on; each
    // read widened to the arithmetic type C, so a plane staged in the storage
    // type gives the same results as one staged in C).  Each thread
    // computes its column's Laplacian for rows -1..RPT in registers and
    // publishes the interior ones to s_lap for its i-neighbours; the
    // workgroup barrier inside separates those writes from the flux reads.
    // The caller must separate one call's s_lap reads from the next call's
    // writes by a barrier.  The same arithmetic as the plane loop of run(),
    // which keeps its own copy: calling this from there changes the register
    // allocation of the float32-storage kernel (126 -> 130 VGPRs, one wave
    // per SIMD fewer, 100 -> 110 us at 512x512x160).
    template <int SW = LW, int LEFT = 2, typename S>
    __device__ static void plane(const S *sin, C *s_lap, const C (&cf)[RPT], C (&res)[RPT], int tx,
                                 int ty, int tid) {
        // 4 c - sum: 4 c of a float32 value is exact in FP64, so the fused form
        // rounds once, as the two operations do
        auto laplacian = [](C c, C sum) {
            if constexpr (sizeof(S) == 4 && sizeof(C) == 8)
                return __builtin_fma(C(4), c, -sum);
            else
                return C(4) * c - sum;
        };
        const int col = tx + LEFT;      // staged column of this thread
        const int row0 = ty * RPT + 2;  // staged row of its first output
        C ic[RPT + 4], il[RPT + 2], ir[RPT + 2], lap[RPT + 2];
    #pragma unroll
        for (int q = 0; q < RPT + 4; ++q) ic[q] = C(sin[(row0 - 2 + q) * SW + col]);
    #pragma unroll
        for (int q = 0; q < RPT + 2; ++q) {
            il[q] = C(sin[(row0 - 1 + q) * SW + col - 1]);
            ir[q] = C(sin[(row0 - 1 + q) * SW + col + 1]);
        }
    #pragma unroll
        for (int q = 0; q < RPT + 2; ++q)
            lap[q] = laplacian(ic[q + 1], ((ir[q] + il[q]) + ic[q + 2]) + ic[q]);
    #pragma unroll
        for (int q = 0; q < RPT; ++q) s_lap[(ty * RPT + q) * PW + tx + 1] = lap[q + 1];
        // Widened float32 fields: the flux at a point's left edge is the
        // right edge of the lane before, so a wave shift of two instructions
        // replaces its six.  Only lane 0 has no such lane; wave 0 publishes
        // its flux, and wave 1 the Laplacian of the halo column on the right.
        // Instructions bound these tiles (397x411x137 51.7 -> 48.8 us); FP64
        // fields are bound by memory and lose by the longer way to the barrier
        // (none gained, the small hdiff and vadv steps up to 4 %).
        constexpr bool SHIFT = sizeof(S) == 4 && sizeof(C) == 8;
        static_assert(!SHIFT || NW >= 2, "two waves share the halo columns");
        auto column = [&](int rr, int c) {
            return laplacian(C(sin[rr * SW + c]),
                             ((C(sin[rr * SW + c + 1]) + C(sin[rr * SW + c - 1])) +
                              C(sin[(rr + 1) * SW + c])) +
                                 C(sin[(rr - 1) * SW + c]));
        };
        if constexpr (SHIFT) {
            if (ty < 2 && tx < TY) {
                const int r = tx, rr = r + 2;
                if (ty == 0)
                    s_lap[r * PW] = limited(column(rr, LEFT) - column(rr, LEFT - 1),
                                            C(sin[rr * SW + LEFT]) - C(sin[rr * SW + LEFT - 1]));
                else
                    s_lap[r * PW + TX + 1] = column(rr, TX + LEFT);
            }
        } else if (tid < 2 * TY) {
            // Laplacian of the tile's halo columns -1 and TX.
            const int side = tid / TY, r = tid - side * TY;
            s_lap[r * PW + (side ? TX + 1 : 0)] = column(r + 2, side ? TX + LEFT : LEFT - 1);
        }
        __syncthreads();
    #pragma unroll
        for (int q = 0; q < RPT; ++q) {
            const int r = ty * RPT + q;
            const C c0 = ic[q + 2];
            const C lc = lap[q + 1];
            const C flx = limited(s_lap[r * PW + tx + 2] - lc, ir[q + 1] - c0);
            C flx_m;
            if constexpr (SHIFT)
                flx_m = from_left_lane(flx, s_lap[r * PW]);
            else
                flx_m = limited(lc - s_lap[r * PW + tx], c0 - il[q + 1]);
            const C fly = limited(lap[q + 2] - lc, ic[q + 3] - c0);
            const C fly_m = limited(lc - lap[q], c0 - ic[q + 1]);
            res[q] = c0 - cf[q] * (((flx - flx_m) + fly) - fly_m);
        }
    }

    template <typename Hook = NoTileHook>
    __device__ static void run(global_ptr<const T> __restrict__ inp,
                               global_ptr<const T> __restrict__ coeff, global_ptr<T> __restrict__ out,
                               const HdiffGeom &a, int64_t i0, int64_t j0,
                               int64_t k_begin, int64_t k_end, C *s_in_base, C *s_lap,
                               Hook hook = Hook{}) {
        C(*s_in)[LH * LW] = reinterpret_cast<C(*)[LH * LW]>(s_in_base);
        // the wave index read as wave-uniform (every caller launches rows of
        // 64 threads): branches on it and row offsets derived from it are scalar
        const int tx = threadIdx.x, ty = __builtin_amdgcn_readfirstlane(threadIdx.y);
        const int tid = ty * TX + tx;
        // ---- per-thread staging offsets (plane-independent) -----------------
        // Byte offsets within a k-plane, 32-bit (a plane of a field below
        // 4 GiB), added to the plane's uniform base: the loads take the
        // scalar-base form with one VGPR of offset each.  Input offsets count
        // from point (-2, -2), the lowest halo point a tile reads, so none is
        // negative; coeff and out offsets count from (0, 0).
        uint32_t off_main[MAIN];
        int lds_main[MAIN];
    #pragma unroll
        for (int m = 0; m < MAIN; ++m) {
            const int r = ty + NW * m;
            const int rr = r < LH ? r : LH - 1;
            const int64_t gi = min(i0 + tx, a.nx + 1);
            const int64_t gj = min(j0 + rr - 2, a.ny + 1);
            off_main[m] = plane_offset_t<T>(gi + 2, gj + 2, a);
            lds_main[m] = r < LH ? rr * LW + tx + 2 : -1;
        }
        const bool has_halo = tid < 4 * LH;
        uint32_t off_halo = 0;
        int lds_halo = -1;
        if (has_halo) {
            const int r = tid >> 2, q = tid & 3;
            const int c = q < 2 ? q : TX + q;  // 0, 1, TX+2, TX+3
            const int64_t gi = min(i0 + c - 2, a.nx + 1);
            const int64_t gj = min(j0 + r - 2, a.ny + 1);
            off_halo = plane_offset_t<T>(gi + 2, gj + 2, a);
            lds_halo = r * LW + c;
        }
        const int64_t gi_out = i0 + tx;
        // coeff (clamped into the domain) and, where in range, out
        uint32_t off_point[RPT];
    #pragma unroll
        for (int q = 0; q < RPT; ++q) {
            const int64_t gi = min(gi_out, a.nx - 1);
            const int64_t gj = min(j0 + ty * RPT + q, a.ny - 1);
            off_point[q] = plane_offset_t<T>(gi, gj, a);
        }

        T pm[MAIN], ph = T(0), pc[RPT];
        auto issue = [&](int64_t k) {
            global_ptr<const T> in_k = inp + (k * a.sk - 2 * a.si - 2 * a.sj);
    #pragma unroll
            for (int m = 0; m < MAIN; ++m) pm[m] = *at(in_k, off_main[m]);
            if (has_halo) ph = *at(in_k, off_halo);
            global_ptr<const T> cf_k = coeff + k * a.sk;
    #pragma unroll
            for (int q = 0; q < RPT; ++q) pc[q] = ld_nt<(FLAGS & 2) != 0>(at(cf_k, off_point[q]));
        };
        auto commit = [&](int buf) {
    #pragma unroll
            for (int m = 0; m < MAIN; ++m)
                if (lds_main[m] >= 0) s_in[buf][lds_main[m]] = C(pm[m]);
            if (has_halo) s_in[buf][lds_halo] = C(ph);
        };

        if (k_begin >= k_end) {
            hook();
            return;
        }
        issue(k_begin);
        commit(0);
        hook();
        const int col = tx + 2;         // staged column of this thread
        const int row0 = ty * RPT + 2;  // staged row of its first output
        for (int64_t k = k_begin; k < k_end; ++k) {
            const int cur = int(k - k_begin) & 1;
            C cf[RPT];
    #pragma unroll
            for (int q = 0; q < RPT; ++q) cf[q] = C(pc[q]);
            __syncthreads();
            const bool more = k + 1 < k_end;
            if (more) issue(k + 1);

            const C *sin = s_in[cur];
            C ic[RPT + 4], il[RPT + 2], ir[RPT + 2], lap[RPT + 2];
    #pragma unroll
            for (int q = 0; q < RPT + 4; ++q) ic[q] = sin[(row0 - 2 + q) * LW + col];
    #pragma unroll
            for (int q = 0; q < RPT + 2; ++q) {
                il[q] = sin[(row0 - 1 + q) * LW + col - 1];
                ir[q] = sin[(row0 - 1 + q) * LW + col + 1];
            }
    #pragma unroll
            for (int q = 0; q < RPT + 2; ++q)
                lap[q] = C(4) * ic[q + 1] - (((ir[q] + il[q]) + ic[q + 2]) + ic[q]);
    #pragma unroll
            for (int q = 0; q < RPT; ++q) s_lap[(ty * RPT + q) * PW + tx + 1] = lap[q + 1];
            if (tid < 2 * TY) {
                // Laplacian of the tile's halo columns -1 and TX.
                const int side = tid / TY, r = tid - side * TY;
                const int c = side ? TX + 2 : 1;
                const int rr = r + 2;
                const C v = C(4) * sin[rr * LW + c] -
                            (((sin[rr * LW + c + 1] + sin[rr * LW + c - 1]) + sin[(rr + 1) * LW + c]) +
                             sin[(rr - 1) * LW + c]);
                s_lap[r * PW + (side ? TX + 1 : 0)] = v;
            }
            __syncthreads();

            C res[RPT];
    #pragma unroll
            for (int q = 0; q < RPT; ++q) {
                const int r = ty * RPT + q;
                const C c0 = ic[q + 2];
                const C lc = lap[q + 1];
                const C flx = limited(s_lap[r * PW + tx + 2] - lc, ir[q + 1] - c0);
                const C flx_m = limited(lc - s_lap[r * PW + tx], c0 - il[q + 1]);
                const C fly = limited(lap[q + 2] - lc, ic[q + 3] - c0);
                const C fly_m = limited(lc - lap[q], c0 - ic[q + 1]);
                res[q] = c0 - cf[q] * (((flx - flx_m) + fly) - fly_m);
            }
            if (gi_out < a.nx) {
                global_ptr<T> out_k = out + k * a.sk;
    #pragma unroll
                for (int q = 0; q < RPT; ++q) {
                    const int64_t gj = j0 + ty * RPT + q;
                    // in range, the clamped point offset is the point's own
                    if (gj < a.ny) st_nt<(FLAGS & 1) != 0>(at(out_k, off_point[q]), T(res[q]));
                }
            }
            if (more) commit(cur ^ 1);
        }
    }
};

// LDS-DMA tile worker, shared by the plain kernel's variant 2 (hdiff.hip) and
// the batched kernel (batch.hip): the calling workgroup (64 x TY/RPT threads)
// computes the 64 x TY output tile at (i0, j0) of plane k.  The staged tile
// is one contiguous LDS array counted from point (i0-LEFT, j0-2), LW elements
// a row; lane l of wave instruction n stages unit 64n + l of it.  A unit is a
// 16-byte chunk of a row (two doubles from column i0-2 on, four floats from
// column i0-4 on) for fields whose tile corners are 16-byte aligned, else a
// 4-byte word, which needs no alignment beyond the element's.  Float32 fields
// gain most from the wide units: FP64 arithmetic bounds the kernel by its
// instructions, and 64x16 tiles take 6 staging instructions instead of 22.
// With HINT the coeff loads are non-temporal (hdiff_dma_hint below), with
// STREAM the stores (hdiff_dma_stream below).
//
// A tile that reaches past the domain's last row or column (EDGE, a uniform
// branch) clamps its unit addresses to the last halo row and to the unit that
// holds column nx + 1, as the register-staged tile does: what is staged there
// only feeds outputs that are not stored.  A 16-byte unit may read more
// columns than the halo of 2: two on the left and up to three on the right of
// float32 fields, one on the right of 8-byte ones; hdiff_dma_unit says where the
// field holds them.
template <typename T, typename C, int TY, int RPT, int UNIT, bool HINT, bool STREAM = true>
struct HdiffDma {
    using Tile = HdiffTile<T, C, TY, RPT, 2>;
    static constexpr int LEFT = UNIT == 16 ? 16 / int(sizeof(T)) : 2;
    static constexpr int LW = Tile::TX + 2 * LEFT, LH = Tile::LH, NW = Tile::NW;
    static constexpr int WORDS = int(sizeof(T)) * LW / UNIT;  // units of a staged row
    static constexpr int UNITS = LH * WORDS;
    static constexpr int STEPS = (UNITS + 63) / 64;  // wave instructions that stage the tile
    static constexpr int TILE_ELEMS = STEPS * 64 * UNIT / int(sizeof(T));
    static_assert(int(sizeof(T)) * LW % UNIT == 0, "a unit must not straddle two rows");

    // Unit of a staged row that holds (the end of) column nx + 1, counted from
    // the first column staged by the tile at i0.
    __host__ __device__ static constexpr uint32_t last_unit(int32_t nx, int32_t i0) {
        return uint32_t(nx + 1 + LEFT - i0) * uint32_t(sizeof(T)) / uint32_t(UNIT) +
               (UNIT < int(sizeof(T)) ? 1u : 0u);
    }

    // `corner` points at the tile's first staged element; wave ty of the NW
    // issues instructions ty, ty + NW, ...
    template <bool EDGE>
    __device__ __forceinline__ static void stage(global_ptr<const T> corner, T *s_tile,
                                                 uint32_t last_row, uint32_t last_unit,
                                                 uint32_t pitch, int tx, int ty) {
        __builtin_assume(tx >= 0 && tx < 64 && ty >= 0 && ty < NW);
        using GP = __attribute__((address_space(1))) const void *;
        using LP = __attribute__((address_space(3))) void *;
    #pragma unroll
        for (int m = 0; m < (STEPS + NW - 1) / NW; ++m) {
            const int n = ty + NW * m;
            const int c = n * 64 + tx;
            if ((m + 1) * NW * 64 <= UNITS || c < UNITS) {
                uint32_t row = uint32_t(c) / WORDS;
                uint32_t unit = uint32_t(c) - __umul24(row, uint32_t(WORDS));
                if constexpr (EDGE) {
                    row = min(row, last_row);
                    unit = min(unit, last_unit);
                }
                const GP src = (GP)at(corner, __umul24(row, pitch) + unit * uint32_t(UNIT));
                LP dst = (LP)((char *)s_tile + n * 64 * UNIT);
                if constexpr (UNIT == 16)
                    __builtin_amdgcn_global_load_lds(src, dst, 16, 0, 0);
                else
                    __builtin_amdgcn_global_load_lds(src, dst, 4, 0, 0);
            }
        }
    }

    // A pointer kept in scalar registers, apart from the offset arithmetic
    // around it: the accesses then take the scalar-base form, one vector
    // register of offset each.
    template <typename P>
    __device__ __forceinline__ static P scalar(P p) {
        uint64_t v = (uint64_t)p;
        __asm__("" : "+s"(v));
        return (P)v;
    }

    // Offsets within a plane are 32-bit (hdiff_dma_band), on a plane's uniform
    // base.
    __device__ static void run(global_ptr<const T> inp, global_ptr<const T> coeff,
                               global_ptr<T> out, int32_t nx, int32_t ny, int32_t sj, int64_t sk,
                               int32_t i0, int32_t j0, int32_t k, T *s_tile, C *s_lap) {
        // the wave index read as wave-uniform: the branches on it and the row
        // offsets derived from it are scalar
        const int tx = threadIdx.x, ty = __builtin_amdgcn_readfirstlane(threadIdx.y);
        const int tid = ty * Tile::TX + tx;
        const bool edge = i0 + Tile::TX > nx || j0 + TY > ny;
        // row pitch below 2^24 bytes (checked on the host): a staged unit's byte
        // offset from the tile corner is one 24-bit multiply and an add
        const uint32_t pitch = uint32_t(sj) * uint32_t(sizeof(T));
        const int64_t plane = k * sk;
        const global_ptr<const T> corner = scalar(inp + plane + ((j0 - 2) * sj + (i0 - LEFT)));
        if (edge) {
            const uint32_t last_row = uint32_t(ny + 3 - j0);
            stage<true>(corner, s_tile, last_row, last_unit(nx, i0), pitch, tx, ty);
        } else {
            stage<false>(corner, s_tile, 0, 0, pitch, tx, ty);
        }
        const int row0 = j0 + ty * RPT;  // this wave's first output row
        const global_ptr<const T> cf_k = scalar(coeff + plane + i0);
        const global_ptr<T> out_k = scalar(out + plane + i0);
        // lanes past the domain re-read its last column, rows its last row
        const uint32_t lane = uint32_t(min(tx, nx - 1 - i0)) * uint32_t(sizeof(T));
        C cf[RPT];
    #pragma unroll
        for (int q = 0; q < RPT; ++q)
            cf[q] = C(ld_nt<HINT>(at(cf_k, uint32_t(min(row0 + q, ny - 1)) * pitch + lane)));
        __syncthreads();  // every wave's staging has landed
        C res[RPT];
        Tile::template plane<LW, LEFT>(s_tile, s_lap, cf, res, tx, ty, tid);
        if (tx < nx - i0) {
    #pragma unroll
            for (int q = 0; q < RPT; ++q)
                if (row0 + q < ny)
                    st_nt<STREAM>(at(out_k, uint32_t(row0 + q) * pitch + lane), T(res[q]));
        }
    }
};

// Whether coeff is loaded non-temporally: not where inp, coeff and out of a
// launch together are small enough to stay in the Infinity Cache until they
// are used again (200x200x80 FP64, 77 MB: 16.1 us with the hint, 13.7 without;
// 400x400x100 float32 storage, 192 MB: 36.8 / 41.1 us).
inline bool hdiff_dma_hint(double points, size_t itemsize) {
    return 3 * points * double(itemsize) > 96.0 * (1 << 20);
}

// Whether the results are stored non-temporally, which keeps the inputs in the
// Infinity Cache for the next launch that reads them: 512x512x160 FP64 174 -> 168
// us over three sets of fields in turn, 397x411x137 float32 storage 57 -> 49 us;
// a vadv launch that reads the result next loses nothing by it.  The price is
// paid by a launch on cold caches, which without the hint ends with up to
// 256 MB of its results still in them: 512x512x160 FP64 155 -> 166 us.
// Rows that start inside a 64-byte line are the exception in fields of more than
// 128 MB: tiles beside each other then share lines that the hint writes in two
// parts, 512x512x160 without padding FP64 173.6 us plain, 177.1 with the hint
// (float32 94.2 / 96.9), 1024x1024x80 333 / 345 and 175 / 186, 1000x700x40 117.5
// / 121.6; smaller ones still gain (397x411x137 float32 storage 55.7 -> 53.1,
// 300x300x120 FP64 51.0 -> 43.8).
inline bool hdiff_dma_stream(const void *out, int64_t sj, double points, size_t itemsize) {
    const bool lines = reinterpret_cast<uintptr_t>(out) % 64 == 0 && sj * int64_t(itemsize) % 64 == 0;
    return lines || points * double(itemsize) <= 128.0 * (1 << 20);
}

// Rows that one launch of the LDS-DMA tile takes: the tile addresses a plane by
// 32-bit byte offsets, so planes of 4 GiB and more go in bands of whole tiles.
// A row pitch below 16 MiB leaves bands of 240 rows and more.
inline int64_t hdiff_dma_band(int64_t nx, int64_t ny, int64_t sj, size_t itemsize) {
    if (hdiff_tile_fits(nx, ny, 1, sj, itemsize)) return ny;
    return (((int64_t(1) << 32) / int64_t(itemsize) - (nx + 4)) / sj - 4) / 16 * 16;
}

// Bytes of the unit that the LDS-DMA tile stages this field by, or 0 where it
// does not take it: unit i stride and a positive row pitch below 16 MiB; 16
// where the tile corners are 16-byte aligned (row and plane strides of whole
// chunks and an aligned interior origin) and the field holds the columns
// beyond the halo of 2 that come with the chunks: column nx + 2 with odd nx
// (8-byte fields, a halo of 3), or columns from -4 on up to the end of the
// chunk of column nx + 1, which is nx + 4 where that column opens a chunk and
// nx + 3 at most elsewhere (4-byte fields; past a row's own halo they are in
// the neighbouring rows or planes).
inline int hdiff_dma_unit(const sb_geom &g, const void *inp, size_t itemsize) {
    if (g.si != 1 || g.sj <= 0 || g.sj * int64_t(itemsize) >= (int64_t(1) << 24)) return 0;
    if (hdiff_dma_band(g.nx, g.ny, g.sj, itemsize) <= 0) return 0;  // rows far beyond the pitch
    const int64_t chunk = 16 / int64_t(itemsize);
    const bool aligned = g.sj % chunk == 0 && g.sk % chunk == 0 &&
                         reinterpret_cast<uintptr_t>(inp) % 16 == 0;
    const bool holds = itemsize == 8 ? g.nx % 2 == 0 || g.hi >= 3
                                     : g.hi >= (g.nx % 4 == 3 ? 5 : 4) || g.hj >= 3 || g.hk >= 1;
    return aligned && holds ? 16 : 4;
}

}  // namespace
}  // namespace sb
