// Variant 5 of the vertical-advection solver: one wave per column group,
// (c', d') of the highest levels in registers and of the rest in LDS.
//
// Why.  A wave that solves one 64-column group alone has no pipeline to fill
// or drain and needs no barrier, so a CU can hold as many groups as its
// registers and LDS have room for: (c', d') of one level are 1 KB of a group
// with FP64 arithmetic, a CU has 512 KB of registers beside its 160 KB of
// LDS, and at nz = 80 with NR = 64 register levels four waves (one per SIMD)
// share a CU, pos of every level kept too.  What bounds such a wave is its own instruction stream: the
// forward recurrence is one serial chain per column, alone on its SIMD.  So
// the loop is arranged for few instructions and a short chain:
//   - the register levels are the highest ones, nz-1-NR .. nz-2, so their
//     unrolled code always ends at the last level, and the levels below run
//     in blocks of PF levels after one partial block; no level needs a
//     select, a clamp or a dropped store;
//   - what a level does not take from the chain (b, c, d of the row) is
//     computed one level ahead, beside the division of the current level;
//   - the terms that repeat from level to level are taken over: a(k) =
//     -c(k-1), and the two products of corr(k) are -P(k-1) and P(k) with
//     P(k) = c(k) (stage(k+1) - stage(k)); negation and scaling by a power of
//     two commute with rounding, so the bits are those of vadv.hip's order;
//   - the reciprocal of the recurrence is column_recip below.
#pragma once

#include <algorithm>
#include <iterator>

#include "vadv_column.h"

namespace sb {
namespace {

// 1 / x, correctly rounded, for the recurrence.  FP64: hardware estimate, two
// Newton steps and the residual correction of Markstein's scheme, which is
// the division's own sequence without the operand scaling that only
// exponents near the ends of the range need; where any lane has such an x
// (also 0, infinity, NaN: extreme()), the wave divides instead.  The test is
// two integer instructions beside the chain and a branch that is not taken.
template <typename C>
struct Recip {
    __device__ __forceinline__ static C estimate(C x) { return C(1) / x; }
    __device__ __forceinline__ static bool extreme(C) { return false; }
};
template <>
struct Recip<double> {
    __device__ __forceinline__ static double estimate(double x) {
        double r = __builtin_amdgcn_rcp(x);
        r = __builtin_fma(__builtin_fma(-x, r, 1.0), r, r);
        r = __builtin_fma(__builtin_fma(-x, r, 1.0), r, r);
        return __builtin_fma(__builtin_fma(-x, r, 1.0), r, r);
    }
    // |x| outside [2^-500, 2^501)
    __device__ __forceinline__ static bool extreme(double x) {
        const uint32_t hi = uint32_t(__builtin_bit_cast(uint64_t, x) >> 32);
        return (hi << 1) - (523u << 21) >= (1001u << 21);
    }
};

// Empty asm that takes and returns its operands: what they are computed from
// is computed before this point (the compiler would sink a level's
// right-hand side, which nothing needs before the backward sweep, below
// hundreds of others and keep every input alive until then).
template <typename V>
__device__ __forceinline__ void settle(V &v) {
    __asm__ volatile("" : "+v"(v));
}

// Levels of loads in flight: 8 levels of six loads stay below the 63
// outstanding vector-memory instructions a wave can count.
constexpr int kRegPf = 8;

// Lanes that a row of nx columns takes in the column groups: rounded up to
// whole 128- or 64-byte chunks of a row where rows and fields are aligned to
// them and that idles at most one lane in nine, so that a group's loads and
// stores touch no line (half line) that another group touches; else nx.  A plane
// stride that is no whole chunk shifts that from level to level, and the padding
// still pays: 313x327x100 float32 storage 53 us with it, 57 without, 100x1024x137
// 99 and 108, FP64 161 and 168.
// Measured on MI355X, float32 storage with the non-temporal hint this allows:
// 500x524x137 196 -> 187 us, 313x327x100 64 -> 49 us, 100x1024x137 92 -> 73
// us; FP64 313x327x100 111 -> 98 us, 100x1024x137 168 -> 146 us.
struct ColumnRow {
    int64_t lanes;
    bool aligned;  // groups are made of whole aligned chunks
};
template <typename P>
inline ColumnRow padded_row(int64_t nx, int64_t si, int64_t sj, size_t itemsize, const P &pointers) {
    if (si != 1) return {nx, false};
    for (size_t bytes : {size_t(128), size_t(64)}) {
        const int64_t chunk = int64_t(bytes / itemsize);
        const int64_t row = (nx + chunk - 1) / chunk * chunk;
        bool fits = sj % chunk == 0 && row * 8 <= nx * 9;
        for (const void *p : pointers) fits = fits && reinterpret_cast<uintptr_t>(p) % bytes == 0;
        if (fits) return {row, true};
    }
    return {nx, false};
}

// Neighbouring items that one XCD takes in a row where every item is a
// workgroup (4, 32, 64 and 128 measured 0-4 % slower).
constexpr uint32_t kRegItemsPerXcd = 16;

// A field's buffer resource in four scalar registers of its own: resources
// that share their size and flag words are otherwise put together anew, three
// scalar moves before most loads.
__device__ __forceinline__ __amdgpu_buffer_rsrc_t own_rsrc(const void *p, uint32_t bytes) {
    int flags = kRsrcWord3;
    __asm__ volatile("" : "+s"(bytes), "+s"(flags));
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<void *>(p), short(0), int(bytes), flags);
}

// Highest columns the variant takes: 201 levels with FP64 arithmetic, 401
// with float32.
template <typename C>
constexpr int64_t reg_max_levels() { return sizeof(C) == 8 ? 201 : 401; }

// Register levels the kernels are built for, and the waves a SIMD holds of
// each: its registers are 512, and a level takes four (two with float32
// arithmetic) beside some 80 (FP64 fields) or 55 (float32 fields) of the
// prefetch ring and the recurrence.  With `pos` every level also keeps its
// pos, in registers or LDS as its (c', d'), so the backward sweep loads
// nothing: the second read of pos is a seventh of a column's traffic, and
// the sweep's loads are a fifth of its instructions.
struct RegLevels {
    int nr, waves_per_simd;
    bool pos;
};
template <typename T, typename C>
struct RegBuilds;
template <>
struct RegBuilds<double, double> {
    static constexpr RegLevels of[] = {{0, 3, false}, {24, 2, false}, {40, 2, false}, {64, 1, false}, {96, 1, false}, {16, 2, true}, {40, 1, true}, {64, 1, true}};
};
template <>
struct RegBuilds<float, double> {
    static constexpr RegLevels of[] = {{0, 4, false}, {24, 3, false}, {48, 2, false}, {112, 1, false}, {16, 3, true}, {40, 2, true}, {88, 1, true}};
};
template <>
struct RegBuilds<float, float> {
    static constexpr RegLevels of[] = {{0, 4, false}, {40, 3, false}, {80, 2, false}};
};

// LDS rows of one wave: levels 0 .. nz-2-NR.
__host__ __device__ constexpr int64_t reg_lds_rows(int64_t nz, int nr) { return nz - 1 - nr; }

// Waves per CU beyond which more of them gain less than keeping pos does: all
// that there are, or four where they run in many rounds (in a few rounds,
// fewer at a time can leave the last round nearly empty: 301x283x60 FP64, 1344
// waves, 47 us with eight a CU, 52 with four).
inline uint64_t reg_waves_needed(uint64_t items, uint64_t cus) {
    return items >= 12 * cus ? 4 : (items + cus - 1) / cus;
}

// A workgroup's LDS is allocated in whole granules of 1280 bytes: three of
// 54272 bytes (float32 arithmetic, nz = 187) would fit 160 KB by their sizes, but
// two are in flight (181x181x187 69 us, 48 at nz = 186).
constexpr size_t kLdsGranule = 1280;

// The build that holds most waves of nz levels on a CU, and how many; one that
// keeps pos where it holds as many or `need`.  Measured on MI355X (us, most
// waves / this choice): FP64 512x512x60 141 / 135, three components 409 / 386,
// 400x400x60 three components 268 / 251, 64x64x160 25.7 / 24.5; float32 storage
// 32x32x80 14.8 / 13.9, 128x128x80 15.7 / 14.8, 301x283x60 three components 65.5 /
// 63, 400x400x60 three components 124 / 128; 512x512x80 FP64, as many waves either
// way, 187 / 180.
struct RegShape {
    int build = 0, per_cu = 0;
    size_t lds_bytes = 0;
};

template <typename T, typename C>
RegShape reg_shape(int64_t nz, size_t lds, uint64_t need) {
    RegShape most, keeps;
    if (nz > reg_max_levels<C>()) return most;
    int build = 0;
    for (const RegLevels &levels : RegBuilds<T, C>::of) {
        const int64_t rows = reg_lds_rows(nz, levels.nr);
        const size_t bytes = size_t(std::max<int64_t>(rows, 0)) * 64 *
                             (sizeof(CD<C>) + (levels.pos ? sizeof(T) : 0));
        if (rows >= 1 && bytes <= lds) {
            const size_t taken = (bytes + kLdsGranule - 1) / kLdsGranule * kLdsGranule;
            const int per_cu = int(std::min<size_t>(4 * levels.waves_per_simd,
                                                    std::max<size_t>(lds / taken, 1)));
            RegShape &best = levels.pos ? keeps : most;
            if (per_cu > best.per_cu) best = RegShape{build, per_cu, bytes};
        }
        ++build;
    }
    return uint64_t(keeps.per_cu) >= std::min(uint64_t(most.per_cu), need) ? keeps : most;
}

// Whether variant 5 loads stage, tens and tensstage (each read once) with the
// non-temporal hint, which leaves L2 and the Infinity Cache to pos, read a
// second time by the backward sweep, and to wcon, shared with the neighbour
// columns (hints on those two as well measured up to 20 % slower than none).
// FP64 fields: always (512x512x160 437 -> 400 us, 256x256x80 54 -> 47 us).
// Float32 fields: where groups are whole chunks of aligned rows, or one
// component is larger than the Infinity Cache (512x512x160 239 -> 217 us,
// 313x327x100 59 -> 49 us): elsewhere neighbouring groups share a line that
// the hint drops too early (301x283x60 without row padding 30.6 -> 32.5 us,
// 500x500x40 all components 150 -> 171 us).
// Short columns, those without register levels, read pos again before it has
// left the caches, so the hint gains only where a call's fields are about as
// large as the Infinity Cache (600x600x12 FP64, 173 MB: 49 us plain, 45 with
// it); smaller fields lose what the cache holds of them from the call before
// (512x512x4 14.2 / 17.4, 600x600x8 float32 storage 14.6 / 18.1), larger ones
// 1 to 14 % (1024x1024x8 three components FP64 264 / 288, float32 123 / 140).
// `points` are the domain's, `field_bytes` include the halo.
template <typename T, typename C>
bool stream_hint(const RegShape &shape, bool aligned, int ncomp, double points,
                 uint64_t field_bytes) {
    if (RegBuilds<T, C>::of[shape.build].nr == 0) {
        const double mb = (4 * ncomp + 1) * points * double(sizeof(T)) / (1 << 20);
        return (sizeof(T) == 8 || aligned) && mb > 128.0 && mb <= 320.0;
    }
    if (sizeof(T) == 8 || aligned) return true;
    return ncomp == 1 && 5 * field_bytes > (uint64_t(256) << 20);
}

// Whether variant 5 is the default for the columns it takes.  Not for
//   - short FP64 columns, those without register levels, beyond what a device
//     holds at once: the single-wave pipeline (variant 3), which loads the next
//     group while the last one finishes, is up to 9 % faster there (450x450x12
//     26.4 us, 28.4 here; 1024x1024x4 three components 155 / 168) and never
//     much slower;
//   - tall columns of float32 arithmetic, whose levels beyond the 80 in
//     registers leave LDS for two waves or one a CU: variants 4 and 3 take nz
//     <= 320 with four waves a CU, or one with two groups in its pipeline.  One
//     wave a CU (us, here / they): 512x512x300 1071 / 529, 128x128x300 64 / 52,
//     but three components of few columns 100x90x300 121 / 149.  Two waves:
//     181x181x201 79 / 58, 512x512x201 396 / 368, 64x64x201 39 / 35, but
//     160x150x201 46 / 57 and three components of 301x283x201 402 / 428.
template <typename T, typename C>
bool reg_default(const RegShape &shape, int ncomp, uint64_t items, uint64_t cus) {
    const uint64_t at_once = uint64_t(shape.per_cu) * cus;
    if (sizeof(T) == 8 && RegBuilds<T, C>::of[shape.build].nr == 0) return items <= at_once;
    if (sizeof(C) == 8 || shape.per_cu > 2) return true;
    if (ncomp == 1) return shape.per_cu == 2 && items > cus && items <= at_once;
    return items <= (shape.per_cu == 2 ? 20 : 2) * cus;
}

// The same where i has no unit stride, so a lane's accesses are lines of their
// own: the lines of all waves in flight have to stay in L2 until their other
// points are used, by the next levels where those are contiguous
// (`levels_inner`), else by the rows beside.  Register columns hold several
// times the waves of the other solvers, so beyond some number of items the lines
// are fetched again and again.  They are the default
//   - up to 96 levels for the `few` column groups that four waves a CU hold, with
//     contiguous levels one item a CU (us, here / the others: 32x33x40 float32
//     15.1 / 15.2, 224x320x43 FP64 283 / 147, 333x293x16 float32 storage 145 / 66;
//     rows beside 301x336x94 float32 467 / 688, 448x717x89 float32 storage 3056 /
//     1435);
//   - above for two items a CU, with contiguous levels half of one (67x22x167
//     three components float32 51 / 131, 78x159x156 FP64 396 / 216; rows beside
//     64x274x134 float32 storage 155 / 216, 391x160x172 float32 992 / 614), but not
//     for one component of float32 arithmetic (`single_float`: 64x128x197 93 / 50).
inline bool reg_default_strided(int64_t nz, bool single_float, bool few, bool levels_inner,
                                uint64_t items, uint64_t cus) {
    if (nz > 96) return !single_float && items <= (levels_inner ? cus / 2 : 2 * cus);
    return few && (!levels_inner || items <= cus);
}

// `shape` with at most `waves` of them on a CU.
inline RegShape reg_limit(RegShape shape, int waves, size_t lds) {
    if (waves < shape.per_cu) {
        shape.per_cu = waves;
        shape.lds_bytes = std::max(shape.lds_bytes, lds / size_t(waves) / kLdsGranule * kLdsGranule);
    }
    return shape;
}

// The kinds of columns in a batch, and whether the subdomains with columns of one
// kind, `groups` together, go to the register columns rather than to the
// warp-specialised solver, whose workgroups take several groups one after the
// other.  One step of n subdomains, in us, register columns / that one:
//   float32 arithmetic, one wave a CU, 128x128x268: n = 6 411 / 498, 8 549 / 526, 10 686 / 550,
//   14 962 / 600
//   two, 128x128x230: n = 24 883 / 1000, 32 1169 / 1084, 40 1450 / 1545, 64 2332 / 2180; x190:
//   32 963 / 897, 48 1434 / 1345, 64 1914 / 1780
//   contiguous levels, FP64: 16 64x64x80 771 / 1125, 8 128x100x140 2440 / 1673, 8 200x200x12 772 / 514
//   rows beside, FP64: 8 200x180x40 1381 / 1557, 8 200x200x12 563 / 505, 6 300x300x80 5291 / 5031
enum BatchColumns { kBatchColumns, kBatchTall1, kBatchTall2, kBatchLevels, kBatchRows, kBatchColumnKinds };

inline BatchColumns batch_columns(int64_t si, int64_t sj, int64_t sk, bool float_arithmetic, int per_cu) {
    if (si != 1) return sk < si && sk < sj ? kBatchLevels : kBatchRows;
    if (!float_arithmetic || per_cu > 2) return kBatchColumns;
    return per_cu == 2 ? kBatchTall2 : kBatchTall1;
}

inline bool batch_reg_default(BatchColumns kind, uint64_t groups, uint64_t cus) {
    constexpr uint64_t kMost[kBatchColumnKinds] = {0, 7, 48, 4, 18};  // groups a CU
    return kind == kBatchColumns || groups <= kMost[kind] * cus;
}

template <typename T, typename C, int NR, int PF, int AUX, bool POS>
struct RegColumn {
    static_assert(NR == 0 || (NR % PF == 0 && NR >= 2 * PF), "register levels: whole prefetch blocks");

    // Row k of the system, apart from the recurrence, and what row k+1 takes
    // over from it.
    struct Row {
        C b, c, d;  // diagonal, upper off-diagonal and right-hand side
        C cp;       // c(k-1) = -a(k)
        C p, st;    // P(k) and stage(k+1)
    };

    __device__ __forceinline__ static Row row(const Level<T> &r, const Row &q) {
        const C dtr = C(3.0 / 20.0);
        const C st_n = C(r.st);
        const C c = C(0.125) * (C(r.wn) + C(r.w));
        const C p = c * (st_n - q.st);
        const C d = ((dtr * C(r.pos) + C(r.tens)) + C(r.ts)) + (-q.p - p);
        return Row{(dtr + q.c) - c, c, d, q.c, p, st_n};
    }

    // c'(k), d'(k) from row k and c'(k-1), d'(k-1); `next` is row k+1, formed
    // from the ring record `r` beside the division
    __device__ __forceinline__ static void recur(const Row &q, C &cc, C &dd, const Level<T> &r,
                                                 Row &next) {
        const C den = q.b + cc * q.cp;
        C rr = Recip<C>::estimate(den);
        C dn = q.d + dd * q.cp;
        next = row(r, q);
        settle(rr);
        settle(dn);
        settle(next.b);
        settle(next.d);
        settle(next.p);
        if (__builtin_expect(__builtin_amdgcn_ballot_w64(Recip<C>::extreme(den)) != 0, 0))
            rr = C(1) / den;
        cc = q.c * rr;
        dd = dn * rr;
    }
    __device__ __forceinline__ static void recur(const Row &q, C &cc, C &dd) {
        const C rr = C(1) / (q.b + cc * q.cp);
        const C dn = q.d + dd * q.cp;
        cc = q.c * rr;
        dd = dn * rr;
    }

    // `lds_raw`: this wave's LDS, level k < nz-1-NR of a lane's column at
    // lds[64 k], with POS followed by pos of the same levels.  Needs nz >= NR + 2.
    __device__ __forceinline__ static void solve(const Rsrc &R, int64_t wshift, const PipeArgs &a,
                                                 int64_t g, unsigned char *lds_raw) {
        const C dtr = C(3.0 / 20.0);
        const int nz = int(a.nz), kl = nz - 1;
        const int low = nz - 2 - NR;            // levels 1 .. low live in LDS beside level 0
        const int part = low % PF;              // of them in the partial block
        CD<C> *const lds = reinterpret_cast<CD<C> *>(lds_raw) + (threadIdx.x & 63);
        T *const lpos = reinterpret_cast<T *>(lds_raw + uint32_t(low + 1) * uint32_t(64 * sizeof(CD<C>))) +
                        (threadIdx.x & 63);
        const uint32_t skb = uint32_t(a.sk * int64_t(sizeof(T)));
        const GroupOff F = group_offsets<T>(a, g, wshift);
        auto at = [&](int k) { return F.row + uint32_t(k) * skb; };
        // pos, tens, tensstage at byte offset `so`; stage, wcon and its
        // neighbour one level above
        auto load = [&](uint32_t so, Level<T> &r) {
            const uint32_t sn = so + skb;
            r.pos = bload<T, 0>(R.pos, F.lane, so);
            r.tens = bload<T, AUX>(R.tens, F.lane, so);
            r.ts = bload<T, AUX>(R.ts, F.lane, so);
            r.st = bload<T, AUX>(R.stage, F.lane, sn);
            r.w = bload<T, 0>(R.w, F.lane, sn);
            r.wn = bload<T, 0>(R.w, F.lane_wn, sn);
            // the loads stay here: sunk to the level that uses them they would
            // be waited on at once
            __asm__ volatile("" ::: "memory");
        };
        // a level's offset, kept running: formed anew at each level, so that
        // no level's offset stays live from the forward to the backward sweep
        auto step_up = [&](uint32_t &so) {
            so += skb;
            __asm__ volatile("" : "+s"(so));
        };
        auto step_down = [&](uint32_t &so) {
            so -= skb;
            __asm__ volatile("" : "+s"(so));
        };

        // ---- first loads: level 0, then the ring ------------------------------
        Level<T> first, ring[PF];
        const T st0 = bload<T, AUX>(R.stage, F.lane, at(0));
        load(at(0), first);
        // slot p starts as level 1 + p of the partial block; slots past it take
        // their level of the first whole block at once
        const int top = max(kl - 1, 0);
#pragma unroll
        for (int p = 0; p < PF; ++p) load(at(min(1 + p + (p < part ? 0 : part), top)), ring[p]);
        T last_pos, last_tens, last_ts;
        auto load_last = [&] {
            last_pos = bload<T, 0>(R.pos, F.lane, at(kl));
            last_tens = bload<T, AUX>(R.tens, F.lane, at(kl));
            last_ts = bload<T, AUX>(R.ts, F.lane, at(kl));
        };
        if constexpr (NR == 0) load_last();

        // ---- level 0 ----------------------------------------------------------
        C cc, dd;
        Row q;
        {
            const C st_n = C(first.st);
            const C c = C(0.125) * (C(first.wn) + C(first.w));
            const C p = c * (st_n - C(st0));
            const C d = ((dtr * C(first.pos) + C(first.tens)) + C(first.ts)) - p;
            const C b = dtr - c;
            cc = c / b;
            dd = d / b;
            lds[0] = CD<C>{cc, dd};
            if constexpr (POS) lpos[0] = first.pos;
            q = Row{b, c, d, C(0), p, st_n};
        }
        // ---- partial block: levels 1 .. part ----------------------------------
#pragma unroll
        for (int p = 0; p < PF - 1; ++p) {
            if (p < part) {
                q = row(ring[p], q);
                recur(q, cc, dd);
                lds[int64_t(1 + p) * 64] = CD<C>{cc, dd};
                if constexpr (POS) lpos[int64_t(1 + p) * 64] = ring[p].pos;
            }
        }
        if (part) {
#pragma unroll
            for (int p = 0; p < PF - 1; ++p)
                if (p < part) load(at(min(1 + p + part, top)), ring[p]);
        }
        // ---- whole blocks in LDS: levels 1 + part .. low -----------------------
        Row done = q;  // the last row that has entered the chain
        q = row(ring[0], q);
        int k = 1 + part;
        uint32_t so = at(k + PF - 1);  // offset of the last level loaded
        for (; k <= low; k += PF) {
            CD<C> *out = lds + int64_t(k) * 64;
            T *pos_out = lpos + int64_t(k) * 64;
#pragma unroll
            for (int p = 0; p < PF; ++p) {
                Row n;
                recur(q, cc, dd, ring[(p + 1) % PF], n);
                if constexpr (POS) pos_out[p * 64] = ring[p].pos;
                step_up(so);
                load(NR >= PF ? so : min(so, at(top)), ring[p]);
                out[p * 64] = CD<C>{cc, dd};
                done = q;
                q = n;
            }
        }
        // ---- register levels: low + 1 .. nz-2 ----------------------------------
        C rc[NR > 0 ? NR : 1], rd[NR > 0 ? NR : 1];
        T pr[PF];  // pos of the levels below, for the backward sweep
        T rp[NR > 0 && POS ? NR : 1];
#pragma unroll
        for (int i = 0; i < NR; ++i) {
            if (i + 1 < NR) {
                Row n;
                recur(q, cc, dd, ring[(i + 1) % PF], n);
                done = q;
                q = n;
            } else {
                recur(q, cc, dd);
                done = q;
            }
            settle(cc);
            settle(dd);
            rc[i] = cc;
            rd[i] = dd;
            if (i + PF < NR) {
                if constexpr (POS) {
                    rp[i] = ring[i % PF].pos;
                    settle(rp[i]);
                }
                step_up(so);
                load(so, ring[i % PF]);
            } else if (i + PF == NR) {
                load_last();
            }
        }
        // ---- level nz-1 ---------------------------------------------------------
        uint32_t sp = at(kl - 1 - PF);  // offset of the last pos level loaded, plus one
        if constexpr (NR >= PF && !POS) {
#pragma unroll
            for (int p = PF - 1; p >= 0; --p) {
                pr[p] = bload<T, 0>(R.pos, F.lane, sp);
                step_down(sp);
            }
        }
        C x;
        {
            const C b = dtr + done.c;
            const C d = ((dtr * C(last_pos) + C(last_tens)) + C(last_ts)) - done.p;
            x = (d + dd * done.c) / (b + cc * done.c);
        }
        uint32_t st = at(kl);
        bstore<T>(R.ts, F.lane, st, T(dtr * (x - C(last_pos))));

        // ---- backward: register levels ------------------------------------------
#pragma unroll
        for (int i = NR - 1; i >= 0; --i) {
            T pos;
            if (i + PF >= NR) {
                pos = ring[i % PF].pos;  // still there from the forward sweep
            } else if constexpr (POS) {
                pos = rp[i];
            } else {
                pos = pr[i % PF];
                pr[i % PF] = bload<T, 0>(R.pos, F.lane, i >= PF ? sp : at(max(low + 1 + i - PF, 0)));
                if (i >= PF) step_down(sp);
            }
            step_down(st);
            x = rd[i] - rc[i] * x;
            bstore<T>(R.ts, F.lane, st, T(dtr * (x - C(pos))));
        }
        // ---- backward: whole blocks in LDS --------------------------------------
        T pp[PF];  // pos of the partial block's levels and of level 0
#pragma unroll
        for (int p = 0; p < PF; ++p)
            pp[p] = POS ? lpos[int64_t(min(p, part)) * 64] : bload<T, 0>(R.pos, F.lane, at(min(p, part)));
        if constexpr (NR == 0 && !POS) {
#pragma unroll
            for (int p = 0; p < PF; ++p)
                pr[p] = bload<T, 0>(R.pos, F.lane, at(max(low - PF + 1 + p, 0)));
        }
        for (k = low - PF + 1; k > part; k -= PF) {
            const CD<C> *in = lds + int64_t(k) * 64;
            const T *pos_in = lpos + int64_t(k) * 64;
            CD<C> cd[PF];
#pragma unroll
            for (int p = PF - 1; p >= 0; --p) {
                cd[p] = in[p * 64];
                if constexpr (POS) pr[p] = pos_in[p * 64];
            }
#pragma unroll
            for (int p = PF - 1; p >= 0; --p) {
                const T pos = pr[p];
                if constexpr (!POS) pr[p] = bload<T, 0>(R.pos, F.lane, at(max(k + p - PF, 0)));
                step_down(st);
                x = cd[p].d - cd[p].c * x;
                bstore<T>(R.ts, F.lane, st, T(dtr * (x - C(pos))));
            }
        }
        // ---- backward: levels part .. 0 ------------------------------------------
#pragma unroll
        for (int p = PF - 1; p >= 0; --p) {
            if (p <= part) {
                const CD<C> cd = lds[int64_t(p) * 64];
                x = cd.d - cd.c * x;
                bstore<T>(R.ts, F.lane, at(p), T(dtr * (x - C(pp[p]))));
            }
        }
    }
};

}  // namespace
}  // namespace sb
