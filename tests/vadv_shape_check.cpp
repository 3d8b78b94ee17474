// Host-side check of the launch rules of the register-column vadv
// (stencil_benchmarks_amd/csrc/vadv_regs.h, sb_internal.h).  Exits non-zero on
// the first rule that does not hold.
#include <array>
#include <cstdio>
#include <vector>

#include "../stencil_benchmarks_amd/csrc/sb_internal.h"
#include "../stencil_benchmarks_amd/csrc/vadv_regs.h"

// Every workgroup takes an item of its own, whatever the run length.
static int check_remap() {
    for (uint32_t xcds : {1u, 2u, 8u})
        for (uint32_t total : {1u, 7u, 8u, 9u, 64u, 127u, 128u, 129u, 256u, 1000u, 2500u, 2048u})
            for (uint32_t chunk : {1u, 3u, 16u, total / xcds, total}) {
                if (chunk == 0) continue;
                std::vector<char> seen(total, 0);
                for (uint32_t b = 0; b < total; ++b) {
                    const uint32_t n = sb::xcd_chunk_remap(b, total, xcds, chunk);
                    if (n >= total || seen[n]++) {
                        std::printf("workgroup %u of %u, %u XCDs, runs of %u: item %u\n", b, total, xcds,
                                    chunk, n);
                        return 1;
                    }
                }
            }
    return 0;
}

constexpr size_t kLds = 160 << 10;  // of a CU
constexpr uint64_t kCus = 256;

template <typename T, typename C>
static sb::RegShape shape_of(int64_t nz, uint64_t items) {
    return sb::reg_shape<T, C>(nz, kLds, sb::reg_waves_needed(items, kCus));
}

// Short columns: the default solver and the cache hint.
static int check_short_columns() {
    const struct { int64_t nz, nx, ny; int ncomp; bool own, hint; } fp64[] = {
        {4, 128, 128, 1, true, false},    {17, 313, 327, 1, true, false},  // all in flight
        {4, 512, 512, 1, false, false},   {17, 512, 512, 1, false, true},  // beyond it
        {4, 1024, 1024, 3, false, false}, {12, 1024, 1024, 3, false, false},
        {40, 512, 512, 1, true, true},    {80, 128, 128, 3, true, true},   // register levels
    };
    for (const auto &c : fp64) {
        const uint64_t items = uint64_t(c.nx * c.ny / 64 * c.ncomp);
        const sb::RegShape s = shape_of<double, double>(c.nz, items);
        const double points = double(c.nx * c.ny * c.nz);
        const uint64_t bytes = uint64_t(points) * 8;
        if (sb::reg_default<double, double>(s, c.ncomp, items, kCus) != c.own ||
            sb::stream_hint<double, double>(s, true, c.ncomp, points, bytes) != c.hint) {
            std::printf("FP64 %lldx%lldx%lld x%d: default %d, hint %d\n", (long long)c.nx, (long long)c.ny,
                        (long long)c.nz, c.ncomp, int(sb::reg_default<double, double>(s, c.ncomp, items, kCus)),
                        int(sb::stream_hint<double, double>(s, true, c.ncomp, points, bytes)));
            return 1;
        }
    }
    // float32 storage keeps the solver; the hint goes by the bytes and the rows
    for (int64_t nz : {8, 12, 60})
        for (bool aligned : {false, true}) {
            const sb::RegShape s = shape_of<float, double>(nz, 1024 * 1024 / 64);
            const double points = 1024.0 * 1024 * double(nz);
            const bool hint = sb::stream_hint<float, double>(s, aligned, 1, points, uint64_t(points) * 4);
            const bool expected = nz == 60 ? true : nz == 8 ? aligned : aligned && 5 * nz * 4 <= 320;
            if (!sb::reg_default<float, double>(s, 1, 1024 * 1024 / 64, kCus) || hint != expected) {
                std::printf("float32 storage nz %lld aligned %d: hint %d\n", (long long)nz, int(aligned), int(hint));
                return 1;
            }
        }
    return 0;
}

// Tall columns: the default solver of float32 arithmetic; FP64 arithmetic has
// no other one beyond the LDS and keeps this one up to there.
static int check_tall_columns() {
    const struct { int64_t nz, groups; int ncomp; bool own; } cases[] = {
        {160, 4096, 1, true},  {186, 4096, 3, true},                         // three waves a CU
        {201, 64, 1, false},   {201, 375, 1, true},   {201, 625, 1, false},  // two
        {201, 625, 3, true},   {201, 4096, 3, false},
        {300, 64, 1, false},   {300, 375, 1, false},  {300, 141, 3, true},   // one
        {300, 4096, 3, false},
    };
    for (const auto &c : cases) {
        const uint64_t items = uint64_t(c.groups * c.ncomp);
        const sb::RegShape s = shape_of<float, float>(c.nz, items);
        if (s.per_cu == 0 || sb::reg_default<float, float>(s, c.ncomp, items, kCus) != c.own) {
            std::printf("float32 nz %lld, %lld groups x%d: %d waves a CU, default %d\n", (long long)c.nz,
                        (long long)c.groups, c.ncomp, s.per_cu, int(!c.own));
            return 1;
        }
        const sb::RegShape d = shape_of<double, double>(std::min<int64_t>(c.nz, 201), items);
        const sb::RegShape m = shape_of<float, double>(std::min<int64_t>(c.nz, 201), items);
        if (!sb::reg_default<double, double>(d, c.ncomp, items, kCus) ||
            !sb::reg_default<float, double>(m, c.ncomp, items, kCus)) {
            std::printf("FP64 arithmetic, %lld groups x%d: not the default\n", (long long)c.groups, c.ncomp);
            return 1;
        }
    }
    return 0;
}

// Fields without unit i stride.
static int check_strided() {
    const struct { int64_t nz; bool single, few, levels; uint64_t items; bool own; } cases[] = {
        {96, true, true, true, 256, true},     {96, true, true, true, 257, false},
        {96, true, true, false, 3072, true},   {40, false, false, false, 513, false},
        {97, false, false, true, 128, true},   {97, false, false, true, 129, false},
        {97, false, false, false, 512, true},  {97, false, false, false, 513, false},
        {97, true, false, true, 1, false},     {200, true, false, false, 1, false},
    };
    for (const auto &c : cases)
        if (sb::reg_default_strided(c.nz, c.single, c.few, c.levels, c.items, kCus) != c.own) {
            std::printf("strided nz %lld: few %d, levels %d, %llu items\n", (long long)c.nz, int(c.few),
                        int(c.levels), (unsigned long long)c.items);
            return 1;
        }
    for (int64_t nz : {30, 90, 201})
        for (int waves : {1, 2, 3, 4}) {
            const sb::RegShape s = sb::reg_shape<double, double>(nz, kLds, 1);
            const sb::RegShape l = sb::reg_limit(s, waves, kLds);
            const size_t taken = (l.lds_bytes + 1279) / 1280 * 1280;
            if (l.build != s.build || l.lds_bytes < s.lds_bytes || l.per_cu > waves || l.per_cu < 1 ||
                size_t(l.per_cu) * taken > kLds || (waves < s.per_cu && size_t(waves + 1) * taken <= kLds)) {
                std::printf("limit of %d waves, nz %lld: %d of %zu bytes\n", waves, (long long)nz, l.per_cu,
                            l.lds_bytes);
                return 1;
            }
        }
    return 0;
}

// The same in a batch, whose subdomains count together.
static int check_batched_columns() {
    const struct { int64_t nz, groups; bool own; } cases[] = {
        {160, 100000, true}, {186, 100000, true},                                  // three waves a CU
        {201, 48 * 256, true}, {230, 20 * 256, true}, {230, 48 * 256 + 1, false},  // two
        {250, 7 * 256, true},  {250, 7 * 256 + 1, false},                          // one
        {300, 64, true},       {320, 4 * 4096, false},
    };
    for (const auto &c : cases) {
        const int per_cu = sb::reg_shape<float, float>(c.nz, kLds, 4).per_cu;
        const sb::BatchColumns kind = sb::batch_columns(1, 100, 10000, true, per_cu);
        if (per_cu == 0 || sb::batch_reg_default(kind, uint64_t(c.groups), kCus) != c.own) {
            std::printf("batch of float32 nz %lld, %lld groups: %d waves a CU\n", (long long)c.nz,
                        (long long)c.groups, per_cu);
            return 1;
        }
    }
    // i, j and k stride: unit i stride, contiguous levels, contiguous rows
    const struct { int64_t si, sj, sk; sb::BatchColumns kind; uint64_t most; } kinds[] = {
        {1, 100, 10000, sb::kBatchColumns, 1000000}, {10000, 100, 1, sb::kBatchLevels, 4 * 256},
        {100, 10000, 1, sb::kBatchLevels, 4 * 256},  {10000, 1, 100, sb::kBatchRows, 18 * 256},
        {100, 1, 10000, sb::kBatchRows, 18 * 256},
    };
    for (const auto &c : kinds) {
        const sb::BatchColumns kind = sb::batch_columns(c.si, c.sj, c.sk, false, 2);
        if (kind != c.kind || !sb::batch_reg_default(kind, c.most, kCus) ||
            (kind != sb::kBatchColumns && sb::batch_reg_default(kind, c.most + 1, kCus))) {
            std::printf("batch of strides %lld %lld %lld: kind %d\n", (long long)c.si, (long long)c.sj,
                        (long long)c.sk, int(kind));
            return 1;
        }
    }
    return 0;
}

// Every build is the choice for some columns, and the choices that the device
// tests name (tests/test_gpu_parity.py).
template <typename T, typename C>
static int check_builds(const char *name, std::initializer_list<std::array<int, 4>> named) {
    std::vector<char> seen(std::size(sb::RegBuilds<T, C>::of), 0);
    for (int64_t nz = 2; nz <= sb::reg_max_levels<C>(); ++nz)
        for (uint64_t need = 1; need <= 20; ++need) seen[size_t(sb::reg_shape<T, C>(nz, kLds, need).build)] = 1;
    for (size_t b = 0; b < seen.size(); ++b)
        if (!seen[b]) {
            std::printf("%s: the build of %d register levels is never chosen\n", name,
                        sb::RegBuilds<T, C>::of[b].nr);
            return 1;
        }
    for (const auto &[nz, items, nr, pos] : named) {
        const sb::RegLevels &of = sb::RegBuilds<T, C>::of[shape_of<T, C>(nz, uint64_t(items)).build];
        if (of.nr != nr || of.pos != bool(pos)) {
            std::printf("%s nz %d, %d items: build of %d register levels\n", name, nz, items, of.nr);
            return 1;
        }
    }
    return 0;
}

// The waves counted on a CU fit its LDS, which is allocated in granules of
// 1280 bytes, and its registers.
template <typename T, typename C>
static int check_waves(const char *name) {
    for (int64_t nz = 2; nz <= sb::reg_max_levels<C>(); ++nz)
        for (uint64_t need = 1; need <= 20; ++need) {
            const sb::RegShape s = sb::reg_shape<T, C>(nz, kLds, need);
            const sb::RegLevels &levels = sb::RegBuilds<T, C>::of[s.build];
            const size_t taken = (s.lds_bytes + 1279) / 1280 * 1280;
            if (s.per_cu < 1 || s.per_cu > 4 * levels.waves_per_simd ||
                size_t(s.per_cu) * taken > kLds || nz < levels.nr + 2) {
                std::printf("%s nz %lld: build %d, %d waves of %zu bytes\n", name, (long long)nz, s.build,
                            s.per_cu, s.lds_bytes);
                return 1;
            }
        }
    return 0;
}

int main() {
    if (check_waves<double, double>("FP64") || check_waves<float, double>("float32 storage") ||
        check_waves<float, float>("float32"))
        return 1;
    // 601 x 140 columns (1315 items) and 601 x 320 (3005)
    if (check_builds<double, double>("FP64", {{26, 1315, 16, 1}, {42, 1315, 24, 0}, {66, 1315, 40, 0},
                                              {98, 1315, 64, 0}, {115, 1315, 96, 0}, {30, 3005, 16, 1},
                                              {31, 3005, 24, 0}, {42, 3005, 24, 0}}) ||
        check_builds<float, double>("float32 storage", {{26, 1315, 16, 1}, {42, 1315, 40, 1},
                                                        {66, 1315, 48, 0}, {98, 1315, 88, 1},
                                                        {122, 1315, 112, 0}, {193, 1315, 112, 0},
                                                        {30, 3005, 24, 0}, {42, 3005, 24, 0}}) ||
        check_builds<float, float>("float32", {{42, 1315, 40, 0}, {98, 1315, 80, 0}}))
        return 1;
    if (check_remap() || check_short_columns() || check_tall_columns() || check_strided() ||
        check_batched_columns())
        return 1;
    std::printf("ok\n");
    return 0;
}
