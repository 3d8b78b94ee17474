// Host-side check of what the LDS-DMA hdiff tile reads
// (stencil_benchmarks_amd/csrc/hdiff_tile.h): over halos, extents and strides,
// every byte of every unit that hdiff_dma_unit lets the tile stage lies in the
// field, from its lowest to its highest halo point, and every launch's rows
// are whole tiles that 32-bit byte offsets cover.  Exits non-zero on the first
// unit or band that does not hold this.
#include <algorithm>
#include <cstdio>

#include "../stencil_benchmarks_amd/csrc/sb_internal.h"
#include "../stencil_benchmarks_amd/csrc/hdiff_tile.h"

static long fields[2];  // fields staged by words and by 16-byte units

template <typename T, int TY, int UNIT>
static int check_units(const sb_geom &g) {
    using Dma = sb::HdiffDma<T, double, TY, TY / 4, UNIT, false>;
    const int64_t size = int64_t(sizeof(T)), top_plane = g.sk > 0 ? g.nz - 1 + g.hk : -g.hk;
    const int64_t low_plane = g.sk > 0 ? -g.hk : g.nz - 1 + g.hk;
    const int64_t low = (low_plane * g.sk - g.hj * g.sj - g.hi) * size;
    const int64_t high =
        (top_plane * g.sk + (g.ny - 1 + g.hj) * g.sj + g.nx - 1 + g.hi + 1) * size;
    for (int64_t k = 0; k < g.nz; ++k)
        for (int32_t j0 = 0; j0 < g.ny; j0 += TY)
            for (int32_t i0 = 0; i0 < g.nx; i0 += 64) {
                const bool edge = i0 + 64 > g.nx || j0 + TY > g.ny;
                const int64_t rows = edge ? std::min<int64_t>(Dma::LH - 1, g.ny + 3 - j0) : Dma::LH - 1;
                const int64_t units =
                    edge ? std::min<int64_t>(Dma::WORDS - 1, Dma::last_unit(int32_t(g.nx), i0))
                         : Dma::WORDS - 1;
                for (int64_t row : {int64_t(0), rows}) {
                    const int64_t first = (k * g.sk + (j0 - 2 + row) * g.sj + i0 - Dma::LEFT) * size;
                    const int64_t end = first + (units + 1) * UNIT;
                    if (first < low || end > high) {
                        std::printf("%zu-byte field %lldx%lldx%lld halo (%lld, %lld, %lld) pitch %lld plane "
                                    "%lld: unit of %d bytes, row %lld, plane %lld reads [%lld, %lld) of "
                                    "[%lld, %lld)\n",
                                    sizeof(T), (long long)g.nx, (long long)g.ny, (long long)g.nz,
                                    (long long)g.hi, (long long)g.hj, (long long)g.hk, (long long)g.sj,
                                    (long long)g.sk, UNIT, (long long)(j0 - 2 + row), (long long)k,
                                    (long long)first, (long long)end, (long long)low, (long long)high);
                        return 1;
                    }
                }
            }
    return 0;
}

template <typename T, int TY>
static int check_field(const sb_geom &g, uintptr_t origin) {
    const int unit = sb::hdiff_dma_unit(g, reinterpret_cast<const void *>(origin), sizeof(T));
    if (unit == 0) return 0;
    ++fields[unit == 16];
    return unit == 16 ? check_units<T, TY, 16>(g) : check_units<T, TY, 4>(g);
}

// Bands of planes around and beyond 4 GiB.
static int check_bands() {
    for (int64_t size : {4, 8})
        for (int64_t pitch : {int64_t(1) << 10, int64_t(123456), int64_t(1) << 20, (int64_t(1) << 24) - 8})
            for (int64_t rows : {int64_t(1), int64_t(240), int64_t(256), int64_t(272), (int64_t(1) << 32) / pitch - 4,
                                 (int64_t(1) << 32) / pitch - 3, (int64_t(1) << 32) / pitch, int64_t(9000000)}) {
                const int64_t sj = pitch / size;
                for (int64_t nx : {int64_t(1), int64_t(64), sj - 4}) {
                    const int64_t band = sb::hdiff_dma_band(nx, rows, sj, size_t(size));
                    const int64_t in_band = std::min(band, rows);
                    const int64_t last = (in_band + 1) * sj + nx + 4;  // row in_band + 1: the halo
                    if (band < 1 || (band < rows && band % 16 != 0) || last * size >= (int64_t(1) << 32)) {
                        std::printf("%lld-byte field, nx %lld, %lld rows of pitch %lld: bands of %lld rows\n",
                                    (long long)size, (long long)nx, (long long)rows, (long long)sj,
                                    (long long)band);
                        return 1;
                    }
                }
            }
    return 0;
}

// Non-temporal stores: rows of whole 64-byte lines, or up to 128 MB of results.
static int check_stores() {
    const struct { uintptr_t out; int64_t sj; double points; size_t size; bool stream; } cases[] = {
        {256, 520, 512.0 * 512 * 160, 8, true},     // padded rows
        {256, 518, 512.0 * 512 * 160, 8, false},    // rows end inside a line
        {264, 520, 512.0 * 512 * 160, 8, false},    // and start inside one
        {256, 528, 512.0 * 512 * 160, 4, true},     {256, 520, 512.0 * 512 * 160, 4, false},
        {256, 403, 397.0 * 411 * 137, 4, true},     {256, 403, 397.0 * 411 * 137, 8, false},
        {256, 134, 128.0 * 128 * 80, 8, true},      {4, 1, 1 << 25, 4, true},
        {4, 1, (1 << 25) + 1, 4, false},
    };
    for (const auto &c : cases)
        if (sb::hdiff_dma_stream(reinterpret_cast<const void *>(c.out), c.sj, c.points, c.size) != c.stream) {
            std::printf("stores of %g points of %zu bytes, pitch %lld, origin %zu: expected %d\n", c.points,
                        c.size, (long long)c.sj, size_t(c.out), int(c.stream));
            return 1;
        }
    return 0;
}

int main() {
    if (check_bands() || check_stores()) return 1;
    const int64_t widths[] = {1, 2, 3, 4, 5, 6, 7, 8, 61, 62, 63, 64, 65, 66, 67, 125, 126, 127, 128, 129, 131};
    const int64_t heights[] = {1, 7, 8, 9, 15, 16, 17, 33};
    for (int64_t nx : widths)
        for (int64_t ny : heights)
            for (int64_t nz : {1, 2})
                for (int64_t hi = 2; hi <= 6; ++hi)
                    for (int64_t hj = 2; hj <= 4; ++hj)
                        for (int64_t hk = 0; hk <= 1; ++hk)
                            for (int64_t pad : {1, 2, 4, 16})   // elements a row is rounded up to
                                for (int64_t gap : {0, 4})      // elements between planes
                                    for (int64_t sign : {1, -1})
                                        for (uintptr_t origin : {uintptr_t(4096), uintptr_t(4104)}) {
                                            const int64_t sj = (nx + 2 * hi + pad - 1) / pad * pad;
                                            const int64_t sk = sign * (sj * (ny + 2 * hj) + gap);
                                            const sb_geom g{nx, ny, nz, 1, sj, sk, hi, hj, hk};
                                            if (check_field<double, 8>(g, origin) ||
                                                check_field<double, 16>(g, origin) ||
                                                check_field<float, 8>(g, origin) ||
                                                check_field<float, 16>(g, origin))
                                                return 1;
                                        }
    std::printf("ok: %ld fields by words, %ld by 16-byte units\n", fields[0], fields[1]);
    return 0;
}
