// Host side of the engine on the runtime of fake_hip.cpp: one check per name.
#include "fake_hip.h"

#include <cmath>
#include <cstdio>
#include <cstring>
#include <functional>
#include <vector>

#include "../../include/icempm.h"

namespace {

int g_failed = 0;

#define EXPECT(cond)                                                                        \
    do {                                                                                    \
        if (!(cond)) {                                                                      \
            std::printf("%s:%d: %s (last error: %s)\n", __FILE__, __LINE__, #cond, icempm_last_error()); \
            g_failed++;                                                                     \
        }                                                                                   \
    } while (0)

icempm_simparams params(int gx, int gy)
{
    icempm_simparams P;
    icempm_params_reset(&P);
    P.GridXTotal = gx;
    P.GridY = gy;
    P.GridHaloSize = 8;
    P.GridXDimension = 0.1 * gx;
    P.nPtsTotal = 100;
    P.ParticleVolume = 1e-3;
    icempm_params_derive(&P);
    return P;
}

icempm_partition *partition(const icempm_simparams &P, int capacity, int precision = ICEMPM_PRECISION_FP64, int device = 0)
{
    icempm_partition *p = nullptr;
    EXPECT(icempm_partition_create(device, 0, precision, &p) == ICEMPM_OK);
    EXPECT(icempm_partition_allocate(p, capacity, P.GridXTotal) == ICEMPM_OK);
    EXPECT(icempm_partition_update_constants(p, &P, sizeof P) == ICEMPM_OK);
    return p;
}

int launched(const char *name)
{
    int n = 0;
    for (auto &l : fake::state().launches) n += l.name.find(name) != std::string::npos;
    return n;
}

// A scene without points steps, also where the runtime cannot tell how many
// workgroups a compute unit holds: its tile table has no tiles.
void empty_scene()
{
    for (int occupancy : {2, 0}) {
        fake::state().occupancy = occupancy;
        const icempm_simparams P = params(64, 32);
        icempm_partition *p = partition(P, 100);
        std::vector<double> soa(16 * 100);
        EXPECT(icempm_partition_transfer_points_from_soa_to_device(p, soa.data(), 100, 0, 0) == ICEMPM_OK);
        EXPECT(icempm_partition_sort_points(p) == ICEMPM_OK);
        EXPECT(icempm_partition_step(p, 3, 0) == ICEMPM_OK);
        EXPECT(launched("k_tiles") > 0);
        for (auto &l : fake::state().launches) EXPECT(l.grid.x > 0);
        icempm_partition_destroy(p);
    }
}

// A table of more than 2^27 tiles (the smallest shape on a grid of 135M cells):
// no launch of 2^32 threads or more, which the runtime refuses, and of the
// table no more than flags and positions (8 bytes) for the places that cannot
// all hold one of the few points.
void huge_tile_table()
{
    const icempm_simparams P = params(16400, 8200);
    icempm_partition *p = partition(P, 100);
    fake::state().allocated.clear();
    EXPECT(icempm_partition_set_tile_shape(p, 1, 1, 1) == ICEMPM_OK);
    for (size_t bytes : fake::state().allocated) EXPECT(bytes < (9ull << 27));
    EXPECT(icempm_partition_sort_points(p) == ICEMPM_OK);
    EXPECT(launched("k_tile_count") == 1 && launched("k_tile_emit") == 1);
    for (auto &l : fake::state().launches) EXPECT((unsigned long long)l.grid.x * l.block.x < 1ull << 32);
    icempm_partition_destroy(p);
}

// A tile shape whose table gets no memory is refused, and the calls after it
// go on with the shape before it; without memory for any table the points are
// stepped in their own order, and sorted again once there is memory.
void no_memory_for_tiles()
{
    const icempm_simparams P = params(2000, 2000);
    icempm_partition *p = partition(P, 100);
    std::vector<double> soa(16 * 100);
    EXPECT(icempm_partition_transfer_points_from_soa_to_device(p, soa.data(), 100, 0, 100) == ICEMPM_OK);
    EXPECT(icempm_partition_set_tile_shape(p, 16, 16, 1) == ICEMPM_OK);
    EXPECT(icempm_partition_sort_points(p) == ICEMPM_OK);
    fake::state().malloc_limit = 24u << 20;   // a table of 1x1 cells takes 32 MB
    EXPECT(icempm_partition_set_tile_shape(p, 1, 1, 0) == ICEMPM_ERR_HIP);
    int tx = 0, ty = 0, margin = 0, spread = 0;
    EXPECT(icempm_partition_get_tile_config(p, &tx, &ty, &margin, &spread) == ICEMPM_OK);
    EXPECT(tx == 16 && ty == 16 && margin == 1);
    EXPECT(icempm_partition_step(p, 3, 0) == ICEMPM_OK && launched("k_tiles") == 4);
    fake::state().malloc_limit = 1;
    EXPECT(icempm_partition_set_tile_shape(p, 1, 1, 0) == ICEMPM_ERR_HIP);
    EXPECT(icempm_partition_step(p, 3, 0) == ICEMPM_OK && launched("k_tiles") == 4);
    EXPECT(icempm_partition_sort_points(p) == ICEMPM_ERR_HIP);
    EXPECT(icempm_partition_step(p, 3, 0) == ICEMPM_OK && launched("k_tiles") == 4);
    fake::state().malloc_limit = ~size_t(0);
    EXPECT(icempm_partition_sort_points(p) == ICEMPM_OK);
    EXPECT(icempm_partition_step(p, 3, 0) == ICEMPM_OK && launched("k_tiles") == 8);
    icempm_partition_destroy(p);
}

// The zero-fill kernel stores 16 bytes at a time: everything it clears is
// aligned to that, also behind tables of odd length (cells + 1 of each scene).
void fill_alignment()
{
    for (int gy : {32, 33}) {
        for (int gx : {64, 65, 67}) {
            const icempm_simparams P = params(gx, gy);
            icempm_partition *p = partition(P, 100);
            std::vector<double> soa(16 * 100);
            EXPECT(icempm_partition_transfer_points_from_soa_to_device(p, soa.data(), 100, 0, 100) == ICEMPM_OK);
            EXPECT(icempm_partition_sort_points(p) == ICEMPM_OK);
            EXPECT(icempm_partition_step(p, 2, ICEMPM_STEP_DIRECT_P2G) == ICEMPM_OK);
            EXPECT(icempm_partition_reset_indenter_force_accumulator(p) == ICEMPM_OK);
            icempm_partition_destroy(p);
        }
    }
    EXPECT(launched("k_fill_zero") > 0);
    for (auto &l : fake::state().launches) EXPECT((size_t)l.pointer % 16 == 0);
}

// The staging memory of the transfers is coherent by its own flags: the host
// reads a chunk that a kernel wrote after the chunk's event.
void coherent_staging()
{
    const icempm_simparams P = params(64, 32);
    icempm_partition *p = partition(P, 100);
    std::vector<double> soa(16 * 100);
    EXPECT(icempm_partition_transfer_points_from_soa_to_device(p, soa.data(), 100, 0, 100) == ICEMPM_OK);
    EXPECT(icempm_partition_transfer_from_device(p, soa.data(), 100, 0) == ICEMPM_OK);
    EXPECT(!fake::state().host_flags.empty());
    for (unsigned f : fake::state().host_flags) EXPECT(f & hipHostMallocCoherent);
    icempm_partition_destroy(p);
}

// One thread drives a partition on each of two devices: transfers of either
// work whichever device is current, and leave it as it is.
void two_devices()
{
    fake::state().n_devices = 2;
    const icempm_simparams P = params(64, 32);
    icempm_partition *a = partition(P, 100, ICEMPM_PRECISION_FP64, 0), *b = partition(P, 100, ICEMPM_PRECISION_FP64, 1);
    std::vector<double> soa(16 * 100);
    for (int current : {0, 1}) {
        for (icempm_partition *p : {a, b}) {
            fake::state().device = current;
            EXPECT(icempm_partition_transfer_points_from_soa_to_device(p, soa.data(), 100, 0, 100) == ICEMPM_OK);
            EXPECT(icempm_partition_transfer_from_device(p, soa.data(), 100, 0) == ICEMPM_OK);
            EXPECT(fake::state().device == current);
        }
    }
    icempm_partition_destroy(a);
    icempm_partition_destroy(b);
}

// Without pinned memory the transfers and the queries still work, with the
// same values: FP64 bits as they were, the mixed form's elements in FP32 (Jp
// and the diagonal of F as differences from 1) and positions to its fixed point.
void no_pinned_memory()
{
    fake::state().host_malloc_fails = true;
    constexpr int n = 700, capacity = 900, offset = 13;
    const icempm_simparams P = params(64, 32);
    std::vector<double> soa(16 * capacity), out(16 * capacity, -1.0);
    for (int line = 0; line < 16; line++)
        for (int i = 0; i < n; i++) {
            double v = 0.25 + 1e-3 * i + 0.1 * line;
            if (line == 0) {
                const long long ud = 1000 + i;
                std::memcpy(&v, &ud, 8);
            }
            soa[line * capacity + offset + i] = v;
        }
    for (int precision : {ICEMPM_PRECISION_FP64, ICEMPM_PRECISION_MIXED}) {
        icempm_partition *p = partition(P, n, precision);
        EXPECT(icempm_partition_transfer_points_from_soa_to_device(p, soa.data(), capacity, offset, n) == ICEMPM_OK);
        uint8_t code = 1;
        EXPECT(icempm_partition_get_error_code(p, &code) == ICEMPM_OK && code == 0);
        EXPECT(icempm_partition_transfer_from_device(p, out.data(), capacity, offset) == ICEMPM_OK);
        for (int line = 0; line < 16; line++)
            for (int i = 0; i < n; i++) {
                const double want = soa[line * capacity + offset + i], got = out[line * capacity + offset + i];
                const bool one = line == 3 || line == 8 || line == 11, pos = line == 4 || line == 5;
                if (precision == ICEMPM_PRECISION_FP64 || line == 0)
                    EXPECT(std::memcmp(&want, &got, 8) == 0);
                else if (pos)
                    EXPECT(std::abs(got - want) <= P.cellsize / (1 << 22));
                else
                    EXPECT(got == (one ? 1.0 + (double)(float)(want - 1.0) : (double)(float)want));
            }
        EXPECT(out[offset - 1] == -1.0 && out[16 * capacity - 1] == -1.0);
        EXPECT(icempm_partition_step(p, 2, 0) == ICEMPM_OK);
        EXPECT(icempm_partition_sort_points(p) == ICEMPM_OK);
        EXPECT(icempm_partition_step(p, 2, 0) == ICEMPM_OK);
        icempm_partition_destroy(p);
    }
}

// The substep launches of a batch have a workgroup for each scene with an
// indenter, as many as there are compute units, and none for the others.
void indenter_workgroups()
{
    unsigned grid[4];
    const int n_scenes = 300, with_indenter[4] = {0, 1, 200, 300};
    for (int c = 0; c < 4; c++) {
        icempm_batch *b = nullptr;
        EXPECT(icempm_batch_create(0, ICEMPM_PRECISION_FP64, &b) == ICEMPM_OK);
        std::vector<double> soa(16);
        for (int i = 0; i < n_scenes; i++) {
            icempm_simparams P = params(64, 32);
            P.IndRSq = i >= n_scenes - with_indenter[c] ? 1.0 : 0.0;
            int id;
            EXPECT(icempm_batch_add_scene(b, &P, sizeof P, soa.data(), 1, 1, &id) == ICEMPM_OK);
        }
        EXPECT(icempm_batch_commit(b) == ICEMPM_OK);
        fake::state().launches.clear();
        EXPECT(icempm_batch_step(b, 2, ICEMPM_STEP_RESORT) == ICEMPM_OK);
        grid[c] = 0;
        for (auto &l : fake::state().launches)
            if (l.name.find("k_tiles") != std::string::npos) grid[c] = l.grid.x;   // of the last, with the indenter
        icempm_batch_destroy(b);
    }
    EXPECT(grid[1] - grid[0] == 1);
    EXPECT(grid[2] - grid[0] == 200);
    EXPECT(grid[3] - grid[0] == 256);
}

// The count of the tiles that decides a scene's tile shape is made by the
// points: few of them on a huge grid take a small launch.
void census_by_points()
{
    const icempm_simparams P = params(8000, 8000);
    icempm_partition *p = partition(P, 1000);
    std::vector<double> soa(16 * 1000);
    EXPECT(icempm_partition_transfer_points_from_soa_to_device(p, soa.data(), 1000, 0, 1000) == ICEMPM_OK);
    EXPECT(icempm_partition_sort_points(p) == ICEMPM_OK);
    EXPECT(launched("k_tile_census") == 1);
    for (auto &l : fake::state().launches)
        if (l.name.find("k_tile_census") != std::string::npos) EXPECT(l.grid.x * l.grid.y <= 4);
    icempm_partition_destroy(p);
}

const struct {
    const char *name;
    void (*check)();
} checks[] = {
    {"empty_scene", empty_scene},
    {"huge_tile_table", huge_tile_table},
    {"no_memory_for_tiles", no_memory_for_tiles},
    {"fill_alignment", fill_alignment},
    {"coherent_staging", coherent_staging},
    {"two_devices", two_devices},
    {"no_pinned_memory", no_pinned_memory},
    {"indenter_workgroups", indenter_workgroups},
    {"census_by_points", census_by_points},
};

}  // namespace

int main(int argc, char **argv)
{
    for (auto &c : checks)
        if (argc == 2 && std::strcmp(argv[1], c.name) == 0) {
            c.check();
            std::printf("%s: %s\n", c.name, g_failed ? "failed" : "ok");
            return g_failed != 0;
        }
    for (auto &c : checks) std::printf("%s\n", c.name);
    return argc == 1 ? 0 : 2;
}
