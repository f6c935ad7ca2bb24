// The 4-bit features (mxfeat.h): every value the digits must hold, the bit
// spread.
#include <algorithm>
#include <cstdio>
#include <random>
#include <string>
#include <vector>

#include "../../immunodbscan_amd/csrc/mxfeat.h"

static const float V[16] = {0, .5f, 1, 1.5f, 2, 3, 4, 6, -0.f, -.5f, -1, -1.5f, -2, -3, -4, -6};
static long fails = 0;

static float value(const std::vector<uint32_t> &f, int d) { return V[(f[d / 8] >> (4 * (d & 7))) & 15u]; }

int main()
{
    for (int v = -185; v <= 185; ++v) {
        const uint32_t g = idb_mx_digits(v, 6);
        float s = 0;
        for (int k = 0; k < 8; ++k) s += V[(g >> (4 * k)) & 15u] * V[(IDB_MX_NT_WEIGHTS >> (4 * k)) & 15u];
        if (s != (float)v) ++fails;
        if (v < -35 || v > 35) continue;
        const uint32_t a = idb_mx_digits(v, 2);
        s = 0;
        for (int k = 0; k < 4; ++k) s += V[(a >> (4 * k)) & 15u] * V[(IDB_MX_AA_WEIGHTS >> (4 * k)) & 15u];
        if (s != (float)v || a >> 16) ++fails;
    }
    for (uint32_t b = 0; b < 256; ++b)
        for (int k = 0; k < 8; ++k)
            if (((idb_mx_spread(b) >> (4 * k)) & 15u) != ((b >> k & 1u) ? 2u : 0u)) ++fails;
    std::printf(fails ? "FAILED %ld\n" : "features ok\n", fails);
    return fails ? 1 : 0;
}
