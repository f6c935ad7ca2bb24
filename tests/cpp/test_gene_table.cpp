// The multi-name automaton (gene_table.h) against a plain search of every
// name, over random names and strings of small alphabets (dense overlaps,
// names inside names, equal names, names that never match) and at the caps.
#include <cstdio>
#include <random>
#include <string>
#include <vector>

#include "../../immunodbscan_amd/csrc/gene_table.h"

static int fails = 0;

static void check(const std::vector<std::string> &names, const std::vector<std::string> &rows, const char *what)
{
    std::vector<uint8_t> data;
    std::vector<uint64_t> off;
    std::vector<uint32_t> len;
    for (auto &n : names) {
        off.push_back(data.size());
        len.push_back((uint32_t)n.size());
        data.insert(data.end(), n.begin(), n.end());
    }
    data.push_back(0);
    idb_gene_table t;
    if (!idb_gene_table_build((uint32_t)names.size(), data.data(), off.data(), len.data(), 1u << 22, t)) {
        std::printf("%s: not built\n", what);
        ++fails;
        return;
    }
    // the cap is exact: one entry fewer is refused
    idb_gene_table u;
    if (idb_gene_table_build((uint32_t)names.size(), data.data(), off.data(), len.data(), t.entries - 1u, u) ||
        !idb_gene_table_build((uint32_t)names.size(), data.data(), off.data(), len.data(), t.entries, u)) {
        std::printf("%s: cap\n", what);
        ++fails;
    }
    for (auto &r : rows) {
        std::vector<char> got(names.size(), 0);
        uint32_t s = 0;
        for (unsigned char ch : r) {
            s = t.trans[s + t.cls[ch]];
            if ((s >= t.out_min) != (t.trans[s + t.ncls] != 0u)) ++fails;
            if (s >= t.out_min)
                for (uint32_t n = t.trans[s + t.ncls]; n; n = t.nodes[n - 1] >> 16) got[t.nodes[n - 1] & 0xFFFFu] = 1;
        }
        for (size_t g = 0; g < names.size(); ++g) {
            const bool want = !names[g].empty() && names[g].size() <= IDB_GENE_NAME_MAX && r.find(names[g]) != std::string::npos;
            if (want != (bool)got[g]) {
                if (++fails < 5) std::printf("%s: name %zu\n", what, g);
                return;
            }
        }
    }
}

int main()
{
    std::mt19937 rng(5);
    auto word = [&](uint32_t lo, uint32_t hi, uint32_t k) {
        std::string s;
        for (uint32_t n = lo + rng() % (hi - lo + 1); n; --n) s.push_back((char)(1 + rng() % k));
        return s;
    };
    for (uint32_t k : {1u, 2u, 3u, 20u, 255u})
        for (int rep = 0; rep < 20; ++rep) {
            std::vector<std::string> names, rows;
            for (int g = 0; g < 90; ++g) names.push_back(word(0, 7, k));
            names.push_back(std::string(1024, 'A'));
            names.push_back(std::string(1025, 'A'));
            names.push_back(names[3]);
            for (int r = 0; r < 60; ++r) rows.push_back(word(0, 90, k < 255 ? k + 1 : k) + std::string(r % 3, '\0'));
            rows.push_back(std::string(1024, 'A'));
            rows.push_back(std::string(3000, 'A'));
            check(names, rows, "random");
        }
    check({}, {"", "abc"}, "no names");
    check({"", std::string(2000, 'x')}, {"", "abc", std::string(2000, 'x')}, "no usable names");
    std::string all;
    for (int b = 1; b <= 256; ++b) all.push_back((char)b);
    idb_gene_table t;
    const uint64_t o = 0;
    const uint32_t l255 = 255, l256 = 256;  // every byte value but 0, then 0 too
    if (!idb_gene_table_build(1, (const uint8_t *)all.data(), &o, &l255, 1u << 20, t)) ++fails;
    if (idb_gene_table_build(1, (const uint8_t *)all.data(), &o, &l256, 1u << 20, t)) ++fails;
    std::printf(fails ? "FAILED %d\n" : "gene table ok\n", fails);
    return fails ? 1 : 0;
}
