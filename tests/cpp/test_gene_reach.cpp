// The quick look at the names (idb_gene_table_in_reach): tables within the cap
// are not turned away, and the build of ones far above it is not begun.
#include <array>
#include <cstdio>
#include <fstream>
#include <random>
#include <string>
#include <vector>

#include "../../immunodbscan_amd/csrc/gene_table.h"

static int fails = 0;

struct Names {
    std::vector<uint8_t> data;
    std::vector<uint64_t> off;
    std::vector<uint32_t> len;
    explicit Names(const std::vector<std::string> &v)
    {
        for (auto &s : v) {
            off.push_back(data.size());
            len.push_back((uint32_t)s.size());
            data.insert(data.end(), s.begin(), s.end());
        }
        data.push_back(0);
    }
    bool reach(uint32_t cap) const
    {
        return idb_gene_table_in_reach((uint32_t)len.size(), data.data(), off.data(), len.data(), cap);
    }
    bool build(uint32_t cap, idb_gene_table &t) const
    {
        return idb_gene_table_build((uint32_t)len.size(), data.data(), off.data(), len.data(), cap, t);
    }
};

static void expect(bool ok, const char *what)
{
    if (!ok) {
        std::printf("%s\n", what);
        ++fails;
    }
}

int main(int, char **argv)
{
    std::mt19937 rng(5);
    // gene lists and their alleles, in order and shuffled: whatever table the
    // cost rule allows for a call is in reach
    for (const char *list : {"VH", "DH", "JH"}) {
        std::vector<std::string> genes, alleles;
        std::ifstream in(std::string(argv[1]) + "/" + list + "genes.txt");
        for (std::string s; std::getline(in, s);)
            if (!s.empty()) genes.push_back(s);
        for (auto &g : genes)
            for (uint32_t k = 1; k < 5 + rng() % 10; ++k) alleles.push_back(g + char('0' + k / 10) + char('0' + k % 10));
        for (auto *v : {&genes, &alleles})
            for (int rep = 0; rep < 20; ++rep) {
                const Names n(*v);
                for (uint32_t calls : {1u, 1000u, 20000u, 1000000u}) {
                    const uint32_t cap = idb_gene_table_cap(calls, (uint32_t)v->size());
                    idb_gene_table t;
                    if (n.build(cap, t)) expect(n.reach(cap), list);
                }
                std::shuffle(v->begin(), v->end(), rng);
            }
    }
    // random names share few letters: half their table is not in reach, all of it is
    auto word = [&](uint32_t lo, uint32_t hi) {
        std::string s;
        for (uint32_t n = lo + rng() % (hi - lo + 1); n; --n) s.push_back((char)('A' + rng() % 23));
        return s;
    };
    for (auto [k, lo, hi] : {std::array<uint32_t, 3>{8000, 8, 12}, {2000, 6, 10}, {260, 6, 9}, {64, 900, 1000}, {20, 200, 400}}) {
        std::vector<std::string> v;
        for (uint32_t g = 0; g < k; ++g) v.push_back(word(lo, hi));
        v[k / 2].clear();
        v[k / 3] = std::string(1100, 'A');
        const Names n(v);
        idb_gene_table t;
        expect(n.build(1u << 22, t), "random names: not built");
        expect(n.reach(t.entries) && n.reach(t.entries + t.entries / 10), "random names: turned away");
        expect(!n.reach(t.entries / 2), "random names: half a table in reach");
    }
    // nothing to look at
    expect(Names({}).reach(0) && Names({""}).reach(0) && Names({"ab"}).reach(100), "few names");
    expect(Names({"", std::string(2000, 'x'), "", ""}).reach(100), "no usable names");
    std::printf(fails ? "FAILED %d\n" : "gene reach ok\n", fails);
    return fails ? 1 : 0;
}
