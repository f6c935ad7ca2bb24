// Which form of the gene scan takes a call: reads "<calls> <names>" and one
// name per line, prints the form, its table's entries and its block's LDS.
#include <cstdio>
#include <iostream>
#include <string>

#include "../../immunodbscan_amd/csrc/gene_table.h"

int main()
{
    uint32_t n, k;
    std::cin >> n >> k;
    std::vector<uint8_t> data;
    std::vector<uint64_t> off;
    std::vector<uint32_t> len;
    std::string s;
    std::getline(std::cin, s);
    for (uint32_t g = 0; g < k; ++g) {
        std::getline(std::cin, s);
        off.push_back(data.size());
        len.push_back((uint32_t)s.size());
        data.insert(data.end(), s.begin(), s.end());
    }
    data.push_back(0);
    idb_gene_table t;
    const uint32_t cap = idb_gene_table_cap(n, k);
    if (!idb_gene_table_in_reach(k, data.data(), off.data(), len.data(), cap) ||
        !idb_gene_table_build(k, data.data(), off.data(), len.data(), cap, t)) {
        std::puts("names 0 0");
        return 0;
    }
    const bool narrow = idb_gene_table_narrow(t, 160 * 1024);
    std::printf("%s %u %zu\n", narrow ? "16" : "32", t.entries, narrow ? idb_gene_table_lds(t) : 256);
}
