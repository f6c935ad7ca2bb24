// Making pages present changes no byte, at odd addresses and lengths, and the
// pool copies as before afterwards.
#include <cstdio>
#include "../../immunodbscan_amd/csrc/copy_pool.h"

int main()
{
    const size_t sizes[] = {1, 4095, 4097, (1u << 20) + 13, (5u << 20) - 1};
    for (size_t n : sizes)
        for (size_t lead : {0, 1, 4095}) {
            std::vector<uint8_t> buf(lead + n + 8192, 0x5A);
            for (size_t k = 0; k < buf.size(); k += 61) buf[k] = (uint8_t)k;
            const std::vector<uint8_t> before = buf;
            const CopyPool::Job present{buf.data() + lead, nullptr, n};
            CopyPool::get().run(&present, 1);
            if (buf != before) return printf("FAIL bytes changed (%zu at %zu)\n", n, lead), 1;
            std::vector<uint8_t> dst(n, 0);
            const CopyPool::Job both[2] = {{dst.data(), nullptr, n}, {dst.data(), before.data() + lead, n}};
            CopyPool::get().run(both, 1);
            CopyPool::get().run(both + 1, 1);
            if (std::memcmp(dst.data(), before.data() + lead, n)) return printf("FAIL copy (%zu)\n", n), 1;
        }
    printf("ok\n");
    return 0;
}
