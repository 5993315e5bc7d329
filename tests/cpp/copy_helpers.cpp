// Unit check of the host copies of the staged transfers (CopyHelpers,
// dxmclib_amd/csrc/hostcopy.hpp): lengths below, at and around 4 MiB
// and the 8 MiB half chunk, odd lengths and unaligned
// addresses, repeated copies on the same helpers, copies without helpers, and
// copies of several blocks (empty, small and large ones, whose ends fall
// anywhere in the threads' parts). Prints "ok" and exits 0, or names the failing case and exits 1.
#include "../../dxmclib_amd/csrc/hostcopy.hpp"

#include <algorithm>
#include <cstdint>
#include <cstdio>
#include <vector>

int main()
{
    using dxmc_backend::CopyHelpers;
    constexpr std::size_t MiB = std::size_t { 1 } << 20;
    const std::size_t lengths[] = { 0, 1, 7, 4 * MiB - 1, 4 * MiB, 4 * MiB + 3, 8 * MiB - 1, 8 * MiB, 8 * MiB + 1, 13 * MiB + 5 };
    const std::size_t maxLen = 13 * MiB + 5 + 64;
    std::vector<unsigned char> src(maxLen), dst(maxLen);
    std::uint64_t x = 0x9E3779B97F4A7C15ULL;
    for (auto& b : src) {
        x ^= x << 13;
        x ^= x >> 7;
        x ^= x << 17;
        b = static_cast<unsigned char>(x);
    }
    CopyHelpers helpers;
    for (int round = 0; round < 3; ++round) {
        if (round == 0 && !helpers.start()) {
            std::printf("helpers did not start\n");
            return 1;
        }
        if (round == 2)
            helpers.stop(); // copies on the calling thread alone
        for (const std::size_t len : lengths)
            for (const std::size_t so : { 0, 3 })
                for (const std::size_t doff : { 0, 5 }) {
                    std::fill(dst.begin(), dst.end(), 0xA5);
                    helpers.copy(dst.data() + doff, src.data() + so, len);
                    for (std::size_t i = 0; i < maxLen; ++i) {
                        const bool inside = i >= doff && i < doff + len;
                        const unsigned char want = inside ? src[i - doff + so] : 0xA5;
                        if (dst[i] != want) {
                            std::printf("round %d len %zu src+%zu dst+%zu: byte %zu differs\n", round, len, so, doff, i);
                            return 1;
                        }
                    }
                }
    }
    using Block = CopyHelpers::Block;
    CopyHelpers many;
    for (int round = 0; round < 2; ++round) {
        if (round == 1 && !many.start()) {
            std::printf("helpers did not start\n");
            return 1;
        }
        const std::size_t sets[][3] = { { 0, 0, 0 }, { 1, 2, 3 }, { 0, MiB, 0 }, { 500 * 1024, 7, 24 * 1024 - 7 }, { 500 * 1024, 7, 24 * 1024 - 8 },
            { 3 * MiB + 1, 0, 5 }, { 5, 2 * MiB + 3, 3 * MiB }, { MiB, MiB / 2, MiB } };
        for (const auto& set : sets) {
            std::fill(dst.begin(), dst.end(), 0xA5);
            Block list[3];
            std::size_t from = 3, to = 5; // gaps between the blocks on both sides
            for (int i = 0; i < 3; ++i) {
                list[i] = { reinterpret_cast<char*>(dst.data() + to), reinterpret_cast<const char*>(src.data() + from), set[i] };
                from += set[i] + 9;
                to += set[i] + 2;
            }
            many.copy(list, 3);
            std::vector<unsigned char> want(maxLen, 0xA5);
            for (const Block& b : list)
                std::copy(b.src, b.src + b.len, want.data() + (b.dst - reinterpret_cast<char*>(dst.data())));
            if (want != dst) {
                std::printf("round %d blocks %zu %zu %zu differ\n", round, set[0], set[1], set[2]);
                return 1;
            }
        }
    }
    std::printf("ok\n");
    return 0;
}
