// Host-side helpers the batch calls share.
#pragma once

#include <stdint.h>

#include <algorithm>
#include <cstring>
#include <functional>
#include <thread>
#include <vector>

namespace dinara {

// Runs body(lo, hi) over [0, count) cut into `threads` contiguous shares, each on a thread of its own; one share
// on the caller's thread when `threads` is one or less.
inline void parallel_for(int64_t count, int64_t threads, const std::function<void(int64_t, int64_t)> &body) {
    const int64_t workers = std::max<int64_t>(1, std::min<int64_t>(threads, count));
    if (workers <= 1) {
        body(0, count);
        return;
    }
    std::vector<std::thread> pool;
    for (int64_t w = 0; w < workers; ++w)
        pool.emplace_back([&, w]() { body(count * w / workers, count * (w + 1) / workers); });
    for (auto &t : pool) t.join();
}

// Sorts `items` by key(item), highest first, equal keys in the order they came: a counting sort 11 bits at a time.
template <typename Key>
void longest_first(std::vector<int32_t> &items, const Key &key) {
    uint32_t longest = 0;
    for (int32_t i : items) longest = std::max<uint32_t>(longest, key(i));
    std::vector<int32_t> sorted(items.size());
    for (int shift = 0; shift < 32 && (longest >> shift) != 0; shift += 11) {
        size_t place[2049] = {0};
        for (int32_t i : items) ++place[2048 - ((key(i) >> shift) & 2047u)];
        for (int d = 1; d < 2049; ++d) place[d] += place[d - 1];
        for (int32_t i : items) sorted[place[2047 - ((key(i) >> shift) & 2047u)]++] = i;
        items.swap(sorted);
    }
}

// Packing letters: A, C, G and T are the 2-bit codes 0, 1, 2 and 3.
struct Dna {
    // Whether `len` letters are A, C, G and T alone. Comparisons rather than the table: the loop vectorizes.
    static bool plain(const char *text, int64_t len) {
        const unsigned char *u = reinterpret_cast<const unsigned char *>(text);
        unsigned char other = 0;
        for (int64_t i = 0; i < len; ++i)
            other |= (unsigned char)!((u[i] == 'A') | (u[i] == 'C') | (u[i] == 'G') | (u[i] == 'T'));
        return other == 0;
    }
    // The codes of eight such letters, in 16 bits: bits 1-2 of A, C, G and T are 0, 1, 3 and 2, and bit 2 flips the last
    // two.
    static uint32_t codes8(uint64_t letters) {
        uint64_t v = ((letters >> 1) ^ (letters >> 2)) & 0x0303030303030303ull;
        v = (v | (v >> 6)) & 0x000F000F000F000Full;
        v = (v | (v >> 12)) & 0x000000FF000000FFull;
        return (uint32_t)(v | (v >> 24)) & 0xFFFFu;
    }
    // Packs `len` letters of A, C, G and T, 16 codes to a 32-bit word (letter i at bits 2i), word w at out[64 w],
    // `words` words in all (zero past the letters); back to front when `reversed`.
    static void pack2(const char *text, int64_t len, bool reversed, uint32_t *out, int32_t words) {
        const unsigned char *u = reinterpret_cast<const unsigned char *>(text);
        const int64_t whole = len / 16;
        for (int64_t w = 0; w < whole; ++w) {
            uint64_t low, high;
            if (reversed) {
                std::memcpy(&low, u + len - 8 - 16 * w, 8);
                std::memcpy(&high, u + len - 16 - 16 * w, 8);
                low = __builtin_bswap64(low);
                high = __builtin_bswap64(high);
            } else {
                std::memcpy(&low, u + 16 * w, 8);
                std::memcpy(&high, u + 16 * w + 8, 8);
            }
            out[w * 64] = codes8(low) | (codes8(high) << 16);
        }
        int64_t w = whole;
        if (w < words && 16 * w < len) {
            uint32_t word = 0;
            for (int64_t i = 0; 16 * w + i < len; ++i) {
                const unsigned char byte = reversed ? u[len - 1 - (16 * w + i)] : u[16 * w + i];
                word |= (uint32_t)((byte >> 1 ^ byte >> 2) & 3) << (2 * i);
            }
            out[w * 64] = word;
            ++w;
        }
        for (; w < words; ++w) out[w * 64] = 0;
    }
};

// The decisions of one sweep launch may take at most this much device memory; a larger launch is cut in pieces.
constexpr size_t ARENA_BUDGET = size_t(16) << 30;

}  // namespace dinara
