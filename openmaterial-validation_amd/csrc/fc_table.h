// fc_table.h -- colour table of an enumerated false-colour subject.
//
// EnumeratedFCSubject (FCSubject.h:153-167) gives every id of a category of
// `size` ids its own colour: `size` distinct 24-bit colours in
// [1, 0xFFFFFF] drawn uniformly, kept in ascending order (a std::set), then
// shuffled; an id >= size paints black.  The reference draws from an
// unseeded generator and shuffles with std::random_shuffle, so its tables
// change from run to run.  Here the draws and the shuffle come from
// splitmix64 (Steele, Lea and Flood 2014) started at (seed << 8 | subject):
// v = 1 + (x mod 0xFFFFFF) until `size` distinct values, ascending sort,
// then Fisher-Yates from the last element down with j = x mod (i + 1).
// The same seed and subject always give the same table.
#ifndef OMV_FC_TABLE_H
#define OMV_FC_TABLE_H

#include <cstdint>
#include <utility>
#include <vector>

namespace omv {

inline uint64_t splitmix64Next(uint64_t& s) {
    uint64_t z = (s += 0x9E3779B97F4A7C15ull);
    z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
    z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
    return z ^ (z >> 31);
}

// false when size exceeds the 0xFFFFFF distinct colours there are (the
// reference's draw loop would not end)
inline bool fcColorTable(uint32_t seed, int subject, uint32_t size, std::vector<uint32_t>& out) {
    out.clear();
    if (size > 0xFFFFFFu) return false;
    uint64_t s = ((uint64_t)seed << 8) | (uint64_t)(subject & 0xFF);
    // The bitmap of drawn colours, read in order, is the ascending set; a bit
    // in `some` for each of its words that holds one.  200 000 colours take
    // 3.0 ms, with a list of the draws and std::sort 18.0 ms.
    std::vector<uint64_t> seen(0x1000000u >> 6, 0), some(0x1000000u >> 12, 0);
    for (uint32_t n = 0; n < size;) {
        const uint32_t v = 1u + (uint32_t)(splitmix64Next(s) % 0xFFFFFFull);
        uint64_t& word = seen[v >> 6];
        n += (uint32_t)(~(word >> (v & 63)) & 1u);
        word |= 1ull << (v & 63);
        some[v >> 12] |= 1ull << ((v >> 6) & 63);
    }
    out.resize(size);
    uint32_t* to = out.data();
    for (uint32_t g = 0; g < (uint32_t)some.size(); ++g)
        for (uint64_t words = some[g]; words; words &= words - 1) {
            const uint32_t w = (g << 6) | (uint32_t)__builtin_ctzll(words);
            for (uint64_t bits = seen[w]; bits; bits &= bits - 1) *to++ = (w << 6) | (uint32_t)__builtin_ctzll(bits);
        }
    for (uint32_t i = size; i > 1; --i) {
        const uint32_t j = (uint32_t)(splitmix64Next(s) % i);
        std::swap(out[i - 1], out[j]);
    }
    return true;
}

}  // namespace omv

#endif
