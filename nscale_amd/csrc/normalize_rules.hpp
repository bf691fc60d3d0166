// Rules of the normalization passes that a host compiler can check (plain C++; constexpr functions serve device
// code too).
#pragma once

namespace nsc {

// q / d as the high half of q * magic, magic = floor((2^64 - 1) / d) + 1.  That is 2^64 / d rounded up, above it by
// less than 1 (exact where d is a power of two), so the product is above q / d by less than q / 2^64, which is below
// 1 / d while q * d < 2^64.  Here d = the groups of four pixels in a row, below 2^29, and q a group's
// number, below 2^35 for an image of up to 400 GB.  d = 1, whose magic would be 2^64, has magic 0: q itself.
constexpr unsigned long long row_magic(unsigned long long d) { return d > 1 ? ~0ull / d + 1 : 0; }
constexpr unsigned long long row_of(unsigned long long q, unsigned long long magic) {
    return magic ? (unsigned long long)((unsigned __int128)q * magic >> 64) : q;
}

}  // namespace nsc
