// Rules that say which kernel may take a call, and the index arithmetic whose range they depend on.
// Plain C++ without HIP, so that a host program can evaluate them as the launchers do.
#pragma once

#include <cstdint>

namespace tqt {

constexpr int kTileCUs = 256;  // compute units of an MI355X

// Whether `blocks` workgroups of `threads` fit one grid dimension: a launch counts its work-items along
// a dimension in 32 bits.
constexpr bool grid_fits(long long blocks, int threads)
{
    return blocks * threads < 0x100000000ll;
}

// ---------------------------------------------------------------------------------------------
// W4A16
// ---------------------------------------------------------------------------------------------

// Scale block of the 32-k block kb, bdiv 32-k blocks to a scale block: kb / bdiv by the rounded-up
// reciprocal inv = ceil(2^32 / bdiv). With inv * bdiv = 2^32 + e, 0 <= e < bdiv, the product kb * inv
// exceeds kb * 2^32 / bdiv by kb * e / bdiv, so the quotient is exact while kb * bdiv <= 2^32. bdiv
// 65537, kb 65536 is the first pair past that line that is wrong.
constexpr uint32_t scale_block_inverse(uint32_t bdiv)
{
    return static_cast<uint32_t>((0x100000000ull + bdiv - 1) / bdiv);
}

constexpr uint32_t scale_block_of(uint32_t kb, uint32_t bdiv, uint32_t inv)
{
    return bdiv == 1 ? kb : static_cast<uint32_t>((static_cast<uint64_t>(kb) * inv) >> 32);
}

// Whether the few-row kernel's scale indexes are exact over k (bl and k multiples of 32).
constexpr bool w4a16_skinny_scales_exact(long long k, long long bl)
{
    return (k / 32) * (bl / 32) <= 0x100000000ll;
}

}  // namespace tqt
