// The two words of a wave's donated range in the depth-first kernel (enum.hip): what is left of a frame's
// candidates, and where the frame starts.  They are stored one after the other without any ordering between
// them, so both carry the version of their publication and are used together only if it is the same.
// A version is 1..65535 and words that were never published are 0, so a cleared word matches none.
#pragma once
#include <cstdint>

namespace csm {

constexpr uint32_t kRangeBits = 24;
constexpr uint32_t kRangeMask = (1u << kRangeBits) - 1;

constexpr uint32_t next_version(uint32_t version) { return version % 0xFFFFu + 1; }

// Candidates [cur, end) still to be explored: version (16 bits) | cur (24) | end (24).
constexpr unsigned long long range_word(uint32_t version, uint32_t cur, uint32_t end) {
    return static_cast<unsigned long long>(version) << (2 * kRangeBits) | static_cast<unsigned long long>(cur) << kRangeBits | end;
}
constexpr uint32_t range_cur(unsigned long long w) { return static_cast<uint32_t>(w >> kRangeBits) & kRangeMask; }
constexpr uint32_t range_end(unsigned long long w) { return static_cast<uint32_t>(w) & kRangeMask; }

// The frame they belong to: version (16 bits) | item group (42) | first item of the group that is in the frame (6).
constexpr unsigned long long frame_word(uint32_t version, uint32_t group, uint32_t first) {
    return static_cast<unsigned long long>(version) << (2 * kRangeBits) | static_cast<unsigned long long>(group) << 6 | first;
}
constexpr uint32_t frame_group(unsigned long long w) { return static_cast<uint32_t>(w >> 6); }
constexpr uint32_t frame_first(unsigned long long w) { return static_cast<uint32_t>(w) & 63u; }

constexpr bool same_publication(unsigned long long range, unsigned long long frame) {
    return range >> (2 * kRangeBits) == frame >> (2 * kRangeBits) && range >> (2 * kRangeBits) != 0;
}

}  // namespace csm
