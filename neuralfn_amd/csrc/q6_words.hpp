// Where the words of a Q6_K block begin.  (No HIP in here: a test compiles it for the host.)
#pragma once

#include <cstdint>

namespace nfn {

// Bytes from the word at or before a Q6_K block of 210 bytes to the block itself, 0 or 2: of a tensor that begins at a word
// every other block of a row begins two bytes past one.  A tensor that does not begin at a word is read as it lies, every
// second of its blocks from past a word: the word before its first block holds bytes that are not its own.
constexpr std::uint32_t q6_past_word(std::uintptr_t tensor, std::uintptr_t block) {
    return (tensor & 3u) == 0 ? static_cast<std::uint32_t>(block) & 2u : 0u;
}

}  // namespace nfn
