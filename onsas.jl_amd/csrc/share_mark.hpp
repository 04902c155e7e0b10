// share_mark.hpp -- the mark of 16 bytes that workgroups of one launch hand to one
// another: 12 bytes of payload and a word that says from which epoch they are.
//
// The mark is the epoch and the payload folded into one word, so that it holds for the
// payload as a whole: a reader that got a part of the words from one store and a part
// from another finds another epoch and reads again.  Rotations by 11 and 22 bits keep
// equal changes of two words from cancelling.  If only one word is stale the mark differs
// for certain, otherwise unless the changes of the words happen to cancel in all 32 bits.
#pragma once

#include <cstdint>

namespace onsas {

constexpr uint32_t rotl32(uint32_t x, int n) { return (x << n) | (x >> (32 - n)); }
constexpr uint32_t share_mark(uint32_t a, uint32_t b, uint32_t c, uint32_t epoch) {
  return epoch ^ a ^ rotl32(b, 11) ^ rotl32(c, 22);
}

}  // namespace onsas
