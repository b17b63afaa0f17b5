// kd_mt_jump.h - jumping ahead in MT19937-64's word sequence.
#pragma once

#include <cstdint>

namespace kd {

constexpr int kMtWords = 312;
constexpr int kMtDegree = 19937;      // of the recurrence's characteristic polynomial
constexpr int kJumpBlocks = 64;       // twists (312 words) from one chain's start to the next
constexpr int kJumpChains = 64;       // chains of a round, the first of which needs no jump

// The polynomials t^(312 * kJumpBlocks * c - 1) modulo the characteristic polynomial for c = 1 .. `count` (below
// kJumpChains), 312 words each, bit k of word k / 64 the coefficient of t^k: with w_0, w_1, ... the generator's words
// from the current ones on,
//   w[312 * kJumpBlocks * c + i] = XOR over the set k of w[k + 1 + i].
// Computed by the first call that asks for them (0.04 ms each) and kept; the pointer is the same for every call.
const uint64_t* mt_jump_polynomials(int count);

} // namespace kd
