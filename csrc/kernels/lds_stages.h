// Blocks of operands moved to LDS by DMA, NST buffers in a ring, waited for by count.  Plain C++: a host program can run it against a model of
// the queue of moves (tests/test_lds_stages_cpu.py).
#pragma once

#include <type_traits>

// stage(buffer, block) issues the MOVES moves of a block; landed(integral_constant n) waits until at most n of the moves issued so far are out and
// then for the other waves; use(buffer) reads a block.  Moves retire in the order in which they are issued, so a block's moves are issued
// together, block after block: when block t is waited for, t .. t + NST - 2 are out, and those after it are (NST - 2) MOVES of them, at
// t = 0 and 1 as later on.  (Past the end the last block is moved again, or the count would not hold.)  The buffer that is
// filled at t is that of block t - 1, which every wave has read before it came to the wait.
template <int NST, int MOVES, class Stage, class Landed, class Use>
constexpr void lds_stages(int blocks, const Stage& stage, const Landed& landed, const Use& use) {
  static_assert(NST >= 2, "one buffer is read while another is filled");
  const auto least = [](int a, int b) { return a < b ? a : b; };
#pragma unroll
  for (int b = 0; b < NST - 1; ++b) stage(b, least(b, blocks - 1));
  int cur = 0;
  for (int t = 0; t < blocks; ++t) {
    landed(std::integral_constant<int, MOVES*(NST - 2)>{});
    stage(cur == 0 ? NST - 1 : cur - 1, least(t + NST - 1, blocks - 1));
    use(cur);
    cur = cur == NST - 1 ? 0 : cur + 1;
  }
}
