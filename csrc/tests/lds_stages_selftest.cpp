// lds_stages (csrc/kernels/lds_stages.h) on a model of a wave's queue of moves: one retires only when a wait needs it to, oldest first.
// A block must be whole in its buffer when it is read, and a buffer is filled again only after every wave has read it.
#include "../kernels/lds_stages.h"

#include <cstdio>
#include <deque>
#include <vector>

namespace {

struct Move {
  int buf, part, block;
};

struct Model {
  int moves;
  std::deque<Move> out;                   // oldest first
  std::vector<std::vector<int>> holds;    // [buffer][part] block, -1: on its way
  std::vector<int> read_at;               // barriers before the buffer's block was read, -1: never
  int barriers = 0, next = 0;
  bool ok = true;

  Model(int nst, int m) : moves(m), holds(nst, std::vector<int>(m, -1)), read_at(nst, -1) {}
  void issue(int buf, int part, int block) {
    bool filled = false;
    for (int h : holds[buf]) filled |= h >= 0;
    if (filled && part == 0 && !(read_at[buf] >= 0 && read_at[buf] < barriers)) ok = false;   // another wave may still read it
    holds[buf][part] = -1;
    out.push_back({buf, part, block});
  }
  void stage(int buf, int block) {
    for (int m = 0; m < moves; ++m) issue(buf, m, block);
  }
  void landed(int most) {
    for (; (int)out.size() > most; out.pop_front()) holds[out.front().buf][out.front().part] = out.front().block;
    ++barriers;
  }
  void use(int buf) {
    for (int h : holds[buf]) ok &= h == next;
    read_at[buf] = barriers;
    ++next;
  }
};

template <int NST, int MOVES>
bool holds_for(int blocks) {
  Model m(NST, MOVES);
  lds_stages<NST, MOVES>(blocks, [&](int buf, int block) { m.stage(buf, block); }, [&](auto n) { m.landed(decltype(n)::value); },
                         [&](int buf) { m.use(buf); });
  return m.ok && m.next == blocks;
}

// A mistake that the model has to see: the first blocks' weights all before their rows, with the counts of whole blocks.
bool weights_first(int nst, int w, int a, int blocks) {
  Model m(nst, w + a);
  const auto least = [](int x, int y) { return x < y ? x : y; };
  for (int b = 0; b < nst - 1; ++b)
    for (int i = 0; i < w; ++i) m.issue(b, i, least(b, blocks - 1));
  for (int b = 0; b < nst - 1; ++b)
    for (int i = 0; i < a; ++i) m.issue(b, w + i, least(b, blocks - 1));
  m.landed(a * (nst - 2));
  for (int t = 0, cur = 0; t < blocks; ++t, cur = (cur + 1) % nst) {
    m.landed((w + a) * (nst - 2));
    m.stage((cur + nst - 1) % nst, least(t + nst - 1, blocks - 1));
    m.use(cur);
  }
  return m.ok;
}

template <int NST>
bool all_moves(int blocks) {
  return holds_for<NST, 1>(blocks) && holds_for<NST, 2>(blocks) && holds_for<NST, 4>(blocks) && holds_for<NST, 6>(blocks) &&
         holds_for<NST, 8>(blocks);
}

}  // namespace

int main() {
  for (int blocks = 1; blocks <= 20; ++blocks) {
    if (!all_moves<2>(blocks) || !all_moves<3>(blocks) || !all_moves<4>(blocks) || !all_moves<5>(blocks)) {
      printf("block read before it landed, or filled too early: %d blocks\n", blocks);
      return 1;
    }
    if (!weights_first(3, 2, 2, blocks)) return printf("three buffers: the model sees a mistake that is none (%d blocks)\n", blocks), 1;
    if (weights_first(4, 2, 2, blocks) != (blocks == 1)) return printf("four buffers: the model misses rows that nothing waits for\n"), 1;
  }
  printf("lds_stages OK\n");
  return 0;
}
