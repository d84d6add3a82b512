// The order in which a block of k_attn_pf fills, reads and refills its LDS
// stages, apart from what it computes, so that the order can also be followed
// on the host (constexpr: callable on both sides).
//
// Key tiles [tb, te); K and V have two stages each. `copy(t, part, stage)`
// starts a wave's share of the DMA of tile t (part 0: K, 1: V) into a stage;
// `arrive` waits for this wave's own copies, `barrier` for all four waves, so
// a stage may be read after arrive + barrier and refilled after a barrier that
// follows its last reads. Per stage, last reader and next writer:
//   K 0: first (tile tb)         | barrier B0                | copy of tile tb + 2 in step tb
//   K s: step t (tile t + 1)     | barrier at step t's end   | copy of tile t + 3 in step t + 1
//   V s: step t (tile t)         | barrier at step t's end   | copy of tile t + 2 in step t + 1
// The last steps copy tile te - 1 again, into a stage that is read no more.
#pragma once

namespace gg {

template <class Copy>
__attribute__((always_inline)) constexpr void pf_schedule_fill(int tb, int te, Copy&& copy) {
  copy(tb, 0, 0);
  copy(tb, 1, 0);
  copy(tb + 1 < te ? tb + 1 : te - 1, 0, 1);
}

// first(t, ks): scores of tile t from K stage ks. step(t, ks, vs): scores of
// tile t + 1 from K stage ks and the weighted sum of tile t from V stage vs.
// last(t, vs): the weighted sum of tile t.
template <class Copy, class Arrive, class Barrier, class First, class Step, class Last>
__attribute__((always_inline)) constexpr void pf_schedule_run(int tb, int te, Copy&& copy, Arrive&& arrive,
                                                              Barrier&& barrier, First&& first, Step&& step,
                                                              Last&& last) {
  arrive();
  barrier();
  first(tb, 0);
  if (tb + 1 < te) barrier();   // B0: every wave has read K stage 0
  for (int t = tb; t + 1 < te; ++t) {
    const int b = (t - tb) & 1;
    copy(t + 1, 1, b ^ 1);
    copy(t + 2 < te ? t + 2 : te - 1, 0, b);
    step(t, b ^ 1, b);
    arrive();
    barrier();
  }
  last(te - 1, (te - 1 - tb) & 1);
}

}  // namespace gg
