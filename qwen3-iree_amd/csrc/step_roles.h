// Which workgroups of the single-launch decode step (dec_step) have a role, and
// how a step that changes that ends.  Constexpr functions and templates over the
// memory they touch, so that the kernel and a CPU check run the same code.
//
// Workgroups 0 .. kStepWgs - 1 have a role at every context, and the end of a
// step depends on each of them.  Workgroups kStepWgs .. kStepGrid - 1 take part
// above kAttnShortCtx positions only (step_long) and end at once below.  They
// read the position themselves, and below the switch nothing else in the step
// waits for them: on a device that is shared, one of them may start after the
// others are done.  The step that moves the position over the switch must
// therefore not store the new position, or the new sequence number, before each
// of them has read the old ones; a late one would take a role in a step that is
// over.  Each of them publishes a tagged word once its reads have returned
// (step_start_extra), and that one step waits for the words (step_crosses).  The
// wait ends without the grid being resident at once: every other workgroup of
// the launch ends by itself and leaves its place to those not yet started.
#ifndef QWEN3_STEP_ROLES_H
#define QWEN3_STEP_ROLES_H

#include <stdint.h>

constexpr int kStepWgs = 448;
constexpr int kStepGrid = 512;
constexpr int kStepExtra = kStepGrid - kStepWgs;
// Contexts up to here have 32 attention splits per kv head, longer ones 64
// (figures beside kAttnSplits in decode_device.h).
constexpr int kAttnShortCtx = 1280;

// at position pos (the context is pos + 1)
constexpr bool step_long(int pos) { return pos >= kAttnShortCtx; }

// Workgroups launched over a cache of max_seq positions: the extra ones only where
// some step can need them.
constexpr int step_grid(int64_t max_seq) {
  return max_seq > kAttnShortCtx ? kStepGrid : kStepWgs;
}

// The last workgroup a step depends on.  Workgroups start in index order, so once
// it runs the whole of the step is resident; it marks the launch as such, and a
// wait that finds the mark missing after about a millisecond gives up instead
// of polling to its limit.
constexpr int step_last_wg(bool is_long) { return (is_long ? kStepGrid : kStepWgs) - 1; }

// Whether the step at position pos leaves it on the other side of the switch.
constexpr bool step_crosses(int pos, int max_seq, bool advance) {
  return advance && pos + 1 < max_seq && !step_long(pos) && step_long(pos + 1);
}

struct StepStart {
  uint32_t seq;     // this launch's sequence number
  uint32_t status;  // the status word
  int32_t pos;
};

// What workgroup kStepWgs + i reads at its start, the sequence word before the
// status word; published once it has them: the word carries the number read
// and the position read, so it cannot leave before both have arrived.
template <class Io>
constexpr StepStart step_start_extra(Io& io, int i) {
  StepStart s{io.load_seq() + 1u, io.load_status(), io.load_pos()};
  io.put_started(i, s.seq, s.pos);
  return s;
}

// Workgroup 0, before the step's token, position and number are stored: false
// if the step was aborted meanwhile.
template <class Io>
constexpr bool step_may_end(Io& io, int pos, int max_seq, bool advance) {
  return !step_crosses(pos, max_seq, advance) || io.wait_started();
}

#endif
