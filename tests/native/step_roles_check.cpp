// Late workgroups of the single-launch step (step_roles.h), on the CPU: the end
// of a step against extra workgroups that start at any point of it, on one
// memory.  What must hold: an extra workgroup takes the role that the step's
// own position gives, and a step it has no role in is not changed by it.
#include <cstdio>
#include <set>

#include "step_roles.h"

struct Memory {
  uint32_t seq = 41, status = 0;
  int32_t pos = 0, max_seq = 0;
  uint32_t started[kStepExtra] = {};  // the number each word carries, 0: none
  bool took_role[kStepExtra] = {};
  std::set<int> late;                 // extra workgroups not started yet

  uint32_t load_seq() const { return seq; }
  uint32_t load_status() const { return status; }
  int32_t load_pos() const { return pos; }
  void put_started(int i, uint32_t n, int32_t) { started[i] = n; }

  void run_extra(int i) {
    const StepStart s = step_start_extra(*this, i);
    const int32_t c = s.pos < 0 ? 0 : (s.pos >= max_seq ? max_seq - 1 : s.pos);
    took_role[i] = step_long(c);
    late.erase(i);
  }
};

// Workgroup 0's view: a wait returns once every word carries this step's
// number; the others have ended, so the late ones are scheduled meanwhile.
struct End {
  Memory& m;
  uint32_t seq;
  bool waits;  // false: a step that does not wait, to see that the check can fail
  bool wait_started() {
    if (!waits) return true;
    for (int i = 0; i < kStepExtra; ++i) {
      if (m.late.count(i)) m.run_extra(i);
      if (m.started[i] != seq) return false;
    }
    return true;
  }
};

// n_between of the late workgroups start between the position's store and the
// sequence number's, the rest after both.  Returns how many took a role that
// the step's own position does not give.
static int run(int pos, int max_seq, bool advance, int n_late, int n_between, bool waits) {
  Memory m;
  m.pos = pos;
  m.max_seq = max_seq;
  const uint32_t seq = m.seq + 1;
  const int32_t c = pos < 0 ? 0 : (pos >= max_seq ? max_seq - 1 : pos);
  const bool is_long = step_long(c);
  for (int i = 0; i < kStepExtra; ++i) m.late.insert(i);
  // a long step needs all of them: none can be late
  const int on_time = is_long ? kStepExtra : kStepExtra - n_late;
  for (int i = 0; i < on_time; ++i) m.run_extra(i);
  End end{m, seq, waits};
  if (!step_may_end(end, pos, max_seq, advance)) return kStepExtra;
  if (advance && pos + 1 < max_seq) m.pos = pos + 1;
  for (int k = 0; k < n_between && !m.late.empty(); ++k) m.run_extra(*m.late.begin());
  m.seq = seq;
  while (!m.late.empty()) m.run_extra(*m.late.begin());
  int wrong = 0;
  for (bool r : m.took_role) wrong += r != is_long;
  return wrong;
}

// The device holds the first `resident` workgroups of the launch: whether the
// mark is there, and whether every workgroup with a role is.
static bool check_mark(int pos, int resident) {
  bool marked = false;
  int roles = 0, running = 0;
  for (int wg = 0; wg < kStepGrid; ++wg) {
    const bool role = wg < kStepWgs || step_long(pos);
    roles += role;
    if (wg >= resident) continue;
    running += role;
    if (wg == step_last_wg(step_long(pos))) marked = true;
  }
  if (marked != (running == roles)) {
    std::printf("pos=%d: %d of the launch resident, %d of %d with a role, marked %d\n", pos,
                resident, running, roles, marked);
    return false;
  }
  return true;
}

// A step at any position of a cache has the workgroups of its roles, and waits
// for late ones only where they are launched.
static bool check_grid(int max_seq) {
  for (int pos = 0; pos < max_seq; ++pos)
    if (step_last_wg(step_long(pos)) >= step_grid(max_seq) ||
        (step_crosses(pos, max_seq, true) && step_grid(max_seq) != kStepGrid)) {
      std::printf("pos=%d max_seq=%d: grid of %d\n", pos, max_seq, step_grid(max_seq));
      return false;
    }
  return step_grid(max_seq) == (step_long(max_seq - 1) ? kStepGrid : kStepWgs);
}

int main() {
  for (int max_seq : {1, kAttnShortCtx - 1, kAttnShortCtx, kAttnShortCtx + 1, 20000})
    if (!check_grid(max_seq)) return 1;
  for (int pos : {0, kAttnShortCtx - 1, kAttnShortCtx, 8 * kAttnShortCtx})
    for (int resident = 0; resident <= kStepGrid; ++resident)
      if (!check_mark(pos, resident)) return 1;
  const int s = kAttnShortCtx;
  const int positions[] = {-5, 0, 1, s - 2, s - 1, s, s + 1, 3 * s, 3 * s + 7};
  const int caches[] = {1, s - 1, s, s + 1, s + 2, 3 * s + 8};
  long cases = 0;
  for (int max_seq : caches)
    for (int pos : positions)
      for (int advance = 0; advance < 2; ++advance)
        for (int late : {0, 1, 7, kStepExtra})
          for (int between : {0, 1, kStepExtra}) {
            const int wrong = run(pos, max_seq, advance != 0, late, between, true);
            if (wrong) {
              std::printf("pos=%d max_seq=%d advance=%d late=%d between=%d: %d wrong roles\n", pos,
                          max_seq, advance, late, between, wrong);
              return 1;
            }
            ++cases;
          }
  // without the wait the crossing step's late workgroups take a role
  if (run(s - 1, s + 2, true, 3, 0, false) != 3 || run(s - 1, s + 2, true, 3, 2, false) != 3) {
    std::printf("the check does not see a step that does not wait\n");
    return 1;
  }
  std::printf("ok %ld cases\n", cases);
  return 0;
}
