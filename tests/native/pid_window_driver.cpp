// Replays, for prefill tiles of every interesting length, which page-table
// entries lie in LDS when an iteration reads them (csrc/pid_window.h).
//
// Wavefronts of a workgroup are at most one barrier apart, so inside iteration
// st one wavefront may read before and another after the chunk that st stages
// is stored: every read has to find its entry in both states.
#include <cstdio>
#include <initializer_list>
#include <vector>

#include "pid_window.h"

using namespace pal;

namespace {

constexpr int kSlots = 2 * kPidChunk;

struct Window {
  std::vector<int> slot = std::vector<int>(kSlots, -1);
  void stage(int chunk, int n_pid) {
    for (int e = chunk * kPidChunk; e < (chunk + 1) * kPidChunk && e < n_pid; ++e) slot[pid_slot(e)] = e;
  }
};

// the step's entries below n_pid all in place?
bool holds(const Window& w, int step, int tp, int n_pid) {
  for (int k = 0; k < (tp == 16 ? 2 : 1); ++k) {
    const int e = step * kKeys / tp + k;
    if (e < n_pid && w.slot[pid_slot(e)] != e) return false;
  }
  return true;
}

int check_tile(bool half, int tp, int keys) {
  const int n_pid = (keys + tp - 1) / tp, nsteps = (keys + kKeys - 1) / kKeys;
  const int lead_ids = half ? kLeadHalf : kLeadK;
  Window w;
  w.stage(0, n_pid);
  w.stage(1, n_pid);
  int next = pid_next_staging(0, tp);
  for (int st = 0; st < nsteps; ++st) {
    const Window before = w;
    const int chunk = pid_chunk_to_stage(st, tp, n_pid);
    if (st > next) next = pid_next_staging(st, tp);
    if (chunk && st != next) {
      std::printf("half=%d tp=%d keys=%d: iteration %d stages, next_staging says %d\n", half, tp, keys, st, next);
      return 1;
    }
    if (chunk) w.stage(chunk, n_pid);
    // page ids of the steps copied, V scales of step st, K scales of step st + 1
    for (int step : {st + lead_ids, st + kLeadV, st, st + 1}) {
      if (step >= nsteps) continue;
      if (!holds(before, step, tp, n_pid) || !holds(w, step, tp, n_pid)) {
        std::printf("half=%d tp=%d keys=%d: iteration %d reads entries of step %d that are not in place\n", half, tp, keys,
                    st, step);
        return 1;
      }
    }
  }
  return 0;
}

}  // namespace

int main() {
  int tiles = 0;
  for (bool half : {false, true})
    for (int tp : {16, 32})
      for (int chunks = 0; chunks <= 7; ++chunks)
        for (int d : {-2 * kKeys - 1, -kKeys, -tp, -1, 0, 1, tp, tp + 1, kKeys, 3 * kKeys, 5 * kKeys + 7, 6 * kKeys}) {
          const int keys = chunks * kPidChunk * tp + d;
          if (keys <= 0) continue;
          if (check_tile(half, tp, keys)) return 1;
          ++tiles;
        }
  std::printf("%d tiles: every entry in place\n", tiles);
  return 0;
}
