// Step geometry of the prefill tiles, and when they stage page-table entries
// into LDS.  Plain constants and arithmetic, so that a host program can replay
// the staging order.
#pragma once

namespace pal {

constexpr int kKeys = 32;              // keys per step
constexpr int kNBuf = 4;               // LDS step buffers, of K and of V
constexpr int kLeadK = 5, kLeadV = 3;  // prefill_tile: iteration st copies K of step st + kLeadK and V of step st + kLeadV
constexpr int kLeadHalf = 3;           // half_tile: iteration st copies K and V of step st + kLeadHalf
constexpr int kPidChunk = 512;         // page ids staged per chunk; two chunks live in LDS

constexpr int pid_slot(int e) { return e & (2 * kPidChunk - 1); }           // LDS slot of page-table entry e
constexpr int pid_chunk_steps(int tp) { return kPidChunk * tp / kKeys; }    // steps of a chunk (page size tp)

// Chunks 0 and 1 are staged before the first step.  Chunk q + 1 overwrites
// chunk q - 1, whose entries are read until V step st takes its pages' scales
// (fp8 pools; the K scales are read one step ahead of it, the page ids up to
// kLeadK ahead).  So it is staged at the end of the iteration whose own step is
// the first of chunk q: at that iteration's barrier every wavefront had read
// the scales of the last step of chunk q - 1.  Nothing reads chunk q + 1 before
// the iterations' barriers have published it: a chunk has 256 steps or more,
// the copies run 5 ahead.
//
// The chunk to stage at the end of iteration st of a tile that reads n_pid
// entries (0: none).
constexpr int pid_chunk_to_stage(int st, int tp, int n_pid) {
  const int steps = pid_chunk_steps(tp);
  const int q = st / steps;
  return st > 0 && st % steps == 0 && (q + 1) * kPidChunk < n_pid ? q + 1 : 0;
}
// The next iteration, from st on, that may stage a chunk.
constexpr int pid_next_staging(int st, int tp) {
  const int steps = pid_chunk_steps(tp);
  return st <= 0 ? steps : (st + steps - 1) / steps * steps;
}

}  // namespace pal
