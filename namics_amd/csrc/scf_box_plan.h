// The launches of a 3-gradient tile chain (scf_box3d.h) as data: which rows a
// launch takes, from which end-point slot it starts and which slots it stores.
// Plain C++, so that the schedule can be walked without a GPU.
#pragma once

#include <algorithm>
#include <vector>

namespace nscf {

constexpr int kBoxH = 4;  // contour steps of a launch at most

// End-point storage of the grid path.  With every row kept (ckpt <= 1) row
// s of the forward recursion is Gf slot s.  With checkpoints every K rows
// (the reference's save_memory, src/molecule.cpp:174-191, on a uniform grid)
// rows 0, K, 2K, ... keep the first ceil(N/K) slots, the other rows of a
// segment share the K - 1 slots after them, and the backward pass
// recomputes a segment's rows from its checkpoint just before it composes
// them, with the forward step itself, so the result does not depend on the
// storage.  The last segment's rows are still there from the forward pass.
struct RowSlots {
  int K;       // checkpoint interval (<= 1: every row)
  int nck;     // checkpoint slots
  int operator()(int r) const { return K <= 1 ? r : (r % K == 0 ? r / K : nck + r % K - 1); }
};

// Forward steps of a launch.
struct BoxForward {
  int n;            // steps
  int src;          // slot of the input row; -1: the segment weight seg0
  int seg0, slot0;  // slot0 >= 0: keep the input row there
  int slot[kBoxH];  // end-point slot of each step's row, -1: not kept
  int seg[kBoxH];
};
// Backward steps of a launch, after the forward steps that bring their rows.
struct BoxRun {
  BoxForward f;
  int n;              // steps
  int src;            // row of Gb to start from; -1: the segment weight seg0
  int seg0, mm0;      // segment and density of the first row
  int slot0;          // >= 0: compose the first row with it
  int dst;            // row of Gb for the last row
  int slot[kBoxH];    // end-point slot of each step's row
  int seg[kBoxH], mm[kBoxH];
};

// A chain of N >= 2 rows with checkpoints every K rows (K <= 1: every row).
struct BoxSchedule {
  int N, K;
  RowSlots loc;
  std::vector<int> seg, mm;  // segment and density of every row
  BoxSchedule(int rows, int ckpt) : N(rows), K(ckpt), loc{ckpt, ckpt > 1 ? (rows + ckpt - 1) / ckpt : rows} {}

  // Rows r0+1 .. r1 of the forward recursion from row r0; the last steps are
  // left in `tail` for the backward launch that follows.  Of the first pass
  // (`pass`) only the rows that outlive it are kept, and the one that the
  // next launch starts from.
  //
  // A launch may not store the slot that it starts from: its workgroups load
  // their halos there while others have already stored.  Rows of one buffer
  // slot are K apart, so with K > kBoxH none are in one launch; with smaller
  // K the first pass's launches end at checkpoints (whose slots are their
  // own), and the recomputation stays within one segment.
  template <typename Launch>
  int forward(int r0, int r1, bool pass, BoxForward &tail, Launch launch) const {
    const int most = pass && K > 1 && K < kBoxH ? kBoxH / K * K : kBoxH;
    for (int r = r0; r < r1;) {
      BoxForward a{};
      a.n = std::min(most, r1 - r);
      a.src = r == 0 ? -1 : loc(r);
      a.seg0 = seg[0];
      a.slot0 = r == 0 ? loc(0) : -1;
      for (int s = 0; s < a.n; s++) {
        const int q = r + 1 + s;
        const bool keep = !pass || K <= 1 || q % K == 0 || q / K == (N - 1) / K || s == a.n - 1;
        a.slot[s] = keep ? loc(q) : -1;
        a.seg[s] = seg[q];
      }
      r += a.n;
      if (r == r1) {
        tail = a;
        break;
      }
      const int e = launch(&a, (const BoxRun *)nullptr);
      if (e != 0) return e;
    }
    return 0;
  }
  // The whole chain: launch(forward, nullptr) or launch(nullptr, run), which
  // returns 0 or an error; gn() launches the sum over row N - 1 (slot
  // loc(N - 1)) while it is held.
  template <typename Launch, typename Gn>
  int run(Launch launch, Gn gn) const {
    int held = K > 1 ? (N - 1) / K : 0;  // the segment whose rows the buffer holds
    int gb = 0;
    for (int s = N - 1; s >= 0;) {
      const bool first = s == N - 1;
      BoxRun a{};
      a.src = first ? -1 : gb;
      a.seg0 = seg[N - 1];
      a.mm0 = mm[N - 1];
      a.slot0 = first ? loc(N - 1) : -1;
      a.dst = gb = 1 - gb;
      int e = 0;
      if (first) {
        e = forward(0, N - 1, true, a.f, launch);
        s--;
      } else if (K > 1 && s % K != 0 && s / K != held) {
        held = s / K;
        e = forward(held * K, held * K + K - 1, false, a.f, launch);
      }
      if (e != 0) return e;
      // rows as long as they are checkpoints or of the segment held
      for (; a.n < kBoxH && s >= 0 && (K <= 1 || s % K == 0 || s / K == held); s--, a.n++) {
        a.slot[a.n] = loc(s);
        a.seg[a.n] = seg[s];
        a.mm[a.n] = mm[s];
      }
      e = launch((const BoxForward *)nullptr, (const BoxRun *)&a);
      if (e != 0) return e;
      if (first) gn();
    }
    return 0;
  }
};

}  // namespace nscf
