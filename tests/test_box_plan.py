"""The launch schedule of the 3-gradient tile chains, walked on the CPU for
every chain length up to 400 and checkpoint interval up to 60: a launch stores
no slot that it starts from (its workgroups load halos there at any time),
every row it starts from or composes is the row held there, every row is
composed exactly once, and nothing lies outside the storage."""
import os
import shutil
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "namics_amd", "csrc")

WALK = r"""
#include <cstdio>
#include <cstdlib>
#include "scf_box_plan.h"
using namespace nscf;

int main() {
  for (int N = 2; N <= 400; N++)
    for (int K = 0; K <= 60; K++) {
      if (K == 1) continue;
      BoxSchedule plan(N, K);
      for (int r = 0; r < N; r++) {  // a segment and a density of its own for every row
        plan.seg.push_back(r);
        plan.mm.push_back(1000 + r);
      }
      const int slots = K <= 1 ? N : (N + K - 1) / K + std::min(K, N) - 1;
      std::vector<int> held(slots, -1), composed(N, 0);
      int gb[2] = {-1, -1};
      bool summed = false;
      auto fail = [&](const char *what) {
        printf("N %d, interval %d: %s\n", N, K, what);
        exit(1);
      };
      auto slot = [&](int s) {
        if (s < 0 || s >= slots) fail("a slot outside the storage");
        return s;
      };
      auto forward = [&](const BoxForward &a) {
        int r = 0;
        if (a.src >= 0) r = held[slot(a.src)];
        if (r < 0) fail("starts from a slot that holds no row");
        if (a.src < 0 && a.seg0 != 0) fail("starts from another row's weight");
        if (a.n < 1 || a.n > kBoxH) fail("steps of a launch");
        if (a.slot0 >= 0) held[slot(a.slot0)] = r;
        for (int i = 0; i < a.n; i++) {
          if (a.seg[i] != ++r) fail("steps to another row");
          if (a.slot[i] < 0) continue;
          if (a.slot[i] == a.src) fail("stores the slot that it starts from");
          if (a.slot0 >= 0 && a.slot[i] == a.slot0) fail("stores the slot of its input row");
          for (int j = 0; j < i; j++)
            if (a.slot[i] == a.slot[j]) fail("stores one slot twice");
          held[slot(a.slot[i])] = r;
        }
      };
      auto compose = [&](int r, int s, int seg, int mm) {
        if (r < 0 || seg != r || mm != 1000 + r) fail("composes with another row's weight or density");
        if (held[slot(s)] != r) fail("composes another row");
        composed[r]++;
      };
      plan.run(
          [&](const BoxForward *f, const BoxRun *b) {
            if (f) {
              forward(*f);
              return 0;
            }
            if (b->f.n > 0) forward(b->f);
            if (b->src == b->dst) fail("stores the backward row that it starts from");
            int r = b->src < 0 ? N - 1 : gb[b->src];
            if (b->src < 0 && b->seg0 != N - 1) fail("starts backward from another row's weight");
            if (b->slot0 >= 0) compose(r, b->slot0, b->seg0, b->mm0);
            for (int i = 0; i < b->n; i++) {
              r--;
              compose(r, b->slot[i], b->seg[i], b->mm[i]);
            }
            gb[b->dst] = r;
            return 0;
          },
          [&] {
            if (held[plan.loc(N - 1)] != N - 1) fail("the last row is not held when it is summed");
            summed = true;
          });
      if (!summed) fail("the last row is not summed");
      for (int r = 0; r < N; r++)
        if (composed[r] != 1) fail("a row is not composed once");
    }
  return 0;
}
"""


def test_schedule_of_every_length_and_interval(tmp_path):
    cxx = shutil.which("g++") or shutil.which("c++")
    if cxx is None:
        pytest.skip("no host C++ compiler")
    src = tmp_path / "walk.cpp"
    src.write_text(WALK)
    exe = tmp_path / "walk"
    subprocess.run([cxx, "-std=c++17", "-O1", "-Wall", "-Werror", "-I", CSRC, str(src), "-o", str(exe)], check=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0, r.stdout
