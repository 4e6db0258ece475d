"""The launches of edge checks (gpuprm_amd/csrc/edge_plan.h), compiled for the
host: an edge's windows hold each of its samples once, and the launches of a
window hold each rank of every edge once, within the item budget, for edges of
one sample up to 2^31 - 1."""
import os
import subprocess
import textwrap

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

SRC = textwrap.dedent(r'''
    #include "edge_plan.h"
    #include <stdio.h>
    #include <stdlib.h>
    #include <string.h>
    using namespace gprm;
    static int fail(const char* what, long long a, long long b, long long c) {
      printf("%s: %lld %lld %lld\n", what, a, b, c);
      return 1;
    }
    // every sample of an edge in one window, ascending in each; windows per
    // level, or one for all
    static int samples(int T) {
      for (int one = 0; one < 2; ++one) {
        std::vector<char> seen(T, 0);
        const int n = one ? 1 : edge_levels(T);
        long long sum = 0;
        for (int l = 0; l < n; ++l) {
          int a, b, cnt, last = -1;
          edge_window(T, l, l + 1 == n ? kLevelAll : l + 1, &a, &b, &cnt);
          if (cnt > edge_window_most(T, l + 1 == n ? kLevelAll : l + 1)) return fail("most", T, l, cnt);
          sum += cnt;
          for (int r = 0; r < cnt; ++r) {
            const int s = edge_window_sample(a, b, r);
            if (s <= last || s >= T || seen[s]) return fail("sample", T, l, r);
            seen[s] = 1;
            last = s;
          }
        }
        if (sum != T) return fail("samples", T, one, sum);
      }
      return 0;
    }
    static int plan(long long budget, int block, int N, int maxT, bool known, unsigned seed) {
      std::vector<int> T(N);
      long long total = 0;
      for (int e = 0; e < N; ++e) {
        seed = seed * 1664525u + 1013904223u;
        const int kind = seed >> 30;
        T[e] = kind == 0 ? 1 + (int)((seed >> 8) % 40u) : 1 + (int)((seed & 0x7fffffffu) % (unsigned)maxT);
        if (T[e] > maxT) T[e] = maxT;
        if (e == N / 2) T[e] = maxT;
        total += T[e];
      }
      const int levels = edge_levels(maxT);
      for (int l = 0; l < levels; ++l) {
        const int l1 = l + 1 == levels ? kLevelAll : l + 1;
        std::vector<EdgeLaunch> p;
        edge_plan_window(budget, block, N, l, l1, maxT, known ? total : -1, &p);
        std::vector<long long> got(N, 0), next(N, 0);
        for (const EdgeLaunch& x : p) {
          if (x.l0 != l || x.l1 != l1 || x.e0 >= x.e1 || x.r0 >= x.r1) return fail("launch", budget, N, maxT);
          if (x.cap <= 0 || x.cap % 64 || x.cap > std::max(budget + 63, 128LL)) return fail("cap", budget, maxT, x.cap);
          long long slots = 0;
          const long long xb = (x.e1 - x.e0 + block - 1) / block;
          const int slice = edge_slice(x.r1 - x.r0, xb), ny = edge_slices(x.r1 - x.r0, xb);
          if (slice < 16 || slice % 16 || xb * ny > std::max(kSliceBlocks, 16 * xb) || ny > 65535) return fail("slice", slice, ny, xb);
          std::vector<long long> packed(xb * ny, 0);  // as the compaction packs a block's runs
          for (int e = x.e0; e < x.e1; ++e) {
            int a, b, cnt;
            edge_window(T[e], l, l1, &a, &b, &cnt);
            long long mine = 0;
            for (int y = 0; y < ny; ++y) {
              const int r0 = x.r0 + y * slice, r1 = r0 + std::min(slice, x.r1 - r0);
              const int run = std::max(std::min(cnt, r1) - r0, 0);
              if (r1 <= r0) return fail("empty slice", y, ny, slice);
              if (run == 0) break;
              mine += run;
              if (run <= kRunShort) packed[y * xb + (e - x.e0) / block] += run;
              else slots += edge_run_slots(run);
            }
            if (mine > 0 && next[e] != x.r0) return fail("ranks", e, x.r0, next[e]);
            if (mine > 0) next[e] = x.r1;
            got[e] += mine;
          }
          for (long long n : packed) slots += (n + 15) / 16 * 16;
          if (slots > x.cap) return fail("slots", slots, x.cap, maxT);
        }
        for (int e = 0; e < N; ++e) {
          int a, b, cnt;
          edge_window(T[e], l, l1, &a, &b, &cnt);
          if (got[e] != cnt) return fail("covered", e, got[e], cnt);
        }
      }
      return 0;
    }
    int main(int argc, char** argv) {
      if (!strcmp(argv[1], "samples")) {
        for (int T = 1; T <= 3000; ++T)
          if (samples(T)) return 1;
        for (int T : {4095, 8191, 8192, 8193, 32768, 32769, 100001, 131073, 2097153, 20000003})
          if (samples(T)) return 1;
        return 0;
      }
      const int maxT = atoi(argv[2]);
      for (long long budget : {1LL << 24, 1LL << 19, 17001LL, 500LL})
        for (int block : {256, 1024})
          for (int N : {1, 2, 255, 1024, 3001}) {
            const long long parts = (long long)maxT / budget * N;
            if (parts > 3000) continue;  // as many launches
            for (int known = 0; known < 2; ++known)
              if (plan(budget, block, N, maxT, known != 0, 77u + N)) return 1;
          }
      return 0;
    }
''')


@pytest.fixture(scope="module")
def checker(tmp_path_factory):
    d = tmp_path_factory.mktemp("edge_plan")
    src = d / "edge_plan_check.cpp"
    src.write_text(SRC)
    exe = d / "edge_plan_check"
    subprocess.run(["g++", "-std=c++17", "-O2", "-fsanitize=signed-integer-overflow", "-fno-sanitize-recover", "-I",
                    os.path.join(ROOT, "gpuprm_amd", "csrc"), str(src), "-o", str(exe)], check=True)
    return str(exe)


def _run(*args):
    out = subprocess.run(args, capture_output=True, text=True)
    assert out.returncode == 0, out.stdout + out.stderr


def test_windows_hold_every_sample_once(checker):
    _run(checker, "samples")


@pytest.mark.parametrize("maxT", [1, 16, 17, 209, 256, 257, 5000, 524288, 700000, 16777215, 30000000, 1000000000,
                                  2147483632, 2147483647])
def test_launches_hold_every_rank_once_within_the_budget(checker, maxT):
    _run(checker, "plan", str(maxT))
