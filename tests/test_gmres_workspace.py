"""Growth of the GMRES workspace when an allocation fails: kernels store into these buffers
by address, so a failed growth must not pass as ready for a later, shorter solve, and must
leave no freed pointer behind.  The library's own function, compiled for the CPU against an
allocator whose k-th call fails."""
import os
import subprocess

from conftest import ROOT

STUB = r"""
#include <cstdio>
#include <cstdlib>
#include <map>
typedef int hipError_t;
typedef void *hipEvent_t;
enum { hipSuccess = 0, hipHostMallocDefault = 0, hipHostMallocCoherent = 1, hipEventDisableTiming = 2 };
#define RED_BLOCKS 256
#define HCK(x) do { if ((x) != hipSuccess) return 0; } while (0)
static std::map<void *, size_t> live;
static int calls, failAt, bad;
static int take(void **p, size_t b) {
  if (++calls == failAt) return 1;   // the pointer is left as it was
  live[*p = malloc(b)] = b;
  return 0;
}
template <class T> static int hipMalloc(T **p, size_t b) { return take((void **)p, b); }
static int hipHostMalloc(void **p, size_t b, int) { return take(p, b); }
static int hipEventCreateWithFlags(hipEvent_t *p, int) { return take(p, 8); }
static int hipFree(void *p) {
  if (!live.erase(p)) bad++;   // freed twice
  free(p);
  return 0;
}
static int hipHostFree(void *p) { return hipFree(p); }
struct fbh_ctx {
  int n = 5, gmRestart = 0, hpinLen = 0;
  double *V = nullptr, *w = nullptr, *r = nullptr, *part = nullptr, *hcol = nullptr, *ydev = nullptr, *scal = nullptr,
         *hpin = nullptr;
  hipEvent_t evDone = nullptr;
};
"""

MAIN = r"""
static int whole(const fbh_ctx &c, size_t restart) {
  auto has = [](void *p, size_t doubles) { return live.count(p) && live[p] >= 8 * doubles; };
  return has(c.V, 2 * c.n * (restart + 1)) && has(c.w, 2 * c.n) && has(c.r, 2 * c.n) && has(c.part, 2 * RED_BLOCKS) &&
         has(c.hcol, restart + 1) && has(c.ydev, restart) && has(c.hpin, restart + 1 > 4 ? restart + 1 : 4) &&
         has(c.evDone, 1);
}
int main() {
  int first = 0, grown = 0;
  for (int k = 1; k <= 12; k++)
    for (int before : {0, 10}) {
      fbh_ctx c;
      failAt = 0;
      if (before && (!ensureGmres(&c, before) || !whole(c, before))) return 1;
      calls = 0;
      failAt = k;
      const int ok = ensureGmres(&c, 20);
      (before ? grown : first) += !ok;
      if (ok && !whole(c, 20)) return printf("allocation %d after %d: not whole\n", k, before), 2;
      failAt = 0;
      for (int again : {10, 20, 5})
        if (!ensureGmres(&c, again) || !whole(c, again))
          return printf("allocation %d failed after restart %d: restart %d passes as ready\n", k, before, again), 3;
      if (bad) return printf("allocation %d after %d: freed twice\n", k, before), 4;
    }
  return first >= 8 && grown >= 4 ? 0 : (printf("%d %d\n", first, grown), 5);   // every allocation was reached
}
"""


def test_failed_growth(tmp_path):
    src = open(os.path.join(ROOT, "cuda-fabipb_amd", "csrc", "fabipb_hip.hip")).read()
    i = src.index("static int ensureGmres(fbh_ctx *c, int restart) {")
    body = src[i:src.index("\n}\n", i) + 3]
    (tmp_path / "t.cpp").write_text(STUB + body + MAIN)
    subprocess.check_call(["g++", "-std=c++17", "-O1", "-Wno-conversion", "-o", str(tmp_path / "t"), str(tmp_path / "t.cpp")])
    p = subprocess.run([str(tmp_path / "t")], capture_output=True, text=True)
    assert p.returncode == 0, p.stdout
