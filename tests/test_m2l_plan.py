"""The plan of the FP64 M2L by tensor slot: the library's own planGamma, compiled for the CPU,
for every order on the smallest shape that holds it.  Every product (gamma, beta <= gamma)
sits in one step of one cell, and every alpha's segments hold exactly its products."""
import os
import re
import subprocess

from conftest import ROOT

MAIN = r"""
int main() {
  for (int p = 0; p <= 8; p++) {
    const int *s = kGamma[p <= 3 ? 0 : p - 3], L = s[1], W = s[2], cells = 64 * W, slotZ = NMOM(s[0]), nm = NMOM(p);
    HostGamma H;
    if (!planGamma(p, L, W, slotZ, H)) return printf("order %d: no plan\n", p), 1;
    std::vector<int> mi(3 * nm);
    for (int d = 0, g = 0; d <= p; d++)
      for (int i1 = 0; i1 <= d; i1++)
        for (int i2 = 0; i2 <= d - i1; i2++, g++) mi[3 * g] = i1, mi[3 * g + 1] = i2, mi[3 * g + 2] = d - i1 - i2;
    std::vector<int> seen(nm * nm), alphaOf(L * cells + 1, -1);
    for (int i = 0; i < cells; i++)
      for (int l = 0; l < L; l++) {
        const int g = H.gamma[i], b = H.beta[l * cells + i];
        if (b == slotZ) continue;
        int a[3];
        for (int k = 0; k < 3; k++)
          if ((a[k] = mi[3 * g + k] - mi[3 * b + k]) < 0) return printf("order %d: beta beyond gamma\n", p), 2;
        seen[g * nm + b]++;
        alphaOf[l * cells + i] = idx3of(a[0], a[1], a[2]);
      }
    long products = 0;
    for (int g = 0; g < nm; g++)
      for (int b = 0; b < nm; b++) {
        const int want = mi[3 * b] <= mi[3 * g] && mi[3 * b + 1] <= mi[3 * g + 1] && mi[3 * b + 2] <= mi[3 * g + 2];
        if (seen[g * nm + b] != want) return printf("order %d: product %d %d is there %d times\n", p, g, b, seen[g * nm + b]), 3;
        products += want;
      }
    if ((int)H.alphaSeg.size() != nm + 1 || (int)H.ent.size() != GAMMA_SEG * H.alphaSeg[nm]) return 4;
    for (int a = 0; a < nm; a++)
      for (int e = GAMMA_SEG * H.alphaSeg[a]; e < GAMMA_SEG * H.alphaSeg[a + 1]; e++) {
        if (H.ent[e] == L * cells) continue;   // the zero entry
        if (alphaOf[H.ent[e]] != a) return printf("order %d: entry of another alpha\n", p), 5;
        alphaOf[H.ent[e]] = -1;
        products--;
      }
    if (products) return printf("order %d: %ld products are in no segment\n", p, products), 6;
  }
  return 0;
}
"""


def test_plan(tmp_path):
    src = open(os.path.join(ROOT, "cuda-fabipb_amd", "csrc", "fabipb_hip.hip")).read()

    def part(a, b):
        i = src.index(a)
        return src[i:src.index(b, i) + len(b)]

    code = ["#include <algorithm>\n#include <cstdio>\n#include <cstring>\n#include <vector>\n"]
    code += [re.search(r"#define %s.*\n" % n, src)[0] for n in (r"NMOM\(p\)", "GAMMA_SEG")]
    code += [part("static int idx3of(", "\n}\n"), part("static constexpr int kGamma", "};\n"),
             part("struct HostGamma {", "\n};\n"), part("static bool planGamma(", "\n}\n"), MAIN]
    (tmp_path / "t.cpp").write_text("".join(code))
    subprocess.check_call(["g++", "-std=c++17", "-O1", "-o", str(tmp_path / "t"), str(tmp_path / "t.cpp")])
    p = subprocess.run([str(tmp_path / "t")], capture_output=True, text=True)
    assert p.returncode == 0, p.stdout
