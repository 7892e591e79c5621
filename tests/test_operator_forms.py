"""What the operator launch accepts does not depend on the volume: the forms that k_dwf
refuses are refused on a small lattice too, where k_dwf_small would run.  No form below
reaches a kernel, so the pointers are never read."""
import os
import shutil
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
LIB = os.path.join(ROOT, "lqcd-dwf-hmc_amd", "dwf_amd")

SOURCE = r"""
#include <cstdio>
#include "dwf_kernels.h"
using namespace dwf;
int main() {
  static double mem[8];
  void* p = mem;
  int bad = 0, n = 0;
  for (int Vh : {8, 1 << 22})
    for (int prec = 0; prec < 4; ++prec)
      for (int Ls : {2, 4, 8, 10, 12, 16, 22, 24, 48})
        for (int op = 0; op < 3; ++op)
          for (int bits = 0; bits < 256; ++bits) {
            Epi e;
            const bool E = bits & 1, X = bits & 2, o2 = bits & 4, G = bits & 8, X2 = bits & 16,
                       upd = bits & 32, nrm = bits & 64, out = bits & 128;
            e.E = e.F = E ? p : nullptr;
            e.X = X ? p : nullptr;
            e.out2 = o2 ? p : nullptr;
            e.G = G ? p : nullptr;
            e.X2 = X2 ? p : nullptr;
            e.upd = upd ? p : nullptr;
            if (nrm) e.nrm_partial = e.nrm_result = mem;
            const bool mfma = E && (Ls == 12 || Ls == 16);
            const bool refuse =
                (!E && (op != K_HOP || X || o2 || G || nrm)) || (op == K_SITE && X && !o2) ||
                (op == K_HOPDAG && o2 && !X) || (G && !X) || (X2 && !o2) ||
                (upd && !(mfma && (op == K_SITE ? X : !o2))) || (!out && !upd && !(mfma && o2));
            if (!refuse) continue;
            ++n;
            const hipError_t r = launch_dwf(prec, op, out ? p : nullptr, p, p, (const int*)p, 0,
                                            Vh, Ls, e, nullptr);
            if (r != hipErrorInvalidValue && ++bad <= 10)
              std::printf("accepted: Vh %d prec %d Ls %d op %d E %d X %d out2 %d G %d X2 %d upd %d "
                          "nrm %d out %d\n", Vh, prec, Ls, op, E, X, o2, G, X2, upd, nrm, out);
          }
  std::printf("%d refused forms, %d accepted\n", n, bad);
  return bad != 0;
}
"""


def test_refused_on_every_volume(tmp_path):
    src, exe = tmp_path / "forms.hip", str(tmp_path / "forms")
    src.write_text(SOURCE)
    hipcc = os.environ.get("HIPCC", shutil.which("hipcc") or "/opt/rocm/bin/hipcc")
    subprocess.run([hipcc, "--offload-arch=gfx950", "-std=c++17", "-I",
                    os.path.join(ROOT, "lqcd-dwf-hmc_amd", "csrc"), str(src), "-L", LIB, "-ldwfhip",
                    f"-Wl,-rpath,{LIB}", "-o", exe], check=True)
    r = subprocess.run([exe], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, r.stdout
