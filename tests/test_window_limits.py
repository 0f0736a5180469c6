"""The largest chains that the window kernels take (win_fits), computed by the
rule's own host code: no GPU needed."""
import importlib.util
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
PROG = """
#include "window_kernels.hpp"
#include <cstdio>
int main()
{
    int dim, tsize, ell, lc;
    while (std::scanf("%d %d %d %d", &dim, &tsize, &ell, &lc) == 4) {
        int n = 0;
        while (n < 4096 && pimc::win_fits(n + 1, ell, lc, dim, tsize)) ++n;
        std::printf("%d\\n", n);
    }
}
"""
# (dim, bytes of a coordinate, ell, slices of a centre-of-mass window): chains up to this N have run on the
# window kernels since they came, four to six times as fast as on the whole-chain kernel
LIMITS = {(1, 4, 2, 8): 2048, (1, 4, 4, 8): 2028, (1, 4, 8, 8): 1448, (1, 4, 16, 8): 920, (1, 4, 32, 8): 532,
          (1, 8, 2, 8): 1278, (1, 8, 4, 8): 1267, (1, 8, 8, 8): 843, (1, 8, 16, 8): 507, (1, 8, 32, 8): 281,
          (2, 4, 2, 8): 1352, (2, 4, 4, 8): 1352, (2, 4, 8, 8): 914, (2, 4, 16, 8): 529, (2, 4, 32, 8): 287,
          (2, 8, 2, 8): 777, (2, 8, 4, 8): 777, (2, 8, 8, 8): 504, (2, 8, 16, 8): 279, (2, 8, 32, 8): 148,
          (2, 4, 8, 100): 188, (1, 8, 8, 199): 97}


def test_largest_window_chains(tmp_path):
    spec = importlib.util.spec_from_file_location("pimc_build", os.path.join(ROOT, "pimc.jl_amd", "build.py"))
    build = importlib.util.module_from_spec(spec)
    spec.loader.exec_module(build)
    try:
        cc = build.hipcc()
    except RuntimeError:
        pytest.skip("no hipcc")
    src, exe = tmp_path / "limits.hip", tmp_path / "limits"
    src.write_text(PROG)
    subprocess.run([cc, "--offload-arch=gfx950", "-std=c++17", "-w", "-I", build.CSRC, str(src), "-o", str(exe)], check=True)
    out = subprocess.run([str(exe)], input="\n".join(" ".join(map(str, k)) for k in LIMITS), capture_output=True, text=True,
                         check=True)
    got = dict(zip(LIMITS, map(int, out.stdout.split())))
    assert not {k: (got[k], n) for k, n in LIMITS.items() if got[k] < n}
