"""bwd_lean_grid (csrc/moc_mfma_launch.h), compiled for the host and run: no range
of the stream backward takes more 32-row steps than its share of the rows needs."""
import random
import subprocess
from pathlib import Path

import pytest

from tests.test_index_model import cdiv, lean_grid, sb_range

ROOT = Path(__file__).resolve().parents[1]
HIPCC = Path("/opt/rocm/bin/hipcc")
SOURCE = """
#include <cstdio>
#include "moc_mfma_launch.h"
int main() {
  long long N, gx, D;
  int S, KC, bf, n_cu;
  while (scanf("%lld %lld %lld %d %d %d %d", &N, &gx, &D, &S, &KC, &bf, &n_cu) == 7) {
    const auto g = moc::mfma::bwd_lean_grid(N, gx, D, S, KC, bf != 0, n_cu);
    printf("%u %u %d %d %d\\n", g.gx, g.gy, g.gy1, g.n_old, g.n_total);
  }
}
"""


def shapes():
    rng = random.Random(5)
    for bf, KC, S in [(1, 1, 2), (1, 1, 3), (1, 1, 4), (1, 1, 5), (1, 1, 8), (1, 2, 2), (1, 2, 4),
                      (1, 2, 7), (0, 1, 2), (0, 1, 8), (0, 2, 2), (0, 2, 5)]:
        own = 33 - S
        lengths = [1, own - 1, own, own + 1, 32, 33, 128, 600, 2000, 16384, 512 * own, 512 * own - 5,
                   65536, *(int(2 ** rng.uniform(0, 17)) for _ in range(12))]
        for N in lengths:
            for D in (2, 128, 130, 520, 2048, 4096, 1 << 20):
                for n_cu in (0, 16, 256):
                    yield N, cdiv(D, 128), D, S, KC, bf, n_cu


@pytest.fixture(scope="module")
def compiled(tmp_path_factory):
    if not HIPCC.exists():
        pytest.skip("no hipcc")
    d = tmp_path_factory.mktemp("grid")
    (d / "grid.hip").write_text(SOURCE)
    subprocess.check_call([str(HIPCC), "--offload-arch=gfx950", "--offload-host-only", "-O1", "-std=c++17",
                           f"-I{ROOT / 'mixture-of-convolutions_amd' / 'csrc'}", str(d / "grid.hip"),
                           "-o", str(d / "grid")])
    cases = list(shapes())
    out = subprocess.run([str(d / "grid")], input="\n".join(" ".join(map(str, c)) for c in cases),
                         capture_output=True, text=True, check=True).stdout
    rows = [dict(zip(("gx", "gy", "gy1", "n_old", "n_total"), map(int, ln.split())))
            for ln in out.splitlines()]
    return list(zip(cases, rows, strict=True))


def test_ranges_take_their_share_of_the_steps(compiled):
    tiers = 0
    for (N, gx, D, S, KC, bf, n_cu), g in compiled:
        own = 33 - S
        steps = [hi - lo for lo, hi in (sb_range(by, g) for by in range(g["gy"]))]
        assert min(steps) >= 1 and sum(steps) == g["n_total"]
        assert 32 * sum(steps) - g["gy"] * (S - 1) >= N  # every row owned
        if g["gy1"] < g["gy"]:
            tiers += 1
        else:  # equal shares of the own rows among the workgroups of one round (two per CU or one)
            four = bf and S <= 4 and KC == 1
            share = cdiv(cdiv(N, own), max((512 if four else n_cu or 256) // gx, 1))
            assert max(steps) <= share, (N, gx, S, KC, bf, n_cu, g)
        # a range's rows are reached by the 32-bit offsets of its buffers
        assert (32 * max(steps) + S - 1) * D * (2 if bf else 4) < 1 << 31
    assert tiers >= 3


def test_index_model_has_the_same_grid(compiled):
    for (N, gx, D, S, KC, bf, n_cu), g in compiled:
        m = lean_grid(N, gx, D, S, KC, bf, n_cu)
        assert {k: m[k] for k in g} == g, (N, gx, D, S, KC, bf, n_cu)
