"""The autotuner's choice of tile counts: no installed table makes a size slower than the default,
the even share of the tiles."""
import os
import subprocess

import numpy as np
import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(os.path.dirname(HERE), "dftbplus_amd", "csrc")
OPTIONS = (2, 4, 8, 16)


@pytest.fixture(scope="module")
def choose(tmp_path_factory):
    exe = str(tmp_path_factory.mktemp("symv") / "model")
    subprocess.run(["g++", "-O2", "-std=c++17", "-I", CSRC, "-o", exe,
                    os.path.join(HERE, "symv_table_model.cpp")], check=True)

    def run(t):
        text = "%d\n%s\n" % (t.shape[1], " ".join(repr(float(x)) for x in t.ravel()))
        out = subprocess.run([exe], input=text, capture_output=True, text=True, check=True).stdout
        rows = [np.array(line.split(), dtype=int).reshape(-1, 2) for line in out.split("\n")[:2]]
        return [[tuple(r) for r in x] for x in rows]
    return run


def _at(rows, bucket):
    return [v for m0, v in rows if m0 <= 256 * bucket][-1]


def test_even_share_stays_where_no_option_gains(choose):
    # an option ahead by 10 %, by 1 %, behind
    t = np.array([[1.0, 1.0, 1.0], [0.9, 0.99, 1.2], [1.0, 1.1, 1.2], [1.3, 1.1, 1.2], [1.0, 1.0, 0.8]])
    fixed, install = choose(t)
    assert fixed == [(0, 4), (512, 2)]
    assert install == [(0, 4), (256, 0)]


@pytest.mark.parametrize("seed", range(8))
def test_never_slower_than_the_default(choose, seed):
    rng = np.random.default_rng(seed)
    nb = int(rng.integers(1, 64))
    t = rng.uniform(0.9, 1.1, (5, nb))
    fixed, install = choose(t)
    for b in range(nb):
        v = _at(install, b)
        assert v in (0, _at(fixed, b))
        took = t[4, b] if v == 0 else t[OPTIONS.index(v), b]
        assert took <= t[4, b]
        assert (v != 0) == (t[OPTIONS.index(_at(fixed, b)), b] < 0.98 * t[4, b])
        assert t[OPTIONS.index(_at(fixed, b)), b] <= t[:4, b].min() / 0.98 * (1 + 1e-12)
    assert all(install[k][1] != install[k + 1][1] for k in range(len(install) - 1))
