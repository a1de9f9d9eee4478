"""The exchange between the workgroups of the tridiagonalisation on a host model that runs the
kernel's own rules (csrc/exchange_ring.h), with any workgroup arbitrarily late: no word is emptied
before everyone who gathers its column has read it, none is read in another column, and nobody
waits for a word that never comes."""
import os
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(os.path.dirname(HERE), "dftbplus_amd", "csrc")


@pytest.fixture(scope="module")
def model(tmp_path_factory):
    exe = str(tmp_path_factory.mktemp("ring") / "model")
    subprocess.run(["g++", "-O2", "-std=c++17", "-I", CSRC, "-o", exe,
                    os.path.join(HERE, "exchange_ring_model.cpp")], check=True)
    return lambda *a: subprocess.run([exe, *map(str, a)], capture_output=True, text=True, timeout=100)


# rows, workgroups: more workgroups than rows left over (the last ones leave), as many, fewer, rows
# that do not divide evenly, one workgroup
SHAPES = [(40, 10, 32), (40, 10, 30), (37, 9, 28), (40, 8, 32), (40, 5, 32), (33, 8, 32), (7, 1, 3),
          (64, 16, 40)]


@pytest.mark.parametrize("m, P, kEnd", SHAPES)
def test_every_word_is_read_in_its_column(model, m, P, kEnd):
    r = model(m, P, kEnd, 0)
    assert r.stdout.strip() == "ok", r.stdout


@pytest.mark.parametrize("m, P, kEnd", [(40, 10, 32), (37, 9, 29)])
def test_model_sees_a_workgroup_that_gathers_its_last_column(model, m, P, kEnd):
    r = model(m, P, kEnd, 1)
    assert r.returncode == 1 and "wait for each other" in r.stdout
