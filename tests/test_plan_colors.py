"""CPU check of the colours of a batch's elements (csrc/msod_plan.h), on which
the freedom from races of the coloured column kernels rests: boxes of every
order, elements in random order, a partial last batch, a full batch of 64 whose
elements share one node, more batches than one thread colours, and a planted
clash that the checker has to see."""
import os
import shutil
import subprocess

import numpy as np
import pytest

import minisod2d_amd as m

HERE = os.path.dirname(os.path.abspath(__file__))
SRC = os.path.join(HERE, "plan_color_check.cpp")
CSRC = os.path.join(os.path.dirname(HERE), "minisod2d_amd", "csrc")
BIN = os.path.join(HERE, "_build", "plan_color_check")
EPB = {1: 64, 2: 28, 3: 16, 4: 10, 5: 7, 6: 5, 7: 4, 8: 3}  # ColShape<P>::EPB in csrc/msod_columns.h


@pytest.fixture(scope="module")
def checker():
    cxx = shutil.which("g++")
    if cxx is None:
        pytest.skip("g++ not available")
    newest = max(os.path.getmtime(SRC), os.path.getmtime(os.path.join(CSRC, "msod_plan.h")))
    if not os.path.exists(BIN) or os.path.getmtime(BIN) < newest:
        os.makedirs(os.path.dirname(BIN), exist_ok=True)
        subprocess.run([cxx, "-std=c++17", "-O1", "-g", "-pthread", "-fsanitize=address,undefined",
                        "-fno-omit-frame-pointer", "-I", CSRC, SRC, "-o", BIN], check=True)
    return BIN


def rounds(checker, tmp_path, connec, npoin, p):
    nelem, nn = connec.shape
    path = str(tmp_path / "mesh.bin")
    with open(path, "wb") as fh:
        np.array([nelem, npoin], np.int64).tofile(fh)
        np.array([nn, EPB[p]], np.int32).tofile(fh)
        (m.hex_tables(p).invAtoIJK.ravel(order="F") - 1).astype(np.int32).tofile(fh)
        np.asfortranarray(connec, dtype=np.int32).ravel(order="F").tofile(fh)
        np.array([p + 1], np.int32).tofile(fh)
    env = dict(os.environ, ASAN_OPTIONS="detect_leaks=0:abort_on_error=0", UBSAN_OPTIONS="halt_on_error=1")
    r = subprocess.run([checker, path], capture_output=True, text=True, env=env)
    assert r.returncode == 0 and r.stdout.startswith("OK rounds="), r.stdout + r.stderr
    return int(r.stdout.split("=")[1])


@pytest.mark.parametrize("shuffled", [False, True])
@pytest.mark.parametrize("p", range(1, 9))
def test_boxes(checker, tmp_path, p, shuffled):
    n = {1: 9, 2: 7, 3: 5, 4: 4, 5: 4, 6: 3, 7: 3, 8: 2}[p]
    prob = m.box_problem(n, p, nz=n + 1)
    connec = prob.connec
    if shuffled:
        connec = connec[np.random.default_rng(p).permutation(prob.nelem)[: prob.nelem - 1]]
    assert 1 <= rounds(checker, tmp_path, connec, prob.npoin, p) <= EPB[p]


def test_a_row_takes_two_rounds(checker, tmp_path):
    prob = m.box_problem(EPB[4], 4, ny=1, nz=1)
    assert rounds(checker, tmp_path, prob.connec, prob.npoin, 4) == 2


def test_64_elements_around_one_node(checker, tmp_path):
    """The most colours that a batch can take, those of its 64-bit masks."""
    nelem = 65  # and a batch of one
    connec = (2 + np.arange(nelem * 8).reshape(nelem, 8)).astype(np.int32)
    connec[:, 3] = 1
    assert rounds(checker, tmp_path, connec, nelem * 8 + 1, 1) == 64


def test_most_colours_in_one_threads_share(checker, tmp_path):
    """5000 batches, coloured by several threads, one of which meets the most colours."""
    nelem = 3 * 5000
    connec = (2 + np.arange(nelem * 729).reshape(nelem, 729)).astype(np.int32)
    connec[9000:9003, 0] = 1
    assert rounds(checker, tmp_path, connec, nelem * 729 + 1, 8) == 3


def test_the_checker_sees_a_clash(tmp_path):
    """The check itself, with the colours all set to one after the plan is built."""
    cxx = shutil.which("g++")
    if cxx is None:
        pytest.skip("g++ not available")
    src = open(SRC).read().replace("if (int st = check(P", "P.ecol.assign(nelem, 0); P.rounds = 1;\n    if (int st = check(P")
    path, exe = tmp_path / "broken.cpp", str(tmp_path / "broken")
    path.write_text(src)
    subprocess.run([cxx, "-std=c++17", "-O1", "-pthread", "-I", CSRC, str(path), "-o", exe], check=True)
    prob = m.box_problem(EPB[4], 4, ny=1, nz=1)
    with pytest.raises(AssertionError, match="share a node"):
        rounds(exe, tmp_path, prob.connec, prob.npoin, 4)


@pytest.mark.parametrize("shuffled", [False, True])
@pytest.mark.parametrize("p", range(1, 9))
def test_whole_plan_with_the_column_batches(checker, tmp_path, p, shuffled):
    """plan_check.cpp's invariants (tests/test_plan.py) at the column kernels' batch sizes."""
    exe = os.path.join(HERE, "_build", "plan_check_columns")
    src = os.path.join(HERE, "plan_check.cpp")
    if not os.path.exists(exe) or os.path.getmtime(exe) < max(os.path.getmtime(src),
                                                              os.path.getmtime(os.path.join(CSRC, "msod_plan.h"))):
        subprocess.run([shutil.which("g++"), "-std=c++17", "-O1", "-g", "-pthread", "-fsanitize=address,undefined",
                        "-fno-omit-frame-pointer", "-I", CSRC, src, "-o", exe], check=True)
    n = {1: 9, 2: 7, 3: 5, 4: 4, 5: 4, 6: 3, 7: 3, 8: 2}[p]
    prob = m.box_problem(n, p, nz=n + 1)
    connec = prob.connec
    if shuffled:  # and the nodes of three elements unreferenced
        connec = connec[np.random.default_rng(p).permutation(prob.nelem)[: prob.nelem - 3]]
    path = str(tmp_path / "mesh.bin")
    with open(path, "wb") as fh:
        np.array([connec.shape[0], prob.npoin], np.int64).tofile(fh)
        np.array([connec.shape[1], EPB[p]], np.int32).tofile(fh)
        (prob.tables.invAtoIJK.ravel(order="F") - 1).astype(np.int32).tofile(fh)
        np.asfortranarray(connec, dtype=np.int32).ravel(order="F").tofile(fh)
    r = subprocess.run([exe, path], capture_output=True, text=True, env=dict(os.environ, ASAN_OPTIONS="detect_leaks=0"))
    assert r.returncode == 0 and r.stdout.startswith("OK ncolors="), r.stdout + r.stderr
