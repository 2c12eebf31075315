"""The composition of row interchanges (zml_amd/csrc/perm.hpp), run on the CPU with
one host thread per GPU thread, against the interchanges applied one after the
other: pivots of every kind, repeated rows, and entries below 1, which name no
row. Such an entry (an ipiv that was cleared, or never written) has to leave its
rows alone and the composition has to end; rows and moves are whole numbers."""
import os
import random
import shutil
import subprocess

import numpy as np
import pytest

from tests.helpers import COL, ROW, P

HERE = os.path.dirname(os.path.abspath(__file__))


@pytest.fixture(scope="module")
def compose(tmp_path_factory):
    exe = str(tmp_path_factory.mktemp("compose") / "compose")
    cxx = os.environ.get("CXX") or shutil.which("g++") or shutil.which("c++")
    assert cxx, "a host C++ compiler"
    subprocess.run([cxx, "-O1", "-std=c++17", "-pthread", "-w", os.path.join(HERE, "compose_swaps_host.cpp"), "-o", exe],
                   check=True)

    def run(rows, ipiv):
        text = f"{len(rows)}\n" + "".join(f"{i} {ip}\n" for i, ip in zip(rows, ipiv))
        r = subprocess.run([exe], input=text, capture_output=True, text=True, timeout=20, check=True)
        return [tuple(map(int, line.split())) for line in r.stdout.splitlines()]
    return run


def one_by_one(rows, ipiv, m):
    at = list(range(m))
    for i, ip in zip(rows, ipiv):
        if ip >= 1:
            at[i], at[ip - 1] = at[ip - 1], at[i]
    return at


CASES = [(1, 0.0), (1, 1.0), (2, 0.5), (33, 0.0), (40, 0.3), (63, 0.9), (64, 0.0), (64, 0.4), (64, 1.0)]


@pytest.mark.parametrize("cnt,unset", CASES)
@pytest.mark.parametrize("backward", [False, True])
def test_moves_are_those_of_the_single_interchanges(compose, cnt, unset, backward):
    r = random.Random(cnt + 7 * backward + int(10 * unset))
    m = cnt + 20
    rows = list(range(cnt))[::-1 if backward else 1]
    ipiv = [r.choice([0, 0, -1, -5, -2 ** 31]) if r.random() < unset else r.randint(1, m) for _ in rows]
    if unset:
        ipiv[0] = 0
    at = list(range(m))
    moves = compose(rows, ipiv)
    assert len({d for d, _ in moves}) == len(moves)
    for dst, src in moves:
        assert 0 <= dst < m and 0 <= src < m
        at[dst] = src
    assert at == one_by_one(rows, ipiv, m)


def test_no_interchanges_at_all(compose):
    assert compose([], []) == []


@pytest.mark.gpu
@pytest.mark.parametrize("order", [ROW, COL])
def test_calls_with_cleared_pivots_end(zh, torch_cuda, order):
    """dlaswp and dgetrs with entries of ipiv below 1: those rows stay (for a cleared
    ipiv the solve is the one with the unpermuted factors)."""
    import ctypes
    torch = torch_cuda
    s = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
    n = 300
    rng = np.random.default_rng(order)
    ip = rng.integers(1, n + 1, n).astype(np.int32)
    ip[::3] = 0
    ip[7::11] = -3
    A = rng.uniform(-1, 1, (n, 5))
    want = A[one_by_one(range(n), ip, n)]
    a = torch.from_numpy(np.ascontiguousarray(A if order == ROW else A.T)).cuda()
    dp = torch.from_numpy(ip).cuda()
    assert zh.zmlhip_dlaswp(order, 5, P(a), 5 if order == ROW else n, 1, n, P(dp), 1, s) == 0
    torch.cuda.synchronize()
    got = a.cpu().numpy()
    assert np.array_equal(got if order == ROW else got.T, want)

    F = np.tril(rng.uniform(-1, 1, (n, n)) / n, -1) + np.triu(rng.uniform(-1, 1, (n, n)) / n, 1) + 2 * np.eye(n)
    B = rng.uniform(-1, 1, (n, 3))
    f = torch.from_numpy(np.ascontiguousarray(F if order == ROW else F.T)).cuda()
    none = torch.zeros(n, dtype=torch.int32, device="cuda")
    LU = (np.tril(F, -1) + np.eye(n)) @ np.triu(F)
    for nrhs in (1, 3):
        b = torch.from_numpy(np.ascontiguousarray(B[:, :nrhs] if order == ROW else B[:, :nrhs].T)).cuda()
        assert zh.zmlhip_dgetrs(order, b"N", n, nrhs, P(f), n, P(none), P(b), nrhs if order == ROW else n, s) == 0
        torch.cuda.synchronize()
        X = b.cpu().numpy()
        X = X if order == ROW else X.T
        R = np.abs(LU @ X - B[:, :nrhs]).max()
        assert R <= 16 * n * 2.0 ** -53 * np.abs(LU).sum(1).max() * np.abs(X).max()
