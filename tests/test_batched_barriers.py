"""The refinement of the batched solver's accumulator-tile kernel: its two kinds of
waves take separate paths through the same barriers (R0 .. R6) and hand results
to each other in LDS. A word that one path writes must not be touched by the
other between the same two barriers, or a late wave reads the wrong decision and
the barriers no longer pair. Read off the source, since a run meets such a race
only when a wave happens to be late."""
import os
import re

import pytest

SOURCE = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "zml_amd", "csrc", "batched.hip")
BARRIER = re.compile(r"__syncthreads\(\);[ ]*// R(\d)")
ACCESS = re.compile(r"\bsh\.(\w+)((?:\[[^\]]*\])*)\s*(=(?!=))?")


def refinement(path):
    """The text of a path's refinement, from its group loop to the end."""
    text = open(SOURCE).read()
    kernel = text[text.index("batched_tile_kernel(BatchArgs g)"):text.index("reset_counters_kernel")]
    helpers, holders = kernel.split("g.status[sid] = worst;")
    part = helpers if path == "helpers" else holders
    part = part[part.rindex("for (int gq = 0;"):]
    return re.sub(r"//(?! R\d).*", "", part)


def phases(path):
    """[(words written, words touched)] between the barriers, in the order of the source."""
    pieces = BARRIER.split(refinement(path))
    assert pieces[1::2] == [str(k) for k in range(7)]
    out = []
    for piece in pieces[0::2]:
        found = ACCESS.findall(piece)
        out.append(({w for w, _, assign in found if assign}, {w for w, _, _ in found}))
    return out


# what can run at the same time: a phase with itself, the end of a step with the
# start of the next one (R5 back to R1), the end of a group with the next (R6 to R0)
PAIRS = [(k, k) for k in range(8)] + [(1, 6), (6, 1), (0, 7), (7, 0)]


@pytest.mark.parametrize("a,b", PAIRS)
def test_no_word_is_written_beside_the_other_paths_use(a, b):
    helpers, holders = phases("helpers"), phases("holders")
    assert any(w for w, _ in helpers) and any(w for w, _ in holders)
    assert not helpers[a][0] & holders[b][1]
    assert not holders[b][0] & helpers[a][1]


@pytest.mark.gpu
@pytest.mark.parametrize("bad", [0, 5, 8])
def test_a_right_hand_side_that_fails_ends_its_system(zh, torch_cuda, bad):
    """Nine right-hand sides (groups of 4, 4 and 1) with one that cannot be solved: both
    paths leave after its group, the earlier solutions stand, other systems go on."""
    import numpy as np
    from tests.test_gpu_batched import Batch

    rng = np.random.default_rng(bad)
    systems = [(rng.uniform(-1, 1, (n, n)) + n / 4.0 * np.eye(n), rng.uniform(-1, 1, (n, 9)), False)
               for n in (70, 128, 200, 256)]
    for _, B, _ in systems[::2]:
        B[3, bad] = np.nan
    bt = Batch(zh, torch_cuda, systems, autotune=0)
    status, hx = bt.run()
    bt.close()
    for i, ((A, B, _), X) in enumerate(zip(systems, bt.solutions(hx))):
        assert (status[i] >= 0) == (i % 2 == 1)
        q = bad if i % 2 == 0 else 9
        R, n = np.abs(B - A @ X)[:, :q].max(axis=0), A.shape[0]
        assert np.all(R <= 16 * n * 2.0 ** -53 * np.abs(A).sum(1).max() * np.abs(X[:, :q]).max(axis=0))
