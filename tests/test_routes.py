"""Which kernels a call launches, seen from the host: the library runs against a stand-in for the HIP runtime that writes
launches down (tests/routes).  The kernels' outputs are compared on the GPU; that those comparisons have two routes to compare
is checked here, with their lists."""
import functools
import json
import os
import re
import subprocess
import sys
import tempfile

import pytest

from patrickstar_amd import _lib

HERE = os.path.join(os.path.dirname(os.path.abspath(__file__)), "routes")
MI = 1 << 20
P, M, V, H = (1 << 40, 2 << 40, 3 << 40, 4 << 40)


_FOLDER = tempfile.TemporaryDirectory()


@functools.lru_cache(maxsize=None)
def _stand_in():
    path = os.path.join(_FOLDER.name, "launches.so")
    subprocess.check_call(["gcc", "-O1", "-fPIC", "-shared", "-o", path, os.path.join(HERE, "launches.c")])
    return path


class Launch:
    def __init__(self, mangled, grid, lds):
        name = re.match(r"_ZN12_GLOBAL__N_1(\d+)", mangled)
        at, n = name.end(), int(name[1])
        self.name, rest = mangled[at : at + n], mangled[at + n :]
        self.near = "NearBatch" in rest
        self.evenly = "even" in self.name or "EvenBatch" in rest
        self.hint = "Lb1EEEv" in rest  # the last template argument
        self.grid, self.lds = grid, lds

    def __repr__(self):
        return f"{self.name}{' near' * self.near}{' hint' * self.hint} {self.grid}"


def launches(entry, rows, numels, gated=False, grad_f32=None):
    call = dict(entry=entry, rows=rows, numels=numels, gated=gated, grad_f32=grad_f32 or [False] * len(rows))
    env = dict(os.environ, HIP_VISIBLE_DEVICES="-1")
    got = subprocess.run([sys.executable, os.path.join(HERE, "record.py"), _stand_in(), _lib.LIB_PATH, _lib.__file__],
                         input=json.dumps([call]), capture_output=True, text=True, env=env)
    assert got.returncode == 0, got.stderr
    return [Launch(*one) for one in json.loads(got.stdout)[0]]


def steps(found):
    return [q for q in found if q.name.startswith("adam_")]


def flat_rows(sizes, phases=(0, 0, 0, 0)):
    """Tensors one after the other in four lists that start at a phase, in elements."""
    rows, at = [], 0
    for n in sizes:
        rows.append([P + 4 * (at + phases[0]), M + 4 * (at + phases[1]), V + 4 * (at + phases[2]), H + 2 * (at + phases[3])])
        at += n
    return rows


# ---------------------------------------------------------------------------------------- the hint of long lists


@pytest.mark.parametrize("gated", [False, True])
@pytest.mark.parametrize("sizes,mirrored", [([33 * MI + 77], False), ([17 * MI] * 2, False), ([17 * MI] * 2, True)])
def test_long_chunk_lists_stream_past_the_caches(sizes, mirrored, gated):
    order = -1 if mirrored else 1
    (aligned,) = steps(launches("chunks", flat_rows(sizes)[::order], sizes, gated))
    (other,) = steps(launches("chunks", flat_rows(sizes, (16,) * 4)[::order], sizes, gated))  # fp16 at half a line
    assert aligned.hint and not other.hint and aligned.name == other.name
    assert ("even" in aligned.name) == (not mirrored)
    (short,) = steps(launches("chunks", flat_rows([27 * MI]), [27 * MI], gated))
    assert not short.hint


@pytest.mark.parametrize("entry", ["tensors", "each"])
@pytest.mark.parametrize("gated", [False, True])
@pytest.mark.parametrize("moved", [False, True])
def test_long_tensor_lists_stream_past_the_caches(entry, gated, moved):
    sizes = [20 * MI, 3, 6 * MI + 1, 255, 6 * MI - 7, 1 * MI, 256, 500_000]
    for phase, hint in ((0, True), (8, False)):  # of momentum and variance alone
        rows = flat_rows(sizes, (0, phase, phase, 0))
        if moved:
            rows[-1][2] += 1 << 38
        found = steps(launches(entry, rows, sizes, gated))
        assert all(q.hint == hint and q.near == (not moved) for q in found) and (moved or len(found) == 1), found
    short = [s // 2 for s in sizes]
    assert not any(q.hint for q in steps(launches(entry, flat_rows(short), short, gated)))


def test_the_lists_that_are_compared_with_the_oracle():
    from test_gpu_streaming_oracle import SIZES

    rows = flat_rows(SIZES)
    assert [(q.hint, q.near) for q in launches("tensors", rows, SIZES)] == [(True, True)]
    rows[-1][2] += 4 * 1024
    found = launches("tensors", rows, SIZES)
    assert len(found) > 1 and all(q.hint and not q.near for q in found)


@pytest.mark.parametrize("n,head,hint", [(256 * 1024, 0, True), (256 * 1024 - 1, 0, False), (300_001, 3, True), (2 * MI + 255, 128, True)])
def test_long_tensors_of_the_operator_stream_past_the_caches(n, head, hint):
    at = (256 - head) % 256
    (aligned,) = launches("operator", flat_rows([n], (at,) * 4), [n])
    (other,) = launches("operator", flat_rows([n], (at, at + 8, at + 8, at)), [n])
    assert aligned.hint == hint and not other.hint


@pytest.mark.parametrize("gated", [False, True])
def test_tensors_with_binary32_gradients_have_no_say_in_the_hint(gated):
    """They never take it: a large one does not move a short list past the caches, and one at another phase does not keep a
    long list there."""
    sizes = [MI, 2 * MI, 40 * MI]
    rows = flat_rows(sizes)
    rows[2][3] = H + (1 << 38)
    found = steps(launches("each", rows, sizes, gated, [False, False, True]))
    assert len([q for q in found if "f32grad" in q.name]) == 1 and not any(q.hint for q in found)
    sizes = [33 * MI, 2 * MI, 300_001]
    rows = flat_rows(sizes)
    rows[2] = [a + 16 for a in rows[2]]
    found = steps(launches("each", rows, sizes, gated, [False, False, True]))
    assert [q.hint for q in found if "f32grad" not in q.name] == [True]


# --------------------------------------------------- chunks at one distance, tensors at the same place of their lists


def test_chunks_at_one_distance_and_the_same_in_the_opposite_order():
    from test_gpu_even_chunk_lists import LISTS

    for chunks, n, last, _ in LISTS.values():
        stride = -(-n // 512) * 512
        rows = [[P + 4 * stride * k, M + 4 * stride * k, V + 4 * stride * k, H + 2 * stride * k] for k in range(chunks)]
        numels = [n] * (chunks - 1) + [last]
        for gated in (False, True):
            short = gated and chunks * -(-n // 256) <= 80  # one workgroup does the whole step
            (even,) = steps(launches("chunks", rows, numels, gated))
            general = steps(launches("chunks", rows[::-1], numels[::-1], gated))
            assert even.name == ("adam_small_step_kernel" if short else "adam_even_chunks_gated_kernel" if gated else "adam_even_chunks_kernel")
            assert even.evenly and not any(q.evenly for q in general), (chunks, n, gated)


def test_tensors_at_the_same_place_of_their_lists_and_one_that_is_not():
    from test_gpu_near_tensor_lists import SHAPES

    for name, sizes in SHAPES.items():
        rows = flat_rows(sizes)
        moved = [list(row) for row in rows]
        moved[max(k for k, n in enumerate(sizes) if n)][2] += 4 + (1 << 38)
        for entry in ("tensors", "each"):
            for gated in (False, True):
                assert all(q.near for q in steps(launches(entry, rows, sizes, gated))), name
                assert len(sizes) == 1 or not any(q.near for q in steps(launches(entry, moved, sizes, gated))), name
