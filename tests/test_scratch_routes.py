"""Which launches device-decided steps with scratch memory take, seen from the host (see test_routes.py): the lists that are compared on
the GPU reach the kernels that they are there for, and the lines lie where include/ps_adam.h says."""
import pytest

from test_routes import H, M, MI, P, V, launches, steps


def rows_of(chunks, n, offset, gap=8):
    stride = n + gap + offset
    return [[P + 4 * (stride * k + offset), M + 4 * (stride * k + offset), V + 4 * (stride * k + offset), H + 2 * (stride * k + offset)] for k in range(chunks)]


def route(chunks, n, used=None, offset=0, even=True):
    rows = rows_of(chunks, n, offset)
    if not even:
        rows[-1][2] += 1 << 38
    return launches("scratch", rows, used or [n] * chunks, True)


def test_the_lists_of_the_many_workgroup_step_take_it():
    from test_gpu_many_workgroups import LISTS, MOST

    for case in LISTS:
        (one,) = route(*case)
        assert one.name == "adam_small_step_kernel" and one.grid[0] > 1, case
    assert len(route(1, MOST + 1)) == 2
    assert {route(*case)[0].evenly for case in LISTS} == {False, True}


@pytest.mark.parametrize("even", [False, True])
def test_where_one_launch_and_two_end(even):
    """The longest chunk's tiles times the number of chunks decide, and 64 chunks are the most of one launch."""
    for chunks, tiles in ((1, 280), (7, 40), (64, 4), (3, 93)):
        used = [tiles * 256] + [3] * (chunks - 1)
        assert [q.name for q in route(chunks, used[0], used, even=even)] == ["adam_small_step_kernel"]
        used[0] += 1
        assert len(route(chunks, used[0], used, even=even)) == 2
    assert len(route(64, 2304, even=even)) == 2 and len(route(65, 2304)) == 2
    assert [q.name for q in route(65, 2304, even=False)][-1] == "scaler_update_kernel" and len(route(65, 2304, even=False)) > 2
    assert len(route(1, 300 * MI)) == 3 and len(route(2, 13 * MI, even=False)) == 2 and len(route(2, 15 * MI, even=False)) == 3
    assert steps(route(2, 15 * MI))[0].name == "adam_even_chunks_closing_kernel"
