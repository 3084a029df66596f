"""ps_adam_update's vector kernel at the ends of its tiles (with and without elements in front of the tile grid and behind it)
leaves the bits of the element-wise kernel, which the same numbers take when the gradients lie at another phase."""
import pytest
import torch

from patrickstar_amd import _lib, adam_op

pytestmark = pytest.mark.gpu
OPT = 7901


@pytest.mark.parametrize("head", [0, 1, 4, 255])
@pytest.mark.parametrize("n", [4096, 4097, 4351, 4352, 4353, 2304 * 256, 2305 * 256 + 255])
@pytest.mark.parametrize("half,out", [(True, False), (True, True), (False, False)])
def test_edges(n, head, half, out):
    lib, s = _lib.load(), _lib.current_stream_handle()
    at = (256 - head) % 256
    gen = torch.Generator(device="cuda").manual_seed(n)
    base = [torch.randn(n + 512, device="cuda", generator=gen) for _ in range(4)]
    base[3].square_()
    results = []
    for phase in (0, 1):
        p, g, m, v = (t.clone() for t in base)
        g = torch.roll(g, phase)
        g = g.half() if half else g
        h = torch.zeros(n + 512, dtype=torch.half, device="cuda")
        adam_op.create_adam(OPT, 1e-3, 0.9, 0.999, 1e-8, 0.01, True, False)
        rc = lib.ps_adam_update(OPT, 3, 1e-3, 0.9, 0.999, 1e-8, 0.01, 1, p[at:].data_ptr(), g[at + phase :].data_ptr(), int(half),
                                m[at:].data_ptr(), v[at:].data_ptr(), n, 8.0, h[at:].data_ptr() if out else None, s)
        _lib.check(rc, "ps_adam_update")
        adam_op.destroy_adam(OPT)
        results.append((p, m, v, h))
    for a, b, before in zip(*results, (base[0], base[2], base[3], None)):
        assert torch.equal(a.view(torch.uint8), b.view(torch.uint8))
        if before is not None:
            assert torch.equal(a[:at], before[:at]) and torch.equal(a[at + n :], before[at + n :])
