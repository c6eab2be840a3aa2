"""Calls just below and on the sizes from which buffers bypass the caches give
the bits of smaller calls, which do not."""
import pytest
import torch

pytestmark = pytest.mark.gpu
N = 65536
LAYOUTS = (([3, 4, 2], [8, 16, 32], 44100), ([4, 3], [12, 48], 48000))


def _x(*shape):
    return torch.randn(*shape, generator=torch.Generator(device="cuda").manual_seed(shape[0]), device="cuda")


@pytest.mark.parametrize("layout,slices", [(0, 124), (0, 126), (1, 138), (1, 140)])
def test_sliced_coefficients(layout, slices):
    """Two signals at once against one after the other."""
    from flash_cqt import SlicedCQT
    octs, bins, fs = LAYOUTS[layout]
    s = SlicedCQT(octs, bins, fs=fs, sl_len=N, device="cuda:0")
    x = _x(2, 1, (slices // 2 - 1) * (N // 2) - 7)
    assert 2 * s._num_slices(x.shape[-1]) == slices
    with torch.no_grad():
        blocks, side = s.fwd(x)
        y = s.bwd(blocks, side, length=x.shape[-1])
        for i in range(2):
            b, d = s.fwd(x[i:i + 1])
            assert all(torch.equal(p[i], q[0]) for p, q in zip([*blocks, *side], [*b, *d]))
            assert torch.equal(y[i], s.bwd(b, d, length=x.shape[-1])[0])
