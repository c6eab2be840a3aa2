"""Calls just below and on the sizes from which buffers bypass the caches give
the bits of smaller calls, which do not."""
import pytest
import torch

pytestmark = pytest.mark.gpu
N = 65536
LAYOUTS = (([3, 4, 2], [8, 16, 32], 44100), ([4, 3], [12, 48], 48000))


def _x(*shape):
    return torch.randn(*shape, generator=torch.Generator(device="cuda").manual_seed(shape[0]), device="cuda")


@pytest.mark.parametrize("layout,slices", [(0, 104), (0, 106), (1, 104), (1, 106)])
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


@pytest.mark.parametrize("layout,batch", [(0, 139), (0, 140), (0, 191), (0, 192), (1, 164), (1, 165), (1, 223), (1, 224)])
def test_coefficient_planes(layout, batch):
    """One call against calls of 50 slices."""
    from flash_cqt import OctCQT
    from flash_cqt.fused import FusedOctCQT
    octs, bins, fs = LAYOUTS[layout]
    f = FusedOctCQT(OctCQT(octs, bins, fs=fs, audio_len=N, device="cuda:0"))
    x = _x(batch, N)
    kr, ki = (k.clone() for k in f.fwd(x))
    y = f.bwd(kr, ki).clone()
    for lo in range(0, batch, 50):
        part = f.fwd(x[lo:lo + 50])
        assert torch.equal(part[0], kr[lo:lo + 50]) and torch.equal(part[1], ki[lo:lo + 50])
        assert torch.equal(f.bwd(*part), y[lo:lo + 50])


@pytest.mark.parametrize("batch", [139, 140])
def test_interleaved_coefficients(batch):
    from flash_cqt import OctCQT
    from flash_cqt.trainable import TrainableCQT
    octs, bins, fs = LAYOUTS[1]
    t = TrainableCQT(OctCQT(octs, bins, fs=fs, audio_len=N, device="cuda:0"), "cuda:0")

    def step(x):
        x = x.clone().requires_grad_(True)
        blocks, side = t.fwd(x)
        y = t.bwd(blocks, side)
        return [c.detach() for c in blocks], y.detach(), torch.autograd.grad((y * y).sum(), x)[0]
    x = _x(batch, N)
    blocks, y, g = step(x)
    for lo in range(0, batch, 50):
        b, p, q = step(x[lo:lo + 50])
        assert all(torch.equal(c, d[lo:lo + 50]) for c, d in zip(b, blocks))
        assert torch.equal(p, y[lo:lo + 50]) and torch.equal(q, g[lo:lo + 50])
