"""Large batches store and load some buffers past the caches (x, y, W, the
coefficients, each from its own batch size on): every slice still gives the
bits it gives in a small batch, on both sides of each of those sizes."""
import pytest
import torch

pytestmark = pytest.mark.gpu
N = 65536


@pytest.fixture(scope="module")
def cqt():
    from flash_cqt import OctCQT
    return OctCQT([3, 4, 2], [8, 16, 32], fs=44100, audio_len=N, device="cuda:0")


def _x(B):
    return torch.randn(B, N, generator=torch.Generator(device="cuda").manual_seed(B), device="cuda")


@pytest.mark.parametrize("B", [104, 105, 123, 124, 139, 140, 191, 192, 257])
def test_streamed_batches_equal_small_ones_bitwise(cqt, B):
    from flash_cqt.fused import FusedOctCQT
    f = FusedOctCQT(cqt)
    x = _x(B)
    kr, ki = (t.clone() for t in f.fwd(x))
    y = f.bwd(kr, ki).clone()
    for lo in range(0, B, 40):
        a, b = f.fwd(x[lo:lo + 40])
        assert torch.equal(a, kr[lo:lo + 40]) and torch.equal(b, ki[lo:lo + 40])
        assert torch.equal(f.bwd(kr[lo:lo + 40], ki[lo:lo + 40]), y[lo:lo + 40])


@pytest.mark.parametrize("B", [105, 140, 192])
def test_streamed_trainable_batches_equal_small_ones_bitwise(cqt, B):
    from flash_cqt.trainable import TrainableCQT
    t = TrainableCQT(cqt, "cuda:0")
    x = _x(B).requires_grad_(True)

    def step(x):
        blocks, side = t.fwd(x)
        y = t.bwd(blocks, side)
        g, = torch.autograd.grad((y * y).sum() + sum(c.abs().square().sum() for c in blocks), x)
        return [*blocks, *side, y, g]
    whole = step(x)
    for lo in range(0, B, 50):
        part = step(x[lo:lo + 50].detach().requires_grad_(True))
        assert all(torch.equal(p, w[lo:lo + 50]) for p, w in zip(part, whole))


@pytest.mark.parametrize("signals,length", [(7, 14 * 32768 - 2), (8, 12 * 32768 + 1), (12, 15 * 32768), (3, 88 * 32768 + 5)])
def test_streamed_sliced_calls_equal_single_signals_bitwise(signals, length):
    """105 slices and more in one call against one signal a call."""
    from flash_cqt import SlicedCQT
    s = SlicedCQT(device="cuda:0")
    x = torch.randn(signals, 1, length, generator=torch.Generator(device="cuda").manual_seed(length), device="cuda")
    with torch.no_grad():
        blocks, side = s.fwd(x)
        y = s.bwd(blocks, side, length=length)
        assert signals * s._num_slices(length) >= 104
        for i in range(signals):
            b1, s1 = s.fwd(x[i:i + 1])
            assert all(torch.equal(p, w[i:i + 1]) for p, w in zip([*b1, *s1], [*blocks, *side]))
            assert torch.equal(s.bwd(b1, s1, length=length), y[i:i + 1])
