"""The inverse column pass loads the overflow slots of a fold list's first
entries ahead of the entries, at the index the builder gives them; tables
whose indices follow another order (images of other builders) and lists
longer than that give the same bits."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu
N = 65536


def _in_bin_order(built, T):
    """The same tables with the overflow indices numbered by ascending bin."""
    out = dict(built)
    for name in ("scat", "scat_a"):
        fold, rec = built["ovf_" + name].copy(), built[name].copy()
        at = np.flatnonzero(fold >= 0)
        at = at[np.argsort(fold[at] & 0xFFFF)]
        new = np.zeros(T.OVF_CAP, dtype=np.int64)
        new[fold[at] >> 16] = np.arange(at.size)
        fold[at] = (fold[at] & 0xFFFF) | (np.arange(at.size) << 16)
        word = rec[:, 0].view(np.uint32).astype(np.int64)
        slot = word & 0x3FFFFFFF
        over = (rec[:, 1] != 0) & (slot >= 2 * T.FSTRIDE)
        k = (slot - 2 * T.FSTRIDE) // 2
        slot[over] += 2 * (new[k[over]] - k[over])
        rec[:, 0] = (slot | (word & 0xC0000000)).astype(np.uint32).view(np.int32)
        out["ovf_" + name], out[name] = fold, rec
    return out


@pytest.mark.parametrize("layout", [([3, 4, 2], [8, 16, 32], 44100), ([2, 5, 2], [4, 8, 64], 44100)])
def test_overflow_index_order_does_not_change_results(monkeypatch, layout):
    from flash_cqt import OctCQT, tables as T
    from flash_cqt.trainable import TrainableCQT
    cqt = OctCQT(layout[0], layout[1], fs=layout[2], audio_len=N, device="cuda:0")
    one, build = TrainableCQT(cqt, "cuda:0"), T.build
    monkeypatch.setattr(T, "build", lambda *a, **k: _in_bin_order(build(*a, **k), T))
    two = TrainableCQT(cqt, "cuda:0")
    assert not torch.equal(one.f.tables["ovf_scat"], two.f.tables["ovf_scat"])
    g = torch.Generator(device="cuda").manual_seed(5)
    for B in (1, 3, 17, 64):                   # the narrow and the wide column pass
        x = torch.randn(B, N, generator=g, device="cuda")
        got = []
        for t in (one, two):
            xg = x.clone().requires_grad_(True)
            blocks, side = t.fwd(xg)
            y = t.bwd(blocks, side)
            got.append((y.detach(), torch.autograd.grad((y * y).sum(), xg)[0]))
        assert torch.equal(got[0][0], got[1][0]) and torch.equal(got[0][1], got[1][1])
