"""The inverse row passes that overlap-add in their stores, whole signals
(tiles of one, two and four hops) and the stream, against the row pass into a
slice buffer and the overlap-add kernels, bit for bit: odd and short lengths,
rows that start on 4-byte boundaries, tiles that end inside a signal."""
import ctypes

import pytest
import torch

pytestmark = pytest.mark.gpu
N, HOP = 65536, 32768


@pytest.fixture(scope="module")
def fused():
    from flash_cqt import OctCQT
    from flash_cqt.fused import FusedOctCQT
    return FusedOctCQT(OctCQT([3, 4, 2], [8, 16, 32], fs=44100, audio_len=N, device="cuda:0"))


def _coef(fused, rows):
    g = torch.Generator(device="cuda").manual_seed(rows)
    return torch.randn(rows * fused.ncoef, dtype=torch.complex64, generator=g, device="cuda")


def _at(words, shift):
    """A fp32 buffer whose start lies `shift` floats past an 8-byte boundary."""
    return torch.full((words + 2,), float("nan"), device="cuda")[shift:shift + words]


def _bits(a, b):
    return torch.equal(a.view(torch.int32), b.view(torch.int32))


@pytest.mark.parametrize("shift", [0, 1])
@pytest.mark.parametrize("nsig,S,length", [(1, 1, 1), (1, 2, HOP + 1), (1, 3, 2 * HOP - 1), (1, 4, 4 * HOP), (2, 9, 8 * HOP + 5),
                                           (1, 17, 17 * HOP - 3), (1, 161, 160 * HOP + 4095), (2, 81, 81 * HOP - 4097),
                                           (1, 323, 322 * HOP + 1), (3, 109, 109 * HOP)])
def test_sliced_synthesis_hop_tiles_same_bits(fused, nsig, S, length, shift):
    from flash_cqt import tables as T
    from flash_cqt.fused import slot_buffer
    B = nsig * S
    coef, f = _coef(fused, B), slot_buffer(B, fused.dev)
    work, y = torch.empty(B, T.L, 2, device="cuda"), torch.empty(B, N, device="cuda")
    ref, got = torch.empty(nsig, length, device="cuda"), _at(nsig * length, shift).view(nsig, length)
    fused.scatter_bands_sliced(coef, f, nsig, S)
    fused.packed_ifft(f, y, work)
    fused.overlap_add(y, ref, nsig, S, length)
    fused.sliced_synthesis(coef, f, work, got, nsig, S, length)
    assert _bits(got, ref)


@pytest.mark.parametrize("shift", [0, 1])
@pytest.mark.parametrize("nsig", [1, 5, 16, 17])
def test_stream_synthesis_same_bits(fused, nsig, shift):
    from flash_cqt import _native, tables as T
    from flash_cqt.fused import slot_buffer
    f = slot_buffer(nsig, fused.dev)
    work, y = torch.empty(nsig, T.L, 2, device="cuda"), torch.empty(nsig, N, device="cuda")
    tail, tail2 = torch.zeros(nsig, HOP, device="cuda"), _at(nsig * HOP, shift).view(nsig, HOP).zero_()
    for k in range(3):
        coef = _coef(fused, nsig) * (k + 1)
        ref, got = torch.empty(nsig, HOP, device="cuda"), _at(nsig * HOP, shift)
        fused.scatter_bands_sliced(coef, f, nsig, 1, first=k)
        fused.packed_ifft(f, y, work)
        fused.stream_overlap(y, tail, ref, nsig, k)
        _native.check(fused.lib.fcqt_stream_synthesis(
            fused._ct, fused._tp["scat"], fused._tp["slice_groups"], fused._tp["ovf_scat"], coef.data_ptr(), f.data_ptr(),
            work.data_ptr(), y.data_ptr(), tail2.data_ptr(), ctypes.c_void_p(got.data_ptr() if k else None), nsig, k,
            _native.stream_handle(0)), "stream_synthesis")
        assert _bits(tail2, tail)
        if k:
            assert _bits(got, ref.view(-1))
