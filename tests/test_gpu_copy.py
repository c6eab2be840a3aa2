"""fcqt_copy_buffers and the copies that Graphed hands out: sizes around a
workgroup's share and a vector's width, ends at every alignment, dtypes, and
outputs that stay as they were when the graph runs again."""
import ctypes

import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shift_src,shift_dst", [(0, 0), (4, 4), (4, 8), (1, 0), (3, 3)])
def test_copy_buffers_sizes_and_alignments(shift_src, shift_dst):
    from flash_cqt import _native
    lib = _native.load()
    sizes = [1, 3, 15, 16, 17, 4095, 8191, 8192, 8193, 100003, 5 * 8192 + 12]
    g = torch.Generator(device="cuda").manual_seed(1)
    src = [torch.randint(0, 255, (n + 48,), dtype=torch.uint8, generator=g, device="cuda") for n in sizes]
    dst = [torch.full((n + 48,), 255, dtype=torch.uint8, device="cuda") for n in sizes]
    want = [d.clone() for d in dst]
    for s, w, n in zip(src, want, sizes):
        w[16 + shift_dst:16 + shift_dst + n] = s[16 + shift_src:16 + shift_src + n]
    array = lambda v, t: (t * len(v))(*v)
    status = lib.fcqt_copy_buffers(array([s.data_ptr() + 16 + shift_src for s in src], ctypes.c_void_p),
                                   array([d.data_ptr() + 16 + shift_dst for d in dst], ctypes.c_void_p),
                                   array(sizes, ctypes.c_int64), len(sizes), _native.stream_handle())
    assert status == 0
    assert all(torch.equal(d, w) for d, w in zip(dst, want))      # and no byte beside them


def test_copy_buffers_refuses_bad_arguments():
    from flash_cqt import _native
    lib, one = _native.load(), (ctypes.c_void_p * 1)(4096)
    none, size, zero = (ctypes.c_void_p * 1)(None), (ctypes.c_int64 * 1)(8), (ctypes.c_int64 * 1)(0)
    for args in ((None, one, size, 1), (one, None, size, 1), (one, one, None, 1), (one, one, size, 0), (one, one, size, 17),
                 (none, one, size, 1), (one, none, size, 1), (one, one, zero, 1)):
        assert lib.fcqt_copy_buffers(*args, None) == 1


def test_graphed_outputs_are_copies_of_every_kind():
    from flash_cqt import Graphed

    def fn(a):
        return (a * 2, [a.t() + 1, torch.complex(a, -a)], (a > 0, a.double()[1:, ::2], a.conj(), torch.complex(a, a).conj()),
                a.sum(), a[:0], 3)
    x = torch.randn(37, 53, device="cuda")
    g = Graphed(fn, x)
    first, kept = g(x), fn(x)
    second = g(x * 5)

    def same(p, q):
        if torch.is_tensor(p):
            return p.shape == q.shape and p.dtype == q.dtype and p.stride() == q.clone().stride() and torch.equal(p, q)
        return type(p) is type(q) and (all(same(a, b) for a, b in zip(p, q)) if isinstance(p, (list, tuple)) else p == q)
    assert same(first, kept) and same(second, fn(x * 5))
    simple = Graphed(lambda a: (a + 1, [a.t() * 2]), x)       # every output plain: one launch
    for s in (1.0, 2.0, 3.0):
        assert same(simple(x * s), (x * s + 1, [(x * s).t() * 2]))


def test_outputs_past_one_launch_are_cloned_one_by_one():
    """More than the copy kernel takes in one launch (here one 5 GiB tensor 13
    times, 65 GiB) is declined before anything is allocated for it; Graphed then
    clones each output."""
    import ctypes as c
    from flash_cqt import _native
    fn = c.cast(_native.load().fcqt_copy_buffers, c.c_void_p).value
    big = torch.empty(5 << 30, dtype=torch.uint8, device="cuda")
    torch.cuda.reset_peak_memory_stats()
    before = torch.cuda.memory_allocated()
    assert _native.load_glue().clones([big] * 13, fn) is None
    assert torch.cuda.max_memory_allocated() == before
    del big
    torch.cuda.empty_cache()


def test_copy_buffers_refuses_more_than_one_launch_takes():
    from flash_cqt import _native
    lib, p = _native.load(), (ctypes.c_void_p * 2)(4096, 4096)
    for sizes in ((1 << 36, 1), ((1 << 36) - 8192, 8193)):
        assert lib.fcqt_copy_buffers(p, p, (ctypes.c_int64 * 2)(*sizes), 2, None) == 1
