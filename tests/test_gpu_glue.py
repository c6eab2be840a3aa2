"""TrainableCQT through the host glue against its Python path: the same bits and
gradients for the calls that the glue takes, and the same answers, errors
included, for those it declines."""
import pytest
import torch

pytestmark = pytest.mark.gpu
N = 65536


@pytest.fixture(scope="module")
def pair():
    """(glue, Python path): two engines of one layout."""
    from flash_cqt import OctCQT
    from flash_cqt.trainable import TrainableCQT
    cqt = OctCQT([3, 4, 2], [8, 16, 32], fs=44100, audio_len=N, device="cuda:0")
    a, b = TrainableCQT(cqt, "cuda:0"), TrainableCQT(cqt, "cuda:0")
    assert a._glue is not None, "the host glue is built by __graft_entry__.build()"
    b._glue = None
    return a, b


def _x(*lead, seed=0, dtype=torch.float32):
    g = torch.Generator(device="cuda").manual_seed(seed)
    return torch.randn(*lead, N, generator=g, device="cuda").to(dtype)


def _same(p, q):
    return len(p) == len(q) and all(a.shape == b.shape and a.dtype == b.dtype and torch.equal(a, b)
                                    for a, b in zip(p, q))


def _step(t, x, edit):
    x = x.detach().requires_grad_(True)
    blocks, side = t.fwd(x)
    if edit == "in place":
        blocks[3].mul_(0.5)
    elif edit == "new":
        blocks = [c * (i + 1.0) for i, c in enumerate(blocks)]
    elif edit == "swap":                       # views of the right buffer in another order of slices
        blocks, side = [c.transpose(0, 1) for c in blocks], [c.transpose(0, 1) for c in side]
        blocks, side = [c.contiguous() for c in blocks], [c.contiguous() for c in side]
    y = t.bwd(blocks, None if edit == "no side" else side)
    loss = (y * y).sum() + blocks[0].abs().sum() + blocks[2].conj().real.sum()
    g, = torch.autograd.grad(loss, x)
    return [*[c.detach() for c in blocks], *[c.detach() for c in side], y.detach(), g]


@pytest.mark.parametrize("edit", ["none", "in place", "new", "no side"])
@pytest.mark.parametrize("lead,dtype", [((1,), torch.float32), ((5,), torch.float32), ((2, 3), torch.float32),
                                        ((), torch.float32), ((2, 1), torch.float64)])
def test_glue_step_equals_python_path(pair, lead, dtype, edit):
    x = _x(*lead, seed=len(lead), dtype=dtype)
    assert _same(_step(pair[0], x, edit), _step(pair[1], x, edit))
    assert _same(_step(pair[0], x, edit), _step(pair[1], x, edit))     # with every buffer of the set there


def test_glue_takes_slices_in_the_order_given(pair):
    assert _same(_step(pair[0], _x(2, 3), "swap"), _step(pair[1], _x(2, 3), "swap"))
    blocks, side = pair[0].fwd(_x(2, 3))
    turned = pair[0].bwd([c.transpose(0, 1) for c in blocks], [c.transpose(0, 1) for c in side])
    assert torch.equal(turned, pair[0].bwd(blocks, side).transpose(0, 1))


def test_glue_no_grad_strided_and_conjugated_inputs(pair):
    for x in (_x(4)[1:3], _x(4)[::2], _x(3).conj().real, -_x(2), torch.complex(_x(2), _x(2, seed=1)).conj().imag):
        with torch.no_grad():
            (b, s), (b2, s2) = pair[0].fwd(x), pair[1].fwd(x)
            assert _same([*b, *s], [*b2, *s2])
            assert torch.equal(pair[0].bwd(b, s), pair[1].bwd(b2, s2))


def test_glue_backward_after_the_engine_and_its_buffers_are_gone():
    from flash_cqt import OctCQT
    from flash_cqt.trainable import TrainableCQT
    cqt = OctCQT([3, 4, 2], [8, 16, 32], fs=44100, audio_len=N, device="cuda:0")
    t = TrainableCQT(cqt, "cuda:0")
    ref = _step(t, _x(3), "none")[-1]
    x = _x(3).requires_grad_(True)
    blocks, side = t.fwd(x)
    loss = (t.bwd(blocks, side) ** 2).sum() + blocks[0].abs().sum() + blocks[2].conj().real.sum()
    t.fwd(_x(6))                               # a larger set replaces the one of the forward pass
    t.f.release_workspace()
    del t
    junk = [torch.full((1 << 22,), float("nan"), device="cuda") for _ in range(16)]
    assert torch.equal(torch.autograd.grad(loss, x)[0], ref)
    del junk


def test_glue_declines_what_the_python_path_refuses(pair):
    for t in pair:
        with pytest.raises(ValueError):
            t.fwd(torch.randn(2, N))
        with pytest.raises(ValueError):
            t.fwd(torch.empty(0, N, device="cuda"))
        b, s = t.fwd(_x(2))
        with pytest.raises(ValueError):
            t.bwd([c[..., :-1] for c in b], s)
        with pytest.raises(RuntimeError):      # no forward-mode rule
            torch.func.jvp(lambda v: t.fwd(v)[0][0], (_x(1),), (_x(1),))
        with pytest.raises(RuntimeError):      # no batching rule
            torch.func.vmap(lambda v: t.fwd(v)[0][0])(_x(2, 1))


def test_glue_step_in_a_graph_and_from_threads(pair):
    from concurrent.futures import ThreadPoolExecutor
    from flash_cqt import Graphed
    t = pair[0]
    x = _x(4)
    want = t.bwd(*t.fwd(x))
    g = Graphed(lambda a: t.bwd(*t.fwd(a)), x)
    t.fwd(_x(9))                               # the recorded set stays with the graph
    for _ in range(3):
        assert torch.equal(g(x), want)
    torch.cuda.synchronize()
    with ThreadPoolExecutor(4) as pool:        # on one stream
        assert all(torch.equal(y, want) for y in pool.map(lambda i: t.bwd(*t.fwd(x)), range(16)))


@pytest.fixture(scope="module")
def cqt():
    from flash_cqt import OctCQT
    return OctCQT([3, 4, 2], [8, 16, 32], fs=44100, audio_len=N, device="cuda:0")


def _engine(cqt, path):
    from flash_cqt.trainable import TrainableCQT
    t = TrainableCQT(cqt, "cuda:0")
    if path == "python":
        t._glue = None
    return t


@pytest.mark.parametrize("path", ["glue", "python"])
def test_turned_views_on_a_first_call_and_later(cqt, path):
    """Slices in the order given, whichever path takes the call: on buffers that
    the engine has released (a first call), and again with them there."""
    t = _engine(cqt, path)
    blocks, side = t.fwd(_x(2, 3))
    want = t.bwd(blocks, side).transpose(0, 1)
    for cold in (True, False):
        if cold:
            t.f.release_workspace()
        assert torch.equal(t.bwd([c.transpose(0, 1) for c in blocks], [c.transpose(0, 1) for c in side]), want)


@pytest.mark.parametrize("path", ["glue", "python"])
def test_blocks_that_are_missing_or_cropped_are_refused(cqt, path):
    t = _engine(cqt, path)
    blocks, side = t.fwd(_x(4))
    with pytest.raises(ValueError):
        t.bwd(blocks, [])
    with pytest.raises(ValueError):
        t.bwd(blocks[:-1], side)
    with pytest.raises(ValueError):
        t.bwd([*blocks[:-1], blocks[-1][:2]], side)


@pytest.mark.parametrize("path", ["glue", "python"])
def test_conjugated_blocks_are_conjugated(cqt, path):
    """Lazily conjugated views of fwd's buffer, against blocks of their own."""
    t = _engine(cqt, path)
    blocks, side = t.fwd(_x(3))
    own = lambda parts: [c.conj().resolve_conj() for c in parts]  # noqa: E731
    want = t.bwd(own(blocks), own(side))
    assert torch.equal(t.bwd([c.conj() for c in blocks], [c.conj() for c in side]), want)
    assert torch.equal(t.bwd([c.conj() for c in blocks], own(side)), want)


def test_sliced_conjugated_blocks_are_conjugated():
    from flash_cqt import SlicedCQT
    s = SlicedCQT(fs=44100, device="cuda:0")
    blocks, side = s.fwd(_x(1, 2))
    own = lambda parts: [c.conj().resolve_conj() for c in parts]  # noqa: E731
    assert torch.equal(s.bwd([c.conj() for c in blocks], [c.conj() for c in side]), s.bwd(own(blocks), own(side)))


@pytest.mark.parametrize("path", ["glue", "python"])
def test_blocks_made_leaves_get_their_gradients(cqt, path):
    """Coefficients of a call without gradients, then optimised themselves."""
    t = _engine(cqt, path)
    x = _x(3)

    def gradients(keep):
        with torch.no_grad():
            blocks, side = t.fwd(x)
        parts = [keep(c) for c in [*blocks, *side]]
        for c in parts[1:]:
            c.requires_grad_(True)
        y = t.bwd(parts[:len(blocks)], parts[len(blocks):])
        return torch.autograd.grad((y ** 3).sum(), parts[1:])
    assert _same(gradients(lambda c: c), gradients(lambda c: c.detach().clone()))


def test_ordinary_calls_are_the_glues(cqt):
    """On a fresh engine, once a call has made its buffers: the directions alone,
    gains learnt between them (no gradient of the signal), coefficients learnt
    themselves, and, after one backward pass, training of the signal."""
    t = _engine(cqt, "glue")
    x = _x(2, 3)
    blocks, side = t.fwd(x)
    assert t._glue.fwd(x) is not None and t._glue.bwd([*blocks, *side]) is not None
    gains = [torch.full((c.shape[-2], 1), 0.5, device="cuda", requires_grad=True) for c in blocks]
    leaves = [c.detach().clone().requires_grad_(True) for c in [*blocks, *side]]
    for parts in ([c * g for c, g in zip(blocks, gains)] + list(side), leaves):
        y = t._glue.bwd(parts)
        assert y is not None and y.requires_grad
    xg = x.clone().requires_grad_(True)
    t.bwd(*t.fwd(xg)).sum().backward()
    assert t._glue.fwd(xg) is not None


def test_both_paths_launch_one_direction_at_a_time(cqt):
    """The two paths share the engine's buffers: while a direction's launches are
    held together, neither path launches another; mixed threads on one stream
    give every caller its own result."""
    import threading
    from concurrent.futures import ThreadPoolExecutor
    from flash_cqt.trainable import TrainableCQT
    t = _engine(cqt, "glue")
    twin = TrainableCQT.__new__(TrainableCQT)              # the Python path on the same engine
    twin.__dict__.update(t.__dict__, _glue=None)
    xs = [_x(2, seed=i) for i in range(4)]
    want = [t.bwd(*t.fwd(x)) for x in xs]
    for e in (t, twin):
        done = threading.Event()
        with t.f._launching:
            worker = threading.Thread(target=lambda: (e.fwd(xs[0]), done.set()))
            worker.start()
            assert not done.wait(0.3)
        assert done.wait(30)
        worker.join()
    with ThreadPoolExecutor(8) as pool:
        got = list(pool.map(lambda i: (t, twin)[i % 2].bwd(*(t, twin)[i // 2 % 2].fwd(xs[i % 4])), range(64)))
    assert all(torch.equal(y, want[i % 4]) for i, y in enumerate(got))


def test_sliced_inverse_of_turned_and_cropped_views():
    """bwd reads fwd's buffer in place for all of its blocks alone: the C++ check
    and the Python one answer alike."""
    from flash_cqt import SlicedCQT
    sliced = SlicedCQT(fs=44100, device="cuda:0")
    x = torch.randn(3, 1, 70001, generator=torch.Generator(device="cuda").manual_seed(4), device="cuda")
    f = sliced.cqt.f
    with torch.no_grad():
        blocks, side = sliced.fwd(x)
        parts, rows = [*blocks, *side], 3 * sliced._num_slices(70001)
        own = [c.clone() for c in parts]
        assert f._glue.block_base(parts, rows).data_ptr() == parts[0].data_ptr()
        assert sliced._block_base(f, parts, rows).data_ptr() == parts[0].data_ptr()
        first = [parts[0][:2], *parts[1:]]
        for bad in (own, [c.conj() for c in parts], [*parts[:-1], parts[-1].conj()], [parts[1], parts[0], *parts[2:]],
                    first, [*parts[:-1], parts[-1][:2]], parts[:-1], [*parts, parts[0]], [c[1:] for c in parts]):
            assert f._glue.block_base(bad, rows) is None and sliced._block_base(f, bad, rows) is None
        ng = len(blocks)
        assert torch.equal(sliced.bwd(parts[:ng], parts[ng:]), sliced.bwd(own[:ng], own[ng:]))
        tail = [c[1:] for c in parts]
        assert torch.equal(sliced.bwd(tail[:ng], tail[ng:]), sliced.bwd(own[:ng], own[ng:])[1:])


@pytest.mark.parametrize("path", ["glue", "python"])
def test_watched_blocks_see_their_gradients(cqt, path):
    """Blocks that keep their gradient, or have a hook, between fwd and bwd."""
    t = _engine(cqt, path)
    seen = []

    def gradients(watched):
        x = _x(3).requires_grad_(True)
        blocks, side = t.fwd(x)
        if watched:
            blocks[2].retain_grad()
            blocks[4].register_hook(lambda g: seen.append(g.clone()))
            own = blocks
        else:
            own = [c.clone() for c in blocks]
            own[2].retain_grad(), own[4].retain_grad()
        y = t.bwd(own, side)
        (y ** 3).sum().backward()
        return [x.grad, own[2].grad] + (seen if watched else [own[4].grad])
    got, want = gradients(True), gradients(False)
    assert len(got) == 3 and all(g is not None and torch.allclose(g, w, rtol=1e-5, atol=1e-5 * float(w.abs().max())) for g, w in zip(got, want))
