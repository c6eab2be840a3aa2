"""Host logic of TrainableCQT that needs no GPU: which block tensors bwd may
read as the coefficient buffer that they are views of."""
import pytest
import torch

GSPEC = [(2, 4, 0), (1, 8, 8), (1, 4, 16)]
NCOEF = 20


@pytest.fixture()
def engine():
    from flash_cqt.trainable import TrainableCQT
    t = TrainableCQT.__new__(TrainableCQT)
    t.dev, t.gspec, t.ncoef, t.ngroups = torch.device("cpu"), GSPEC, NCOEF, 2
    return t


def _kc(rows=6):
    return torch.randn(rows, NCOEF, dtype=torch.complex64, generator=torch.Generator().manual_seed(rows))


def _views(kc, *lead):
    return [kc.narrow(1, off, b * M).view(*lead, b, M) for b, M, off in GSPEC]


@pytest.mark.parametrize("lead", [(6,), (2, 3), (1, 6), (6, 1), (3, 1, 2)])
def test_fwd_views_are_read_as_their_buffer(engine, lead):
    kc = _kc()
    assert engine._base_of(_views(kc, *lead), 6) is kc


@pytest.mark.parametrize("lead,turn", [((2, 3), (1, 0)), ((3, 2), (1, 0)), ((3, 1, 2), (2, 1, 0)), ((1, 2, 3), (0, 2, 1))])
def test_views_in_another_slice_order_are_not_the_buffer(engine, lead, turn):
    n = len(lead)
    parts = [c.permute(*turn, n, n + 1) for c in _views(_kc(), *lead)]
    assert engine._base_of(parts, 6) is None


def test_part_of_the_views_is_not_the_buffer(engine):
    """Fewer slices in one block, or fewer blocks, than the buffer holds."""
    parts = _views(_kc(), 6)
    for i in range(3):
        assert engine._base_of([c[:2] if j == i else c for j, c in enumerate(parts)], 6) is None
    assert engine._base_of(parts[:2], 6) is None
    assert engine._base_of(parts[:2] + [parts[1], parts[2]], 6) is None


def test_conjugated_views_are_not_the_buffer(engine):
    """conj() is a view with the buffer's address and strides and a flag."""
    parts = _views(_kc(), 6)
    for i in range(3):
        assert engine._base_of([c.conj() if j == i else c for j, c in enumerate(parts)], 6) is None


def test_sliced_conjugated_views_are_not_the_buffer():
    import types
    from flash_cqt.sliced import SlicedCQT
    s = SlicedCQT.__new__(SlicedCQT)
    f = types.SimpleNamespace(gspec=GSPEC, ncoef=NCOEF, dev=torch.device("cpu"))
    coef = _kc(6).flatten().clone()
    views = [coef[6 * off:6 * (off + b * M)].view(1, 3, b, 2 * M) for b, M, off in GSPEC]
    for i in range(3):
        turned = [c.conj() if j == i else c for j, c in enumerate(views)]
        got = s._block_buffer(f, turned[:2], turned[2:], 3, 2)
        assert got is not coef and torch.equal(got, torch.cat([c.flatten().resolve_conj() for c in turned]))


@pytest.mark.parametrize("base_grad", [False, True])
def test_leaf_views_are_not_the_buffer(engine, base_grad):
    """Views made without a gradient and then made to want one of their own."""
    kc = _kc().requires_grad_(base_grad) * 1
    with torch.no_grad():
        parts = _views(kc, 6)
    parts[1].requires_grad_(True)
    assert engine._base_of(parts, 6) is None
    with torch.no_grad():
        assert engine._base_of(parts, 6) is kc


def test_replaced_directions_and_engines_are_not_passed_by(monkeypatch):
    """The C++ path serves the class's own directions on the engine that it was
    attached to, nothing else."""
    import types
    from flash_cqt.trainable import TrainableCQT
    glue, lib = object(), object()

    def make(cls):
        t = cls.__new__(cls)
        t.f, t._lib, t._glue = types.SimpleNamespace(lib=lib, _glue=glue), lib, glue
        return t

    class Same(TrainableCQT):
        extra = 1

    class Other(TrainableCQT):
        def _synthesis(self, kc):
            return super()._synthesis(kc) * 2
    x = (torch.zeros(1),)
    assert make(TrainableCQT)._plain(x) is glue and make(Same)._plain(x) is glue
    assert make(Other)._plain(x) is None
    t = make(TrainableCQT)
    t._analysis = lambda v: v
    assert t._plain(x) is None
    t = make(TrainableCQT)
    t.f = types.SimpleNamespace(lib=lib, _glue=None)               # another engine on the same library
    assert t._plain(x) is None
    t.f = types.SimpleNamespace(lib=lib, _glue=object())
    assert t._plain(x) is None
    monkeypatch.setattr(TrainableCQT, "_adj_analysis", lambda self, g: g)
    assert make(TrainableCQT)._plain(x) is None


def test_glue_of_another_build_is_refused(monkeypatch, tmp_path):
    from flash_cqt import _native
    mod = _native.load_glue()
    assert mod is not None and (mod.abi_version, mod.torch_version) == (_native.ABI_VERSION, str(torch.__version__))
    monkeypatch.setattr(_native, "_glue", None)
    with monkeypatch.context() as m:
        m.setattr(_native, "ABI_VERSION", _native.ABI_VERSION + 1)
        with pytest.raises(_native.NativeError, match="rebuild"):
            _native.load_glue()
    with monkeypatch.context() as m:
        m.setattr(torch, "__version__", "0.0.0")
        with pytest.raises(_native.NativeError, match="torch"):
            _native.load_glue()
    broken = tmp_path / "_fcqt_torch.so"
    broken.write_bytes(b"not a library")
    monkeypatch.setattr(_native, "GLUE_PATH", broken)
    with pytest.raises(_native.NativeError, match="rebuild"):
        _native.load_glue()
    monkeypatch.setattr(_native, "GLUE_PATH", tmp_path / "absent.so")
    assert _native.load_glue() is None


def test_failed_glue_build_leaves_none_behind(monkeypatch, tmp_path):
    """build() with a host compiler that fails removes an earlier build's glue."""
    import importlib.util
    import pathlib
    root = pathlib.Path(__file__).resolve().parents[1]
    spec = importlib.util.spec_from_file_location("flashcqt_build_test", root / "flash-cqt_amd" / "build.py")
    b = importlib.util.module_from_spec(spec)
    spec.loader.exec_module(b)
    old = tmp_path / "_fcqt_torch.so"
    old.write_bytes(b"old")
    monkeypatch.setattr(b, "GLUE", old)
    monkeypatch.setattr(b, "OUT", tmp_path / "libflashcqt.so")
    monkeypatch.setattr(b, "VARIANTS", {})
    monkeypatch.setattr(b, "glue_command", lambda out: ["false"])
    with pytest.raises(RuntimeError, match="glue"):
        b.build()
    assert not old.exists()


def test_sliced_part_of_the_views_is_not_the_buffer():
    """A block cropped to fewer signals, or blocks left out: refused, as blocks of
    their own are, or taken as zero, not completed from the buffer."""
    import types
    from flash_cqt.sliced import SlicedCQT
    s = SlicedCQT.__new__(SlicedCQT)
    f = types.SimpleNamespace(gspec=GSPEC, ncoef=NCOEF, dev=torch.device("cpu"))
    coef = _kc(6).flatten().clone()
    views = [coef[6 * off:6 * (off + b * M)].view(3, 1, b, 2 * M) for b, M, off in GSPEC]
    assert s._block_buffer(f, views[:2], views[2:], 3, 2) is coef
    for i in range(1, 3):
        cut = [c[:2] if j == i else c for j, c in enumerate(views)]
        with pytest.raises(RuntimeError):
            s._block_buffer(f, cut[:2], cut[2:], 3, 2)
    got = s._block_buffer(f, views[:2], [], 3, 2)
    assert torch.equal(got[:96], coef[:96]) and not got[96:].any()


@pytest.mark.parametrize("watch", [lambda c: c.retain_grad(), lambda c: c.register_hook(lambda g: g)])
def test_watched_views_are_not_the_buffer(engine, watch):
    kc = _kc().requires_grad_(True) * 1
    parts = _views(kc, 6)
    assert engine._base_of(parts, 6) is kc
    watch(parts[1])
    assert engine._base_of(parts, 6) is None
