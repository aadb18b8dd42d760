"""The C++ form of the wrappers' plain calls (csrc/host_calls.cpp) against the Python bodies behind it: which calls it
takes, the same results to the bit where it does, the Python body's own decision where it does not."""
import contextlib
import sys

import pytest
import torch

import parrotserve_amd
from parrotserve_amd import build, kernels, mem


@contextlib.contextmanager
def _python_only():
    host, kernels._host = kernels._host, kernels._TakesNothing()
    try:
        yield
    finally:
        kernels._host = host


class _Subclass(torch.Tensor):
    pass


def test_what_is_not_plain_is_left_to_python():
    host = kernels._load_host()
    x, w = torch.zeros(2, 8, dtype=torch.float16), torch.zeros(8, dtype=torch.float16)
    assert host.rms_norm(x, w, 1e-6, True, "x") is None  # host memory
    assert host.rms_norm(x.as_subclass(_Subclass), w, 1e-6, True, "x") is None
    assert host.rms_norm(None, w, 1e-6, True, "x") is None
    assert host.rms_norm(x, w) is None
    assert host.add_rms_norm(x, x, w, 1e-6, True) is None
    assert host.silu_mul(x, 3) is None
    assert host.sample_top_p(x, None, None, w) is None
    assert host.rope_append(x, x, x, x, x, 8, x, x, x, True) is None
    assert host.decode_attention(x, x, x, None, None, None, 0) is None
    assert host.prefill_attention(x, x, x, None, None) is None
    for call in (lambda: kernels.vllm_rms_norm(x, w, 1e-6), lambda: kernels.silu_mul(x, x),
                 lambda: kernels.fused_add_rms_norm(x, x, w, 1e-6)):
        with pytest.raises(RuntimeError, match="CPU tensor"):
            call()


def test_without_the_module_the_python_bodies_serve(monkeypatch):
    """_host.so is bound to one interpreter and one torch; where it does not load, a warning names the build command and
    every call is the Python body's, as it was before there was such a module."""
    monkeypatch.setattr(kernels, "_host", None)
    monkeypatch.delattr(parrotserve_amd, "_host", raising=False)
    monkeypatch.setitem(sys.modules, "parrotserve_amd._host", None)  # the import fails
    x, w = torch.zeros(2, 8, dtype=torch.float16), torch.zeros(8, dtype=torch.float16)
    with pytest.warns(RuntimeWarning, match="python -m parrotserve_amd.build"):
        with pytest.raises(RuntimeError, match="CPU tensor"):
            kernels.vllm_rms_norm(x, w, 1e-6)
    assert kernels._host.decode_attention(x, x, x, None, None, None, 0) is None
    with pytest.raises(RuntimeError, match="CPU tensor"):
        kernels.silu_mul(x, x)


def test_the_module_is_built_without_gcc_and_left_out_without_headers(monkeypatch, tmp_path):
    monkeypatch.delenv("CXX", raising=False)
    monkeypatch.setattr(build.shutil, "which", lambda name: None)
    assert build._host_compiler() == [build.HIPCC, "-x", "c++"]
    stale = tmp_path / "_host.so"
    stale.write_bytes(b"of an earlier build")
    monkeypatch.setattr(build, "HOST_LIB_PATH", str(stale))
    monkeypatch.setattr(build.sysconfig, "get_paths", lambda: {"include": str(tmp_path)})
    assert build._build_host() is False and not stale.exists()


class _Recorder:
    """The C++ form with a note of every call: taken (it returned a result or raised), or left to Python (None)."""

    def __init__(self, host):
        self.host, self.taken = host, []

    def __getattr__(self, name):
        def call(*args):
            self.taken.append(True)
            out = getattr(self.host, name)(*args)
            self.taken[-1] = out is not None
            return out
        return call


@contextlib.contextmanager
def _recording():
    host = kernels._host or kernels._load_host()
    assert host.__name__ == "parrotserve_amd._host"
    kernels._host = _Recorder(host)
    try:
        yield kernels._host
    finally:
        kernels._host = host


def _both(call, takes):
    """The call's outputs (or the class of what it raised) with the C++ form and without; ``takes``: the C++ form takes
    the call, and does not leave it to Python."""
    seen = []
    for ctx in (_recording(), _python_only()):
        with ctx as recorder:
            try:
                out = call()
            except Exception as e:  # noqa: BLE001 -- what is compared is the class
                out = type(e)
            if recorder:
                assert recorder.taken == [takes]
        seen.append(out)
    a, b = seen
    if isinstance(a, type) or isinstance(b, type):
        assert a is b
        return
    for x, y in zip(a, b):
        assert x.shape == y.shape and x.dtype == y.dtype and x.stride() == y.stride()
        assert torch.equal(x.view(torch.uint8) if x.dim() else x, y.view(torch.uint8) if y.dim() else y)


_FORMS = {
    "plain": lambda t: t,
    "columns": lambda t: torch.cat([t, t], dim=-1)[..., : t.shape[-1]],
    "one_row": lambda t: t[3:4],
    "no_rows": lambda t: t[:0],
    "3d": lambda t: t.view(-1, 5, t.shape[-1]),
    "transposed": lambda t: t.t().contiguous().t(),
    "subclass": lambda t: t.as_subclass(_Subclass),
    "int": lambda t: t.to(torch.int16),
    "float": lambda t: t.float(),
    "host": lambda t: t.cpu(),
    "grad": lambda t: t.clone().requires_grad_(),
}


@pytest.mark.gpu
@pytest.mark.parametrize("form", sorted(_FORMS))
def test_rows_through_both(dev, form):
    f, g = _FORMS[form], torch.Generator(device=dev).manual_seed(5)
    x, r, up = (torch.randn(40, 136, generator=g, device=dev, dtype=torch.float16) for _ in range(3))
    w = torch.randn(136, generator=g, device=dev, dtype=torch.float16)
    if form in ("int", "float"):
        w = f(w)
    t, p, u = (torch.full((40,), v, device=dev) for v in (0.8, 0.9, 0.37))
    n = f(x).shape[0]
    plain = form in ("plain", "columns", "one_row", "float", "grad")
    _both(lambda: [kernels.vllm_rms_norm(f(x), w, 1e-6)], plain)
    _both(lambda: [kernels.rmsnorm_forward(f(x), w, 1)], plain)
    _both(lambda: [kernels.silu_mul(f(x), f(up))], plain)
    _both(lambda: [kernels.silu_mul(f(x), up)], plain and form not in ("one_row", "float"))
    _both(lambda: [kernels.sample_top_p(f(x), t[:n], p[:n], u[:n])], plain)
    _both(lambda: [kernels.sample_top_p(f(x), None, None, u)], plain and form != "one_row")

    def add():
        res = f(r.clone())
        return [kernels.fused_add_rms_norm(f(x), res, w, 1e-6), res.detach()]

    if form != "grad":  # (a leaf that takes a gradient is refused by neither and written by both)
        _both(add, plain)


@pytest.mark.gpu
@pytest.mark.parametrize("form", ["plain", "chunks", "heads", "int64_slots", "wrong_heads", "short_slots", "host_positions"])
def test_rope_through_both(dev, form):
    g = torch.Generator(device=dev).manual_seed(6)
    T, H, D = 9, 4, 64
    qkv = torch.randn(T, 3 * H * D, generator=g, device=dev, dtype=torch.bfloat16)
    pos = torch.randint(0, 50, (T,), generator=g, device=dev)
    cs = mem.make_cos_sin_cache(50, D, 10000.0, torch.bfloat16, dev)
    slots = torch.randperm(30, generator=g, device=dev)[:T].to(torch.int64 if form == "int64_slots" else torch.int32)

    def call():
        q, k, v = (c if form == "chunks" else c.contiguous() for c in torch.chunk(qkv.clone(), 3, dim=-1))
        if form == "heads":
            q, k, v = (c.view(T, H, D) for c in (q, k, v))
        kc, vc = (torch.zeros(30, H + (form == "wrong_heads"), D, device=dev, dtype=torch.bfloat16) for _ in range(2))
        kernels.rope_and_cache(pos.cpu() if form == "host_positions" else pos, q, k, v, cs, D, kc, vc,
                               slots[:5] if form == "short_slots" else slots)
        return [q.contiguous(), k.contiguous(), kc, vc]

    _both(call, form in ("plain", "chunks", "int64_slots"))


@pytest.mark.gpu
@pytest.mark.parametrize("form", ["plain", "scale", "no_prefix", "grouped", "strided_query", "wrong_batch",
                                  "wrong_dtype"])
def test_attention_through_both(dev, form):
    g = torch.Generator(device=dev).manual_seed(7)
    H, D, own = 8, 128, [17, 3, 40, 9, 1]
    G = 2 if form == "grouped" else H
    kc, vc = (torch.randn(300, G, D, generator=g, device=dev, dtype=torch.float16) for _ in range(2))
    slots = torch.randperm(300, generator=g, device=dev).tolist()
    lists, at = [], 130
    for n in own:
        lists.append(slots[at:at + n])
        at += n
    q = torch.randn(len(own), H + 1, D, generator=g, device=dev, dtype=torch.float16)
    q = q[:, :H] if form == "strided_query" else q[:, :H].contiguous()
    q = q[:4] if form == "wrong_batch" else q.bfloat16() if form == "wrong_dtype" else q
    prefix = [] if form == "no_prefix" else [slots[:130]]
    tables = kernels.DecodeTables.build(prefix, [0, len(own)], lists, dev, num_heads=H, kv_group=H // G)
    heads = {} if G == H else dict(head_mapping=torch.arange(G, dtype=torch.int32, device=dev).repeat_interleave(H // G),
                                   kv_group=H // G)
    scale = 0.05 if form == "scale" else None
    plain = not form.startswith("wrong")
    _both(lambda: [kernels.decode_attention(q, kc, vc, tables, scale=scale, **heads)], plain)
    if form == "grouped":
        return
    new = [4, 1]
    pre = kernels.PrefillTables.build(new, [slots[:60], slots[60:61]], dev)
    _both(lambda: [kernels.prefill_attention(q, kc, vc, pre, scale=scale)], plain)


@pytest.mark.gpu
def test_an_error_of_the_library_is_the_wrappers(dev):
    x = torch.zeros(4, 12, device=dev, dtype=torch.float32)  # no norm-and-add of 32-bit elements
    w = torch.zeros(12, device=dev, dtype=torch.float32)
    _both(lambda: [kernels.fused_add_rms_norm(x, x.clone(), w, 1e-6)], True)
    with pytest.raises(RuntimeError, match="fused_add_rms_norm: unsupported data type"):
        kernels.fused_add_rms_norm(x, x.clone(), w, 1e-6)


@pytest.mark.gpu
def test_a_whole_number_beyond_a_double_is_refused_as_by_python(dev):
    """``float()`` of it raises OverflowError; the C++ form leaves the call to the body that says so."""
    huge = 10 ** 400
    x, w = torch.ones(4, 64, device=dev, dtype=torch.float16), torch.ones(64, device=dev, dtype=torch.float16)
    q, kc, vc = (torch.ones(n, 2, 128, device=dev, dtype=torch.float16) for n in (2, 40, 40))
    tables = kernels.DecodeTables.build([], [], [[1, 2, 3], [4, 5]], dev, num_heads=2)
    pre = kernels.PrefillTables.build([2], [[1, 2, 3]], dev)
    for call in (lambda: kernels.vllm_rms_norm(x, w, huge), lambda: kernels.rmsnorm_forward(x, w, -huge),
                 lambda: kernels.fused_add_rms_norm(x, x.clone(), w, huge),
                 lambda: kernels.decode_attention(q, kc, vc, tables, scale=huge),
                 lambda: kernels.prefill_attention(q, kc, vc, pre, scale=huge)):
        with pytest.raises(OverflowError):
            call()
