"""The native form of the wrappers' common case (respect_amd/_calls, csrc/calls.cpp): which
calls it takes, and that it and the Python wrappers' own path give the same results."""
import pytest
import torch


def test_calls_leaves_what_it_does_not_take():
    """CPU tensors, other dtypes, non-tensors and wrong argument counts come back as None, so
    that the Python wrapper decides (on the CPU: no kernel is called)."""
    from respect_amd import _lib
    if not _lib.LIB_PATH.exists():
        pytest.skip("librespect_amd.so not built")
    c = _lib.calls()
    x = torch.zeros(4, 16, dtype=torch.bfloat16)
    assert c.silu_mul(x, x) is None and c.silu_mul(x) is None and c.silu_mul(1, "a") is None
    assert c.rmsnorm(x, x[0], 1e-6) is None and c.rmsnorm(x.float(), x[0], 1e-6) is None
    assert c.linear(x, x, 0, 0, False, False, {}, "linear") is None
    assert c.trie_attn(x, x, x, x, x, x, None, {}, "attn") is None
    assert c.rope(x, x, x) is None and c.add_sq(x, x) is None and c.rope_vision(x, x, x) is None
    assert c.norm_apply(x, x, x, 1e-6) is None and c.qk_norm_rope(x, x, x, x, 1e-6, x, x) is None
    assert c.rmsnorm_qk_norm_rope(x, x, 1e-6, x, x, x, x, 1e-6, x, x) is None


def test_calls_missing_or_of_another_build(monkeypatch):
    """Without the extension module the wrappers take their own path, with one warning; a module
    compiled for another library or torch raises instead of being called."""
    import sys
    import types
    import respect_amd
    from respect_amd import _lib
    from respect_amd.system import fused as F
    if not _lib.LIB_PATH.exists():
        pytest.skip("librespect_amd.so not built")
    version, tv = _lib.lib().rspx_version().decode(), torch.__version__.split("+")[0]
    x = torch.zeros(4, 16, dtype=torch.bfloat16)
    with monkeypatch.context() as m:
        m.setattr(_lib, "_calls", None)
        m.delattr(respect_amd, "_calls", raising=False)
        m.setitem(sys.modules, "respect_amd._calls", None)   # the import fails
        with pytest.warns(RuntimeWarning, match="respect_amd.build"):
            assert _lib.calls().silu_mul(x, x) is None
        with pytest.raises(RuntimeError, match="GPU tensor"):
            F.silu_mul(x, x)                                 # the wrapper's own checks
    for v, t in ((version + "0", tv), (version, "1.0.0")):
        with monkeypatch.context() as m:
            mod = types.SimpleNamespace(VERSION=v, TORCH=t)
            m.setattr(_lib, "_calls", None)
            m.setattr(respect_amd, "_calls", mod, raising=False)
            m.setitem(sys.modules, "respect_amd._calls", mod)
            with pytest.raises(RuntimeError, match="respect_amd.build"):
                _lib.calls()
    assert _lib.calls().VERSION == version


@pytest.mark.gpu
def test_calls_equal_the_wrappers_own_path(monkeypatch):
    """Each wrapper with and without the native call: equal results, shapes and dtypes, for the
    layouts the native call takes (it does take them) and for views, paddings and dtypes it
    leaves to Python."""
    from respect_amd import _lib
    from respect_amd.kernels.attention import fused_attn_hyb
    from respect_amd.kernels.gemm import linear, tile_weight
    from respect_amd.kernels.rmsnorm import rmsnorm
    from respect_amd.system import fused as F

    class Leave:
        def __getattr__(self, name):
            return lambda *a: None

    g = torch.Generator(device="cuda")
    g.manual_seed(1)

    def r(*s, dtype=torch.bfloat16):
        return torch.randn(*s, generator=g, device="cuda").to(dtype)

    x, w, w2 = r(2, 5, 512), r(512), r(768, 512)
    q, k, wq = r(7, 4, 128), r(7, 2, 128), r(128)
    cos, sin = r(7, 128), r(7, 128)
    gu = r(7, 2048)
    kp, kn = r(2, 40, 64), r(2, 32, 64)
    qa, msk = r(4, 9, 64), torch.ones(9, 32, dtype=torch.bool, device="cuda").tril()
    xr = r(1, 9, 4, 128)
    tw = tile_weight(w2)
    taken = [
        lambda: F.silu_mul(gu[:, :1024], gu[:, 1024:]),
        lambda: F.silu_mul(gu[0, :1024], gu[0, 1024:]),
        lambda: rmsnorm(x, w, 1e-6),
        lambda: F.qk_norm_rope(q, k, wq, wq, 1e-6, cos, sin),
        lambda: F.rmsnorm_qk_norm_rope(x, w, 1e-6, q, k, wq, wq, 1e-5, cos, sin),
        lambda: linear(x, w2),
        lambda: linear(x, w2, out_dtype=torch.float32),
        lambda: linear(x[0, 1:], tw),
        lambda: linear(r(70, 512) * 0 + x[0, :1], torch.nn.Parameter(w2)),
        lambda: fused_attn_hyb(qa, kp, kp, kn, kn, msk),
        lambda: fused_attn_hyb(qa, kp, kp, kn, kn, msk.to(torch.uint8), 0.1),
        lambda: F.rope(xr.transpose(1, 2), cos[None, :7].expand(1, 7, 128).repeat(1, 2, 1)[:, :9],
                       sin[None, :7].repeat(1, 2, 1)[:, :9]),
        lambda: F.add_sq(x[0], x[1]),
        lambda: F.norm_from(x[0], x[0].float() ** 2, w, 1e-6),
        lambda: F.rope_vision(q, cos.float(), sin.float()),
    ]
    left = [   # a copy, a dtype or a shape that the wrapper makes or converts
        lambda: F.silu_mul(gu[:, 1:1001], gu[:, 1001:2001]),
        lambda: rmsnorm(q[:, 1:3], wq, 1e-5),
        lambda: rmsnorm(x[..., :500], w[:500], 1e-6),
        lambda: F.rmsnorm_qk_norm_rope(x, w, 1e-6, q, k, wq, wq, 1e-5, cos[:, None], sin[:, None]),
        lambda: linear(x[..., :100], w2[:, :100]),
        lambda: fused_attn_hyb(qa, kp, kp, kn, kn, msk.to(torch.int32), 0.1),
        lambda: F.rope_vision(q, cos, sin),
    ]
    native = _lib.calls()
    answers = []

    class Record:
        def __getattr__(self, name):
            def call(*a):
                answers.append(getattr(native, name)(*a))
                return answers[-1]
            return call

    def taken_by(fn):
        answers.clear()
        with monkeypatch.context() as m:
            m.setattr(_lib, "calls", lambda: Record())
            y = fn()
        assert len(answers) == 1
        return answers[0] is not None, y

    for i, fn in enumerate(taken + left):
        print(f"[calls] {i}", flush=True)
        fn()                       # the stream's scratch is made
        took, a = taken_by(fn)
        assert took == (i < len(taken)), i
        with monkeypatch.context() as m:
            m.setattr(_lib, "calls", lambda: Leave())
            b = fn()
        for u, v in zip(a if isinstance(a, tuple) else (a,), b if isinstance(b, tuple) else (b,)):
            assert u.dtype == v.dtype and u.shape == v.shape and torch.equal(u, v), i
    # a scratch that is missing or too small is made by the wrapper; the next call is taken
    for fn, tag in ((lambda: linear(x[0], w2), "linear"), (lambda: fused_attn_hyb(qa, kp, kp, kn, kn, msk), "attn")):
        key = next(k for k in _lib._WORKSPACES if k[2] == tag)
        for start in ({}, {key: torch.zeros(16, dtype=torch.uint8, device="cuda")}):
            with monkeypatch.context() as m:
                m.setattr(_lib, "_WORKSPACES", start)
                (first, a), (second, b) = taken_by(fn), taken_by(fn)
            assert not first and second and torch.equal(a, b)
    # errors are the wrappers' own
    with pytest.raises(TypeError):
        F.silu_mul(gu.float(), gu.float())
    with pytest.raises(ValueError):
        F.silu_mul(gu, gu[:, :1024])
    with pytest.raises(TypeError):
        linear(x.float(), w2)
    with pytest.raises(ValueError):
        fused_attn_hyb(qa, kp, kp, kn, kn, msk[:, :16])
    # rows of no elements are refused, no rows are not
    for fn in (lambda t: F.silu_mul(t, t), lambda t: rmsnorm(t, t[0], 1e-6), lambda t: F.add_sq(t, t)):
        with pytest.raises(RuntimeError):
            fn(gu[:, :0])
    assert F.silu_mul(gu[:0], gu[:0]).shape == (0, 2048) and rmsnorm(x[:0], w, 1e-6).shape == (0, 5, 512)
    assert F.add_sq(x[0, :0], x[0, :0])[0].shape == (0, 512) and linear(x[:0], w2).shape == (0, 5, 768)


@pytest.mark.gpu
def test_calls_raise_where_torch_refuses_the_memory():
    """An output whose memory torch refuses to hand out (an allocation made under a dispatch
    mode that fakes it) is an ordinary error from inside the native call, and the thread
    holds the interpreter afterwards: later calls work."""
    from torch.utils._python_dispatch import TorchDispatchMode
    from respect_amd.kernels.gemm import linear
    from respect_amd.system import fused as F

    class NoMemory(TorchDispatchMode):
        def __torch_dispatch__(self, func, types, args=(), kwargs=None):
            r = func(*args, **(kwargs or {}))
            if func is torch.ops.aten.empty.memory_format:
                torch._C._set_throw_on_mutable_data_ptr(r)
            return r

    x, w = (torch.randn(n, 512, device="cuda").bfloat16() for n in (4, 2048))
    want = F.silu_mul(x, x)
    y = linear(x, w)
    for fn in (lambda: F.silu_mul(x, x), lambda: linear(x, w)):
        with pytest.raises(RuntimeError, match="data pointer"), NoMemory():
            fn()
    assert torch.equal(F.silu_mul(x, x), want) and torch.equal(linear(x, w), y)
