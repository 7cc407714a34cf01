"""The native way of the short calls (csrc/host_calls.cpp) against the general way through DLPack capsules: the same outputs for
every form of argument it takes, the same exceptions for what the library refuses, and hands off what is not plain."""
import pytest
import torch

from longcontext_sqattn_paddle_amd import _native as N

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


class _Nothing:
    """Stands in for the module: leaves every call to the general way."""

    def __getattr__(self, name):
        return lambda *a: None


def _both(monkeypatch, call):
    """(outcome of the call as it is, outcome of the general way): outputs as a list of tensors, or the exception."""
    outcomes = []
    monkeypatch.undo()
    real = N.host_calls()
    taken = []

    class Spy:
        def __getattr__(self, name):
            def f(*a):
                r = getattr(real, name)(*a)
                taken.append(r is not None)
                return r
            return f

    for module in (Spy(), _Nothing()):
        monkeypatch.setattr(N, "host_calls", lambda module=module: module)
        try:
            res = call()
            torch.cuda.synchronize()
            outcomes.append([t.clone() for t in (res if isinstance(res, tuple) else (res,))])
        except Exception as e:   # noqa: BLE001 (compared below)
            outcomes.append(e)
    return outcomes[0], outcomes[1], taken


def _same(a, b):
    if isinstance(a, Exception) or isinstance(b, Exception):
        assert type(a) is type(b) and str(a) == str(b), (a, b)
        return
    assert len(a) == len(b)
    for x, y in zip(a, b):
        assert x.dtype == y.dtype and x.shape == y.shape and x.stride() == y.stride() and x.device == y.device
        assert torch.equal(x.view(torch.uint8) if x.is_contiguous() else x, y.view(torch.uint8) if y.is_contiguous() else y)


def _qkv(dtype, layout, nq, nk, B=2, Hq=6, Hkv=2, D=128):
    g = torch.Generator(device=DEV).manual_seed(nq + nk)
    mk = lambda H, n: torch.randn((B, n, H, D) if layout == "NHD" else (B, H, n, D), device=DEV, generator=g).to(dtype)
    return mk(Hq, nq), mk(Hkv, nk), mk(Hkv, nk)


@pytest.mark.parametrize("layout", ["NHD", "HND"])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_calls_that_are_taken_give_the_same_outputs(monkeypatch, layout, dtype):
    from longcontext_sqattn_paddle_amd.cache_hub.kmeans import topk_select
    from longcontext_sqattn_paddle_amd.sqattn.attn_triton import attn_causal
    from longcontext_sqattn_paddle_amd.sqattn.attn_triton_decode import attn_decode, attn_decode_selected

    print(f"case host calls {layout} {dtype}", flush=True)
    q, k, v = _qkv(dtype, layout, 1, 300)
    dim = 1 if layout == "NHD" else 2
    lens = torch.tensor([300, 17], dtype=torch.int32, device=DEV)
    ids = torch.randint(0, 300, (4, 50), device=DEV, dtype=torch.int32)
    wide = torch.cat([q, q], dim=0)
    calls = [
        lambda: attn_decode(q, k, v, layout, dtype),
        lambda: attn_decode(q, k, v, layout, torch.float32, True, seqlens=lens),
        lambda: attn_decode(q, k, v, layout, dtype, is_P_fp8_quant=True, num_splits=3),
        lambda: attn_decode(q, k, v, layout, dtype, workspace=torch.empty(1 << 20, device=DEV), out=torch.empty_like(q)),
        lambda: attn_decode(wide[1:3], k.narrow(dim, 0, 256), v.narrow(dim, 0, 256), layout, dtype),
        lambda: attn_decode(q[:1], k[1:], v[1:], layout, dtype),
        lambda: attn_decode_selected(q, k, v, ids, layout, dtype, True),
        lambda: attn_decode_selected(q, k, v, ids[:, :40], layout, dtype, seqlens=torch.tensor([40, 0], dtype=torch.int32, device=DEV)),
    ]
    qp, kp, vp = _qkv(dtype, layout, 130, 194)
    calls += [
        lambda: attn_causal(qp, kp, vp, layout, dtype, q_offset=64),
        lambda: attn_causal(qp, kp.narrow(dim, 0, 130), vp.narrow(dim, 64, 130), layout, torch.float32, True),
        lambda: attn_causal(qp, kp, vp, layout, dtype, p_quant=5, q_offset=64),
        lambda: attn_causal(qp, kp, vp, layout, dtype, q_offset=64, workspace=torch.empty(1 << 21, dtype=torch.uint8, device=DEV), out=torch.empty_like(qp)),
    ]
    if dtype == torch.bfloat16:
        cent = torch.randn(4, 64, 128, device=DEV).bfloat16()
        table = torch.randint(0, 300, (4, 64, 9), device=DEV, dtype=torch.int32)
        size = torch.randint(0, 10, (4, 64), device=DEV, dtype=torch.int32)
        query = torch.randn(2, 6, 128, device=DEV).bfloat16()
        calls += [lambda: topk_select(query, cent, table, size, 100, 3),
                  lambda: topk_select(query, cent, table, size, 100, 3, out=torch.empty(4, 120, dtype=torch.int32, device=DEV)[:, :100])]
    for i, call in enumerate(calls):
        a, b, taken = _both(monkeypatch, call)
        assert taken == [True], i
        assert not isinstance(a, Exception), (i, a)
        _same(a, b)


def test_refused_and_unusual_calls_end_as_on_the_general_way(monkeypatch):
    from longcontext_sqattn_paddle_amd.cache_hub.kmeans import topk_select
    from longcontext_sqattn_paddle_amd.sqattn.attn_triton import attn_causal
    from longcontext_sqattn_paddle_amd.sqattn.attn_triton_decode import attn_decode, attn_decode_selected

    q, k, v = _qkv(torch.bfloat16, "NHD", 1, 300)
    q64, k64, v64 = _qkv(torch.bfloat16, "NHD", 1, 300, D=64)
    qp, kp, vp = _qkv(torch.bfloat16, "NHD", 130, 130)
    ids = torch.randint(0, 300, (4, 50), device=DEV, dtype=torch.int32)
    cent = torch.randn(4, 64, 128, device=DEV).bfloat16()
    table = torch.randint(0, 300, (4, 64, 9), device=DEV, dtype=torch.int32)
    size = torch.randint(0, 10, (4, 64), device=DEV, dtype=torch.int32)
    query = torch.randn(2, 6, 128, device=DEV).bfloat16()
    calls = {
        "head_dim 64": lambda: attn_decode(q64, k64, v64, "NHD", torch.bfloat16),
        "layout": lambda: attn_decode(q, k, v, "XYZ", torch.bfloat16),
        "cpu": lambda: attn_decode(q.cpu(), k, v, "NHD", torch.bfloat16),
        "dtypes": lambda: attn_decode(q.half(), k, v, "NHD", torch.bfloat16),
        "fp32": lambda: attn_decode(q.float(), k.float(), v.float(), "NHD", torch.float32),
        "out dtype": lambda: attn_decode(q, k, v, "NHD", torch.float64),
        "heads": lambda: attn_decode(q[:, :, :5], k, v, "NHD", torch.bfloat16),
        "two queries": lambda: attn_decode(torch.cat([q, q], 1), k, v, "NHD", torch.bfloat16),
        "seqlens": lambda: attn_decode(q, k, v, "NHD", torch.bfloat16, seqlens=torch.tensor([3, 4], device=DEV)),
        "seqlens on the host": lambda: attn_decode(q, k, v, "NHD", torch.bfloat16, seqlens=torch.tensor([3, 4], dtype=torch.int32)),
        "small workspace": lambda: attn_decode(q, k, v, "NHD", torch.bfloat16, workspace=torch.empty(4, device=DEV)),
        "negative splits": lambda: attn_decode(q, k, v, "NHD", torch.bfloat16, num_splits=-2),
        "many splits": lambda: attn_decode(q, k, v, "NHD", torch.bfloat16, num_splits=5000),
        "gradient": lambda: attn_decode(q.clone().requires_grad_(), k, v, "NHD", torch.bfloat16),
        "parameter": lambda: attn_decode(q, torch.nn.Parameter(k, requires_grad=False), v, "NHD", torch.bfloat16),
        "truth value": lambda: attn_decode(q, k, v, "NHD", torch.bfloat16, 1),
        "channels": lambda: attn_decode(q[..., ::2], k[..., ::2], v[..., ::2], "NHD", torch.bfloat16),
        "ids 1-d": lambda: attn_decode_selected(q, k, v, ids[0], "NHD", torch.bfloat16),
        "ids int64": lambda: attn_decode_selected(q, k, v, ids.long(), "NHD", torch.bfloat16),
        "ids None": lambda: attn_decode_selected(q, k, v, None, "NHD", torch.bfloat16),
        "offset": lambda: attn_causal(qp, kp, vp, "NHD", torch.bfloat16, q_offset=3),
        "mode": lambda: attn_causal(qp, kp, vp, "NHD", torch.bfloat16, p_quant=9),
        "negative mode": lambda: attn_causal(qp, kp, vp, "NHD", torch.bfloat16, p_quant=-1),
        "lengths": lambda: attn_causal(qp, kp[:, :100], vp[:, :100], "NHD", torch.bfloat16),
        "v shape": lambda: attn_causal(qp, kp, vp[:, :100], "NHD", torch.bfloat16),
        "3-d": lambda: attn_causal(qp[0], kp[0], vp[0], "NHD", torch.bfloat16),
        "prefill 64": lambda: attn_causal(*_qkv(torch.float16, "HND", 70, 70, D=64), "HND", torch.float16, True),
        "groups": lambda: topk_select(query, cent, table, size, 100, 4),
        "k 0": lambda: topk_select(query, cent, table, size, 0, 3),
        "centroids 2-d": lambda: topk_select(query, cent[0], table, size, 100, 3),
        "query fp16": lambda: topk_select(query.half(), cent, table, size, 100, 3),
        "sizes int64": lambda: topk_select(query, cent, table, size.long(), 100, 3),
    }
    for name, call in calls.items():
        print(f"case host calls {name}", flush=True)
        a, b, _ = _both(monkeypatch, call)
        _same(a, b)


def test_modes_and_transforms_see_what_they_saw(monkeypatch):
    """Under a dispatch mode, and inside vmap, the native way stands aside."""
    from torch.utils._python_dispatch import TorchDispatchMode

    from longcontext_sqattn_paddle_amd.sqattn.attn_triton_decode import attn_decode

    q, k, v = _qkv(torch.bfloat16, "NHD", 1, 300)

    class Log(TorchDispatchMode):
        def __init__(self):
            super().__init__()
            self.seen = []

        def __torch_dispatch__(self, func, types, args=(), kwargs=None):
            self.seen.append(str(func))
            return func(*args, **(kwargs or {}))

    logs = []

    def under_mode():
        with Log() as log:
            res = attn_decode(q, k, v, "NHD", torch.bfloat16)
        logs.append(log.seen)
        return res

    a, b, taken = _both(monkeypatch, under_mode)
    assert taken == [False] and logs[0] == logs[1] and any("empty" in f for f in logs[0])
    _same(a, b)
    a, b, taken = _both(monkeypatch, lambda: torch.vmap(lambda x: attn_decode(x, k, v, "NHD", torch.bfloat16))(torch.stack([q, q])))
    assert taken in ([], [False])
    _same(a, b)


def _linear_case():
    g = torch.Generator(device=DEV).manual_seed(5)
    mk = lambda *s: torch.randn(s, device=DEV, generator=g).bfloat16()
    return mk(2, 20, 512), mk(256, 512), mk(256)


@pytest.mark.parametrize("which", ["x", "weight", "bias"])
def test_linear_of_a_prompt_keeps_forward_mode_tangents(which):
    """A dual tensor is an ordinary GPU tensor without gradient; its tangent goes through the product."""
    import torch.autograd.forward_ad as fwd

    from longcontext_sqattn_paddle_amd.model_hub.utils import linear

    args = dict(zip(("x", "weight", "bias"), _linear_case()))
    tangent = torch.ones_like(args[which])
    with fwd.dual_level():
        args[which] = fwd.make_dual(args[which], tangent)
        got, want = fwd.unpack_dual(linear(**args)), fwd.unpack_dual(torch.nn.functional.linear(args["x"], args["weight"], args["bias"]))
    assert got.tangent is not None and torch.equal(got.tangent, want.tangent) and torch.equal(got.primal, want.primal)


def test_linear_of_a_prompt_is_seen_by_a_trace():
    from longcontext_sqattn_paddle_amd.model_hub.utils import linear

    x, w, b = _linear_case()
    traced = torch.jit.trace(lambda t: linear(t, w, b), (x,), check_trace=False)
    assert "linear" in str(traced.graph)
    other = x.flip(0) * 2
    assert torch.equal(traced(other), torch.nn.functional.linear(other, w, b))


def test_linear_of_a_prompt_takes_the_type_autocast_names():
    from longcontext_sqattn_paddle_amd.model_hub.utils import linear

    x, w, b = _linear_case()
    with torch.autocast("cuda", dtype=torch.float16):
        got, want = linear(x, w, b), torch.nn.functional.linear(x, w, b)
    assert got.dtype == torch.float16 and torch.equal(got, want)
    with torch.autocast("cuda", dtype=torch.bfloat16):   # the type the operands have: nothing to convert
        got = linear(x, w, b)
    assert got.dtype == torch.bfloat16 and torch.equal(got, linear(x, w, b))


def test_linear_of_a_prompt_on_a_gpu_that_is_not_current():
    """`sq_linear` refuses tensors of another GPU than the current one, torch's linear does not.  One GPU is enough to see it: the
    library's product is replaced by one that returns that refusal."""
    import ctypes

    from longcontext_sqattn_paddle_amd.model_hub.utils import linear

    x, w, b = _linear_case()
    m = N.host_calls()
    addresses = [ctypes.cast(getattr(N.lib(), name), ctypes.c_void_p).value for name in N._HOST_CALLS_USE]
    refuse = ctypes.CFUNCTYPE(ctypes.c_int, *[ctypes.c_void_p] * 6)(lambda *a: N.SQ_EDEVICE)
    other = list(addresses)
    other[N._HOST_CALLS_USE.index("sq_linear")] = ctypes.cast(refuse, ctypes.c_void_p).value
    try:
        m.bind(*other)
        assert m.linear(x, w, b, N.current_stream(x.device)) is None
        assert torch.equal(linear(x, w, b), torch.nn.functional.linear(x, w, b))
    finally:
        m.bind(*addresses)
    assert m.linear(x, w, b, N.current_stream(x.device)) is not None


def test_linear_of_a_prompt_without_memory_for_the_parts():
    """The split product wants scratch that torch's linear does not (4 x 512 x 3584 fp32 here, 29 MB): where there is no room for it, the
    product is torch's."""
    from longcontext_sqattn_paddle_amd.model_hub.utils import linear

    x, w = torch.randn(512, 18944, device=DEV).bfloat16(), torch.randn(3584, 18944, device=DEV).bfloat16()
    want = torch.nn.functional.linear(x, w)   # and the BLAS library's own scratch is there
    torch.cuda.empty_cache()
    torch.cuda.set_per_process_memory_fraction((torch.cuda.memory_reserved() + (48 << 20)) / torch.cuda.get_device_properties(0).total_memory)
    taken = []
    try:
        with pytest.raises(torch.OutOfMemoryError):
            while True:
                taken.append(torch.empty(12 << 20, dtype=torch.uint8, device=DEV))
        taken.pop()
        got = linear(x, w)
    finally:
        torch.cuda.set_per_process_memory_fraction(1.0)
    assert torch.equal(got, want)
    assert N.host_calls().linear(x, w, None, N.current_stream(x.device)) is not None
