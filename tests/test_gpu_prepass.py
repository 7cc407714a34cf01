"""GPU parity of `sq_fake_quant_prepass` (through the C ABI) with the oracle's restatement of the operand pre-pass
of sqattn/attn_replacer.py:334-365: bit-exact outputs, both layouts and dtypes, ragged sizes, error paths, and
sampled rows at the benchmark shape."""
import math

import pytest
import torch

from oracle import fake_quant as FQ
from oracle import plugin

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _inputs(B, N, Hq, Hkv, seed, dtype=torch.bfloat16, outliers=True):
    g = torch.Generator().manual_seed(seed)
    q = torch.randn(B, N, Hq, 128, generator=g)
    k = torch.randn(B, N, Hkv, 128, generator=g) + torch.randn(1, 1, Hkv, 128, generator=g)   # a per-channel offset to centre away
    v = torch.randn(B, N, Hkv, 128, generator=g)
    if outliers:
        k[..., 5] *= 8
        q[:, ::7] = 0   # all-zero rows: the scale clamp
    return q.to(dtype), k.to(dtype), v.to(dtype)


@pytest.mark.parametrize("B,N,Hq,Hkv,dtype,want4", [(1, 257, 4, 1, torch.bfloat16, True), (2, 1000, 8, 2, torch.bfloat16, True),
                                                  (1, 4096, 28, 4, torch.bfloat16, False), (2, 333, 6, 3, torch.float16, True),
                                                  (3, 64, 40, 40, torch.bfloat16, True)])
def test_prepass_is_bit_exact(B, N, Hq, Hkv, dtype, want4):
    from longcontext_sqattn_paddle_amd.sqattn.fake_quant import fused_int_prepass

    print(f"case prepass B={B} N={N} Hq={Hq} Hkv={Hkv} {dtype} want4={want4}", flush=True)
    q, k, v = _inputs(B, N, Hq, Hkv, seed=N, dtype=dtype)
    got = fused_int_prepass(q.to(DEV), k.to(DEV), v.to(DEV), want_4bit=want4, tensor_layout="NHD")
    torch.cuda.synchronize()
    ref = plugin.int_prepass(q, k, v, want_4bit=want4)
    for name, a, b in zip(("q8", "q4", "k8", "k4", "v8"), got, ref):
        if b is None:
            assert a is None
            continue
        assert a.dtype == dtype and a.shape == b.shape
        assert torch.equal(a.cpu(), b), (name, float((a.cpu().float() - b.float()).abs().max()))
        # ... and to the bit, which torch.equal does not see for the sign of zero
        assert torch.equal(a.cpu().contiguous().view(torch.int16), b.contiguous().view(torch.int16)), name


@pytest.mark.parametrize("qk,vq,dtype", [("e4m3", "e4m3", torch.bfloat16), ("e5m2", "int", torch.bfloat16), ("int", "e5m2", torch.float16)])
def test_prepass_float_quantiser_types(qk, vq, dtype):
    """The closure's e4m3 / e5m2 quantisers (sqattn/attn_replacer.py:340-358, float simulation of fake_quant.py:151-204)
    in the fused pre-pass.  Every operation of the simulation is exact in fp32 except `floor(log2(|t| + 1e-30))`, which
    the kernel reads from the exponent field: where a library's fp32 log2 rounds a value a few units in the last place
    below a power of two up to the integer, the two differ by one grid step.  Stated tolerance: at most 1e-4 of the
    elements differ, each by at most one step of its grid (2^-3 relative for e4m3, 2^-2 for e5m2); the integer outputs
    of the same call stay bit-exact."""
    from longcontext_sqattn_paddle_amd.sqattn.fake_quant import fused_int_prepass

    print(f"case prepass float quantisers qk={qk} v={vq} {dtype}", flush=True)
    q, k, v = _inputs(2, 700, 8, 2, seed=5, dtype=dtype)
    got = fused_int_prepass(q.to(DEV), k.to(DEV), v.to(DEV), want_4bit=True, tensor_layout="NHD", qk_qtype=qk, v_qtype=vq)
    torch.cuda.synchronize()
    ref = plugin.int_prepass(q, k, v, want_4bit=True, qk_qtype=qk, v_qtype=vq)
    for name, a, b, qt in zip(("q8", "q4", "k8", "k4", "v8"), got, ref, (qk, "int", qk, "int", vq)):
        a = a.cpu()
        if qt == "int":
            assert torch.equal(a.contiguous().view(torch.int16), b.contiguous().view(torch.int16)), name
            continue
        diff = a != b
        assert float(diff.float().mean()) <= 1e-4, (name, float(diff.float().mean()))
        step = 2.0 ** -3 if qt == "e4m3" else 2.0 ** -2
        rel = (a.float() - b.float()).abs() / b.float().abs().clamp(min=1e-30)
        assert float(rel[diff].max()) <= step * 1.01 if bool(diff.any()) else True, name
    with pytest.raises(ValueError):
        fused_int_prepass(q.to(DEV), k.to(DEV), v.to(DEV), qk_qtype="e3m4")


def test_prepass_hnd_views_and_strides():
    from longcontext_sqattn_paddle_amd.sqattn.fake_quant import fused_int_prepass

    q, k, v = _inputs(2, 300, 4, 2, seed=9)
    ref = plugin.int_prepass(q, k, v)
    # HND tensors that are permuted views of NHD storage (non-compact strides) ...
    got = fused_int_prepass(*(t.to(DEV).permute(0, 2, 1, 3) for t in (q, k, v)), tensor_layout="HND")
    for a, b in zip(got, ref):
        assert torch.equal(a.permute(0, 2, 1, 3).cpu(), b)
    # ... and compact HND tensors
    got = fused_int_prepass(*(t.to(DEV).permute(0, 2, 1, 3).contiguous() for t in (q, k, v)), tensor_layout="HND")
    for a, b in zip(got, ref):
        assert a.is_contiguous() and torch.equal(a.permute(0, 2, 1, 3).cpu(), b)


def test_prepass_benchmark_shape_sampled_rows():
    """128K tokens, 28/4 heads: rows sampled across the tensor must equal the oracle run on the same tokens
    (query rows and value columns are independent of other tokens; the key needs the global mean, checked first)."""
    from longcontext_sqattn_paddle_amd.sqattn.fake_quant import fused_int_prepass

    N = 131072
    g = torch.Generator(device=DEV).manual_seed(3)
    q = torch.randn(1, N, 28, 128, generator=g, device=DEV).bfloat16()
    k = (torch.randn(1, N, 4, 128, generator=g, device=DEV) + 0.5).bfloat16()
    v = torch.randn(1, N, 4, 128, generator=g, device=DEV).bfloat16()
    q8, q4, k8, k4, v8 = fused_int_prepass(q, k, v)
    torch.cuda.synchronize()
    kc_mean = plugin.key_mean_exact(k.cpu().permute(0, 2, 1, 3))          # [1,4,1,128]
    tok = torch.randint(0, N, (512,), generator=torch.Generator().manual_seed(1))
    tok = torch.cat([tok, torch.tensor([0, N - 1])])
    qs, ks, vs = q[:, tok].cpu(), k[:, tok].cpu(), v[:, tok].cpu()
    rq8, rq4, _, _, rv8 = plugin.int_prepass(qs, ks, vs)
    assert torch.equal(q8[:, tok].cpu(), rq8) and torch.equal(q4[:, tok].cpu(), rq4) and torch.equal(v8[:, tok].cpu(), rv8)
    from oracle import fake_quant as FQ
    kc = ks.permute(0, 2, 1, 3) - kc_mean
    assert torch.equal(k8[:, tok].cpu(), FQ.int_fake_quant(kc, 8, True, "per_token").permute(0, 2, 1, 3))
    assert torch.equal(k4[:, tok].cpu(), FQ.int_fake_quant(kc, 4, True, "per_token").permute(0, 2, 1, 3))


def test_prepass_errors():
    from longcontext_sqattn_paddle_amd.sqattn.fake_quant import fused_int_prepass

    q, k, v = (t.to(DEV) for t in _inputs(1, 64, 4, 2, seed=1))
    with pytest.raises(ValueError):
        fused_int_prepass(q, k, v, tensor_layout="XYZ")
    with pytest.raises(ValueError):
        fused_int_prepass(q[..., :64], k[..., :64], v[..., :64])
    with pytest.raises(AssertionError):
        fused_int_prepass(q, k[:, :32], v)            # token counts disagree
    with pytest.raises(ValueError):
        fused_int_prepass(q, k.half(), v)             # mixed dtypes
    with pytest.raises(RuntimeError):
        fused_int_prepass(q.cpu(), k, v)


@pytest.mark.parametrize("layout", ["NHD", "HND"])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_int8qk_prepass_codes_and_scales_are_the_quantisers_factors(layout, dtype):
    """sq_fake_quant_prepass_int8qk: the int8 codes and fp32 scales of the centred key equal the oracle's factors exactly
    (codes * scale rounded to the tensor dtype is the fake-quantised key of the other pre-pass), v8 is unchanged, the query
    is not touched."""
    from longcontext_sqattn_paddle_amd.sqattn.fake_quant import fused_int8qk_prepass, fused_int_prepass

    B, N, Hq, Hkv, D = 2, 333, 8, 2, 128
    g = torch.Generator().manual_seed(17)
    q = torch.randn(B, N, Hq, D, generator=g).to(dtype)
    k = (torch.randn(B, N, Hkv, D, generator=g) * torch.logspace(-4, 1, N)[None, :, None, None] + 0.25).to(dtype)
    v = torch.randn(B, N, Hkv, D, generator=g).to(dtype)
    kh = k.permute(0, 2, 1, 3)
    kc = kh - plugin.key_mean_exact(kh)
    codes_ref, scale_ref = FQ.int_quant_codes(kc, 8)                      # HND
    if layout == "HND":
        qd, kd, vd = (t.permute(0, 2, 1, 3).contiguous().to(DEV) for t in (q, k, v))
    else:
        qd, kd, vd = q.to(DEV), k.to(DEV), v.to(DEV)
    q_before = qd.clone()
    k_codes, k_scale, v8 = fused_int8qk_prepass(qd, kd, vd, layout)
    _, _, k8, _, v8_ref = fused_int_prepass(qd, kd, vd, want_4bit=False, tensor_layout=layout)
    torch.cuda.synchronize()
    assert torch.equal(qd, q_before) and torch.equal(v8, v8_ref)
    got_codes = k_codes.cpu() if layout == "HND" else k_codes.cpu().permute(0, 2, 1, 3)
    assert k_codes.dtype == torch.int8 and torch.equal(got_codes.float(), codes_ref)
    assert k_scale.shape == (B, Hkv, 384) and torch.equal(k_scale.cpu()[:, :, :N], scale_ref[..., 0]) and not bool(k_scale[:, :, N:].any())
    deq = (got_codes.float() * k_scale.cpu()[:, :, :N, None]).to(dtype)
    k8h = k8.cpu() if layout == "HND" else k8.cpu().permute(0, 2, 1, 3)
    assert torch.equal(deq.view(torch.int16), k8h.contiguous().view(torch.int16))


@pytest.mark.parametrize("B,Hkv", [(1, 1), (1, 4), (2, 3), (1, 8), (3, 3)])      # 1, 4 | 6, 8 in registers | 9 rows read twice
@pytest.mark.parametrize("N,layout,vq", [(1, "NHD", "int"), (64, "HND", "int"), (131, "NHD", "e4m3"), (190, "HND", "int"), (257, "NHD", "e5m2")])
def test_value_tiles_are_the_tiles_of_v8(B, Hkv, N, layout, vq):
    """The value as V^T tiles: v8's rounded values as fp16, transposed, keys 4 i .. 4 i + 3 of a group of 16 at 4 perm(i) with
    perm = 0 2 1 3, zeros past N -- bit for bit, since every step after v8's rounding is exact or the same rounding.  The other
    outputs of the call and an attention call over the tiles have the bits of the call with rows."""
    from longcontext_sqattn_paddle_amd.sqattn._prefill import run_prefill
    from longcontext_sqattn_paddle_amd.sqattn.fake_quant import fused_int_prepass

    print(f"case value tiles B={B} Hkv={Hkv} N={N} {layout} {vq}", flush=True)
    q, k, v = (t.to(DEV) for t in _inputs(B, N, 2 * Hkv, Hkv, seed=N + B, dtype=torch.bfloat16))
    if layout == "HND":
        q, k, v = (t.permute(0, 2, 1, 3).contiguous() for t in (q, k, v))
    rows = fused_int_prepass(q, k, v, tensor_layout=layout, v_qtype=vq)
    tiled = fused_int_prepass(q, k, v, tensor_layout=layout, v_qtype=vq, value_tiles=True)
    torch.cuda.synchronize()
    for a, b in zip(rows[:4], tiled[:4]):
        assert torch.equal(a.view(torch.int16), b.view(torch.int16))
    v8 = rows[4] if layout == "HND" else rows[4].permute(0, 2, 1, 3)
    nT = (N + 63) // 64
    pad = torch.zeros(B, Hkv, nT * 64, 128, dtype=torch.float16)
    pad[:, :, :N] = v8.cpu().half()
    want = pad.view(B, Hkv, nT, 4, 4, 4, 128)[:, :, :, :, [0, 2, 1, 3]].reshape(B, Hkv, nT, 64, 128).transpose(3, 4).contiguous()
    assert torch.equal(tiled[4].cpu().view(torch.int16), want.view(torch.int16))
    a, b = (run_prefill(rows[0], rows[2], rows[4] if t is None else None, tensor_layout=layout, output_dtype=torch.float32, v_tiles=t)
            for t in (None, tiled[4]))
    torch.cuda.synchronize()
    assert torch.equal(a, b)
    with pytest.raises(ValueError, match="bf16"):
        fused_int_prepass(q.half(), k.half(), v.half(), tensor_layout=layout, v_qtype=vq, value_tiles=True)


def test_value_tiles_of_another_shape_or_type_are_refused():
    """The kernel finds a tile by the call's own tile count, so tiles made for a longer prompt (more bytes than needed, other
    strides), of another type or as a flat buffer are an error, not another answer."""
    from longcontext_sqattn_paddle_amd.sqattn._prefill import run_prefill

    q, k, v = (t.to(DEV) for t in _inputs(1, 200, 4, 2, seed=5, dtype=torch.bfloat16))
    tiles = lambda *shape, dtype=torch.float16: torch.zeros(*shape, dtype=dtype, device=DEV)
    run_prefill(q, k, None, tensor_layout="NHD", v_tiles=tiles(1, 2, 4, 128, 64))
    for bad in (tiles(1, 2, 5, 128, 64), tiles(1, 2, 3, 128, 64), tiles(1, 3, 4, 128, 64), tiles(2, 2, 4, 128, 64), tiles(1, 2, 4, 64, 128),
                tiles(1, 2, 4 * 64 * 128), tiles(1, 2, 4, 64, 128).transpose(3, 4)):
        with pytest.raises(AssertionError, match="v_tiles must be"):
            run_prefill(q, k, None, tensor_layout="NHD", v_tiles=bad)
    for dtype in (torch.bfloat16, torch.float32):
        with pytest.raises(ValueError, match="v_tiles must be fp16"):
            run_prefill(q, k, None, tensor_layout="NHD", v_tiles=tiles(1, 2, 4, 128, 64, dtype=dtype))
    with pytest.raises(ValueError, match="not v_tiles"):
        run_prefill(q, k.to(torch.int8), v, tensor_layout="NHD", k_scale=torch.zeros(1, 2, 256, device=DEV), v_tiles=tiles(1, 2, 4, 128, 64))
    torch.cuda.synchronize()


@pytest.mark.parametrize("B,Hkv", [(1, 4), (2, 4), (3, 3)])
def test_value_tiles_of_special_values(B, Hkv):
    """NaN, infinities, values past fp16's range, signed zeros and subnormals come out of the tile pass as out of the rows."""
    from longcontext_sqattn_paddle_amd.sqattn.fake_quant import fused_int_prepass

    print(f"case value tiles special values B={B} Hkv={Hkv}", flush=True)
    N = 130
    q, k, v = _inputs(B, N, Hkv, Hkv, seed=9, dtype=torch.bfloat16)
    special = torch.tensor([math.nan, math.inf, -math.inf, 3.3e38, -3.3e38, 1e5, 7e4, -0.0, 0.0, 1e-40, -1e-39, 65504.0, 1e-5]).bfloat16()
    g = torch.Generator().manual_seed(10)
    at = torch.rand(v.shape, generator=g) < 0.1
    v[at] = special[torch.randint(0, len(special), (int(at.sum()),), generator=g)]
    v[:, :, 0] = 0                                                 # rows without a value and a whole NaN row
    v[:, 5] = math.nan
    q, k, v = (t.to(DEV) for t in (q, k, v))
    for vq in ("int", "e4m3", "e5m2"):
        rows = fused_int_prepass(q, k, v, tensor_layout="NHD", v_qtype=vq)[4].permute(0, 2, 1, 3)
        tiles = fused_int_prepass(q, k, v, tensor_layout="NHD", v_qtype=vq, value_tiles=True)[4].cpu()
        nT = (N + 63) // 64
        pad = torch.zeros(B, Hkv, nT * 64, 128, dtype=torch.float16)
        pad[:, :, :N] = rows.cpu().half()
        want = pad.view(B, Hkv, nT, 4, 4, 4, 128)[:, :, :, :, [0, 2, 1, 3]].reshape(B, Hkv, nT, 64, 128).transpose(3, 4).contiguous()
        assert torch.equal(tiles.isnan(), want.isnan()) and not bool(want.isfinite().all())
        assert torch.equal(tiles.view(torch.int16)[~want.isnan()], want.view(torch.int16)[~want.isnan()])
