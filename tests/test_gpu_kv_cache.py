"""KV-cache row kernels and the `flash_attn_cache` mirror against oracle/kv_cache.py: bit-exact (pure copies).

Follows the call pattern of the reference runtime (model_hub/LLM.py:64-68 prefill, :102-105 decode)."""
import pytest
import torch

from oracle import attention as A
from oracle import kv_cache as KC

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _cache(valid_start, layers=2, batch=2, max_length=300, kv_heads=4, heads=28, dim=128, dtype=torch.bfloat16):
    from longcontext_sqattn_paddle_amd.cache_hub.flash_attn_cache import flash_attn_cache

    mapping = {str(i): DEV for i in range(layers)}
    return flash_attn_cache(valid_start, layers, batch, max_length, kv_heads, heads, dim, dtype, mapping, 1, 7)


def _rand(shape, seed, dtype=torch.bfloat16):
    return torch.randn(*shape, generator=torch.Generator().manual_seed(seed)).to(dtype)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_prefill_store_and_decode_append_match_oracle(dtype):
    print(f"case kv-cache store/append {dtype}", flush=True)
    layers, B, L, H, D = 2, 2, 300, 4, 128
    starts = [0, 37]
    lens_prompt = [200, 261]
    cache = _cache(starts, layers, B, L, H, 28, D, dtype)
    for kc, vc in zip(cache.key_cache, cache.value_cache):   # recognisable background: untouched rows must keep it
        kc.fill_(3.0)
        vc.fill_(-3.0)
    ref_k = [torch.full((B, L, H, D), 3.0, dtype=dtype) for _ in range(layers)]
    ref_v = [torch.full((B, L, H, D), -3.0, dtype=dtype) for _ in range(layers)]
    ref_len = torch.zeros(B, dtype=torch.int32)
    for b in range(B):
        for layer in range(layers):
            ks, vs = _rand((1, lens_prompt[b], H, D), 10 * b + layer, dtype), _rand((1, lens_prompt[b], H, D), 50 + 10 * b + layer, dtype)
            rk, rv = cache.prefill_update_kv_cache(None, ks.to(DEV), vs.to(DEV), layer, b)
            cache.sync(layer, b)
            assert torch.equal(rk.cpu(), ks[:, starts[b]:]) and torch.equal(rv.cpu(), vs[:, starts[b]:])
            ref_len[b] = KC.prefill_store(ref_k[layer], ref_v[layer], ks, vs, b, starts[b])
    torch.cuda.synchronize()
    assert cache.valid_length.cpu().tolist() == ref_len.tolist()
    assert cache.context == lens_prompt[-1]
    for step in range(3):
        for layer in range(layers):
            kn, vn = _rand((B, 1, H, D), 100 + 7 * step + layer, dtype), _rand((B, 1, H, D), 200 + 7 * step + layer, dtype)
            kc, vc = cache.decode_update_kv_cache(kn.to(DEV), vn.to(DEV), layer)
            assert kc is cache.key_cache[layer] and vc is cache.value_cache[layer]
            att = KC.decode_append(ref_k[layer], ref_v[layer], kn, vn, ref_len, advance=layer == layers - 1)
            assert cache.attend_length.cpu().tolist() == att.tolist()
        assert cache.valid_length.cpu().tolist() == ref_len.tolist()
    for layer in range(layers):
        assert torch.equal(cache.key_cache[layer].cpu(), ref_k[layer]), f"key cache of layer {layer}"
        assert torch.equal(cache.value_cache[layer].cpu(), ref_v[layer]), f"value cache of layer {layer}"
    assert cache.context == lens_prompt[-1] + 3


def test_store_reads_strided_views_of_a_fused_projection():
    """key/value states are usually views into one [1, T, (Hq + 2 Hkv) * D] projection output."""
    print("case kv-cache strided store", flush=True)
    T, Hq, H, D = 333, 8, 2, 128
    qkv = _rand((1, T, (Hq + 2 * H) * D), 5).to(DEV)
    ks = qkv[:, :, Hq * D:(Hq + H) * D].view(1, T, H, D)
    vs = qkv[:, :, (Hq + H) * D:].view(1, T, H, D)
    assert not ks.is_contiguous()
    cache = _cache(5, layers=1, batch=1, max_length=400, kv_heads=H, heads=Hq)
    cache.prefill_update_kv_cache(None, ks, vs, 0, 0)
    cache.sync(0, 0)
    torch.cuda.synchronize()
    assert torch.equal(cache.key_cache[0][0, :T - 5], ks[0, 5:]) and torch.equal(cache.value_cache[0][0, :T - 5], vs[0, 5:])


def test_decode_attention_over_the_cache_uses_the_valid_prefix_only():
    """append + decode attention with `attend_length` == exact attention over each sequence's own tokens; the rows
    behind them hold NaN and must not leak in."""
    from longcontext_sqattn_paddle_amd.sqattn.attn_triton_decode import attn_decode

    print("case kv-cache decode attention", flush=True)
    B, L, Hq, H, D = 2, 1024, 28, 4, 128
    lens = [700, 401]
    cache = _cache(0, layers=1, batch=B, max_length=L, kv_heads=H, heads=Hq)
    cache.key_cache[0].fill_(float("nan"))
    cache.value_cache[0].fill_(float("nan"))
    ks = [_rand((1, n, H, D), 20 + i) for i, n in enumerate(lens)]
    vs = [_rand((1, n, H, D), 30 + i) for i, n in enumerate(lens)]
    for b in range(B):
        cache.prefill_update_kv_cache(None, ks[b].to(DEV), vs[b].to(DEV), 0, b)
        cache.sync(0, b)
    kn, vn, q = _rand((B, 1, H, D), 40), _rand((B, 1, H, D), 41), _rand((B, 1, Hq, D), 42)
    kc, vc = cache.decode_update_kv_cache(kn.to(DEV), vn.to(DEV), 0)
    out = attn_decode(q.to(DEV), kc, vc, "NHD", torch.float32, seqlens=cache.attend_length)
    torch.cuda.synchronize()
    for b in range(B):
        kb = torch.cat([ks[b], kn[b:b + 1]], dim=1).permute(0, 2, 1, 3)
        vb = torch.cat([vs[b], vn[b:b + 1]], dim=1).permute(0, 2, 1, 3)
        ref, _ = A.exact_attention(q[b:b + 1].permute(0, 2, 1, 3), kb, vb, causal=False)
        err = float((out[b].cpu().double() - ref[0].permute(1, 0, 2)).abs().max())
        assert err < 2e-3, f"sequence {b}: max abs err {err}"   # bf16 inputs, fp32 accumulation (decode tests use 2e-4 * rms)


def test_store_runs_on_the_callers_stream_and_sync_joins_another_one():
    """One hardware queue per request: the copy is queued where the caller's work is, and a reader on a second stream sees the
    rows after `sync`, without a device-wide wait."""
    print("case kv-cache store stream", flush=True)
    T, H, D = 4096, 4, 128
    ks, vs = _rand((1, T, H, D), 61).to(DEV), _rand((1, T, H, D), 62).to(DEV)
    cache = _cache(0, layers=1, batch=1, max_length=T, kv_heads=H)
    cache.sync(0, 0)                                                  # nothing to wait for yet
    queued = []

    class Spy:
        def __getattr__(self, name, lib=cache._lib):
            def call(*args):
                queued.append((name, args[-1]))
                return getattr(lib, name)(*args)
            return call

    cache._lib = Spy()
    first, second = torch.cuda.Stream(), torch.cuda.Stream()
    torch.cuda.synchronize()
    with torch.cuda.stream(first):
        x = torch.randn(4096, 4096, device=DEV)
        for _ in range(20):
            x = x @ x * 1e-3                                          # keeps the first stream busy while the second one reads
        cache.prefill_update_kv_cache(None, ks, vs, 0, 0)
    with torch.cuda.stream(second):
        cache.sync(0, 0)
        k, v, n = cache.key_cache[0].clone(), cache.value_cache[0].clone(), cache.valid_length.clone()
    torch.cuda.synchronize()
    assert queued == [("sq_kv_cache_store", first.cuda_stream)]
    assert torch.equal(k, ks) and torch.equal(v, vs) and int(n) == T


def test_full_size_store_128k():
    """A prompt of 131072 tokens with 4 kv heads: 268 MB into the cache, checked on the device."""
    print("case kv-cache store 128K", flush=True)
    T, H, D = 131072, 4, 128
    g = torch.Generator(device=DEV).manual_seed(9)
    ks = torch.randn(1, T, H, D, generator=g, device=DEV).bfloat16()
    vs = torch.randn(1, T, H, D, generator=g, device=DEV).bfloat16()
    cache = _cache(128, layers=1, batch=1, max_length=T + 64, kv_heads=H)
    cache.key_cache[0].zero_()
    cache.value_cache[0].zero_()
    cache.prefill_update_kv_cache(None, ks, vs, 0, 0)
    cache.sync(0, 0)
    torch.cuda.synchronize()
    n = T - 128
    assert torch.equal(cache.key_cache[0][0, :n], ks[0, 128:]) and torch.equal(cache.value_cache[0][0, :n], vs[0, 128:])
    assert float(cache.key_cache[0][0, n:].abs().sum()) == 0.0 and float(cache.value_cache[0][0, n:].abs().sum()) == 0.0


def test_errors():
    from longcontext_sqattn_paddle_amd.cache_hub.flash_attn_cache import flash_attn_cache

    print("case kv-cache errors", flush=True)
    cache = _cache(0, layers=1, batch=1, max_length=64, kv_heads=2, heads=4)
    ks = torch.zeros(1, 65, 2, 128, dtype=torch.bfloat16, device=DEV)
    with pytest.raises(AssertionError, match="exceeds max length"):
        cache.prefill_update_kv_cache(None, ks, ks, 0, 0)
    with pytest.raises(AssertionError, match="single batch"):
        cache.prefill_update_kv_cache(None, ks[:, :8].expand(2, -1, -1, -1), ks[:, :8].expand(2, -1, -1, -1), 0, 0)
    with pytest.raises(ValueError, match="same dtype|one 16-bit dtype|must share"):
        cache.prefill_update_kv_cache(None, ks[:, :8].half(), ks[:, :8].half(), 0, 0)
    full = torch.zeros(1, 64, 2, 128, dtype=torch.bfloat16, device=DEV)
    cache.prefill_update_kv_cache(None, full, full, 0, 0)
    cache.sync(0, 0)
    with pytest.raises(IndexError, match="full"):
        cache.decode_update_kv_cache(full[:, :1], full[:, :1], 0)
    with pytest.raises(ValueError, match="one GPU"):
        flash_attn_cache(0, 1, 1, 64, 2, 4, 128, torch.bfloat16, {"0": DEV}, 2, 7)
    with pytest.raises(MemoryError):
        _cache(0, layers=64, batch=64, max_length=1 << 20, kv_heads=8)
