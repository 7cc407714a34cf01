"""GPU parity: prefill kernel (through the C ABI) against the CPU oracle.

Stated tolerances.  Kernel vs the same-algorithm oracle (identical quantisation points; only v_exp_f32 and
fp32 summation order differ): without P quantisation max|d| <= 2e-3 * rms(out) + 2^-11 * max|out| -- the second term
because the kernel rounds p to fp16 relative to a reference point that may trail the row's running maximum by up to
2^8 (the same probability with the same relative rounding error 2^-11 as the reference's, but a dominant key no longer
has p = 1 exactly); with e4m3 P a few
probabilities sit within an ulp of a rounding boundary and flip to the neighbouring e4m3 value, so the
check is cosine >= 0.99999, 99.9 % of elements within 2e-3 * rms and every element within 0.25 * rms.
Kernel vs exact attention: cosine >= 0.999 (the bar of the benchmark configuration).
"""
import math

import pytest
import torch

from oracle import attention as A
from oracle import inputs

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _cos(a, b):
    a, b = a.double().flatten(), b.double().flatten()
    return float(a @ b / (a.norm() * b.norm()))


def _check(out, ref, quantised, q_tol=2e-3):
    out, ref = out.double().cpu(), ref.double()
    rms = float(ref.pow(2).mean().sqrt())
    d = (out - ref).abs()
    if not quantised:
        assert float(d.max()) <= 2e-3 * rms + 2.0 ** -11 * float(ref.abs().max()), (float(d.max()), rms)
    else:
        assert _cos(out, ref) >= 0.99999
        assert float(torch.quantile(d.flatten()[:: max(1, d.numel() // 1000000)], 0.999)) <= q_tol * rms
        assert float(d.max()) <= 0.25 * rms, (float(d.max()), rms)


def _rand(B, Hq, Hkv, N, D, seed, dtype=torch.bfloat16, scale=1.0):
    g = torch.Generator().manual_seed(seed)
    q = (torch.randn(B, Hq, N, D, generator=g) * scale).to(dtype)
    k = (torch.randn(B, Hkv, N, D, generator=g) * scale).to(dtype)
    v = (torch.randn(B, Hkv, N, D, generator=g) * scale).to(dtype)
    return q, k, v


@pytest.mark.parametrize("B,Hq,Hkv,N", [(1, 4, 2, 512), (2, 14, 2, 700), (1, 2, 1, 64), (1, 3, 3, 1000)])
@pytest.mark.parametrize("mode", [A.P_NONE, A.P_STATIC448, A.P_BLOCK_ABSMAX, 3])
def test_causal_matches_oracle(B, Hq, Hkv, N, mode):
    from longcontext_sqattn_paddle_amd.sqattn.attn_triton import attn_causal

    print(f"case prefill causal B={B} Hq={Hq} Hkv={Hkv} N={N} p_quant={mode}", flush=True)
    q, k, v = _rand(B, Hq, Hkv, N, 128, 100 + N)
    # kernel mode 3 is the static-448 grid with the scale folded into the exponent: same oracle, same tolerance
    ref, lse_ref = A.prefill_blockwise(q, k, v, p_quant=A.P_STATIC448 if mode == 3 else mode, out_dtype=torch.float32)
    out, lse = attn_causal(q.to(DEV), k.to(DEV), v.to(DEV), "HND", torch.float32, return_lse=True, p_quant=mode)
    torch.cuda.synchronize()
    _check(out, ref, mode != A.P_NONE)
    assert torch.allclose(lse.cpu(), lse_ref, atol=2e-4)
    exact, _ = A.exact_attention(q, k, v)
    assert _cos(out.cpu(), exact) >= 0.999


@pytest.mark.parametrize("mode", [4, 5])
@pytest.mark.parametrize("B,Hq,Hkv,N,layout", [(1, 4, 2, 512, "HND"), (2, 14, 2, 700, "NHD"), (1, 7, 1, 2048, "HND")])
def test_fp8_pv_mode_matches_oracle(B, Hq, Hkv, N, layout, mode):
    """Modes 4 and 5 (no reference counterpart): e4m3 P *and* e4m3 V (per batch/kv-head/channel scale) on the fp8
    MFMA; mode 5 adds one power-of-two scale per query row and 64-key tile to P."""
    from longcontext_sqattn_paddle_amd.sqattn.attn_triton import attn_causal

    print(f"case prefill fp8-pv mode={mode} B={B} Hq={Hq} Hkv={Hkv} N={N} {layout}", flush=True)
    q, k, v = inputs.prefill_inputs(B, Hq, Hkv, N, 128, seed=200 + N) if N == 2048 else _rand(B, Hq, Hkv, N, 128, 200 + N)
    ref, lse_ref = A.prefill_blockwise(q, k, v, p_quant=A.P_STATIC448_GRID if mode == 4 else A.P_MX_ROW, v_quant="e4m3_channel",
                                       out_dtype=torch.float32)
    args = [t.to(DEV) for t in (q, k, v)]
    if layout == "NHD":
        args = [t.permute(0, 2, 1, 3).contiguous() for t in args]
    out, lse = attn_causal(*args, layout, torch.float32, return_lse=True, p_quant=mode)
    torch.cuda.synchronize()
    if layout == "NHD":
        out = out.permute(0, 2, 1, 3)
    # 99.9 % of elements within 5e-3 * rms here (2e-3 for the fp16 P.V modes): the fp8 matrix instruction sums its 64
    # products with its own internal alignment, which shows on near-uniform rows of thousands of keys
    _check(out, ref, True, q_tol=5e-3)
    assert torch.allclose(lse.cpu(), lse_ref, atol=2e-4)
    exact, _ = A.exact_attention(q, k, v)
    assert _cos(out.cpu(), exact) >= 0.999   # thin margin by construction: e4m3 on both operands (about 0.9995)


def test_block_scaled_p_keeps_small_probabilities_the_static_scale_flushes():
    """Attention sink: key 0 outscores every other key by about 2^17, so all later tiles hold probabilities near
    2^-17 whose 448-fold lies in the subnormal range of e4m3 (steps of 2^-9) and partly rounds to zero under the
    static scale (modes 3 and 4), although the 8192 of them together carry a few percent of the row.  The per-row
    block scale of mode 5 moves each tile's row sum to [128, 256), i.e. its probabilities back to three mantissa bits."""
    from longcontext_sqattn_paddle_amd.sqattn.attn_triton import attn_causal

    N, D = 8192, 128
    g = torch.Generator().manual_seed(77)
    q = torch.randn(1, 4, N, D, generator=g) * 0.3
    k = torch.randn(1, 2, N, D, generator=g) * 0.3
    v = torch.randn(1, 2, N, D, generator=g)
    q[..., 0] = 4.0
    k[..., 0] *= 0.1
    k[:, :, 0, :] = 0.0
    k[:, :, 0, 0] = 17.0 / (4.0 * 1.44269504 / D ** 0.5)   # score of key 0 in log2 units: 17 above the rest
    v[:, :, 0, :] = 0.0   # the sink carries no value, so the output is made of the small probabilities alone
    q, k, v = q.to(torch.bfloat16), k.to(torch.bfloat16), v.to(torch.bfloat16)
    exact, _ = A.exact_attention(q, k, v)
    errs = {}
    for mode in (3, 4, 5):
        print(f"case prefill sink mode={mode}", flush=True)
        out = attn_causal(q.to(DEV), k.to(DEV), v.to(DEV), "HND", torch.float32, p_quant=mode)
        torch.cuda.synchronize()
        errs[mode] = float((out.cpu().double()[:, :, N // 2:] - exact[:, :, N // 2:]).pow(2).mean().sqrt())
    print("rms error vs exact attention, rows N/2..N:", errs, flush=True)
    assert errs[5] <= 0.5 * errs[4]


def _climbing_scores(step_up, jump):
    N, D = 1536, 128
    g = torch.Generator().manual_seed(91)
    q = torch.randn(1, 4, N, D, generator=g) * 0.5
    k = torch.randn(1, 2, N, D, generator=g) * 0.5
    v = torch.randn(1, 2, N, D, generator=g)
    ramp = torch.arange(N, dtype=torch.float32) / 64.0 * step_up
    ramp[700:] += jump          # key 700 sits in the middle of a tile, 1000 on a tile that is a diagonal tile for some rows
    ramp[1000:] += jump / 2
    q[..., 0] = 1.0
    k[:, :, :, 0] = (ramp * (D ** 0.5 / 1.44269504))[None, None]
    return q.bfloat16(), k.bfloat16(), v.bfloat16()


@pytest.mark.parametrize("step_up,jump", [(6.0, 40.0), (0.0, 140.0), (3.0, 17.0)])
def test_block_scaled_p_reference_moves_and_overflows(step_up, jump):
    """Mode 5 forms a tile's probabilities against the standing reference point without looking at the scores first.
    Scores that climb by `step_up` (log2) per 64-key tile push the row sums past 2^16 every few tiles (the reference then
    moves up by whole binades, which rescales the tile packed just before as well); one key that leads everything before
    it by `jump` does the same in one step, and by 140 it overflows 2^(s - reference): the tile is formed again from the
    key rows in memory.  Against the oracle's restatement of the same rule, and against exact attention."""
    from longcontext_sqattn_paddle_amd.sqattn.attn_triton import attn_causal

    print(f"case prefill mode 5 reference moves step_up={step_up} jump={jump}", flush=True)
    q, k, v = _climbing_scores(step_up, jump)
    ref, lse_ref = A.prefill_blockwise(q, k, v, p_quant=A.P_MX_ROW, v_quant="e4m3_channel", out_dtype=torch.float32)
    out, lse = attn_causal(q.to(DEV), k.to(DEV), v.to(DEV), "HND", torch.float32, return_lse=True, p_quant=5)
    torch.cuda.synchronize()
    assert bool(torch.isfinite(out).all()) and bool(torch.isfinite(lse).all())
    # The scores here reach 200 and more (log2), so their fp32 rounding (1e-4, and the MFMA adds the products in another
    # order than the oracle) moves a probability by 1e-4 relative -- enough to send one in a thousand across an e4m3
    # rounding boundary, a step of 6 %.  Rows like these hang on a dozen leading keys each, so such a flip shows in the
    # row (up to 0.1 rms) where on random data it disappears: a few percent of the rows differ visibly, none grossly.
    err = (out.cpu().double() - ref.double()).abs()
    rms = float(ref.double().pow(2).mean().sqrt())
    assert float(torch.quantile(err.flatten()[:: 7], 0.90)) <= 5e-3 * rms
    assert float(err.max()) <= 0.25 * rms
    assert _cos(out.cpu(), ref) >= 0.9995
    assert torch.allclose(lse.cpu(), lse_ref, atol=2e-4, rtol=1e-6)       # the log-sum-exp has no quantised quantity in it
    exact, lse_exact = A.exact_attention(q, k, v)
    assert _cos(out.cpu(), exact) >= 0.999
    assert torch.allclose(lse.cpu(), lse_exact.float(), atol=2e-2, rtol=5e-3)


def _pattern_scores(pattern, N):
    D = 128
    g = torch.Generator().manual_seed(1001)
    q = torch.randn(1, 4, N, D, generator=g) * 0.5
    k = torch.randn(1, 2, N, D, generator=g) * 0.5
    v = torch.randn(1, 2, N, D, generator=g)
    pos = torch.arange(N, dtype=torch.float32)
    r = torch.zeros(N)
    if pattern == "spikes":
        r[torch.randint(0, N, (6,), generator=g)] = torch.tensor([20.0, 45.0, 90.0, 135.0, 170.0, 60.0])
    elif pattern == "late_giant":
        r[N * 3 // 4:] = 150.0
        r[N // 3: N // 3 + 5] = 30.0
    elif pattern == "alternating":
        r = ((pos // 64) % 2) * 85.0
    elif pattern == "edge_spikes":
        r[63::64] = 90.0
        r[64::128] = 100.0
    else:
        r = -pos / 64.0 * 7.0
    q[..., 0] = 1.0
    k[:, :, :, 0] = (r * (D ** 0.5 / 1.44269504))[None, None]
    return q.bfloat16(), k.bfloat16(), v.bfloat16()


@pytest.mark.parametrize("pattern", ["spikes", "late_giant", "alternating", "edge_spikes", "ramp_down"])
@pytest.mark.parametrize("N,window", [(777, None), (1536, (64, 128, 256)), (2304, (0, 64, 64))])
def test_block_scaled_p_score_patterns_with_and_without_windows(pattern, N, window):
    """Mode 5 on score patterns chosen against its rare paths, full causal and with sink + windows (where a wave leaves
    and re-enters its key range with a tile pending): lone keys 20 to 170 (log2) above the rest, a block of keys 150 above
    everything before it, tiles that alternate between two levels 85 apart, spikes on the last key of a tile and the
    first of the next, scores that fall by 7 per tile.  Same criteria as the test above."""
    from longcontext_sqattn_paddle_amd.sqattn._prefill import run_prefill

    print(f"case prefill mode 5 pattern={pattern} N={N} window={window}", flush=True)
    q, k, v = _pattern_scores(pattern, N)
    kw = {} if window is None else dict(block_m=64, sink=window[0], w8=[window[1]] * 4, w4=[window[2]] * 4)
    ref, lse_ref = A.prefill_blockwise(q, k, v, p_quant=A.P_MX_ROW, v_quant="e4m3_channel", out_dtype=torch.float32, **kw)
    out, lse = run_prefill(q.to(DEV), k.to(DEV), v.to(DEV), tensor_layout="HND", output_dtype=torch.float32, return_lse=True,
                           p_quant=5, window=kw or None)
    torch.cuda.synchronize()
    assert bool(torch.isfinite(out).all()) and bool(torch.isfinite(lse).all())
    # (a leading probability that lands on the other side of an e4m3 rounding boundary than in the oracle moves a row
    # that hangs on two or three keys by up to 0.06 |v|, which is most of the output's rms here: no bound on single
    # elements, a tight one on their bulk and on the whole)
    err = (out.cpu().double() - ref.double()).abs()
    rms = float(ref.double().pow(2).mean().sqrt())
    assert float(torch.quantile(err.flatten()[:: 3], 0.90)) <= 5e-3 * rms
    assert float(err.max()) <= 1.0 * rms
    assert _cos(out.cpu(), ref) >= 0.9999
    assert torch.allclose(lse.cpu(), lse_ref, atol=3e-4, rtol=2e-6)


def test_nhd_layout_bf16_out_and_gqa_7():
    from longcontext_sqattn_paddle_amd.sqattn.attn_triton import attn_causal

    q, k, v = _rand(1, 28, 4, 384, 128, 7)
    ref, _ = A.prefill_blockwise(q, k, v, p_quant=A.P_STATIC448, out_dtype=torch.float32)
    qn, kn, vn = (t.permute(0, 2, 1, 3).contiguous().to(DEV) for t in (q, k, v))
    out = attn_causal(qn, kn, vn, "NHD", torch.bfloat16, is_P_fp8_quant=True)
    torch.cuda.synchronize()
    assert out.shape == (1, 384, 28, 128) and out.dtype == torch.bfloat16
    o = out.permute(0, 2, 1, 3).float().cpu()
    assert _cos(o, ref) >= 0.9999
    assert float((o - ref).abs().max()) <= 2 ** -7 * float(ref.abs().max()) + 0.25 * float(ref.pow(2).mean().sqrt())


@pytest.mark.parametrize("mode", [0, 2, 5])
@pytest.mark.parametrize("N,heads", [(1, 2), (31, 2), (257, 2), (290, 128)])
def test_16_bit_outputs_are_the_rounded_fp32_ones_and_stay_in_their_rows(mode, N, heads):
    """16-bit outputs leave through LDS, fp32 ones from the accumulators: the same values, rounded once.  (290 rows of 128 heads:
    workgroups of 256 rows, the others of 128.)  The output is a view with other rows and channels around it."""
    from longcontext_sqattn_paddle_amd.sqattn._prefill import run_prefill

    print(f"case 16-bit outputs mode={mode} N={N} heads={heads}", flush=True)
    q, k, v = (t.to(DEV).transpose(1, 2).contiguous() for t in _rand(1, heads, 2, N, 128, 40 + N))
    for dt in (torch.bfloat16, torch.float16):
        qd, kd, vd = q.to(dt), k.to(dt), v.to(dt)
        ref = run_prefill(qd, kd, vd, tensor_layout="NHD", output_dtype=torch.float32, p_quant=mode)
        around = torch.full((1, N + 40, heads + 1, 136), -7.0, dtype=dt, device=DEV)
        view = around[:, :N, :heads, :128]
        run_prefill(qd, kd, vd, tensor_layout="NHD", output_dtype=dt, p_quant=mode, out=view)
        torch.cuda.synchronize()
        assert torch.equal(view, ref.to(dt))
        view.fill_(-7.0)
        assert bool((around == -7.0).all())


# 256-row workgroups with windows, those of two query blocks (separate 4-bit operands, 128-row blocks), and 64-row workgroups
@pytest.mark.parametrize("mode", [0, 2])
@pytest.mark.parametrize("N", [513, 770])
@pytest.mark.parametrize("block_m,own4", [(64, False), (128, True), (64, True)])
def test_16_bit_outputs_of_windowed_launches(mode, N, block_m, own4):
    from longcontext_sqattn_paddle_amd.sqattn._prefill import prefill_workspace, run_prefill

    heads = 64
    print(f"case 16-bit outputs mode={mode} N={N} block_m={block_m} own4={own4}", flush=True)
    q, k, v = (t.to(DEV).transpose(1, 2).contiguous() for t in _rand(1, heads, 2, N, 128, 60 + N))
    for dt in (torch.bfloat16, torch.float16):
        qd, kd, vd = q.to(dt), k.to(dt), v.to(dt)
        kw = dict(tensor_layout="NHD", p_quant=mode, workspace=prefill_workspace(1, 2, N, qd.device),
                  window=dict(block_m=block_m, sink=64, w8=[128] * heads, w4=[256] * heads))
        if own4:
            kw.update(q4=(qd * 0.9).contiguous(), k4=(kd * 1.1).contiguous())
        ref = run_prefill(qd, kd, vd, output_dtype=torch.float32, **kw)
        around = torch.full((1, N + 40, heads + 1, 136), -7.0, dtype=dt, device=DEV)
        view = around[:, :N, :heads, :128]
        run_prefill(qd, kd, vd, output_dtype=dt, out=view, **kw)
        torch.cuda.synchronize()
        assert torch.equal(view, ref.to(dt))
        view.fill_(-7.0)
        assert bool((around == -7.0).all())


def test_fp16_inputs_and_head_dim_64():
    from longcontext_sqattn_paddle_amd.sqattn.attn_triton import attn_causal

    q, k, v = _rand(1, 4, 2, 320, 64, 9, dtype=torch.float16)
    ref, lse_ref = A.prefill_blockwise(q, k, v, out_dtype=torch.float32)
    out, lse = attn_causal(q.to(DEV), k.to(DEV), v.to(DEV), "HND", torch.float32, return_lse=True)
    torch.cuda.synchronize()
    assert out.shape == (1, 4, 320, 64)
    _check(out, ref, False)
    assert torch.allclose(lse.cpu(), lse_ref, atol=2e-4)


def test_config2_style_inputs_with_k_outliers():
    from longcontext_sqattn_paddle_amd.sqattn.attn_triton import attn_causal

    q, k, v = inputs.prefill_inputs(1, 7, 1, 2048, 128, seed=2)
    ref, _ = A.prefill_blockwise(q, k, v, p_quant=A.P_STATIC448, out_dtype=torch.float32)
    out = attn_causal(q.to(DEV), k.to(DEV), v.to(DEV), "HND", torch.float32, is_P_fp8_quant=True)
    torch.cuda.synchronize()
    _check(out, ref, True)
    exact, _ = A.exact_attention(q, k, v)
    assert _cos(out.cpu(), exact) >= 0.999


def test_chunked_prefill_offset():
    from longcontext_sqattn_paddle_amd.sqattn.attn_triton import attn_causal

    q, k, v = _rand(1, 4, 2, 768, 128, 11)
    ref, lse_ref = A.prefill_blockwise(q, k, v, out_dtype=torch.float32)
    out, lse = attn_causal(q[:, :, 512:].contiguous().to(DEV), k.to(DEV), v.to(DEV), "HND", torch.float32,
                           return_lse=True, q_offset=512)
    torch.cuda.synchronize()
    _check(out, ref[:, :, 512:], False)
    assert torch.allclose(lse.cpu(), lse_ref[:, :, 512:], atol=2e-4)


@pytest.mark.parametrize("B,Hq,Hkv,N,offset,window", [
    (1, 4, 1, 4096, 0, None),            # shares of unequal blocks
    (1, 2, 2, 1217, 0, None),            # ragged: last block of 193 rows, last tile of one key
    (1, 2, 1, 1025, 0, None),            # last block of a single row: seven of its waves have none
    (3, 2, 1, 300, 2048, None),          # a chunk behind a context, several sequences
    (1, 2, 1, 64, 4096, None),           # one 64-row block over 65 tiles
    (1, 4, 2, 4000, 0, (256, 0.125, 0.75)),   # sink and windows: a share may begin inside the sink or at the jump behind it
    (1, 2, 1, 3008, 0, (64, 512, 2048)),     # absolute windows with their own 4-bit operands (tiles walked twice)
])
def test_split_key_ranges_match_unsplit_launch_and_oracle(B, Hq, Hkv, N, offset, window):
    """Launches too small to fill the chip split the key range of a query block over several workgroups (given the workspace
    for it).  A row's parts start from reference points of their own, so p differs by its fp16 rounding: the unquantised
    criterion of this file, against the oracle and against the unsplit launch (twice that criterion: both sides round)."""
    from longcontext_sqattn_paddle_amd import _native as NV
    from longcontext_sqattn_paddle_amd.sqattn._prefill import prefill_workspace
    from longcontext_sqattn_paddle_amd.sqattn.attn_triton import attn_causal
    from longcontext_sqattn_paddle_amd.sqattn.attn_triton_mix_bad import attn_hierarchical_window
    from longcontext_sqattn_paddle_amd.sqattn.attn_triton_mix_relative import attn_hierarchical_relative_window
    from oracle import fake_quant as FQ

    print(f"case prefill split B={B} Hq={Hq} Hkv={Hkv} N={N} offset={offset} window={window}", flush=True)
    _, k, v = _rand(B, Hq, Hkv, offset + N, 128, 300 + N)
    q = _rand(B, Hq, Hkv, N, 128, 301 + N)[0]
    qd, kd, vd = q.to(DEV), k.to(DEV), v.to(DEV)
    small = prefill_workspace(B, Hkv, offset + N, qd.device)     # no room for parts: the unsplit launch
    if window is None:
        ref, lse_ref = A.exact_attention(A.fold_scale(q, 128), k, v, causal=True, q_offset=offset, score_scale=math.log(2.0))
        call = lambda **kw: attn_causal(qd, kd, vd, "HND", torch.float32, return_lse=True, q_offset=offset, **kw)
        assert NV.lib().sq_prefill_workspace_bytes_split(B, Hq, Hkv, N, offset + N, NV.PrefillParams(q_offset=offset)) > small.numel() * 2
    elif isinstance(window[1], float):
        w8, w4 = ([A.window_size_relative(r, N)] * Hq for r in window[1:])
        ref, lse_ref = A.prefill_blockwise(q, k, v, block_m=64, sink=window[0], w8=w8, w4=w4, out_dtype=torch.float32)
        call = lambda **kw: attn_hierarchical_relative_window(qd, kd, qd, kd, vd, window[1], window[2], window[0], "HND", torch.float32,
                                                              return_lse=True, **kw)
    else:
        q4, k4 = FQ.int_fake_quant(q, 4, True, "per_token"), FQ.int_fake_quant(k, 4, True, "per_token")
        ref, lse_ref = A.prefill_blockwise(q, k, v, block_m=128, sink=window[0], w8=[window[1]] * Hq, w4=[window[2]] * Hq, q4=q4, k4=k4,
                                           out_dtype=torch.float32)
        q4d, k4d = q4.to(DEV), k4.to(DEV)
        call = lambda **kw: attn_hierarchical_window(qd, kd, q4d, k4d, vd, window[1], window[2], window[0], "HND", torch.float32,
                                                     return_lse=True, **kw)
    out, lse = call()
    whole, lse_whole = call(workspace=small)
    torch.cuda.synchronize()
    _check(out, ref.reshape(out.shape), False)
    _check(whole, ref.reshape(out.shape), False)
    assert torch.allclose(lse.cpu(), lse_ref.reshape(lse.shape).float(), atol=2e-4)
    assert torch.allclose(lse, lse_whole, atol=2e-4)
    assert not torch.equal(out, whole)     # the workspace the wrapper takes by itself does split these launches


@pytest.mark.parametrize("mode", [1, 2, 3, 4])
@pytest.mark.parametrize("N,offset", [(3010, 0), (200, 3072)])
def test_split_key_ranges_keep_the_e4m3_grid(mode, N, offset):
    """The parts of a split row start from the reference point the whole row would have had there (a pass that forms the
    parts' row maxima), so the e4m3 grid is the unsplit launch's: what differs is a score's last bit, which moves the few
    probabilities that sit on a rounding boundary by one step of the grid (up to 2^-3 of themselves).  With scores of unit
    variance a row of n keys averages about n / e of them, so one such step moves an output element by about
    2^-3 / sqrt(n / e) of its rms: 4e-3 at n = 3000.  Against the unsplit launch: cosine, 99.9 % of the elements within two
    such steps (8e-3 rms), all within 0.25 rms."""
    from longcontext_sqattn_paddle_amd.sqattn._prefill import prefill_workspace
    from longcontext_sqattn_paddle_amd.sqattn.attn_triton import attn_causal

    print(f"case prefill split grid mode={mode} N={N} offset={offset}", flush=True)
    _, k, v = _rand(1, 3, 1, offset + N, 128, 41)
    q = _rand(1, 3, 1, N, 128, 42)[0]
    qd, kd, vd = q.to(DEV), k.to(DEV), v.to(DEV)
    out, lse = attn_causal(qd, kd, vd, "HND", torch.float32, return_lse=True, p_quant=mode, q_offset=offset)
    whole, lse_whole = attn_causal(qd, kd, vd, "HND", torch.float32, return_lse=True, p_quant=mode, q_offset=offset,
                                   workspace=prefill_workspace(1, 1, offset + N, qd.device))
    torch.cuda.synchronize()
    assert not torch.equal(out, whole)
    _check(out, whole.cpu(), True, q_tol=8e-3)
    assert torch.allclose(lse, lse_whole, atol=2e-4)
    exact, _ = A.exact_attention(A.fold_scale(q, 128), k, v, causal=True, q_offset=offset, score_scale=math.log(2.0))
    assert _cos(out.cpu(), exact) >= 0.999


@pytest.mark.parametrize("mode,B,Hq,Hkv,N,offset", [
    (2, 2, 4, 2, 2048, 0), (3, 2, 4, 2, 2048, 0),      # one round of value tiles, batch and kv heads to tell apart
    (2, 1, 8, 8, 2048, 0), (2, 2, 4, 4, 2000, 0), (3, 2, 4, 4, 2000, 0), (2, 1, 14, 2, 300, 2048),   # two rounds
    (1, 1, 28, 4, 512, 16384)])                        # ten
@pytest.mark.parametrize("layout", ["HND", "NHD"])
def test_value_tiles_formed_beside_the_row_maximum_pass(mode, B, Hq, Hkv, N, offset, layout):
    """The split launches whose value tiles the row-maximum pass forms (test_prefill_plan_cpu.py shows that these do): every
    (sequence, kv head, tile) in its place, against the unsplit launch, whose tiles have a kernel of their own.  Values are independent, so a tile of
    another place moves the outputs by about its share of their rms (1 / sqrt(256) at the most tiles here, 0.06); tolerance as in the test above (0.008)."""
    from longcontext_sqattn_paddle_amd.sqattn._prefill import prefill_workspace
    from longcontext_sqattn_paddle_amd.sqattn.attn_triton import attn_causal

    print(f"case prefill tiles beside the pass mode={mode} B={B} {Hq}/{Hkv} N={N} offset={offset} {layout}", flush=True)
    g = torch.Generator(device=DEV).manual_seed(N + offset)
    mk = lambda H, n: torch.randn(B, H, n, 128, device=DEV, generator=g)
    q, k, v = mk(Hq, N), mk(Hkv, offset + N), mk(Hkv, offset + N)
    q, k, v = (t.bfloat16() if layout == "HND" else t.bfloat16().permute(0, 2, 1, 3).contiguous() for t in (q, k, v))
    out = attn_causal(q, k, v, layout, torch.float32, p_quant=mode, q_offset=offset)
    whole = attn_causal(q, k, v, layout, torch.float32, p_quant=mode, q_offset=offset, workspace=prefill_workspace(B, Hkv, offset + N, q.device))
    torch.cuda.synchronize()
    assert not torch.equal(out, whole)
    _check(out, whole.cpu(), True, q_tol=8e-3)


@pytest.mark.parametrize("mode", [0, 1, 2, 3, 4])
@pytest.mark.parametrize("window", [None, (64, 0.125, 0.75)])
@pytest.mark.parametrize("tensor,value", [("k", math.nan), ("k", math.inf), ("v", math.nan), ("v", math.inf)])
def test_split_key_ranges_keep_nan_and_infinity(mode, window, tensor, value):
    """One poisoned element of a key or value row: the outputs and log-sum-exps that are not finite are the unsplit launch's,
    wherever the row lies among the parts (first, middle, last)."""
    from longcontext_sqattn_paddle_amd.sqattn._prefill import prefill_workspace
    from longcontext_sqattn_paddle_amd.sqattn.attn_triton import attn_causal
    from longcontext_sqattn_paddle_amd.sqattn.attn_triton_mix_relative import attn_hierarchical_relative_window

    print(f"case prefill split poison mode={mode} window={window} {tensor}={value}", flush=True)
    N = 3010
    q, k, v = (t.to(DEV) for t in _rand(1, 3, 1, N, 128, 43))

    def call(k, v, **kw):
        if window is None:
            return attn_causal(q, k, v, "HND", torch.float32, return_lse=True, p_quant=mode, **kw)
        return attn_hierarchical_relative_window(q, k, q, k, v, window[1], window[2], window[0], "HND", torch.float32, return_lse=True,
                                                 p_quant=mode, **kw)

    small = prefill_workspace(1, 1, N, q.device)
    clean, clean_whole = call(k, v)[0], call(k, v, workspace=small)[0]
    assert not torch.equal(clean, clean_whole)                       # the first call is split
    for at in (20, 1500, 2000, 2990):
        kp, vp = k.clone(), v.clone()
        (kp if tensor == "k" else vp)[0, 0, at, 5] = value
        parts, whole = call(kp, vp), call(kp, vp, workspace=small)
        torch.cuda.synchronize()
        for a, b in zip(parts, whole):
            assert torch.equal(a.isfinite(), b.isfinite()), (at, int(a.isfinite().sum()), int(b.isfinite().sum()))
        assert tensor == "v" and mode == 4 or not bool(whole[0].isfinite().all())   # (mode 4 clamps the value to its e4m3 range)
        assert bool(whole[0].isfinite().any())


@pytest.mark.parametrize("mode", [0, 1, 2, 3, 4])
@pytest.mark.parametrize("value", [-3.38e38, -math.inf, -3e6])
@pytest.mark.parametrize("window", [None, (64, 0.25, 0.75)])
def test_split_key_ranges_over_masked_keys(mode, value, window):
    """Keys masked out through a channel of their own (query 1, masked keys the type's lowest value, -infinity or just far below
    the others) in runs that some parts begin inside of: a part's reference point must not come from them.  The unmasked keys
    in front set the unsplit launch's reference; exact attention over the unmasked keys is the result."""
    from longcontext_sqattn_paddle_amd.sqattn._prefill import prefill_workspace, run_prefill

    print(f"case prefill split masked keys mode={mode} value={value} window={window}", flush=True)
    N = 3010
    q, k, v = _rand(1, 3, 1, N, 128, 44)
    q[..., 7] = 1.0
    k[..., 7] = 0.0
    k *= torch.linspace(0.5, 2.0, N)[None, None, :, None].bfloat16()      # (no two tiles with the same maximum)
    masked = torch.zeros(N, dtype=torch.bool)
    for lo, hi in ((300, 800), (900, 1100), (1250, 1900), (2000, 2400), (2500, 2700)):
        masked[lo:hi] = True
    km = k.clone()
    km[:, :, masked, 7] = value
    w = None if window is None else {"block_m": 64, "sink": window[0], "w8": [A.window_size_relative(window[1], N)] * 3,
                                     "w4": [A.window_size_relative(window[2], N)] * 3}
    qd, kd, vd = q.to(DEV), km.to(DEV), v.to(DEV)
    parts = run_prefill(qd, kd, vd, output_dtype=torch.float32, p_quant=mode, window=w, return_lse=True)
    whole = run_prefill(qd, kd, vd, output_dtype=torch.float32, p_quant=mode, window=w, return_lse=True, workspace=prefill_workspace(1, 1, N, qd.device))
    torch.cuda.synchronize()
    rows = ~masked                                            # a masked key's own row may see nothing else in its first tiles
    assert not torch.equal(parts[0], whole[0])
    for t in (*parts, *whole):
        assert bool(t[:, :, rows].isfinite().all())
    _check(parts[0][:, :, rows], whole[0][:, :, rows].cpu(), mode != 0, q_tol=8e-3)
    assert torch.allclose(parts[1][:, :, rows], whole[1][:, :, rows], atol=2e-4)
    if window is None:
        qs = A.fold_scale(q, 128)
        s = torch.matmul(qs[0].float(), k[0, 0].float().T) * math.log(2.0)
        s = s.masked_fill(masked[None, None, :] | torch.ones(N, N, dtype=torch.bool).triu(1)[None], -math.inf)
        exact = torch.matmul(torch.softmax(s.double(), -1), v[0, 0].double())
        assert _cos(parts[0][0, :, rows].cpu(), exact[:, rows]) >= 0.999


@pytest.mark.parametrize("scale", [2.6e36, 1e3])
@pytest.mark.parametrize("window", [None, (64, 768, 2304)])
def test_split_key_ranges_over_masked_codes(scale, window):
    """The same for the integer Q.K^T form: masked keys are a code of -127 in a channel where the query is 1, with a scale that takes
    the score to -4e37 or to a few thousand below the others."""
    from longcontext_sqattn_paddle_amd.sqattn._prefill import prefill_workspace, run_prefill

    print(f"case prefill split masked codes scale={scale} window={window}", flush=True)
    N = 3010
    q, _, v = _rand(1, 3, 1, N, 128, 45)
    g = torch.Generator().manual_seed(46)
    codes = torch.randint(-127, 128, (1, 1, N, 128), generator=g, dtype=torch.int8)
    codes[..., 7] = 0
    k_scale = torch.full((1, 1, 3072), 0.012)
    q[..., 7] = 1.0
    masked = torch.zeros(N, dtype=torch.bool)
    for lo, hi in ((300, 800), (900, 1100), (1250, 1900), (2000, 2400), (2500, 2700)):
        masked[lo:hi] = True
    codes[:, :, masked] = 0
    codes[:, :, masked, 7] = -127
    k_scale[:, :, :N][:, :, masked] = scale
    w = None if window is None else {"block_m": 64, "sink": window[0], "w8": [window[1]] * 3, "w4": [window[2]] * 3}
    qd, kd, vd, sd = q.to(DEV), codes.to(DEV), v.to(DEV), k_scale.to(DEV)
    kw = dict(output_dtype=torch.float32, window=w, return_lse=True, k_scale=sd)
    parts, whole = run_prefill(qd, kd, vd, **kw), run_prefill(qd, kd, vd, workspace=prefill_workspace(1, 1, N, qd.device), **kw)
    torch.cuda.synchronize()
    rows = ~masked
    assert not torch.equal(parts[0], whole[0])
    for t in (*parts, *whole):
        assert bool(t[:, :, rows].isfinite().all())
    _check(parts[0][:, :, rows], whole[0][:, :, rows].cpu(), False)
    assert torch.allclose(parts[1][:, :, rows], whole[1][:, :, rows], atol=2e-4)


@pytest.mark.parametrize("mode", [0, 2, 4])
def test_split_key_ranges_in_a_graph_and_on_two_streams(mode):
    """A split call (row maxima, parts and merge behind each other, scratch of its own) recorded into a graph and replayed on new
    inputs with eager work in between, and two of them at once on different streams: the bits of the eager call."""
    from longcontext_sqattn_paddle_amd.sqattn.attn_triton import attn_causal

    print(f"case prefill split graph mode={mode}", flush=True)
    inputs_ = [tuple(t.to(DEV) for t in _rand(1, 3, 1, 2100, 128, 50 + i)) for i in range(4)]
    call = lambda x: attn_causal(*x, "HND", torch.float32, return_lse=True, p_quant=mode)
    want = [call(x) for x in inputs_]
    held = tuple(t.clone() for t in inputs_[0])
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out, lse = call(held)
    for x, (o, l) in list(zip(inputs_, want)) * 2:
        for a, b in zip(held, x):
            a.copy_(b)
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, o) and torch.equal(lse, l)
        assert torch.equal(call(x)[0], o)                        # eager work between the replays
    streams = [torch.cuda.Stream() for _ in range(2)]
    torch.cuda.synchronize()
    got = []
    for i in range(8):
        with torch.cuda.stream(streams[i & 1]):
            got.append(call(inputs_[i & 3]))
    torch.cuda.synchronize()
    for i, (o, l) in enumerate(got):
        assert torch.equal(o, want[i & 3][0]) and torch.equal(l, want[i & 3][1])


@pytest.mark.parametrize("mode", [0, 1, 2, 5])
@pytest.mark.parametrize("N,window", [(257, None), (640, (64, 128, 256))])
def test_rows_do_not_depend_on_the_workgroup_size(mode, N, window):
    """Short launches run in workgroups of 128 rows, launches that fill the chip in workgroups of 256; a row's arithmetic is the same in
    both (mode 2: the same 64-row groups), so a sequence alone gives the bits it gives in a batch of 130."""
    from longcontext_sqattn_paddle_amd.sqattn._prefill import prefill_workspace, run_prefill

    print(f"case prefill workgroup size mode={mode} N={N} window={window}", flush=True)
    q, k, v = (t.to(DEV) for t in _rand(1, 4, 2, N, 128, 77))
    w = None if window is None else {"block_m": 64, "sink": window[0], "w8": [window[1]] * 4, "w4": [window[2]] * 4}
    one = run_prefill(q, k, v, output_dtype=torch.float32, p_quant=mode, window=w, workspace=prefill_workspace(1, 2, N, q.device))
    many = run_prefill(*(t.repeat(130, 1, 1, 1) for t in (q, k, v)), output_dtype=torch.float32, p_quant=mode, window=w,
                       workspace=prefill_workspace(130, 2, N, q.device))
    torch.cuda.synchronize()
    assert torch.equal(one[0], many[0]) and torch.equal(one[0], many[129])


@pytest.mark.parametrize("mode", [0, 1, 2, 5])
@pytest.mark.parametrize("case", ["climb", "overflow", "step", "spikes", "late_giant", "alternating", "edge_spikes", "ramp_down", "sink", "chunk"])
@pytest.mark.parametrize("window", [None, (64, 128, 256), (0, 64, 64)])
def test_score_patterns_in_workgroups_of_256_rows(mode, case, window):
    """The score patterns of the tests above run in 128-row workgroups at their sizes; launches that fill the chip, the long
    prompts among them, run in 256-row ones, whose instantiations are others.  The same sequence in a batch too large for the small
    workgroups (they are taken for at most 512 of them) gives the bits it gives alone."""
    from longcontext_sqattn_paddle_amd.sqattn._prefill import prefill_workspace, run_prefill

    print(f"case prefill 256 rows mode={mode} {case} window={window}", flush=True)
    offset = 0
    if case in ("climb", "overflow", "step"):
        q, k, v = _climbing_scores(*{"climb": (6.0, 40.0), "overflow": (0.0, 140.0), "step": (3.0, 17.0)}[case])
    elif case == "sink":
        q, k, v = _rand(1, 4, 2, 777, 128, 79, scale=0.3)
        q[..., 0] = 4.0
        k[:, :, 0] = 0.0
        k[:, :, 0, 0] = 33.0
    elif case == "chunk":
        q, k, v = _rand(1, 4, 2, 2560, 128, 31)
        q, offset = q[:, :, 2048:].contiguous(), 2048
    else:
        q, k, v = _pattern_scores(case, 1536 if window else 777)
    w = None if window is None else {"block_m": 64, "sink": window[0], "w8": [window[1]] * 4, "w4": [window[2]] * 4}
    copies = 512 // (4 * ((q.shape[2] + 127) // 128)) + 1

    def run(reps):
        qd, kd, vd = (t.to(DEV).repeat(reps, 1, 1, 1) for t in (q, k, v))
        return run_prefill(qd, kd, vd, output_dtype=torch.float32, p_quant=mode, window=w, return_lse=True, q_offset=offset,
                           workspace=prefill_workspace(reps, 2, k.shape[2], qd.device))   # no room for parts

    one, many = run(1), run(copies)
    torch.cuda.synchronize()
    for a, b in zip(one, many):
        assert bool(a.isfinite().all())
        assert torch.equal(a[0], b[0]) and torch.equal(a[0], b[copies - 1])


@pytest.mark.parametrize("sink,r8,r4", [(128, 0.25, 0.25), (256, [0.125, 0.5], [0.5, 0.5]), (0, 0.0, 0.0), (64, 2.0, 2.0)])
def test_relative_window_matches_oracle(sink, r8, r4):
    from longcontext_sqattn_paddle_amd.sqattn.attn_triton_mix_relative import attn_hierarchical_relative_window

    N = 1024
    q, k, v = _rand(1, 2, 1, N, 128, 13)
    l8 = r8 if isinstance(r8, list) else [r8, r8]
    l4 = r4 if isinstance(r4, list) else [r4, r4]
    w8 = [A.window_size_relative(x, N) for x in l8]
    w4 = [A.window_size_relative(x, N) for x in l4]
    ref, lse_ref = A.prefill_blockwise(q, k, v, block_m=64, sink=sink, w8=w8, w4=w4, out_dtype=torch.float32)
    qd, kd, vd = q.to(DEV), k.to(DEV), v.to(DEV)
    out, lse = attn_hierarchical_relative_window(qd, kd, qd, kd, vd, r8, r4, sink, "HND", torch.float32, return_lse=True)
    torch.cuda.synchronize()
    _check(out, ref, False)
    assert torch.allclose(lse.cpu(), lse_ref, atol=2e-4)


@pytest.mark.parametrize("sink,w8,w4,distinct", [(128, 256, 512, True), (64, 128, 128, True), (256, [128, 384], [640, 384], True),
                                                 (128, 256, 512, False), (0, 0, 0, False),
                                                 (64, 192, 320, True), (192, [192, 64], [320, 64], True)])   # multiples of 64 but not of 128: walked as written
def test_absolute_window_matches_oracle(sink, w8, w4, distinct):
    from longcontext_sqattn_paddle_amd.sqattn.attn_triton_mix_bad import attn_hierarchical_window
    from oracle import fake_quant as FQ

    N = 1152
    q, k, v = _rand(1, 2, 1, N, 128, 17)
    q4 = FQ.int_fake_quant(q, 4, True, "per_token") if distinct else q
    k4 = FQ.int_fake_quant(k, 4, True, "per_token") if distinct else k
    l8 = w8 if isinstance(w8, list) else [w8, w8]
    l4 = w4 if isinstance(w4, list) else [w4, w4]
    ref, lse_ref = A.prefill_blockwise(q, k, v, block_m=128, sink=sink, w8=l8, w4=l4, q4=q4, k4=k4, out_dtype=torch.float32)
    qd, kd, vd = q.to(DEV), k.to(DEV), v.to(DEV)
    q4d, k4d = (q4.to(DEV), k4.to(DEV)) if distinct else (qd, kd)
    arg8 = torch.tensor(l8, dtype=torch.int32) if isinstance(w8, list) else w8
    arg4 = torch.tensor(l4, dtype=torch.int32) if isinstance(w4, list) else w4
    out, lse = attn_hierarchical_window(qd, kd, q4d, k4d, vd, arg8, arg4, sink, "HND", torch.float32, return_lse=True)
    torch.cuda.synchronize()
    _check(out, ref, False)
    assert torch.allclose(lse.cpu(), lse_ref, atol=2e-4)


def test_unaligned_window_and_sink_sizes_follow_the_documented_rounding():
    """Sizes the reference's kernel has no defined behaviour for (its block loops promise multiples of the query block):
    windows and the sink are rounded up to the next multiple of 64, and an 8-bit window below
    the query block under a wider 4-bit window is raised to the block (the reference's 4-bit range would read keys behind
    the query rows).  Expected values: the oracle on the sizes written out by hand."""
    from longcontext_sqattn_paddle_amd.sqattn.attn_triton_mix_bad import attn_hierarchical_window
    from longcontext_sqattn_paddle_amd.sqattn.attn_triton_mix_relative import attn_hierarchical_relative_window
    from oracle import fake_quant as FQ

    N = 1152
    q, k, v = _rand(1, 2, 1, N, 128, 19)
    q4, k4 = FQ.int_fake_quant(q, 4, True, "per_token"), FQ.int_fake_quant(k, 4, True, "per_token")
    dev = [t.to(DEV) for t in (q, k, q4, k4, v)]
    # absolute: sink 100 -> 128; windows (1, 1000) -> (64, 1024) -> 8-bit window raised to the 128-row block; (300, 200) -> (320, 256)
    out, lse = attn_hierarchical_window(*dev, torch.tensor([1, 300], dtype=torch.int32), torch.tensor([1000, 200], dtype=torch.int32), 100,
                                        "HND", torch.float32, return_lse=True)
    torch.cuda.synchronize()
    ref, lse_ref = A.prefill_blockwise(q, k, v, block_m=128, sink=128, w8=[128, 320], w4=[1024, 256], q4=q4, k4=k4, out_dtype=torch.float32)
    _check(out, ref, False)
    assert torch.allclose(lse.cpu(), lse_ref, atol=2e-4)
    # relative: ratios (0, 0.3) -> 8-bit window 0 raised to the 64-row query block, 4-bit window ceil128(345) = 384; sink 1 -> 64
    out, lse = attn_hierarchical_relative_window(dev[0], dev[1], dev[0], dev[1], dev[4], 0.0, 0.3, 1, "HND", torch.float32, return_lse=True)
    torch.cuda.synchronize()
    ref, lse_ref = A.prefill_blockwise(q, k, v, block_m=64, sink=64, w8=[64, 64], w4=[384, 384], out_dtype=torch.float32)
    _check(out, ref, False)
    assert torch.allclose(lse.cpu(), lse_ref, atol=2e-4)
    with pytest.raises(ValueError):
        attn_hierarchical_window(*dev, -5, 128, 0)


@pytest.mark.parametrize("mode", [3, 4, 5])
@pytest.mark.parametrize("sink,r8,r4,N", [(128, 0.25, 0.25, 1024), (256, [0.125, 0.5], [0.5, 0.5], 1600), (64, 2.0, 2.0, 777)])
def test_relative_window_quantised_modes(mode, sink, r8, r4, N):
    """The folded-scale e4m3 mode and the two fp8 P.V modes walk the same sink/window/diagonal schedule."""
    from longcontext_sqattn_paddle_amd.sqattn.attn_triton_mix_relative import attn_hierarchical_relative_window

    print(f"case prefill relative window mode={mode} sink={sink} N={N}", flush=True)
    q, k, v = _rand(1, 2, 1, N, 128, 23 + N)
    l8 = r8 if isinstance(r8, list) else [r8, r8]
    l4 = r4 if isinstance(r4, list) else [r4, r4]
    w8 = [A.window_size_relative(x, N) for x in l8]
    w4 = [A.window_size_relative(x, N) for x in l4]
    ref, lse_ref = A.prefill_blockwise(q, k, v, p_quant=A.P_MX_ROW if mode == 5 else A.P_STATIC448_GRID, block_m=64, sink=sink,
                                       w8=w8, w4=w4, out_dtype=torch.float32, v_quant="e4m3_channel" if mode >= 4 else None)
    qd, kd, vd = q.to(DEV), k.to(DEV), v.to(DEV)
    out, lse = attn_hierarchical_relative_window(qd, kd, qd, kd, vd, r8, r4, sink, "HND", torch.float32, return_lse=True,
                                                 p_quant=mode)
    torch.cuda.synchronize()
    _check(out, ref, True, q_tol=5e-3 if mode >= 4 else 2e-3)
    assert torch.allclose(lse.cpu(), lse_ref, atol=2e-4)


@pytest.mark.parametrize("mode", [0, 1, 2, 3, 4, 5])
def test_chunked_prefill_offset_all_modes(mode):
    """512 rows behind 2K keys, in the workgroups the launch plan takes for them (mode 5: four waves; the others: eight, with
    split key ranges): every wave runs interior (unmasked) pairs, its own diagonal tiles and idle steps."""
    from longcontext_sqattn_paddle_amd.sqattn.attn_triton import attn_causal

    print(f"case prefill chunked mode={mode}", flush=True)
    N, off = 2560, 2048
    q, k, v = _rand(1, 4, 2, N, 128, 31)
    omode = {0: A.P_NONE, 1: A.P_STATIC448, 2: A.P_BLOCK_ABSMAX, 3: A.P_STATIC448_GRID, 4: A.P_STATIC448_GRID, 5: A.P_MX_ROW}[mode]
    ref, lse_ref = A.prefill_blockwise(q, k, v, p_quant=omode, out_dtype=torch.float32, v_quant="e4m3_channel" if mode >= 4 else None)
    out, lse = attn_causal(q[:, :, off:].contiguous().to(DEV), k.to(DEV), v.to(DEV), "HND", torch.float32,
                           return_lse=True, q_offset=off, p_quant=mode)
    torch.cuda.synchronize()
    # mode 3/4: exp2(x + log2 448) and 448 * exp2(x) differ in the last bits, which moves a probability across an e4m3
    # rounding boundary now and then; with 2K+ keys per row most output elements contain such a flip (each worth
    # about p * 2^-4 * |v|), so the 99.9 % band is a little wider than for short rows
    # mode 2: the scale 448 / maximum of a block comes from an approximate reciprocal, so its products too differ in the last bits
    _check(out, ref[:, :, off:], mode != 0, q_tol={0: 2e-3, 1: 2e-3, 2: 3e-3, 3: 3e-3, 4: 5e-3, 5: 5e-3}[mode])
    assert torch.allclose(lse.cpu(), lse_ref[:, :, off:], atol=2e-4)


def test_prefill_argument_errors():
    from longcontext_sqattn_paddle_amd.sqattn.attn_triton import attn_causal
    from longcontext_sqattn_paddle_amd.sqattn.attn_triton_mix_relative import attn_hierarchical_relative_window

    q = torch.zeros(1, 2, 128, 128, dtype=torch.bfloat16, device=DEV)
    k = torch.zeros(1, 1, 128, 128, dtype=torch.bfloat16, device=DEV)
    with pytest.raises(ValueError):
        attn_causal(q, k, k, "DNH")
    with pytest.raises(ValueError):
        attn_causal(torch.zeros(1, 2, 128, 256, dtype=torch.bfloat16, device=DEV), k, k)
    with pytest.raises(AssertionError):   # qo_len != kv_len (attn_triton.py:272)
        attn_causal(q, k[:, :, :64].contiguous(), k[:, :, :64].contiguous())
    with pytest.raises(AssertionError):   # last dim not contiguous (attn_triton.py:245-247)
        attn_causal(q.transpose(2, 3).contiguous().transpose(2, 3), k, k)
    with pytest.raises(ValueError):       # sink must be a non-negative int (attn_triton_mix_relative.py:367-368)
        attn_hierarchical_relative_window(q, k, q, k, k, 0.1, 0.1, -1)
    with pytest.raises(ValueError):
        attn_hierarchical_relative_window(q, k, q, k, k, 0.1, 0.1, 2.5)
    with pytest.raises(RuntimeError):     # no CPU path
        attn_causal(q.cpu(), k.cpu(), k.cpu())


@pytest.mark.parametrize("mode,peaked", [(0, False), (5, False), (0, True)])
def test_full_size_128k_sampled_rows(mode, peaked):
    """The benchmark shape (1 x 28/4 heads x 131072 x 128): rows sampled over the whole sequence (first row, tile and
    block edges, middle, last) against exact attention of that row on the CPU, plus the base-2 LSE.  Modes 0 (the
    reference's own numerics) and 5 (the benchmark's default) on the benchmark configuration's own inputs, mode 0 also on
    a more peaked distribution."""
    from longcontext_sqattn_paddle_amd.sqattn.attn_triton import attn_causal

    print(f"case prefill 128K sampled rows mode={mode} peaked={peaked}", flush=True)
    N, Hq, Hkv, D = 131072, 28, 4, 128
    if not peaked:  # the benchmark configuration's own generator: N(0,1)/sqrt(128), three key channels per kv head x 8
        q, k, v = (t.to(DEV) for t in inputs.prefill_inputs(1, Hq, Hkv, N, D, seed=2))
    else:           # scores with a spread of a few units instead of a few tenths
        g = torch.Generator(device=DEV).manual_seed(5)
        q = (torch.randn(1, Hq, N, D, device=DEV, generator=g) * 0.7).bfloat16()
        k = (torch.randn(1, Hkv, N, D, device=DEV, generator=g) * 0.7).bfloat16()
        v = torch.randn(1, Hkv, N, D, device=DEV, generator=g).bfloat16()
    out, lse = attn_causal(q, k, v, "HND", torch.float32, return_lse=True, p_quant=mode)
    torch.cuda.synchronize()
    assert bool(torch.isfinite(out).all())
    kc, vc = k.cpu().double(), v.cpu().double()
    rows = [0, 1, 63, 64, 255, 256, 4095, 65535, 65536, 100000, 131071]
    worst = 0.0
    for h in (0, 6, 7, 27):
        kvh = h // (Hq // Hkv)
        for i in rows:
            qi = A.fold_scale(q[:, h:h + 1, i:i + 1].cpu(), D).double()[0, 0, 0]       # carries log2e / sqrt(D)
            s = kc[0, kvh, :i + 1] @ qi
            m = s.max()
            p = torch.exp2(s - m)
            ref = (p[:, None] * vc[0, kvh, :i + 1]).sum(0) / p.sum()
            ref_lse = float(m + torch.log2(p.sum()))
            got = out[0, h, i].cpu().double()
            err = float((got - ref).abs().max())
            # a row that averages thousands of keys of similar weight has an output far below a single value's size:
            # its e4m3 rounding errors are a random sum measured against rms(V) / sqrt(keys), not against the output
            scale = max(float(ref.abs().max()), 3.0 * float(vc[0, kvh].pow(2).mean().sqrt()) / math.sqrt(i + 1)) + (1e-3 if mode == 0 else 0.0)
            worst = max(worst, err / scale)
            # exact mode: fp16 P and V.  Mode 5: e4m3 P (block-scaled) and e4m3 V, whose elements sit within half a
            # spacing (2^-4 relative) of the true value: a row with one key reproduces a quantised V row
            assert err <= (4e-3 if mode == 0 else 8e-2) * scale, (h, i, err, scale)
            assert abs(float(lse[0, h, i]) - ref_lse) <= 2e-3, (h, i, float(lse[0, h, i]), ref_lse)
    print(f"  worst relative row error {worst:.2e}", flush=True)


def test_window_configurations_drawn_at_random():
    """A seeded sweep over what the window entry points take: sequence lengths that are not multiples of the tile, sink
    sizes from none to longer than the sequence, per-head windows from nothing to everything (8-bit wider or narrower than
    4-bit), 1 to 7 q heads per kv head, both layouts, relative and absolute sizes -- each case against the oracle's
    block-wise restatement over `kv_ranges` (2e-3 rms) and its LSE."""
    from longcontext_sqattn_paddle_amd.sqattn.attn_triton_mix_bad import attn_hierarchical_window
    from longcontext_sqattn_paddle_amd.sqattn.attn_triton_mix_relative import attn_hierarchical_relative_window

    rng = torch.Generator().manual_seed(2024)

    def pick(options):
        return options[int(torch.randint(0, len(options), (1,), generator=rng))]

    for case in range(24):
        N = int(torch.randint(65, 2100, (1,), generator=rng))
        group = pick([1, 2, 4, 7])
        Hkv = pick([1, 2])
        Hq = Hkv * group
        sink = pick([0, 64, 128, 256, 512, 4096])
        layout = pick(["HND", "NHD"])
        relative = case % 2 == 0
        q, k, v = _rand(1, Hq, Hkv, N, 128, 1000 + case)
        if relative:
            r8 = [pick([0.0, 0.05, 0.1, 0.25, 0.5, 1.0, 2.0]) for _ in range(Hq)]
            r4 = [pick([0.0, 0.1, 0.3, 0.5, 1.0]) for _ in range(Hq)]
            w8 = [A.window_size_relative(x, N) for x in r8]
            w4 = [A.window_size_relative(x, N) for x in r4]
            # the documented rule for a 4-bit window wider than an 8-bit window below the query block: the 8-bit window is
            # raised to the block (the reference's ranges would read future keys unmasked there)
            w8 = [max(a8, 64) if a4 > a8 else a8 for a8, a4 in zip(w8, w4)]
            block_m = 64
        else:
            w8 = [pick([0, 128, 256, 384, 1024, 4096]) for _ in range(Hq)]
            w4 = [pick([0, 128, 512, 640, 2048]) for _ in range(Hq)]
            w8 = [max(a8, 128) if a4 > a8 else a8 for a8, a4 in zip(w8, w4)]   # (a 4-bit window wider than an 8-bit window below the query block is refused)
            block_m = 128
        print(f"case windows #{case}: N={N} Hq={Hq} Hkv={Hkv} sink={sink} {layout} {'relative' if relative else 'absolute'} w8={w8} w4={w4}", flush=True)
        ref, lse_ref = A.prefill_blockwise(q, k, v, block_m=block_m, sink=sink, w8=w8, w4=w4, out_dtype=torch.float32)
        if layout == "NHD":
            qd, kd, vd = (t.permute(0, 2, 1, 3).contiguous().to(DEV) for t in (q, k, v))
        else:
            qd, kd, vd = q.to(DEV), k.to(DEV), v.to(DEV)
        if relative:
            out, lse = attn_hierarchical_relative_window(qd, kd, qd, kd, vd, r8, r4, sink, layout, torch.float32, return_lse=True)
        else:
            out, lse = attn_hierarchical_window(qd, kd, qd, kd, vd, torch.tensor(w8, dtype=torch.int32), torch.tensor(w4, dtype=torch.int32),
                                                sink, layout, torch.float32, return_lse=True)
        torch.cuda.synchronize()
        if layout == "NHD":
            out = out.permute(0, 2, 1, 3)
        _check(out, ref, False)
        assert torch.allclose(lse.cpu(), lse_ref, atol=2e-4), case


def test_causal_configurations_drawn_at_random():
    """A seeded sweep over the full-causal entry point: P modes 0, 1, 3, 4, 5 (the last cases: 2), lengths that are not multiples of the tile,
    1 to 7 q heads per kv head, batch 1 to 3, both layouts, bf16 and fp16 inputs, head_dim 64 / 96 / 128 (padded by the
    host as the reference pads), chunked calls with a query offset -- each against the oracle's block-wise restatement
    with the tolerances stated at the top (fp8 P.V modes: 99.9 % within 5e-3 rms)."""
    from longcontext_sqattn_paddle_amd.sqattn.attn_triton import attn_causal

    rng = torch.Generator().manual_seed(4242)

    def pick(options):
        return options[int(torch.randint(0, len(options), (1,), generator=rng))]

    for case in range(24):
        mode = [0, 1, 3, 4, 5][case % 5] if case < 16 else 2
        B = pick([1, 1, 2, 3])
        Hkv = pick([1, 2])
        Hq = Hkv * pick([1, 2, 4, 7])
        N = int(torch.randint(33, 1800, (1,), generator=rng))
        D = pick([128, 128, 64, 96])
        dtype = pick([torch.bfloat16, torch.bfloat16, torch.float16])
        layout = pick(["HND", "NHD"])
        off = pick([0, 0, 64 * int(torch.randint(0, max(1, N // 64), (1,), generator=rng))])
        print(f"case causal #{case}: mode={mode} B={B} Hq={Hq} Hkv={Hkv} N={N} D={D} {dtype} {layout} q_offset={off}", flush=True)
        q, k, v = _rand(B, Hq, Hkv, N, D, 3000 + case, dtype=dtype)
        omode = {0: A.P_NONE, 1: A.P_STATIC448, 2: A.P_BLOCK_ABSMAX, 3: A.P_STATIC448_GRID, 4: A.P_STATIC448_GRID, 5: A.P_MX_ROW}[mode]
        ref, lse_ref = A.prefill_blockwise(q, k, v, p_quant=omode, out_dtype=torch.float32, v_quant="e4m3_channel" if mode >= 4 else None)
        qc = q[:, :, off:].contiguous()
        args = [t.to(DEV) for t in (qc, k, v)]
        if layout == "NHD":
            args = [t.permute(0, 2, 1, 3).contiguous() for t in args]
        out, lse = attn_causal(*args, layout, torch.float32, return_lse=True, p_quant=mode, q_offset=off)
        torch.cuda.synchronize()
        if layout == "NHD":
            out = out.permute(0, 2, 1, 3)
        assert out.shape == (B, Hq, N - off, D)
        _check(out, ref[:, :, off:], mode != 0, q_tol={0: 2e-3, 1: 2e-3, 2: 3e-3, 3: 3e-3, 4: 5e-3, 5: 5e-3}[mode])
        assert torch.allclose(lse.cpu(), lse_ref[:, :, off:], atol=2e-4), case
