"""Drop-in for the reference's sqattn/attn_replacer.py: same entry points, HIP kernels underneath.

`process_model(model, "SQAttn", window_sizes, args)` binds `mp_triton_wrapper(...)` as
`layer.prefill_attention` exactly like the reference (:12-34); the closure does what the reference's does
(:323-452) -- GQA handling, K mean-centring, 8-/4-bit fake-quant of Q/K, 8-bit fake-quant of V, sink +
hierarchical-window prefill, reshape to [B, N, Hq*D] -- with two deliberate differences:
  * K and V are never expanded to the 28 q-heads (`repeat_kv`, :335-336): the kernel maps q-head -> kv-head
    itself.  Every per-token / per-(token, channel) quantisation range is unchanged by the expansion
    (per-token ranges are per head; the "per_channel" range reduces over batch and heads, fake_quant.py:30-32,
    and duplicated heads add nothing to a min/max), so the results are identical at 1/7 of the traffic;
  * the dead `seq_len == 1` branch (:369-420, it uses names deleted three lines earlier) is replaced by the
    split-KV decode kernel.
"""
from __future__ import annotations

import math
import types

import torch

from .. import _native as N
from .attn_triton_decode import attn_decode
from .attn_triton_mix_bad import attn_hierarchical_window
from .attn_triton_mix_relative import attn_hierarchical_relative_window
from .fake_quant import FloatQuantizer, IntegerQuantizer, fused_int8qk_prepass, fused_int_prepass
from .sdpa_attention import sdpa_attention_forward


def process_model(model, method, window_sizes=None, args=None, patch_decode=False):
    """attn_replacer.py:12-34.  `patch_decode=True` (extension) also binds the split-KV decode kernel as
    `layer.decode_attention` on every layer."""
    if method == "SQAttn":
        for i in range(len(model.layers)):
            if i in window_sizes.keys():
                layer = model.layers[i]
                bit8_window_sizes = window_sizes[i]["bit8"]
                bit4_window_sizes = window_sizes[i]["bit4"]
                sink_size = window_sizes[i]["sink"]  # read and, as in the reference (:19,24), overridden by 256
                layer.prefill_attention = types.MethodType(
                    mp_triton_wrapper(i, args=args, bit8_window_sizes=bit8_window_sizes,
                                      bit4_window_sizes=bit4_window_sizes, sink_window_size=256), layer)
                model.layers[i] = layer
        if patch_decode:
            for layer in model.layers:
                layer.decode_attention = types.MethodType(decode_attention_fn, layer)
    elif method == "SDPA":
        print("use sdpa")
    elif method == "FlashAttn":
        print("use full flash attn")
    else:
        raise ValueError(f"Unsupported attention type: {method}")
    return model


def decode_attention_fn(module, query_states, key_states, value_states, layer_idx=None, seqlens=None):
    """`layer.decode_attention(q [B,1,Hq,D], Kcache, Vcache [B,L,Hkv,D], None)[0]` slot (model_hub/LLM.py:105):
    returns a 1-tuple so that the caller's `[0]` picks the [B,1,Hq*D] output."""
    cache = getattr(module, "kv_cache", None)
    if seqlens is None and cache is not None:
        seqlens = cache.attend_length   # this package's cache knows how many rows of the buffers are valid
    out = attn_decode(query_states, key_states, value_states, "NHD", query_states.dtype, seqlens=seqlens)
    b, n, h, d = out.shape
    return (out.reshape(b, n, h * d),)


def _normalise_windows(bit8_window_sizes, bit4_window_sizes):
    """attn_replacer.py:299-321."""
    is_per_head = isinstance(bit8_window_sizes, list) or isinstance(bit4_window_sizes, list)
    if is_per_head:
        num_heads = len(bit8_window_sizes) if isinstance(bit8_window_sizes, list) else len(bit4_window_sizes)
        if isinstance(bit8_window_sizes, int):
            bit8_window_sizes = [bit8_window_sizes] * num_heads
        if isinstance(bit4_window_sizes, int):
            bit4_window_sizes = [bit4_window_sizes] * num_heads
        if bit8_window_sizes is None:
            bit8_window_sizes = [0] * num_heads
        if bit4_window_sizes is None:
            bit4_window_sizes = [0] * num_heads
    else:
        bit8_window_sizes = bit8_window_sizes or 0
        bit4_window_sizes = bit4_window_sizes or 0
    return bit8_window_sizes, bit4_window_sizes


def _quantizers(args):
    """attn_replacer.py:340-358."""
    if args.qk_qtype == "int":
        bit8_qk = IntegerQuantizer(8, True, "per_token")
    elif args.qk_qtype in ("e4m3", "e5m2"):
        bit8_qk = FloatQuantizer(args.qk_qtype, True, "per_token")
    else:
        raise ValueError(f"Invalid quantization type: {args.qk_qtype}")
    bit4_qk = IntegerQuantizer(4, True, "per_token")
    if args.v_qtype == "int":
        bit8_v = IntegerQuantizer(8, True, "per_channel")
    elif args.v_qtype in ("e4m3", "e5m2"):
        bit8_v = FloatQuantizer(args.v_qtype, True, "per_channel")
    else:
        raise ValueError(f"Invalid quantization type: {args.v_qtype}")
    return bit8_qk, bit4_qk, bit8_v


def mp_triton_wrapper(layer_idx, bit8_window_sizes=0, bit4_window_sizes=0, sink_window_size=0, args=None):
    """attn_replacer.py:296-454: builds the `prefill_attention` closure of one layer."""
    bit8_window_sizes, bit4_window_sizes = _normalise_windows(bit8_window_sizes, bit4_window_sizes)

    def attention_fn(module, query, key, value, attention_mask, dropout=0.0, scaling=1.0, sliding_window=None, **kwargs):
        # query [B,N,Hq,D], key/value [B,N,Hkv,D]; the kv heads are never expanded (the kernels take GQA as is)
        nhd = hasattr(module, "num_key_value_groups")
        layout = "NHD" if nhd else "HND"
        seq_dim = 1 if nhd else 2
        seq_len = query.shape[seq_dim]
        if seq_len == 1:
            if not nhd:
                query, key, value = (t.permute(0, 2, 1, 3) for t in (query, key, value))
            out = attn_decode(query, key, value, "NHD", torch.bfloat16)
            b, n, h, d = out.shape
            return out.reshape(b, n, h * d)
        p_quant = kwargs.get("p_quant", None)
        relative = bool(args.use_relative_distance)
        known = ("int", "e4m3", "e5m2")
        if args.qk_qtype not in known or args.v_qtype not in known:
            raise ValueError(f"Invalid quantization type: {args.qk_qtype if args.qk_qtype not in known else args.v_qtype}")
        if query.size(-1) == 128:
            # one fused HIP pre-pass instead of the reference's tensor passes (:338-365), for every quantiser type.  The
            # relative launch aliases the 4-bit operands to the 8-bit ones (attn_triton_mix_relative.py:441-444), so
            # they are only produced for the absolute variant.
            # With the integer quantiser and relative windows the query does not go through the pre-pass at all: the
            # attention kernel quantises its rows while loading them (same bits), which saves writing and re-reading q8.
            q_in_kernel = relative and args.qk_qtype == "int"
            if getattr(args, "int8_qk", False):
                # extension (off unless args.int8_qk is set): Q.K^T as a real integer product on the int8 matrix
                # instruction -- the pre-pass hands over the key's codes and scales instead of the fake-quantised key
                if not (q_in_kernel and args.v_qtype == "int"):
                    raise ValueError("int8_qk needs use_relative_distance and the integer quantiser types")
                k_codes, k_scale, v_bit8 = fused_int8qk_prepass(query, key, value, tensor_layout=layout)
                attn_output = attn_hierarchical_relative_window(
                    query, k_codes, query, k_codes, v_bit8, int8_window_ratios=bit8_window_sizes,
                    int4_window_ratios=bit4_window_sizes, sink_size=sink_window_size, tensor_layout=layout,
                    output_dtype=torch.bfloat16, k_scale=k_scale)
                del query, key, value
                if layout == "HND":
                    attn_output = attn_output.transpose(1, 2).contiguous()
                bs, seq_len, head, head_dim = attn_output.shape
                return attn_output.reshape(bs, seq_len, head * head_dim)
            # bf16: the value goes straight into the tiles the attention kernel reads (the fp8 P.V modes make their own from
            # rows).  Up to 8 (batch, kv head) rows, which the tile pass holds in registers; with more it reads them twice, one
            # workgroup per 64 keys: 700 tokens of 32 rows 128 - 160 us a call against 95 - 115 with the value as rows, level at 8192
            tiled = (query.dtype == torch.bfloat16 and (p_quant is None or p_quant < N.P_E4M3_FP8_PV)
                     and value.size(0) * value.size(2 if nhd else 1) <= 8)
            q_bit8, q_bit4, k_bit8, k_bit4, v_bit8 = fused_int_prepass(query, key, value, want_4bit=not relative, tensor_layout=layout,
                                                                       qk_qtype=args.qk_qtype, v_qtype=args.v_qtype, skip_query=q_in_kernel,
                                                                       value_tiles=tiled)
            if q_in_kernel:
                q_bit8 = query
        else:
            q_in_kernel = tiled = False
            bit8_qk, bit4_qk, bit8_v = _quantizers(args)
            if nhd:   # the quantisers' "per_channel" range is over dims (0, 1) of [B,H,N,D]: quantise HND views
                query, key, value = (t.permute(0, 2, 1, 3) for t in (query, key, value))
            key = key - key.mean(dim=2, keepdim=True)
            q_bit8 = bit8_qk.fake_quant_tensor(query)
            k_bit8 = bit8_qk.fake_quant_tensor(key)
            v_bit8 = bit8_v.fake_quant_tensor(value)
            q_bit4 = k_bit4 = None
            if not relative:
                q_bit4 = bit4_qk.fake_quant_tensor(query)
                k_bit4 = bit4_qk.fake_quant_tensor(key)
            layout = "HND"
        del query, key, value
        v_bit8, v_tiles = (None, v_bit8) if tiled else (v_bit8, None)
        if relative:
            attn_output = attn_hierarchical_relative_window(
                q_bit8, k_bit8, q_bit8, k_bit8, v_bit8, int8_window_ratios=bit8_window_sizes,
                int4_window_ratios=bit4_window_sizes, sink_size=sink_window_size, tensor_layout=layout,
                output_dtype=torch.bfloat16, p_quant=p_quant, q_quant=8 if q_in_kernel else 0, v_tiles=v_tiles)
        else:
            attn_output = attn_hierarchical_window(
                q_bit8, k_bit8, q_bit4, k_bit4, v_bit8, int8_window_sizes=bit8_window_sizes,
                int4_window_sizes=bit4_window_sizes, sink_size=sink_window_size, tensor_layout=layout,
                output_dtype=torch.bfloat16, p_quant=p_quant, v_tiles=v_tiles)
        if layout == "HND":
            attn_output = attn_output.transpose(1, 2).contiguous()
        bs, seq_len, head, head_dim = attn_output.shape
        return attn_output.reshape(bs, seq_len, head * head_dim)

    return attention_fn


def construct_mix_bit_mask(kv_len, bit8_window_sizes, bit4_window_sizes, sink_window_size, device):
    """attn_replacer.py:63-112 (`construct_mix_bit_mask` and its per-head variant, called with seq_len = 2 * kv_len):
    bool [kv_len, 2 kv_len] (or [H, kv_len, 2 kv_len] for per-head lists), True = attend; columns [0, kv_len) are the
    8-bit keys, [kv_len, 2 kv_len) their 4-bit copies."""
    L = 2 * kv_len
    q_idx = torch.arange(L, device=device).unsqueeze(1)
    kv_idx = torch.arange(L, device=device).unsqueeze(0)
    w8, w4 = bit8_window_sizes, bit4_window_sizes
    if isinstance(w8, list) or isinstance(w4, list):
        w8 = torch.tensor(w8, device=device).view(-1, 1, 1)
        w4 = torch.tensor(w4, device=device).view(-1, 1, 1)
        q_idx, kv_idx = q_idx.unsqueeze(0), kv_idx.unsqueeze(0)
    fp8_mask = (kv_idx <= q_idx) & ((kv_idx < sink_window_size) | (kv_idx > q_idx - w8))
    kv_idx_4bit = kv_idx - L // 2
    int4_mask = (kv_idx_4bit >= sink_window_size) & (kv_idx_4bit <= q_idx - w8) & (kv_idx_4bit > q_idx - w8 - w4)
    is_bit8_part = kv_idx < L // 2
    return ((is_bit8_part & fp8_mask) | (~is_bit8_part & int4_mask))[..., : L // 2, :]


def delayed_sdpa_wrapper(layer_idx, bit8_window_sizes=0, bit4_window_sizes=0, sink_window_size=0, args=None):
    """attn_replacer.py:36-250: the masked-SDPA emulation of the mixed-precision windows, on dense [L, 2L] masks (a tool
    for short sequences).  q, k, v are [B, H, L, D] here, heads already expanded as the reference's branch assumes.
    Plain branch (`args.quant` false): SDPA with the caller's mask.  Quantised branch: the reference builds the
    concatenated operands and the mask, then passes the unconcatenated operands to SDPA and stops in a debugger
    (:173-189); this closure finishes what it sets up -- the 8-bit queries attend to [8-bit keys ; 4-bit keys] with values
    [v8 ; v8] under the mask -- and returns [B, L, H * D]."""
    bit8_window_sizes, bit4_window_sizes = _normalise_windows(bit8_window_sizes, bit4_window_sizes)

    def attention_fn(module, q, k, v, attn_mask, dropout=0.0, scaling=1.0, sliding_window=None, **kwargs):
        if not getattr(args, "quant", False):
            return sdpa_attention_forward(module, q, k, v, attention_mask=attn_mask, dropout=dropout, scaling=scaling, **kwargs)
        q_len, kv_len = q.shape[2], k.shape[2]
        k = k - k.mean(dim=2, keepdim=True)
        bit8_qk, bit4_qk, _ = _quantizers(args)
        if args.v_qtype == "int":
            bit8_v = IntegerQuantizer(8, False, "per_channel")          # this branch quantises V asymmetrically (:141)
        else:
            bit8_v = FloatQuantizer(args.v_qtype, True, "per_channel")
        q_bit8 = bit8_qk.fake_quant_tensor(q)
        k_bit8_bit4 = torch.cat([bit8_qk.fake_quant_tensor(k), bit4_qk.fake_quant_tensor(k)], dim=2)
        v_bit8 = bit8_v.fake_quant_tensor(v)
        v_bit8_bit8 = torch.cat([v_bit8, v_bit8], dim=2)
        mask = construct_mix_bit_mask(kv_len, bit8_window_sizes, bit4_window_sizes, sink_window_size, q.device)[..., -q_len:, :]
        if mask.ndim == 3:
            mask = mask[None]
        return sdpa_attention_forward(None, q_bit8, k_bit8_bit4, v_bit8_bit8, attention_mask=mask, dropout=dropout, scaling=scaling,
                                      is_causal=False, tensor_layout="HND")

    return attention_fn


def cal_attn_weight(module, query, key, is_causal=True, attn_mask=None):
    """Dense softmax attention map used by calibration (attn_replacer.py:253-278)."""
    if hasattr(module, "num_key_value_groups"):
        key = repeat_kv(key, module.num_key_value_groups)
        query = query.permute(0, 2, 1, 3)
    query, key = query.contiguous(), key.contiguous()
    L, S = query.shape[-2], key.shape[-2]
    attn_bias = torch.zeros(L, S, dtype=query.dtype, device=query.device)
    if is_causal:
        assert attn_mask is None
        keep = torch.ones(L, S, dtype=torch.bool, device=query.device).tril(diagonal=0)
        attn_bias.masked_fill_(keep.logical_not(), float("-inf"))
    if attn_mask is not None:
        if attn_mask.dtype == torch.bool:
            attn_bias.masked_fill_(attn_mask.logical_not(), float("-inf"))
        else:
            attn_bias = attn_mask + attn_bias
    attn_weight = query @ key.transpose(-2, -1) * (1 / math.sqrt(query.shape[-1]))
    attn_weight += attn_bias
    return torch.softmax(attn_weight, dim=-1)


def repeat_kv(hidden_states: torch.Tensor, n_rep: int) -> torch.Tensor:
    """[B,N,Hkv,D] -> [B,Hkv*n_rep,N,D], each kv head repeated n_rep times (attn_replacer.py:281-293)."""
    batch, slen, num_key_value_heads, head_dim = hidden_states.shape
    hidden_states = hidden_states.permute(0, 2, 1, 3)
    if n_rep == 1:
        return hidden_states
    hidden_states = hidden_states[:, :, None, :, :].expand(batch, num_key_value_heads, n_rep, slen, head_dim)
    return hidden_states.reshape(batch, num_key_value_heads * n_rep, slen, head_dim)
