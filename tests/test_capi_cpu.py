"""CPU-side checks of the C ABI: the library loads, exports every symbol the header declares, and
rejects bad arguments with error codes (no compute call is made here)."""
import ctypes
import os
import re

import pytest
import torch

from longcontext_sqattn_paddle_amd import _native as N

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def _declared_symbols():
    text = open(os.path.join(ROOT, "include", "sqattn.h")).read()
    text = re.sub(r"/\*.*?\*/", "", text, flags=re.S)
    return sorted(set(re.findall(r"\b(sq_[a-z0-9_]+)\s*\(", text)))


def test_library_exports_every_declared_symbol():
    names = _declared_symbols()
    assert "sq_prefill_fwd" in names and "sq_decode_fwd" in names and "sq_kmeans_train" in names
    handle = ctypes.CDLL(N.LIB_PATH)
    for n in names:
        assert hasattr(handle, n), f"{n} declared in include/sqattn.h but not exported"
    assert set(names) == set(N.SYMBOLS), "ctypes table and header disagree"
    assert N.lib().sq_abi_version() == 3


def test_sizes_and_split_heuristic():
    lib = N.lib()
    assert lib.sq_prefill_workspace_bytes(1, 4, 131072, 128) == 4 * 131072 * 128 * 2
    assert lib.sq_prefill_workspace_bytes(1, 4, 100, 128) == 4 * 2 * 64 * 128 * 2     # rounded up to 64-key tiles
    s = lib.sq_decode_num_splits(1, 4, 131072)
    assert 1 <= s <= 131072 * 4 // 256      # at least 4 tiles of 16 tokens for each of the 4 waves (one kv head each)
    assert lib.sq_decode_num_splits(8, 4, 131072) <= s
    assert lib.sq_decode_workspace_bytes(2, 28, 128, 16) == 2 * 28 * 16 * 129 * 4
    assert lib.sq_decode_num_splits(1, 4, 10) == 1


def test_split_workspace_size_of_calls_that_are_refused():
    """The size of a call that sq_prefill_fwd refuses is the plain one, whatever its arguments: an unknown window mode with a
    block of 0 rows, offsets and lengths that do not fit each other or 32-bit tile counts."""
    lib = N.lib()
    w = (ctypes.c_int32 * 4)(128, 128, 128, 128)
    wp = ctypes.cast(w, ctypes.POINTER(ctypes.c_int32))

    def size(batch=1, Hq=4, Hkv=1, Nq=4096, Nk=4096, **fields):
        p = N.PrefillParams(**fields)
        return lib.sq_prefill_workspace_bytes_split(batch, Hq, Hkv, Nq, Nk, ctypes.byref(p))

    plain = lambda batch=1, Nk=4096: lib.sq_prefill_workspace_bytes(batch, 1, Nk, 128)
    assert size() > plain()                                            # this call is split
    for mode in (2, 7, -1):
        for block_m in (0, 64):
            assert size(window_mode=mode, block_m=block_m) == plain()
    sizes = dict(window_mode=N.WINDOW_SIZES, num_heads_w=4, w8=wp, w4=wp)
    for block_m in (0, -64, 1, 32, 256):
        assert size(**sizes, block_m=block_m) == plain()
    assert size(window_mode=N.WINDOW_SIZES, block_m=64) == plain()     # no windows
    for offset in (-64, 64, 1 << 40, (1 << 63) - 1):
        assert size(q_offset=offset) == plain()
    assert size(Nq=1 << 40) == plain()
    assert size(Nq=4096, Nk=1 << 40, q_offset=(1 << 40) - 4096) == plain(Nk=1 << 40)
    assert size(batch=1 << 40) == plain(batch=1 << 40)
    assert size(p_quant=9) == plain() and size(p_quant=-1) == plain()
    assert lib.sq_prefill_workspace_bytes_split(0, 4, 1, 4096, 4096, ctypes.byref(N.PrefillParams())) == 0


def _dec(q, k, v, out, ws, layout=0, p_quant=0):
    lib = N.lib()
    b = [N.dl(t) for t in (q, k, v, None, out, None, ws)]
    return lib.sq_decode_fwd(*[N.ptr(x) for x in b], N.DecodeParams(layout, p_quant, 0, 0), None), \
        lib.sq_last_error().decode()


def test_decode_rejects_cpu_tensors_and_bad_arguments():
    q = torch.zeros(1, 4, 1, 128, dtype=torch.bfloat16)
    k = torch.zeros(1, 2, 64, 128, dtype=torch.bfloat16)
    ws = torch.zeros(4096)
    rc, msg = _dec(q, k, k, q.clone(), ws)
    assert rc == N.SQ_EDEVICE and "ROCm" in msg
    rc, msg = _dec(q, k, k, q.clone(), ws, layout=7)
    assert rc == N.SQ_EINVAL and "tensor_layout" in msg
    rc, _ = _dec(q, k, k, q.clone(), ws, p_quant=2)
    assert rc == N.SQ_EINVAL
    lib = N.lib()
    assert lib.sq_decode_fwd(None, None, None, None, None, None, None, N.DecodeParams(0, 0, 0, 0), None) == N.SQ_EINVAL
    assert lib.sq_decode_fwd(None, None, None, None, None, None, None, None, None) == N.SQ_EINVAL


def test_prefill_rejects_cpu_tensors_and_bad_arguments():
    lib = N.lib()
    q = torch.zeros(1, 2, 64, 128, dtype=torch.bfloat16)
    b = [N.dl(t) for t in (q, q, q, None, None, q.clone(), None, torch.zeros(64))]
    p = N.PrefillParams()
    assert lib.sq_prefill_fwd(*[N.ptr(x) for x in b], ctypes.byref(p), None) == N.SQ_EDEVICE
    p.layout = 5
    assert lib.sq_prefill_fwd(*[N.ptr(x) for x in b], ctypes.byref(p), None) == N.SQ_EINVAL
    p.layout, p.p_quant = 0, 9
    assert lib.sq_prefill_fwd(*[N.ptr(x) for x in b], ctypes.byref(p), None) == N.SQ_EINVAL
    assert lib.sq_prefill_fwd(None, None, None, None, None, None, None, None, None, None) == N.SQ_EINVAL


@pytest.mark.parametrize("M,N_,K,taken", [
    (5, 3584, 3584, 1), (64, 4608, 3584, 1), (256, 8192, 3584, 1), (2048, 3584, 18944, 1), (1024, 4096, 14336, 1), (640, 1024, 4096, 1),   # faster here
    (16, 8192, 8192, 0), (24, 4096, 16384, 0), (8, 6144, 8192, 0), (200, 6144, 4096, 0), (176, 8192, 3584, 0),                            # few rows; half-empty blocks
    (1024, 1024, 4096, 0), (777, 3584, 8192, 0), (1024, 3072, 6144, 0), (64, 14336, 4096, 0), (512, 4096, 4096, 0), (1500, 2048, 8192, 0),
    (65, 8192, 8192, 1), (17, 6144, 8192, 1), (192, 6144, 4096, 1), (224, 8192, 3584, 1), (256, 6144, 4096, 1),                           # the edges
    (0, 256, 512, 0), (16, 255, 512, 0), (16, 256, 100, 0), (2049, 3584, 18944, 0)])
def test_prompt_products_go_to_the_faster_side(M, N_, K, taken):
    assert N.lib().sq_linear_preferred(M, N_, K) == taken


def test_error_mapping():
    with pytest.raises(ValueError):
        _ = N.check(N.SQ_EINVAL)
    with pytest.raises(AssertionError):
        N.check(N.SQ_ESHAPE)
    with pytest.raises(RuntimeError):
        N.check(N.SQ_EHIP)
    N.check(N.SQ_OK)


def test_wrappers_refuse_cpu_tensors():
    from longcontext_sqattn_paddle_amd.sqattn.attn_triton import attn_causal

    q = torch.zeros(1, 2, 64, 128, dtype=torch.bfloat16)
    with pytest.raises(RuntimeError, match="no CPU path"):
        attn_causal(q, q, q)
