"""The C ABI: the shared library loads and exports every function the header declares, and the
ctypes signatures cover exactly that set.  No compute call is made (runs without a GPU)."""
import ctypes
import re
from pathlib import Path

import pytest

from fastcache_amd import _lib

ROOT = Path(__file__).resolve().parent.parent
HEADER = ROOT / "include" / "fastcache_hip.h"


def declared_functions():
    text = re.sub(r"/\*.*?\*/", "", HEADER.read_text(), flags=re.S)
    return sorted(set(re.findall(r"\b(fc_[a-z0-9_]+)\s*\(", text)))


def test_header_declares_functions():
    names = declared_functions()
    assert "fc_snapkv_score" in names and "fc_decode_attn" in names and len(names) >= 14


def test_library_exports_every_declared_symbol():
    if not _lib.LIB_PATH.exists():
        pytest.fail(f"{_lib.LIB_PATH} missing: run `python -m fastcache_amd.build`")
    lib = ctypes.CDLL(str(_lib.LIB_PATH))
    missing = [n for n in declared_functions() if not hasattr(lib, n)]
    assert not missing, f"not exported: {missing}"


def test_signatures_cover_the_header():
    assert sorted(_lib.SIGNATURES) == declared_functions()
    for name in _lib.SIGNATURES:
        _lib.fn(name)          # binds restype/argtypes; raises if the symbol is absent


def test_abi_version_and_error_text():
    assert _lib.fn("fc_abi_version")() == 1
    assert isinstance(_lib.fn("fc_last_error")(), bytes)


def test_argument_validation_without_gpu():
    """Bad arguments are rejected on the host before any launch."""
    rc = _lib.fn("fc_topk_select")(None, 0, 1, 1, None, 1, 1, 1, None, None, 1, None)
    assert rc == -1
    assert b"null" in _lib.fn("fc_last_error")()
    v = _lib.FcKvView()
    rc = _lib.fn("fc_knorm_score")(ctypes.byref(v), None, 0, None)
    assert rc == -1
    v.base = 16
    v.dtype, v.head_dim, v.num_layers, v.batch, v.num_kv_heads = 2, 64, 1, 1, 1
    rc = _lib.fn("fc_knorm_score")(ctypes.byref(v), None, 0, None)
    assert rc == -2 and b"head_dim" in _lib.fn("fc_last_error")()


def _dense_view(seq_len, dtype=2, heads=2):
    """A view of nothing real (base 256): enough for the host-side checks, which never touch the memory."""
    v = _lib.FcKvView()
    v.base, v.dtype, v.head_dim, v.num_layers, v.batch, v.num_kv_heads = 256, dtype, 128, 1, 1, heads
    v.stride_layer = v.stride_batch = heads * seq_len * 128
    v.stride_head, v.stride_token, v.block_size, v.max_seq_len = seq_len * 128, 128, 1, seq_len
    return v


def test_one_launch_presses_validate_on_the_host():
    """fc_knorm_press / fc_select_compact / fc_snapkv_press refuse what they cannot take before any launch: missing
    outputs, kept counts beyond the index row, columns too long for LDS, kept counts inside the window."""
    err = lambda: _lib.fn("fc_last_error")()
    k, v = _dense_view(1024), _dense_view(1024)
    B = ctypes.byref
    assert _lib.fn("fc_knorm_press")(B(k), B(v), None, 1024, 10, None, None, 10, None) == -1 and b"null" in err()
    assert _lib.fn("fc_knorm_press")(B(k), B(v), 16, 1000, 10, None, 16, 10, None) == -1 and b"score_stride" in err()
    assert _lib.fn("fc_select_compact")(B(k), B(v), 16, 1024, 20, None, 16, 10, None) == -1 and b"index_stride" in err()
    other = _dense_view(1024, heads=4)
    assert _lib.fn("fc_select_compact")(B(k), B(other), 16, 1024, 10, None, 16, 10, None) == -1 and b"disagree" in err()
    kl, vl = _dense_view(40000), _dense_view(40000)
    assert _lib.fn("fc_select_compact")(B(kl), B(vl), 16, 40000, 10, None, 16, 10, None) == -2 and b"LDS" in err()
    press = _lib.fn("fc_snapkv_press")
    args = lambda kk, vv, k_keep, stride: (B(kk), B(vv), 16, None, 8, 64, 7, 1, 0.1, 1.0, 16, kk.max_seq_len, 16, k_keep, None,
                                           16, stride, None)
    assert press(*args(k, v, 64, 64)) == -1 and b"exceed the window" in err()
    assert press(*args(kl, vl, 5000, 5000)) == -2 and b"fc_select_compact" in err()
    f32 = _dense_view(1024, dtype=0)
    assert press(*args(f32, f32, 100, 100)) == -2 and b"fp16/bf16" in err()


def test_select_in_one_pass_validates_on_the_host():
    """fc_snapkv_select_once refuses what it cannot take before any launch, fc_snapkv_once_workspace_bytes says so."""
    err = lambda: _lib.fn("fc_last_error")()
    B, call, room = ctypes.byref, _lib.fn("fc_snapkv_select_once"), _lib.fn("fc_snapkv_once_workspace_bytes")
    k = _dense_view(1024)
    need = room(B(k), 8, 64)
    args = lambda v=k, q=16, hq=8, W=64, ksz=7, keep=100, wgs=0, ws=16, nbytes=need: call(
        B(v), q, hq, W, ksz, 1, 0.1, 1.0, keep, None, 16, keep, wgs, ws, nbytes, None)
    assert need > 0 and args(nbytes=need - 1) == -1 and b"workspace" in err()
    assert args(q=None) == -1 and args(q=24) == -1 and args(hq=7, keep=200) in (-1, -2) and args(ksz=4) == -1
    assert args(keep=64) == -1 and b"exceed the window" in err()
    assert args(wgs=-1) == -1 and b"workgroups" in err()
    long, f32 = _dense_view(12289), _dense_view(1024, dtype=0)
    for v, hq, W in ((long, 8, 64), (f32, 8, 64), (k, 8, 64 * 40)):
        assert room(B(v), hq, W) == -1
    assert args(v=long) == -2 and args(v=f32) == -2


def test_one_pass_pays_where_it_can_run():
    """The rule never asks for a shape that the kernel does not take, hooks of more than 8192 keys a column or 32 768 in all keep their sweeps,
    and so do batches whose columns fill the chip."""
    B = ctypes.byref

    def pays(L, batch, H, hq, S, W, mean=None, paged=True, **kw):
        v = _lib.FcKvView(**dict(dict(dtype=2, num_layers=L, batch=batch, num_kv_heads=H, max_seq_len=S, block_size=256 if paged else 1,
                                      block_tables=1 if paged else None, stride_token=H * 128), **kw))
        got = _lib.fn("fc_snapkv_once_pays")(B(v), hq, W, S if mean is None else mean)
        assert not got or _lib.fn("fc_snapkv_once_workspace_bytes")(B(v), hq, W) > 0
        return got

    assert pays(1, 1, 8, 32, 4096, 64, paged=False) and not pays(1, 2, 8, 32, 250, 64, paged=False)
    assert not pays(1, 1, 8, 32, 4097, 64, paged=False) and not pays(1, 4, 8, 32, 4096, 64, paged=False)
    assert not pays(1, 1, 3, 21, 8193, 64, paged=False) and pays(1, 1, 3, 21, 8192, 64, paged=False)
    assert pays(36, 1, 8, 32, 4096, 64) and not pays(36, 8, 8, 32, 4096, 64) and not pays(28, 13, 4, 28, 2300, 32, mean=1200)
    assert pays(28, 3, 4, 28, 1000, 64) and not pays(28, 16, 4, 28, 4096, 64)
    assert not pays(36, 1, 8, 32, 4096, 64, dtype=0) and not pays(36, 1, 8, 32, 1000, 64, block_size=48)
    assert not pays(36, 1, 8, 32, 1000, 64, stride_token=1 << 24) and not pays(1, 1, 1, 17, 4096, 32, paged=False)
    for L, batch, H, hq, W in ((36, 2, 8, 32, 32), (28, 5, 4, 28, 64), (32, 16, 32, 32, 32), (1, 8, 32, 32, 64), (1, 64, 8, 32, 64)):
        for S in (1, 33, 450, 4096, 4097, 9216, 9217, 12289, 40000):
            pays(L, batch, H, hq, S, W, paged=L > 1)


def test_one_pass_over_a_pool_counts_the_rows_that_stay():
    """Against key ranges the kept rows do not matter; against the one launch a pass that keeps much, fills the chip's rounds or
    has lengths that differ stays there, and a route that refuses the shape is not overruled."""
    B = ctypes.byref

    def pays(L, batch, H, hq, S, W, kept, route=0, mean=None):
        v = _lib.FcKvView(dtype=2, num_layers=L, batch=batch, num_kv_heads=H, max_seq_len=S, block_size=256, block_tables=1,
                          stride_token=H * 128)
        return bool(_lib.fn("fc_snapkv_rows_once_pays")(B(v), hq, W, S if mean is None else mean, kept, route))

    for kept in (100, 700, 1400):
        assert pays(36, 2, 8, 32, 2000, 32, kept, route=2) and not pays(36, 2, 8, 32, 2000, 32, kept, route=-1)
    for (L, batch, H, hq, W), S in (((36, 6, 8, 32, 32), 1951), ((32, 4, 32, 32, 32), 1941), ((28, 13, 4, 28, 64), 1968)):
        assert not pays(L, batch, H, hq, S, W, S * 7 // 10) and pays(L, batch, H, hq, min(S, 1300), W, S // 10)
    assert pays(36, 1, 8, 32, 651, 64, 455) and not pays(36, 2, 8, 32, 3245, 64, 2271) and not pays(28, 6, 4, 28, 590, 32, 413)
    assert not pays(12, 5, 8, 8, 671, 64, 402) and pays(12, 5, 8, 8, 671, 64, 200) and not pays(28, 2, 4, 28, 809, 64, 200)
    assert not pays(36, 4, 8, 32, 2939, 32, 700, mean=1270) and pays(36, 2, 8, 32, 2074, 32, 500, mean=1935)


def test_missing_library_fails_loudly(monkeypatch, tmp_path):
    monkeypatch.setattr(_lib, "_lib", None)
    monkeypatch.setattr(_lib, "LIB_PATH", tmp_path / "nope.so")
    with pytest.raises(_lib.FastcacheError):
        _lib.load()
