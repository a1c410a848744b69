"""The C-ABI library and the host-side logic, on the CPU (no compute calls on a GPU).

- librelay_hip.so loads and exports every function include/relay_hip.h declares;
- without a device the package refuses to run (there is no CPU fallback);
- config parsing matches relay's ModelConfig on the reference fixtures;
- the synthetic generator is deterministic and has the stated moments;
- relay's comparison schedule is self-consistent on the CPU oracle (its CPU-vs-CPU
  run agrees exactly, test_attention.cpp:169-175).
"""
import os
import re

import numpy as np
import pytest

from relay_amd import _lib
from relay_amd.model import HostWeights, ModelConfig, llama3_8b, read_safetensors

REPO = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
HEADER = os.path.join(REPO, "include", "relay_hip.h")
FIX = os.path.join(REPO, "tests", "golden", "fixtures")


def declared_functions():
    text = open(HEADER).read()
    text = re.sub(r"/\*.*?\*/", "", text, flags=re.S)
    return sorted(set(re.findall(r"\b((?:rh|relay_hip)_\w+)\s*\(", text)))


def test_header_declares_the_abi():
    names = declared_functions()
    for want in ("rh_paged_decode_attention", "rh_flash_prefill", "rh_gemv_int8", "rh_gemv_f16", "relay_hip_backend_forward",
                 "relay_hip_backend_read_kv_layer", "relay_hip_backend_update_weight"):
        assert want in names


def test_library_exports_every_declared_symbol():
    lib = _lib.lib()
    missing = [n for n in declared_functions() if not hasattr(lib, n)]
    assert not missing, f"not exported: {missing}"
    assert set(declared_functions()) == set(_lib.SIGNATURES), "the ctypes table and the header disagree"


def test_no_device_means_an_error_not_a_fallback():
    if _lib.lib().rh_device_available():
        pytest.skip("a GPU is present")
    with pytest.raises(_lib.RelayHipError):
        _lib.require_device()
    from relay_amd import HipBackend

    w = HostWeights.load(os.path.join(FIX, "llama-mha"))
    with pytest.raises(_lib.RelayHipError):
        HipBackend(w, 8, 16)


@pytest.mark.parametrize("T,K,N", [(32, 4096, 262080), (32, 4096, 262081), (32, 4096, 262100), (32, 4096, 262142),
                                   (32, 4096, 262143), (32, 4096, 262144), (17, 8192, 131070), (17, 8192, 131071),
                                   (17, 8192, 131072), (262143, 4096, 64), (262144, 4096, 64), (20, 64, 16777215),
                                   (20, 64, 16777216), (33, 576, 1864135), (33, 576, 1864136)])
def test_gemm_f16_takes_every_shape_that_fits_says(T, K, N):
    """rh_gemm_f16_fits says whether rh_gemm_f16 takes a shape with ldw = K, on both sides of N * K and
    T * K = 2^30. y is misaligned, so that the call ends in a refusal whatever the shape."""
    lib = _lib.lib()
    assert lib.rh_gemm_f16(16, K, 16, 4, T, K, N, 0.0, None) != 0
    refused = "too large" in _lib.last_error()
    assert refused or "y must be 16-byte aligned" in _lib.last_error()
    assert lib.rh_gemm_f16_fits(T, K, N) == (0 if refused else 1)
    assert refused == (max(T, N) * K >= 1 << 30)


@pytest.mark.parametrize("n,kv_heads,group,D,ctx,keys", [
    # 32 to 63 (context, kv head) groups of head size 64: slices of 4 chunks only where that makes three.
    (12, 3, 3, 64, 460, 128), (16, 3, 3, 64, 512, 128), (12, 4, 8, 64, 512, 128), (16, 3, 3, 64, 513, 256), (8, 4, 8, 64, 640, 256),
    # Past 128 groups rounds are filled by the slices that there are, at least 8 chunks each: a third
    # slice fills no more of them (192 groups), or does (144).
    (48, 4, 8, 64, 1500, 768), (64, 3, 3, 64, 1500, 768), (24, 8, 4, 128, 700, 352), (48, 3, 3, 64, 1500, 512),
    (48, 4, 8, 64, 4096, 1024), (48, 4, 8, 64, 2048, 512)])
def test_decode_slices(n, kv_heads, group, D, ctx, keys):
    assert _lib.lib().rh_decode_slice_keys(n, kv_heads, group, D, ctx) == keys


PLAIN, RANGES, SILU = 0, 1, 2  # RH_F16_*


@pytest.mark.parametrize("T,K,N,form,pays", [
    # A plain product that the plan would split has no one to add its ranges: o and down of widths
    # past the merging RMSNorm's 4096 (library / tile us: 39 / 76, 44 / 62, 37 / 76).
    (32, 13824, 5120, PLAIN, 0), (64, 8192, 8192, PLAIN, 0), (17, 13824, 5120, PLAIN, 0), (32, 5632, 2048, PLAIN, 0),
    (32, 5632, 2048, RANGES, 1), (560, 576, 960, PLAIN, 1), (560, 4096, 6144, RANGES, 1),
    # 4 M outputs (1536 x 6144: 84 / 114; 3072 x 2048, K 5632: 80 / 93).
    (1536, 4096, 6144, RANGES, 0), (1536, 14336, 4096, RANGES, 0), (3072, 5632, 2048, RANGES, 0), (3999, 1024, 1000, RANGES, 1),
    (4000, 1024, 1000, RANGES, 0),
    # SiLU in the epilogue: 10 M outputs where K is past 2048.
    (512, 2048, 11264, SILU, 1), (2048, 2048, 11264, SILU, 1), (256, 4096, 28672, SILU, 1), (384, 4096, 28672, SILU, 0),
    # The same with 100 M weights and more at up to 64 tokens (44 / 47, 57 / 64).
    (32, 4096, 28672, SILU, 0), (64, 5120, 27648, SILU, 0), (65, 4096, 28672, SILU, 1), (64, 2048, 11264, SILU, 1),
    # LM heads, for their first pass's sake.
    (32, 2048, 32000, PLAIN, 1), (17, 4096, 128256, PLAIN, 1), (32, 4096, 128256, PLAIN, 0),
    # Shapes that the kernel cannot take.
    (32, 96, 64, RANGES, 0), (20, 64, 1 << 24, PLAIN, 0)])
def test_f16_tile_kernel_is_chosen_where_it_is_level_or_ahead(T, K, N, form, pays):
    assert _lib.lib().rh_gemm_f16_pays(T, K, N, form) == pays


def test_kernel_launchers_validate_shapes_before_launching():
    lib = _lib.lib()
    assert lib.rh_gemv_int8(None, 64, None, 0, None, None, 0, 64, 64, 0.0, None) != 0
    assert lib.rh_gemv_int8_row_stride(4096) == 4096 + 256 and lib.rh_gemv_int8_row_stride(576) == 576
    assert lib.rh_gemv_int8_row_stride(14336) == 14336 + 256 and lib.rh_gemv_int8_row_stride(100) == 112
    assert "T must be" in _lib.last_error()
    assert lib.rh_flash_prefill(None, 64, None, None, None, None, 1, 4, 3, 64, 16, 0.1, None, 64, None) != 0
    assert lib.rh_prefill_tile_rows() == 128
    assert lib.rh_gemv_int8_max_tokens() == 64
    # a null weight pointer (an int8-only matrix passed to the fp16 product) is an error, not a launch
    assert lib.rh_gemv_f16_rmsnorm(None, 576, 16, 32, 1e-5, 48, 1, 576, 3072, 0.0, None) != 0
    assert "missing pointer" in _lib.last_error()
    assert lib.rh_gemv_int8(None, 576, 16, 0, 32, 48, 1, 576, 960, 0.0, None) != 0
    assert "missing pointer" in _lib.last_error()


def test_config_parsing_of_the_fixtures():
    c = ModelConfig.from_json_text(open(os.path.join(FIX, "llama3-rope", "config.json")).read())
    assert c.rope_llama3 and c.rope_factor > 1
    q = ModelConfig.from_json_text(open(os.path.join(FIX, "qwen2-bias", "config.json")).read())
    assert q.qkv_bias
    g = ModelConfig.from_json_text(open(os.path.join(FIX, "llama-gqa-tied-bf16", "config.json")).read())
    assert g.tie_embeddings and g.heads > g.kv_heads and g.head_dim == 8
    t = read_safetensors(os.path.join(FIX, "llama-gqa-tied-bf16", "model.safetensors"))
    assert all(a.dtype == np.float32 for a in t.values())


def test_synthetic_generator_is_deterministic_with_the_stated_moments():
    n = 1 << 20
    a, b = np.empty(n, np.float32), np.empty(n, np.float32)
    _lib.lib().rh_synth_normal_f32(a.ctypes.data, n, 0, 5, 0.0, 0.02)
    _lib.lib().rh_synth_normal_f32(b.ctypes.data, n, 0, 5, 0.0, 0.02)
    assert np.array_equal(a, b)
    c = np.empty(n, np.float32)
    _lib.lib().rh_synth_normal_f32(c.ctypes.data, n, 0, 6, 0.0, 0.02)
    assert not np.array_equal(a, c)
    assert abs(a.mean()) < 5 * 0.02 / np.sqrt(n) and abs(a.std() - 0.02) < 2e-4
    # the first elements do not depend on n (counter-based, any thread count)
    s = np.empty(1000, np.float32)
    _lib.lib().rh_synth_normal_f32(s.ctypes.data, 1000, 0, 5, 0.0, 0.02)
    assert np.array_equal(s, a[:1000])


def test_llama3_config_matches_the_stated_shape():
    c = llama3_8b()
    assert (c.hidden, c.layers, c.heads, c.kv_heads, c.head_dim, c.intermediate, c.vocab) == \
        (4096, 32, 32, 8, 128, 14336, 128256)


@pytest.mark.parametrize("heads", [4, 32])
def test_prefill_plan_covers_every_row_once(heads):
    """rh_prefill_plan (host code): every row of every chunk in exactly one block of at
    most rh_prefill_tile_rows() rows, blocks inside their chunk with the chunk's positions
    and table, records heaviest first; a large step pairs light with heavy blocks."""
    rows = _lib.lib().rh_prefill_tile_rows()
    chunks = [(0, 2048, 0, 0), (2048, 300, 700, 130), (2348, 2, 5, 200), (2350, 129, 0, 210)]
    work = _lib.prefill_work(chunks, heads)
    seen, cost = [], []
    for rec in work:
        c = 0
        for t0, n, p0 in (rec[0:3], rec[3:6]):
            if n == 0:
                continue
            assert 0 < n <= rows
            ch = [x for x in chunks if x[0] <= t0 < x[0] + x[1]]
            assert len(ch) == 1 and t0 + n <= ch[0][0] + ch[0][1] and rec[6] == ch[0][3]
            assert p0 == ch[0][2] + (t0 - ch[0][0])
            seen.extend(range(t0, t0 + n))
            c += int(n) * int(p0 + n)
        cost.append(c)
    assert sorted(seen) == list(range(2479))
    assert cost == sorted(cost, reverse=True)
    paired = sum(1 for rec in work if rec[4] > 0)
    assert (paired > 0) == (heads == 32)


def test_prefill_plan_rejects_small_capacity():
    import numpy as np

    a = np.array([0], np.int32)
    n = np.array([1000], np.int32)
    work = np.zeros((1, 8), np.int32)
    assert _lib.lib().rh_prefill_plan(a.ctypes.data, n.ctypes.data, a.ctypes.data, a.ctypes.data, 1, 4,
                                      work.ctypes.data, 1) < 0
    assert "capacity" in _lib.last_error()


def test_work_planners_follow_their_rules():
    """The host-side planners (no device needed): rh_decode_slice_keys cuts contexts into
    whole chunks, kMergeBatch (8) slices of 2 to 8 chunks for few groups at head sizes 64 and
    128, one slice for a handful of
    short contexts, at least two otherwise, never below 8 chunks; rh_gemv_f16_split_plan splits K in two only for long K on few row tiles above 16 tokens;
    rh_gemv_int8_row_stride pads rows that are a multiple of 2 KB."""
    L = _lib.lib()
    for D in (16, 32, 64, 128):
        chunk = L.rh_decode_chunk_keys(D)
        assert chunk == {16: 128, 32: 128, 64: 64, 128: 32}[D]
        for n, kvh, g, ctx in [(32, 4, 8, 2048), (48, 8, 4, 8192), (1, 3, 3, 640), (1, 8, 4, 65536), (200, 8, 4, 100)]:
            sk = L.rh_decode_slice_keys(n, kvh, g, D, ctx)
            assert sk > 0 and sk % chunk == 0
            groups = n * kvh * ((g + 15) // 16)
            small = max(2 * chunk, -(-ctx // (8 * chunk)) * chunk)
            if D in (64, 128) and small <= 8 * chunk and groups * -(-ctx // small) <= 256:
                assert sk == small and -(-ctx // sk) <= 8  # few groups: short slices, one merge round
            elif groups <= 16 and ctx <= 16 * chunk:
                assert sk >= ctx  # one slice
            else:
                assert sk >= 8 * chunk and (ctx + sk - 1) // sk >= min(2, (ctx + 8 * chunk - 1) // (8 * chunk))
    assert L.rh_decode_slice_keys(32, 4, 8, 64, 2048) == 1024  # config 2: two slices of 1024 keys
    assert L.rh_decode_slice_keys(1, 3, 3, 64, 640) == 128  # config 1: five slices of 2 chunks
    assert L.rh_decode_slice_keys(1, 8, 4, 128, 2048) == 256  # 8 slices of 8 chunks at D128
    assert L.rh_decode_chunk_keys(96) == -1
    assert [L.rh_gemv_f16_split_plan(T, K, N) for T, K, N in
            [(32, 5632, 2048), (1, 5632, 2048), (32, 2048, 2048), (32, 4096, 4096), (8, 14336, 4096), (1, 4096, 1024)]] \
        == [2, 1, 1, 1, 1, 1]
    assert L.rh_gemv_f16_split_plan(0, 64, 64) == -1
    assert [L.rh_gemv_int8_row_stride(K) for K in (4096, 14336, 2048, 576, 100)] == [4352, 14592, 2304, 576, 112]
