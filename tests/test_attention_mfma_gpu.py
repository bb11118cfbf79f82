"""Decode attention outside the one-launch grids: chunk partials and the fold
(attn_mfma_kernel, attn_kvchunk_kernel, attn_fold_kernel) bit for bit against the oracle, for every number of
query heads per KV head, both head dimensions and KV types, capacities that end inside a
chunk, strided caches, garbage past the count, one token and several fold blocks."""

from __future__ import annotations

import numpy as np
import pytest
import torch

import oracle
from tests.helpers import bf16_bits, bf16_to_f32, f16_normal, from_torch_bits, rng, to_torch
from tests.test_gemv_gpu import assert_bits_equal
from thintensor_amd import _lib

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("heads,kv_heads,dim,tokens,cap,bf16,sinks,pad", [
    (40, 10, 128, 130, 200, True, False, 0),     # four heads per KV head, capacity inside a chunk
    (2, 2, 128, 1, 1, False, True, 0),           # one head, one token, one-row cache
    (1, 1, 128, 130, 130, False, False, 0),      # three chunk rows: partials off a 16-byte boundary
    (6, 3, 128, 64, 64, True, True, 0),          # two heads, exactly one chunk
    (8, 1, 64, 8257, 8300, False, True, 0),      # 130 chunks: a second fold block of two
    (16, 1, 64, 2050, 2050, False, False, 0),    # sixteen heads, four waves
    (16, 2, 128, 1041, 1100, True, False, 0),    # eight heads, 17 chunks
    (264, 33, 64, 700, 704, False, False, 0),    # whole chunks, more workgroups than CUs
    (4, 1, 64, 77, 100, True, False, 8),         # token stride above the head dimension
    (4, 1, 96, 77, 128, False, True, 0),         # other head dimension: scalar loads
    (4, 1, 64, 77, 128, False, False, 1),        # misaligned rows: scalar loads
])
def test_attention_partials_and_fold(backend, device, heads, kv_heads, dim, tokens, cap, bf16, sinks, pad):
    g = rng(heads + tokens + dim)

    def values(*shape):
        v = g.standard_normal(shape).astype(np.float32)
        if bf16:
            return torch.from_numpy(v).to(torch.bfloat16).view(torch.int16).numpy().view(np.uint16)
        return v.astype(np.float16)

    q, sk = values(heads * dim), values(heads) if sinks else None
    keys, vals = values(kv_heads, cap, dim + pad), values(kv_heads, cap, dim + pad)
    code, dtype = (oracle.BF16, torch.bfloat16) if bf16 else (oracle.F16, torch.float16)
    nan, inf = (0x7fc0, 0x7f80) if bf16 else (np.float16(np.nan), np.float16(np.inf))
    keys[:, tokens:], vals[:, tokens:] = nan, inf             # past the count: never used
    qd, kd, vd = (to_torch(a, device, bf16) for a in (q, keys, vals))
    kd, vd = kd[:, :, :dim], vd[:, :, :dim]
    skd = to_torch(sk, device, bf16) if sinks else None
    out = torch.empty(heads * dim, device=device, dtype=dtype)
    stride = (cap * (dim + pad), dim + pad)
    for n, count in ((tokens, torch.tensor([tokens], dtype=torch.int32, device=device)), (max(1, tokens // 2), None)):
        backend.single_token_gqa_attention(qd, kd, vd, out, heads, kv_heads, dim, sinks=skd,
                                           active_tokens=n if count is None else count)
        want = np.empty(heads * dim, dtype=q.dtype)
        oracle.lib().tto_attention(q.ctypes.data, keys.ctypes.data, vals.ctypes.data, code, *stride, *stride,
                                   sk.ctypes.data if sinks else None, code, n, heads, kv_heads, dim, want.ctypes.data)
        got = out.cpu().view(torch.int16).numpy().view(np.uint16)
        assert_bits_equal(got, want.view(np.uint16), f"{n} tokens")


@pytest.mark.parametrize("heads,kv_heads,dim,cap,sinks", [
    (64, 8, 64, 4096, True),      # one launch up to 20 known chunks, then one wave per head and the fold
    (8, 8, 64, 4160, False),      # 65 chunks: the count read before the rows
    (256, 32, 64, 4096, True),    # more than 12288 waves: matrix-core partials, unless the host knows the count
    (512, 64, 64, 640, False),    # 640 workgroups in one launch
    (16, 4, 128, 8192, True),
    (2, 1, 128, 5000, False),     # capacity inside a chunk
    (16, 1, 64, 4200, True),      # sixteen heads, four waves
])
def test_counts_of_a_long_cache(backend, device, heads, kv_heads, dim, cap, sinks):
    """Every form gives the oracle's bits on one cache and scratch, the counts going up and
    down across the borders of the dispatch, known to the host and only on the device; each
    call leaves the arrival counters at zero."""
    g = rng(cap + heads)
    q, sk = f16_normal(g, heads * dim), f16_normal(g, heads) if sinks else None
    keys, vals = f16_normal(g, (kv_heads, cap, dim)), f16_normal(g, (kv_heads, cap, dim))
    qd, kd, vd = (to_torch(a, device) for a in (q, keys, vals))
    skd = to_torch(sk, device) if sinks else None
    out = torch.empty(heads * dim, device=device, dtype=torch.float16)
    want = np.empty(heads * dim, dtype=np.float16)
    for n in sorted({min(cap, n) for n in (1, 64, 65, 1280, 1281, 4096, 4097, cap)}, key=lambda n: (n % 3, n)):
        oracle.lib().tto_attention(q.ctypes.data, keys.ctypes.data, vals.ctypes.data, oracle.F16, cap * dim, dim, cap * dim,
                                   dim, sk.ctypes.data if sinks else None, oracle.F16, n, heads, kv_heads, dim,
                                   want.ctypes.data)
        for count in (torch.tensor([n], dtype=torch.int32, device=device), n):
            out.fill_(7.0)
            backend.single_token_gqa_attention(qd, kd, vd, out, heads, kv_heads, dim, sinks=skd, active_tokens=count)
            assert_bits_equal(from_torch_bits(out), want, f"{n} tokens, {type(count).__name__}")
            assert not backend._attention_partials[:1024].view(torch.int32).any()


@pytest.mark.parametrize("heads,kv_heads,dim,tokens,max_tokens", [(8, 2, 128, 130, 1000), (40, 10, 128, 64, 4500),
                                                                  (8, 8, 64, 77, 200)])
def test_rows_past_the_count_need_not_exist(backend, device, heads, kv_heads, dim, tokens, max_tokens):
    """max_tokens bounds the count and sizes the scratch; caches that are not contiguous
    head_dim-64 rows of whole chunks are read below the count only.  Here the last KV head
    ends with the tensor, `tokens` rows long, so a read past the count leaves the
    allocation."""
    g = rng(heads + dim)
    q, keys, vals = (f16_normal(g, s) for s in ((heads * dim,), (kv_heads, tokens, dim), (kv_heads, tokens, dim)))
    qd, kd, vd = (to_torch(a, device) for a in (q, keys, vals))
    out = torch.empty(heads * dim, device=device, dtype=torch.float16)
    floats = backend.lib.tt_attention_scratch_floats(heads, max_tokens, dim)
    scratch = torch.zeros(floats, device=device)
    count = torch.tensor([tokens], dtype=torch.int32, device=device)
    want = np.empty(heads * dim, dtype=np.float16)
    oracle.lib().tto_attention(q.ctypes.data, keys.ctypes.data, vals.ctypes.data, oracle.F16, tokens * dim, dim,
                               tokens * dim, dim, None, oracle.F16, tokens, heads, kv_heads, dim, want.ctypes.data)
    for dev, n in ((None, tokens), (count.data_ptr(), 0)):
        out.fill_(7.0)
        rc = backend.lib.tt_single_token_gqa_attention(
            qd.data_ptr(), kd.data_ptr(), vd.data_ptr(), _lib.F16, tokens * dim, dim, tokens * dim, dim, None, _lib.F16,
            dev, n, max_tokens, heads, kv_heads, dim, scratch.data_ptr(), floats, out.data_ptr(),
            torch.cuda.current_stream(device).cuda_stream)
        _lib.check(rc, "single_token_gqa_attention")
        assert_bits_equal(from_torch_bits(out), want, "device count" if dev else "host count")


@pytest.mark.parametrize("kind", ["tiny values", "late weights", "inf and nan"])
@pytest.mark.parametrize("dim,cap", [(128, 200), (64, 200), (64, 192), (64, 4096), (96, 192)])
def test_subnormals_and_non_finite_values(backend, device, kind, dim, cap):
    """Every form keeps binary32 subnormals (the oracle's fmaf chains do): values whose products
    with the weights and their sums are subnormal, and weights near the smallest normal number
    on the only tokens with values; infinities and NaN of K and V rows inside the count reach
    the same outputs."""
    heads, kv_heads, tokens = 16, 4, 150
    g = rng(dim + cap + len(kind))
    q = g.standard_normal((heads, dim))
    keys, vals = g.standard_normal((kv_heads, cap, dim)), g.standard_normal((kv_heads, cap, dim))
    if kind == "tiny values":
        vals *= 2.0 ** -g.integers(122, 133, (kv_heads, cap, 1))
    elif kind == "late weights":
        # scores from 0 down to -87 below the first token's; values from token 100 on
        q[:] = 1.0
        keys[:] = -np.linspace(0.0, 86.5, tokens).repeat(cap // tokens + 1)[:cap, None] / np.sqrt(dim)
        keys[:, 140:tokens] = -86.0 / np.sqrt(dim)
        vals[:, :100] = 0.0
        vals[:, 100:] *= 2.0 ** -g.integers(0, 8, (kv_heads, cap - 100, 1))
        vals[:, 100:140] = 0.0
    else:
        keys[1, 70, 3], keys[2, 5, 0], vals[3, 149, 7], vals[3, 0, 9] = np.nan, np.inf, -np.inf, np.nan
    q, keys, vals = (bf16_bits(a.astype(np.float32)) for a in (q, keys, vals))
    out = torch.empty(heads * dim, device=device, dtype=torch.bfloat16)
    want = np.empty(heads * dim, dtype=np.uint16)
    oracle.lib().tto_attention(q.ctypes.data, keys.ctypes.data, vals.ctypes.data, oracle.BF16, cap * dim, dim, cap * dim, dim,
                               None, oracle.BF16, tokens, heads, kv_heads, dim, want.ctypes.data)
    w = bf16_to_f32(want)
    if kind == "inf and nan":
        assert np.isnan(w).any() and np.isinf(w).any() and np.isfinite(w).any()
    else:
        assert ((w != 0) & (np.abs(w) < 2.0 ** -126)).any()
    qd, kd, vd = (to_torch(a, device, True) for a in (q, keys, vals))
    count = torch.tensor([tokens], dtype=torch.int32, device=device)
    backend.single_token_gqa_attention(qd.view(-1), kd, vd, out, heads, kv_heads, dim, active_tokens=count)
    got = from_torch_bits(out)
    nan = np.isnan(w)
    assert np.array_equal(np.isnan(bf16_to_f32(got)), nan)
    assert_bits_equal(np.where(nan, 0, got).astype(np.uint16), np.where(nan, 0, want).astype(np.uint16), kind)
