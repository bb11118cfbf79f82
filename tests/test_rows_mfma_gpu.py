"""Several activation rows on the binary32 matrix cores (rows_mfma.hip) and, where those are
slower (few weight rows), as slots of the single-row kernel: fp16 GEMV + bias, the fp16
lm_head argmax and the fp8 GEMM must give every row the single-row operator's bits, at the edges of the row tiles (16 or 32 weight rows, passes of 32 activation rows,
the 4-, 8- and 16-row forms), of the chunk groups (ragged last group, each lanes-per-row
value) and of the tile schedule (more tiles than workgroups, one tile, two row tiles per
wave)."""

from __future__ import annotations

import numpy as np
import pytest
import torch

import oracle
from oracle.decode_ref import lanes
from tests.helpers import f16_normal, from_torch_bits, rng, to_torch
from tests.test_gemv_gpu import assert_bits_equal

pytestmark = pytest.mark.gpu


def _dense_rows(w, x):
    return [oracle.gemv("f16w", "none", w.view(np.uint8).reshape(w.shape[0], -1), None, v, cols=w.shape[1],
                        lpr=lanes(w.shape[1])) for v in x]


@pytest.mark.parametrize("m,rows,cols", [
    (3, 1, 32),          # one row, one chunk
    (4, 17, 512),        # 16 lanes per row; a tile of one row
    (5, 40, 1056),       # ragged last group (33 chunks)
    (8, 300, 2880),      # 32 lanes, 90 chunks
    (9, 130, 4096),      # 64 lanes, eight waves per workgroup
    (16, 4113, 2048),    # more 16-row tiles than CUs
    (17, 33, 5152),      # two activation tiles, 161 chunks
    (33, 70, 5120),      # a second pass of one row
    (3, 12400, 64),      # more tiles than workgroups
])
def test_bias_rows(backend, device, m, rows, cols):
    g = rng(m * 1000 + rows)
    w, x, bias = f16_normal(g, (rows, cols), 0.05), f16_normal(g, (m, cols)), f16_normal(g, rows)
    out = torch.full((m, rows + 3), 7.0, device=device, dtype=torch.float16)
    backend.matvec_bias_rows(to_torch(w, device), to_torch(bias, device), to_torch(x, device), out[:, :rows])
    got = from_torch_bits(out)
    for r, y in enumerate(_dense_rows(w, x)):
        want = (y.astype(np.float32) + bias.astype(np.float32)).astype(np.float16)
        assert_bits_equal(got[r, :rows], want, f"row {r}")
    assert np.all(got[:, rows:] == np.float16(7.0))


@pytest.mark.parametrize("m,rows,cols", [(3, 33, 2048), (8, 32801, 512), (16, 32801, 96), (35, 900, 2880), (64, 40, 160)])
def test_lm_head_rows(backend, device, m, rows, cols):
    """Tokens and logits; equal logits in different tiles go to the lower row, a NaN row wins."""
    g = rng(m + rows)
    w, x = f16_normal(g, (rows, cols), 0.05), f16_normal(g, (m, cols))
    w[rows - 1] = w[rows // 3] = w[rows // 2] = x[1] * np.float16(0.25)   # row 1's maximum, three times
    x[2, 5], w[rows // 2 + 1, 5] = np.float16(np.inf), np.float16(0.0)     # inf * 0 in row 2
    wd = to_torch(w, device)
    logits = torch.empty((m, rows), device=device, dtype=torch.float16)
    idx = backend.matvec_argmax_batched(wd, to_torch(x, device), logits).cpu().numpy()
    for r, want in enumerate(_dense_rows(w, x)):
        got = from_torch_bits(logits[r])
        assert np.array_equal(np.isnan(got), np.isnan(want))
        assert_bits_equal(np.where(np.isnan(got), 0, got).astype(np.float16), np.where(np.isnan(want), 0, want).astype(np.float16),
                          f"logits row {r}")
        assert idx[r] == int(oracle.lib().tto_argmax(want.ctypes.data, oracle.F16, rows)), f"row {r}"
    assert idx[1] == rows // 3 and idx[2] == rows // 2 + 1
    only = backend.matvec_argmax_batched(wd, to_torch(x, device)).cpu().numpy()   # without logits
    assert np.array_equal(only, idx)


@pytest.mark.parametrize("m,rows,cols", [(3, 1, 256), (4, 530, 512), (7, 32900, 256), (8, 300, 8192), (15, 4200, 2816)])
def test_fp8_rows(backend, device, m, rows, cols):
    g = rng(m + cols)
    bits = g.integers(0, 256, size=(rows, cols), dtype=np.uint8)
    bits[(bits & 0x7F) == 0x7F] = 0x3C
    scales = (np.abs(g.standard_normal(rows)) * 0.01 + 1e-3).astype(np.float32)
    x = f16_normal(g, (m, cols))
    out = torch.empty((m, rows), device=device, dtype=torch.float16)
    backend.scaled_batched_matvec(torch.from_numpy(bits).to(device).view(torch.float8_e4m3fn), to_torch(scales, device),
                                  to_torch(x, device), out)
    for r in range(m):
        want = oracle.gemv("fp8", "row", bits, scales, x[r], cols=cols, lpr=lanes(cols), s_row=1)
        assert_bits_equal(from_torch_bits(out[r]), want, f"row {r}")


# Sizes that the matrix-core kernel serves rather than slots of the single-row kernel, compared
# with the single-row operators (which other tests compare with the oracle): 16, 32 and 64
# lanes per row in four- and eight-wave workgroups, each activation form.
@pytest.mark.parametrize("m,rows,cols", [
    (3, 1840, 2880), (4, 1375, 8192),     # four rows of activations, eight waves
    (5, 4200, 2048), (8, 4130, 2880),     # eight rows, four waves, 64 and 32 lanes
    (8, 1124, 4096), (8, 1125, 4096),     # the last size of the slots, the first past it
    (12, 1050, 96), (16, 4113, 4096),     # sixteen rows, 16 and 64 lanes
    (17, 5000, 2880), (32, 5000, 2048),   # two activation tiles, more tiles than CUs
    (33, 930, 5152), (35, 1000, 16384),   # a second pass of one and of three rows
    (3, 32801, 512), (20, 1000, 32768),
    (64, 64, 5120), (31, 780, 32768),     # slots
    (2, 3300, 5152), (2, 2056, 8192), (2, 2048, 8192),   # two rows: engine, engine, slots
])
def test_bias_rows_match_single_rows(backend, device, m, rows, cols):
    g = torch.Generator(device=device).manual_seed(rows + cols + m)
    w, x, bias = (torch.randn(s, generator=g, device=device).mul_(f).half()
                  for s, f in (((rows, cols), 0.05), ((m, cols), 1.0), ((rows,), 1.0)))
    out, one = (torch.empty((m, rows), device=device, dtype=torch.float16) for _ in range(2))
    backend.matvec_bias_rows(w, bias, x, out)
    for t in range(m):
        backend.multi_matvec_bias((w,), (bias,), x[t], one[t])
    assert torch.equal(out.view(torch.int16), one.view(torch.int16))


@pytest.mark.parametrize("m,rows,cols", [(3, 32801, 2048), (4, 32801, 2880), (7, 32801, 2880), (16, 32801, 2048),
                                         (16, 32801, 2880), (20, 32801, 2048), (32, 5000, 2880), (32, 5000, 2048),
                                         (64, 5000, 4096)])
def test_lm_head_matches_single_rows(backend, device, m, rows, cols):
    """Two weight tiles per wave at each lanes-per-row value, and two activation tiles in four-wave
    workgroups."""
    g = torch.Generator(device=device).manual_seed(rows + cols + m)
    w = torch.randn((rows, cols), generator=g, device=device).mul_(0.05).half()
    x = torch.randn((m, cols), generator=g, device=device).half()
    logits, one = (torch.empty((m, rows), device=device, dtype=torch.float16) for _ in range(2))
    idx = backend.matvec_argmax_batched(w, x, logits)
    for t in range(m):
        assert int(backend.matvec_argmax_tensor(w, x[t])) == int(idx[t]), f"row {t}"
        one[t] = backend.logits_buffer(rows, torch.float16)
    assert torch.equal(logits.view(torch.int16), one.view(torch.int16))


@pytest.mark.parametrize("m,rows,cols", [(4, 4200, 4096), (12, 4200, 4096), (4, 32900, 4096), (12, 32900, 4096),
                                         (7, 32900, 2816), (8, 1124, 2048), (8, 1125, 2048), (15, 900, 8192)])
def test_fp8_rows_match_single_rows(backend, device, m, rows, cols):
    g = torch.Generator(device=device).manual_seed(rows + cols + m)
    w = torch.randn((rows, cols), generator=g, device=device).mul_(100).clamp_(-448, 448).to(torch.float8_e4m3fn)
    scales = torch.rand(rows, generator=g, device=device) * 0.01 + 1e-3
    x = torch.randn((m, cols), generator=g, device=device).half()
    out, one = (torch.empty((m, rows), device=device, dtype=torch.float16) for _ in range(2))
    backend.scaled_batched_matvec(w, scales, x, out)
    for t in range(m):
        backend.scaled_matvec(w, scales, x[t], one[t])
    assert torch.equal(out.view(torch.int16), one.view(torch.int16))


@pytest.mark.parametrize("m", [3, 4, 7])
def test_activation_rows_64_mib_apart(backend, device, m):
    """Row strides past the matrix-core kernel's 32-bit offsets take the GEMV engine, four, two
    and one rows a launch, with the bits of the same rows side by side."""
    rows, cols = 3000, 512
    g = torch.Generator(device=device).manual_seed(m)
    w, bias = (torch.randn(s, generator=g, device=device).mul_(0.05).half() for s in ((rows, cols), (rows,)))
    w8 = torch.randn((rows, cols), generator=g, device=device).mul_(100).clamp_(-448, 448).to(torch.float8_e4m3fn)
    scales = torch.rand(rows, generator=g, device=device) * 0.01 + 1e-3
    x = torch.randn((m, cols), generator=g, device=device).half()
    w[rows // 2] = w[rows - 1] = x[m - 1] * 0.25          # a tied maximum of the last row
    far = torch.empty((m, 1 << 25), device=device, dtype=torch.float16)[:, :cols]
    far.copy_(x)
    results = []
    for a in (far, x):
        y, y8, logits = (torch.empty((m, rows), device=device, dtype=torch.float16) for _ in range(3))
        backend.matvec_bias_rows(w, bias, a, y)
        backend.scaled_batched_matvec(w8, scales, a, y8)
        tokens = backend.matvec_argmax_batched(w, a, logits)
        results.append((y.view(torch.int16), y8.view(torch.int16), logits.view(torch.int16), tokens))
    for got, want in zip(*results):
        assert torch.equal(got, want)
