"""GPU: the MFMA form of ``linear`` (csrc/linear_mfma.hip) at the edges of its token tiles
(4, 16 and 32 tokens), weight-row tiles and K splits (2 to 94 K tiles over 2, 4 or 8 waves).

Reference: the dequantized weights times x in float64, rounded once to bf16.  The kernel's
fp32 sums are within (K + 64) * 2^-23 * sum |x w| of that before its one rounding, so every
output is within one bf16 step of the reference plus that bound."""

from __future__ import annotations

import numpy as np
import pytest

from oracle import bfp16 as B
from oracle.bf16 import bf16_to_f32, f32_to_bf16
from oracle.q4nx import dequantize_simple, pack_gemv, quantize

pytestmark = pytest.mark.gpu

# (128, 512) and (768, 2048) in q4nx are shapes whose one-token device calls run the GEMV.
SHAPES = [(128, 256), (384, 768), (2176, 2560), (128, 12032), (128, 512), (768, 2048)]


def _matrix(gpu_ctx, fmt, M, K, seed):
    rng = np.random.default_rng(seed)
    w = rng.normal(0.0, 0.02, (M, K)).astype(np.float32)
    if fmt == "q4nx":
        c, s, m = quantize(w)
        return gpu_ctx.upload_matrix(pack_gemv(c, s, m), M, K), dequantize_simple(c, s, m).astype(np.float64), rng
    blob = B.pack_gemv(w)
    return gpu_ctx.upload_matrix(blob, M, K, fmt="bfp16"), B.dequantize_packed(blob, K, M).astype(np.float64), rng


def _check(y, x, w):
    xf = bf16_to_f32(x).astype(np.float64)
    ref = xf @ w.T
    slack = (w.shape[1] + 64) * 2.0**-23 * (np.abs(xf) @ np.abs(w.T))
    assert np.all(np.abs(bf16_to_f32(y) - ref) <= np.abs(ref) * 2.0**-8 + slack)


@pytest.mark.parametrize("fmt", ["q4nx", "bfp16"])
@pytest.mark.parametrize("M,K", SHAPES)
def test_batches_are_stacked_rows(gpu_ctx, fmt, M, K):
    """Every batch size against float64, and a row's bytes the same in all of them, a batch
    of one row included."""
    mat, w, rng = _matrix(gpu_ctx, fmt, M, K, M + 3 * K)
    x = f32_to_bf16(rng.standard_normal((70, K)).astype(np.float32))
    full = mat.linear(x)
    _check(full, x, w)
    for T in (2, 4, 5, 15, 16, 17, 31, 32, 33, 64, 65):
        np.testing.assert_array_equal(mat.linear(x[:T]), full[:T], err_msg=f"T={T}")
    for t in range(70):
        np.testing.assert_array_equal(mat.linear(x[t:t + 1])[0], full[t], err_msg=f"row {t} alone")
    mat.free()


@pytest.mark.parametrize("fmt", ["q4nx", "bfp16"])
def test_largest_tile_of_eight_waves(gpu_ctx, fmt):
    """K = 8,192 (eight waves) with enough tokens for the 32 x 64 tiles: the most LDS of all."""
    T = 3553
    mat, w, rng = _matrix(gpu_ctx, fmt, 256, 8192, 11)
    x = f32_to_bf16(rng.standard_normal((T, 8192), dtype=np.float32))
    _check(mat.linear(x), x, w)
    mat.free()


@pytest.mark.parametrize("fmt", ["q4nx", "bfp16"])
@pytest.mark.parametrize("T", [3, 20])
def test_operands_at_odd_addresses(gpu_ctx, fmt, T):
    """x that the 16-byte loads cannot take runs the K-split kernels; y that the 8-byte stores
    cannot take is stored by halves, the same bytes as in place."""
    import torch

    M, K = 256, 768
    mat, w, rng = _matrix(gpu_ctx, fmt, M, K, 5)
    mat.reserve(T)
    x = f32_to_bf16(rng.standard_normal((T, K)).astype(np.float32))
    for ox, oy in ((2, 0), (0, 1), (0, 2), (6, 3)):
        xb = torch.zeros(T * K + 16, dtype=torch.int16, device="cuda")
        yb = torch.zeros(T * M + 16, dtype=torch.int16, device="cuda")
        xd, yd = xb[ox:ox + T * K].view(T, K), yb[oy:oy + T * M].view(T, M)
        xd.copy_(torch.from_numpy(x.view(np.int16)))
        mat.linear_dev(xd, T, yd, stream=torch.cuda.current_stream())
        torch.cuda.synchronize()
        y = yd.cpu().numpy().view(np.uint16)
        _check(y, x, w)
        if ox == 0:
            np.testing.assert_array_equal(y, mat.linear(x))
        assert not yb[:oy].any() and not yb[oy + T * M:].any()
    mat.free()


@pytest.mark.parametrize("fmt", ["q4nx", "bfp16"])
def test_batch_larger_than_one_launch(gpu_ctx, fmt):
    """x of more than 4 GiB runs as several launches: every row as in batches of 65,536 tokens."""
    import torch

    K, T = 8192, 262144 + 77
    mat, _, _ = _matrix(gpu_ctx, fmt, 128, K, 13)
    mat.reserve(T)
    g = torch.Generator(device="cuda").manual_seed(14)
    x = torch.empty(T, K, dtype=torch.int16, device="cuda")
    for t0 in range(0, T, 65536):
        rows = x[t0:t0 + 65536]
        rows.copy_(torch.randn(rows.shape, device="cuda", generator=g).to(torch.bfloat16).view(torch.int16))
    y, want = (torch.zeros(T, 128, dtype=torch.int16, device="cuda") for _ in range(2))
    st = torch.cuda.current_stream()
    mat.linear_dev(x, T, y, stream=st)
    for t0 in range(0, T, 65536):
        n = min(65536, T - t0)
        mat.linear_dev(x[t0:t0 + n], n, want[t0:t0 + n], stream=st)
    torch.cuda.synchronize()
    assert torch.equal(y, want) and bool((y != 0).any(1).all())
    mat.free()


def test_non_finite_rows_stay_in_their_row(gpu_ctx):
    """Rows of x with an infinity or a NaN are not finite; the other rows of the tile are as without them."""
    for fmt in ("q4nx", "bfp16"):
        mat, w, rng = _matrix(gpu_ctx, fmt, 128, 512, 9)
        x = f32_to_bf16(rng.standard_normal((18, 512)).astype(np.float32))
        want = mat.linear(x)
        bad = x.copy()
        bad[3, 7], bad[17, 300] = 0x7F80, 0x7FC0
        y = mat.linear(bad)
        keep = [t for t in range(18) if t not in (3, 17)]
        np.testing.assert_array_equal(y[keep], want[keep])
        assert not np.isfinite(bf16_to_f32(y[[3, 17]])).any()
        mat.free()
