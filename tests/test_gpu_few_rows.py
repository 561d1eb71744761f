"""GPU: the grouped GEMM for groups of few rows (csrc/few_rows_gemm.h) against the general one.

Both kernels take a row's products in the same order, so a token's output is the same bytes
in a batch of few rows per expert and in one of many.  The batches put groups on both sides
of the 16-, 32- and 48-row tile edges; I = 320 leaves half of the last gate/up tile and of
the last down K tile empty; some token rows are scaled so that their h chunks carry
different exponents."""

from __future__ import annotations

import numpy as np
import pytest

from raon_npu_amd import geometry as G

from moe_fixtures import compare_bf16, make_layer, random_tokens
from oracle import bfp16 as B
from oracle import moe as om

pytestmark = pytest.mark.gpu

GEOM = dict(hidden=512, inter=320, n_routed=16, n_shared=1, top_k=2)
FEW, MANY = 200, 1200  # 25 and 150 rows per expert: below and above the line at 46


def _routes(rng, T):
    """Skewed routing: expert e is drawn ~ 1 / (1 + e), so group sizes span the tile edges."""
    p = 1.0 / (1.0 + np.arange(16))
    return np.stack([rng.choice(16, 2, replace=False, p=p / p.sum()) for _ in range(T)]).astype(np.int32)


def _tokens(T, seed, hidden=512):
    x = random_tokens(T, hidden, seed)
    u = x.astype(np.uint32)
    # rows 5, 25, 45, ...: a hundred times 2^12 larger, rows 6, 26, ... 2^-14 smaller
    for r0, shift in ((5, 12), (6, -14)):
        e = (u[r0::20] >> 7) & 0xFF
        u[r0::20] = (u[r0::20] & ~np.uint32(0xFF << 7)) | (np.clip(e.astype(np.int64) + shift, 1, 250).astype(np.uint32) << 7)
    return u.astype(np.uint16)


@pytest.mark.parametrize("layout", ["q4nx", "weights-d"])
@pytest.mark.parametrize("betas", [(None, None), (4.0, 25.0)])
def test_few_rows_equals_many_rows(gpu_ctx, layout, betas):
    geom = G.MoeGeometry(**GEOM)
    syn = make_layer(geom, seed=71)
    rng = np.random.default_rng(72)
    if layout == "q4nx":
        lyr = gpu_ctx.create_layer(1700, geom)
        lyr.upload_experts(syn.gate_up, syn.down)
    else:
        lyr = gpu_ctx.create_layer_d(1700, geom)
        lyr.upload_d(1, 0, syn.gate_up[: geom.n_routed * geom.gu_bytes])
        w = rng.normal(0.0, 0.02, (geom.n_experts, geom.hidden, geom.inter_pad)).astype(np.float32)
        lyr.upload_d(2, 0, b"".join(B.pack_gemv(m) for m in w))
    x, ids = _tokens(MANY, 73), _routes(rng, MANY)
    wts = rng.uniform(0.1, 0.9, ids.shape).astype(np.float32)
    sgu = random_tokens(MANY, 2 * geom.inter, 74)
    want_r, want_s = lyr.moe_experts_grouped(x, ids, wts, sgu, *betas)
    assert len(set(np.bincount(ids[:FEW].reshape(-1), minlength=16) // 16)) > 2  # several tile classes
    for T in (1, 2, 17, 33, 48, 49, FEW):
        r, s = lyr.moe_experts_grouped(x[:T], ids[:T], wts[:T], sgu[:T], *betas)
        np.testing.assert_array_equal(r, want_r[:T], err_msg=f"routed, T={T}")
        np.testing.assert_array_equal(s, want_s[:T], err_msg=f"shared, T={T}")
    lyr.free()


def test_few_rows_prefill_equals_many_rows(gpu_ctx):
    """The device-routed form (the shared expert's gate/up in the layer) over the same line."""
    import torch

    geom = G.MoeGeometry(**GEOM)
    syn = make_layer(geom, seed=75)
    lyr = gpu_ctx.create_layer(1701, geom)
    lyr.upload_experts(syn.gate_up, syn.down)
    lyr.set_router(syn.router, score="softmax")
    lyr.reserve(MANY)
    x = torch.from_numpy(_tokens(MANY, 76).view(np.int16)).cuda()

    def run(T):
        out = torch.empty(T, geom.hidden, dtype=torch.int16, device="cuda")
        lyr.moe_prefill_dev(x[:T].contiguous(), T, out, stream=torch.cuda.current_stream())
        torch.cuda.synchronize()
        return out.cpu().numpy()

    want = run(MANY)
    for T in (1, 16, 47, FEW):
        np.testing.assert_array_equal(run(T), want[:T], err_msg=f"T={T}")
    lyr.free()


# Blocks of 32 groups in the correction: one, two and a quarter, three and a quarter (the widest
# whose scales stay in LDS), three and a half, eight; the same for the down GEMM, whose width is
# not limited (8,704: with its scales in LDS a workgroup would take more than a CU has); rows per
# group for each tile class.
@pytest.mark.parametrize("hidden,inter", [(1024, 64), (2304, 64), (3328, 64), (3584, 64), (8192, 64), (256, 3328),
                                          (256, 3392), (256, 8704)])
def test_few_rows_widths(gpu_ctx, hidden, inter):
    geom = G.MoeGeometry(hidden=hidden, inter=inter, n_routed=4, n_shared=1, top_k=1)
    syn = make_layer(geom, seed=77)
    lyr = gpu_ctx.create_layer(1702, geom)
    lyr.upload_experts(syn.gate_up, syn.down)
    x = _tokens(260, 78, hidden)
    ids = np.repeat(np.arange(4), [5, 16, 30, 209]).astype(np.int32)[:, None]
    wts = np.ones(ids.shape, np.float32)
    sgu = random_tokens(260, 2 * inter, 79)
    want_r, want_s = lyr.moe_experts_grouped(x, ids, wts, sgu)  # 65 rows per expert: the general kernel
    for T in (5, 51, 98):  # the last groups hold 5, 30 and 47 rows
        r, s = lyr.moe_experts_grouped(x[:T], ids[:T], wts[:T], sgu[:T])
        np.testing.assert_array_equal(r, want_r[:T], err_msg=f"routed, T={T}")
        np.testing.assert_array_equal(s, want_s[:T], err_msg=f"shared, T={T}")
    bank = syn.bank()
    for t in (0, 21, 97):
        _, rel, _ = compare_bf16(want_r[t], om.moe_experts(bank, x[t], ids[t], wts[t], 4.0, 25.0))
        assert rel <= 4e-3, (t, rel)  # one bf16 rounding per element: 2^-8
    lyr.free()


# The shared group's last tile in each class (12, 32 and 47 rows of 48; 24, 60 and 100 of 128), which
# the gate/up GEMM leaves out of its tiles: 16 experts (table by the scatter launch), 256 (its own).
@pytest.mark.parametrize("experts", [16, 256])
def test_shared_tiles_left_out_of_gate_up(gpu_ctx, experts):
    geom = G.MoeGeometry(hidden=256, inter=64, n_routed=experts, n_shared=1, top_k=1)
    syn = make_layer(geom, seed=91)
    lyr = gpu_ctx.create_layer(1703, geom)
    lyr.upload_experts(syn.gate_up, syn.down)
    few, many = (300, 320, 335), tuple(128 * (experts // 2) + r for r in (24, 60, 100))
    T = max(many)
    rng = np.random.default_rng(92)
    x, ids = random_tokens(T, 256, 93), rng.integers(0, experts, (T, 1)).astype(np.int32)
    wts = np.ones(ids.shape, np.float32)
    sgu = random_tokens(T, 128, 94)
    want_r, want_s = lyr.moe_experts_grouped(x, ids, wts, sgu)
    bank = syn.bank()
    for t in (0, 150, T - 1):
        _, rel, _ = compare_bf16(want_r[t], om.moe_experts(bank, x[t], ids[t], wts[t], 4.0, 25.0))
        assert rel <= 4e-3, (t, rel)  # one bf16 rounding per element: 2^-8
    for n in few + many:
        r, s = lyr.moe_experts_grouped(x[:n], ids[:n], wts[:n], sgu[:n])
        np.testing.assert_array_equal(r, want_r[:n], err_msg=f"routed, T={n}")
        np.testing.assert_array_equal(s, want_s[:n], err_msg=f"shared, T={n}")
    lyr.free()
