"""GPU: the padding of the h rows and the combine's width in the grouped prefill.

The gate/up GEMM's last n-tile clears a row's columns past I, their group sums and the
exponents of the chunks past the last live one; the combine takes one workgroup of
H / 8 threads per token.  Down weights that are not zero past I make whatever stands there
visible: the columns and exponents to both formats, the group sums to the q4nx down, whose
scales and mins multiply the sums of all groups.  Each result is computed again after a call
that leaves large values in the whole scratch, and compared with the oracle over weights cut
at I."""

from __future__ import annotations

import numpy as np
import pytest

from raon_npu_amd import geometry as G

from moe_fixtures import compare_bf16, make_layer, random_tokens
from oracle import bfp16 as B
from oracle import moe as om
from oracle.q4nx import pack_gemv, quantize

pytestmark = pytest.mark.gpu


# I: 320 -> Ipad 512 (a half-live chunk, one dead), 64 -> 256, 448 -> 512; T on both sides
# of the line between the two grouped kernels (46 rows per expert).
@pytest.mark.parametrize("inter", [64, 320, 448])
@pytest.mark.parametrize("T", [3, 300])
@pytest.mark.parametrize("layout", ["weights-d", "q4nx"])
def test_padding_is_cleared_on_every_call(gpu_ctx, inter, T, layout):
    geom = G.MoeGeometry(hidden=256, inter=inter, n_routed=8, n_shared=1, top_k=2)
    full = G.MoeGeometry(hidden=256, inter=geom.inter_pad, n_routed=8, n_shared=1, top_k=2)
    rng = np.random.default_rng(81)
    downs = rng.normal(0.0, 0.02, (9, 256, geom.inter_pad)).astype(np.float32)

    def pack(mats):
        return b"".join(B.pack_gemv(m) if layout == "weights-d" else bytes(pack_gemv(*quantize(m))) for m in mats)

    lyrs = []
    for i, g in enumerate((geom, full)):
        syn = make_layer(g, seed=82 + i)
        if layout == "weights-d":
            lyr = gpu_ctx.create_layer_d(1710 + i, g)
            lyr.upload_d(1, 0, syn.gate_up[: 8 * g.gu_bytes])
            lyr.upload_d(2, 0, pack(downs))
        else:
            lyr = gpu_ctx.create_layer(1710 + i, g)
            lyr.upload_experts(syn.gate_up, pack(downs))
        lyrs.append((lyr, syn.gate_up))
    cut = downs.copy()
    cut[:, :, inter:] = 0.0  # I % 64 == 0: whole groups and blocks, the others keep their bytes
    gate_up = lyrs[0][1]
    if layout == "weights-d":
        bank = om.DExpertBank(gate_up[: 8 * geom.gu_bytes], pack(cut), 8, 256, inter)
    else:
        bank = om.ExpertBank(gate_up, pack(cut), 9, 256, inter)
    ids = np.stack([rng.choice(8, 2, replace=False) for _ in range(T)]).astype(np.int32)
    wts = rng.uniform(0.1, 0.9, ids.shape).astype(np.float32)
    x = random_tokens(T, 256, 84)
    big = ((x & 0x8000) | 0x4400).astype(np.uint16)  # +-512
    sgu, sgu_big = random_tokens(T, 2 * inter, 85), np.full((T, 2 * geom.inter_pad), 0x4400, np.uint16)
    want = lyrs[0][0].moe_experts_grouped(x, ids, wts, sgu, 4.0, 25.0)
    lyrs[1][0].moe_experts_grouped(big, ids, wts, sgu_big, None, None)
    again = lyrs[0][0].moe_experts_grouped(x, ids, wts, sgu, 4.0, 25.0)
    np.testing.assert_array_equal(again[0], want[0])
    np.testing.assert_array_equal(again[1], want[1])
    for t in range(0, T, 97):
        err, rel, _ = compare_bf16(again[0][t], om.moe_experts(bank, x[t], ids[t], wts[t], 4.0, 25.0))
        assert err <= 1e-2 and rel <= 4e-3, (t, err, rel)  # one bf16 rounding per element: 2^-8
    for lyr, _ in lyrs:
        lyr.free()


# 256: 32 live threads of 64; 768: two waves, the second half full; 8192: the widest.
@pytest.mark.parametrize("hidden", [256, 768, 8192])
def test_combine_widths(gpu_ctx, hidden):
    geom = G.MoeGeometry(hidden=hidden, inter=64, n_routed=4, n_shared=1, top_k=2)
    syn = make_layer(geom, seed=86)
    lyr = gpu_ctx.create_layer(1712, geom)
    lyr.upload_experts(syn.gate_up, syn.down)
    x = random_tokens(5, hidden, 87)
    rng = np.random.default_rng(88)
    ids = np.stack([rng.choice(4, 2, replace=False) for _ in range(5)]).astype(np.int32)
    wts = rng.uniform(0.1, 0.9, ids.shape).astype(np.float32)
    sgu = random_tokens(5, 128, 89)
    got, _ = lyr.moe_experts_grouped(x, ids, wts, sgu)
    for t in range(5):
        err, rel, _ = compare_bf16(got[t], lyr.moe_experts(x[t], ids[t], wts[t]))
        assert err <= 1e-2 and rel <= 4e-3, (t, err, rel)
    lyr.free()
