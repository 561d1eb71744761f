"""GPU: q4nx upload re-layout round trips and the device quantizer vs the oracle (bit-exact)."""

from __future__ import annotations

import numpy as np
import pytest

from oracle.q4nx import pack_gemv, quantize

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("M,K", [(128, 256), (768, 2048), (2176, 2560), (2048, 1280), (1536, 2048)])
def test_upload_download_round_trip(gpu_ctx, M, K):
    rng = np.random.default_rng(M + K)
    blob = rng.integers(0, 256, M * K * 5 // 8, dtype=np.uint8)
    # scales/mins are arbitrary bf16 bits: the layout must move every byte unchanged
    mat = gpu_ctx.upload_matrix(blob, M, K)
    assert mat.download() == blob.tobytes()
    mat.free()


def _quantize_on_gpu(gpu_ctx, w):
    import torch

    wd = torch.from_numpy(w).cuda()
    mat = gpu_ctx.quantize_matrix(wd, *w.shape)
    out = mat.download()
    mat.free()
    return out


@pytest.mark.parametrize("M,K,scale", [(128, 256, 0.02), (768, 2048, 0.02), (256, 512, 2.5), (128, 1024, 1e-30)])
def test_device_quantizer_matches_oracle(gpu_ctx, M, K, scale):
    rng = np.random.default_rng(99)
    w = (rng.standard_normal((M, K)) * scale).astype(np.float32)
    assert _quantize_on_gpu(gpu_ctx, w) == pack_gemv(*quantize(w))


def test_device_quantizer_edge_groups(gpu_ctx):
    w = np.zeros((128, 256), np.float32)
    w[:, 32:64] = 5.0
    w[:, 64:96] = -12.5
    w[:, 96:128] = np.linspace(1.0, 10.0, 32, dtype=np.float32)
    w[:, 128:160] = 0.1
    w[0, 160] = -3e38
    w[0, 161] = 3e38
    w[1:, 160:192] = np.linspace(1001.0, 1001.1, 32, dtype=np.float32)
    w[:, 192:] = np.random.default_rng(1).standard_normal((128, 64)).astype(np.float32) * 1e-40
    assert _quantize_on_gpu(gpu_ctx, w) == pack_gemv(*quantize(w))


def test_device_quantizer_rejects_non_finite(gpu_ctx):
    w = np.ones((128, 256), np.float32)
    w[3, 7] = np.nan
    with pytest.raises(ValueError, match="non-finite"):
        _quantize_on_gpu(gpu_ctx, w)


def test_expert_quantizer_pads_down_columns(gpu_ctx):
    import torch

    import raon_npu_amd.geometry as G
    from oracle.q4nx import pad

    geom = G.MoeGeometry(hidden=256, inter=192, n_routed=2, n_shared=1, top_k=1)  # Ipad = 256
    rng = np.random.default_rng(5)
    gu = (rng.standard_normal((2 * geom.inter, geom.hidden)) * 0.02).astype(np.float32)
    dn = (rng.standard_normal((geom.hidden, geom.inter)) * 0.02).astype(np.float32)
    lyr = gpu_ctx.create_layer(900, geom)
    lyr.quantize_expert(1, torch.from_numpy(gu).cuda(), torch.from_numpy(dn).cuda())
    got_gu, got_dn = lyr.download_expert(1)
    assert got_gu == pack_gemv(*quantize(gu))
    assert got_dn == pack_gemv(*quantize(pad(dn, 128, 256)[0]))
    lyr.free()


@pytest.mark.parametrize("M, K, offset", [(128, 256, 1), (384, 768, 3), (256, 2304, 0)])
def test_quantize_and_download_tiles(gpu_ctx, M, K, offset):
    """Tile and block edges of the LDS transposes; a source that is 4-byte aligned only."""
    import torch

    rng = np.random.default_rng(M + K)
    w = rng.normal(0.0, 0.02, (M, K)).astype(np.float32)
    buf = torch.zeros(M * K + 4, dtype=torch.float32, device="cuda")
    buf[offset : offset + M * K] = torch.from_numpy(w).cuda().reshape(-1)
    torch.cuda.synchronize()
    mat = gpu_ctx.quantize_matrix(buf[offset : offset + M * K].view(M, K), M, K)
    assert bytes(mat.download()) == pack_gemv(*quantize(w))
    mat.free()
    blob = rng.integers(0, 256, M * K * 5 // 8, dtype=np.uint8).tobytes()
    mat = gpu_ctx.upload_matrix(blob, M, K)
    assert bytes(mat.download()) == blob
    mat.free()


def test_quantize_weights_still_being_written(gpu_ctx):
    """Without a stream argument, quantizing waits for work queued on any stream before the call
    (here 50 ms of it ahead of the copies that fill the weights)."""
    import torch

    import raon_npu_amd.geometry as G

    rng = np.random.default_rng(61)
    w = rng.normal(0.0, 0.02, (128, 256)).astype(np.float32)
    want = pack_gemv(*quantize(w))
    src = torch.from_numpy(w).cuda()
    buf, gu = torch.zeros_like(src), torch.zeros_like(src)
    dn = torch.zeros(256, 64, device="cuda")
    lyr = gpu_ctx.create_layer(61, G.MoeGeometry(hidden=256, inter=64, n_routed=1, n_shared=0, top_k=1))
    torch.cuda.synchronize()
    torch.cuda._sleep(100_000_000)
    buf.copy_(src)
    mat = gpu_ctx.quantize_matrix(buf, 128, 256)
    torch.cuda._sleep(100_000_000)
    gu.copy_(src)
    lyr.quantize_expert(0, gu, dn)
    assert bytes(mat.download()) == bytes(want)
    assert bytes(lyr.download_expert(0)[0]) == bytes(want)
    mat.free()
    lyr.free()


# q4nx: 51 blocks of 10,240 bytes are one chunk of the download; 50, 52, 204 (the whole ring)
# and 206 blocks.  bfp16: the same sizes at nine bits, chunks cut anywhere.
@pytest.mark.parametrize("fmt, bits", [("q4nx", 5), ("bfp16", 9)])
@pytest.mark.parametrize("blocks", [50, 52, 204, 206])
def test_download_chunk_edges(gpu_ctx, fmt, bits, blocks):
    M, K = 128, 128 * blocks
    blob = np.random.default_rng(blocks).integers(0, 256, M * K * bits // 8, dtype=np.uint8).tobytes()
    mat = gpu_ctx.upload_matrix(blob, M, K, fmt=fmt)
    for _ in range(2):
        assert mat.download() == blob
    mat.free()
