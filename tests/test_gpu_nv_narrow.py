"""GPU parity of the NVFP4 kernel on 128-column tiles: both tile heights, whole stages and every kind of K tail, K split
into slices, ragged tiles, and the shapes where dispatch changes over to it."""
import numpy as np
import pytest
import torch

from avelang_amd import _lib
from oracle import fp4_oracle as orc
from tests import helpers as H
from tests.onehot_patterns import nv_expect, nv_onehot, nv_varied, same_bits

pytestmark = pytest.mark.gpu
NARROW = 4


def _narrow(gpu, ops, tile_rows, slice_stages):
    a, a_s, a_g, b, b_s, b_g = ops
    m, k, n = a.shape[0], a.shape[1] * 2, b.shape[0]
    slices = -(-(k // 256) // slice_stages) if slice_stages else 1
    ws = torch.full((slices * m * n,), float("nan"), dtype=torch.float32, device=gpu)
    out = torch.full((m, n), float("nan"), dtype=torch.bfloat16, device=gpu)
    da, das, db, dbs = (H.to_dev(x, gpu) for x in (a, a_s, b, b_s))
    ag, bg = (torch.tensor([g], dtype=torch.float32, device=gpu) for g in (a_g, b_g))
    _lib.check(_lib.load().ave_fp4_debug_gemm_nvfp4_narrow(
        da.data_ptr(), das.data_ptr(), ag.data_ptr(), db.data_ptr(), dbs.data_ptr(), bg.data_ptr(), out.data_ptr(), m, n, k,
        ws.data_ptr(), ws.numel() * 4, tile_rows, slice_stages, torch.cuda.current_stream(gpu).cuda_stream))
    torch.cuda.synchronize(gpu)
    return H.bits(out)


# one stage to more than the ring holds; tails of 1, 2, 3, 4, 5, 8, 12, 13 and 15 blocks of 16; one row, one column, part tiles
@pytest.mark.parametrize("m,n,k", [(1, 1, 256), (64, 128, 512), (65, 129, 768), (128, 256, 1024), (129, 5, 1536), (130, 300, 1792),
                                   (200, 130, 272), (3, 200, 288), (64, 257, 304), (100, 128, 320), (70, 140, 848), (128, 136, 896),
                                   (33, 264, 1216), (260, 100, 1488), (77, 200, 1520)])
@pytest.mark.parametrize("tile_rows", [64, 128])
def test_nv_narrow_random_bytes_and_scales(gpu, m, n, k, tile_rows):
    """Random codes under random finite E4M3 scales that differ per row and 16-block, unsplit and in slices of one to three
    stages; with unit scales the sums are exact in fp32 whatever their order, so the result is exact too."""
    rng = np.random.default_rng(m + n + k)
    a = rng.integers(0, 256, size=(m, k // 2), dtype=np.uint8)
    b = rng.integers(0, 256, size=(n, k // 2), dtype=np.uint8)
    a_s = rng.integers(0x20, 0x50, size=(m, k // 16), dtype=np.uint8)
    b_s = rng.integers(0x20, 0x50, size=(n, k // 16), dtype=np.uint8)
    one_a, one_b = np.full_like(a_s, 0x38), np.full_like(b_s, 0x38)
    exact = orc.f64_to_bf16_bits(orc.gemm_nvfp4_fp64(a, one_a, 1.0, b, one_b, 1.0))
    for slice_stages in (0, 1, 2, 3):
        if slice_stages > k // 256:
            break
        H.assert_nv_close(_narrow(gpu, (a, a_s, 0.5, b, b_s, 0.25), tile_rows, slice_stages), a, a_s, 0.5, b, b_s, 0.25)
        assert np.array_equal(_narrow(gpu, (a, one_a, 1.0, b, one_b, 1.0), tile_rows, slice_stages), exact)


@pytest.mark.parametrize("k", [512, 560])
def test_nv_narrow_every_scale_byte_both_sides(gpu, k):
    g = (0.5, 4.0)
    for rows in (528, 64):
        b, b_s = nv_varied(rows, k)
        a, a_s = nv_onehot(0, k, k)
        same_bits(H.run_nv(gpu, a, a_s, g[0], b, b_s, g[1], variant=NARROW), nv_expect(a, a_s, g[0], b, b_s, g[1]))
        a, a_s = nv_varied(rows, k)
        b, b_s = nv_onehot(0, k, k)
        same_bits(H.run_nv(gpu, a, a_s, g[0], b, b_s, g[1], variant=NARROW), nv_expect(a, a_s, g[0], b, b_s, g[1]))


@pytest.mark.parametrize("m,n,k", [(64, 3600, 4096), (32, 2048, 6912), (48, 600, 3584), (16, 256, 4176), (320, 1024, 2048), (200, 300, 1040),
                                   (700, 520, 1152)])
def test_nv_dispatch_around_the_narrow_kernel(gpu, m, n, k):
    a, a_s, a_g = H.nv_operand(m, k, seed=m)
    b, b_s, b_g = H.nv_operand(n, k, seed=n, std=0.02)
    H.assert_nv_close(H.run_nv(gpu, a, a_s, a_g, b, b_s, b_g), a, a_s, a_g, b, b_s, b_g)
