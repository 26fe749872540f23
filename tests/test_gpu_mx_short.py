"""GPU parity of the MXFP4 kernel for small calls: every number of MFMAs per wave, K that ends in any wave, ragged rows and columns,
scale tensors and outputs at odd addresses, and the shapes at which dispatch changes to it and away from it."""
import numpy as np
import pytest
import torch

from avelang_amd import _lib, gemm_mxfp4_transposed_b
from tests import helpers as H

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("k", [32, 64, 96, 224, 256, 288, 480, 512, 544, 1024, 1056, 1280, 2016, 2048])
@pytest.mark.parametrize("m,n", [(1, 1), (33, 36), (64, 95), (97, 256)])
def test_short_matches_oracle(gpu, m, n, k):
    a, a_s = H.mx_operand(m, k, seed=m + k, outliers=True)
    b, b_s = H.mx_operand(n, k, seed=n + k, std=0.05)
    H.assert_mx_close(H.run_mx(gpu, a, a_s, b, b_s, variant=_lib.SHORT), a, a_s, b, b_s)


@pytest.mark.parametrize("k", [256, 512, 1024, 2048])
def test_short_takes_scales_and_outputs_at_any_address(gpu, k):
    m, n = 40, 68
    a, a_s = H.mx_operand(m, k, seed=k)
    b, b_s = H.mx_operand(n, k, seed=k + 1, std=0.05)
    want = H.run_mx(gpu, a, a_s, b, b_s, variant=_lib.SHORT)

    def moved(x):   # one byte behind an aligned address
        t = torch.empty(x.size + 1, dtype=torch.uint8, device=gpu)
        t[1:] = H.to_dev(x.reshape(-1), gpu)
        return t[1:].reshape(x.shape)

    out = torch.empty(m * n + 1, dtype=torch.bfloat16, device=gpu)[1:].reshape(m, n)
    gemm_mxfp4_transposed_b(H.to_dev(a, gpu), moved(a_s), H.to_dev(b, gpu), moved(b_s), out=out, variant=_lib.SHORT)
    assert np.array_equal(H.bits(out), want)


# around the lines of the dispatch rule: K 256 / 288 / 512 / 1024 / 1280, and rounds of blocks that it takes and leaves
@pytest.mark.parametrize("m,n,k", [(256, 256, 256), (48, 4096, 288), (16, 4096, 512), (600, 2560, 256), (600, 4096, 256), (64, 4096, 1024),
                                   (64, 8224, 1024), (100, 2048, 1280), (100, 2080, 1280), (2048, 1024, 160)])
def test_dispatch_around_the_small_calls(gpu, m, n, k):
    a, a_s = H.mx_operand(m, k, seed=m)
    b, b_s = H.mx_operand(n, k, seed=n, std=0.05)
    H.assert_mx_close(H.run_mx(gpu, a, a_s, b, b_s), a, a_s, b, b_s)
