"""GPU parity of the grouped MXFP4 kernel for a few rows per expert: every tile height, tiles of two and more stages with
every kind of K tail, experts around a tile's rows, plain, with SwiGLU and with SwiGLU and the quantiser."""
import numpy as np
import pytest
import torch

from avelang_amd import (_lib, gemm_mxfp4_swiglu_quant_transposed_b, gemm_mxfp4_swiglu_transposed_b,
                         grouped_gemm_mxfp4_swiglu_quant_transposed_b, grouped_gemm_mxfp4_swiglu_transposed_b,
                         grouped_gemm_mxfp4_transposed_b, quantize_mxfp4)
from oracle import fp4_oracle as orc
from tests import helpers as H

pytestmark = pytest.mark.gpu
NARROW = 4
BY_LINES, CHUNKS, PAIRS = 0x1000, 0x2000, 0x4000   # include/ave_fp4_debug.h


def _stream(gpu, ops, ro, n, tile_rows, swiglu, quant):
    m, k, e = ops[0].shape[0], ops[0].shape[1] * 2, ops[2].shape[0]
    c = torch.full((m, n), float("nan"), dtype=torch.bfloat16, device=gpu)
    q = torch.full((m, n // 2), 0xEE, dtype=torch.uint8, device=gpu)
    qs = torch.full((m, n // 32), 0xEE, dtype=torch.uint8, device=gpu)
    _lib.check(_lib.load().ave_fp4_debug_grouped_gemm_mxfp4_stream(
        *(t.data_ptr() for t in ops), ro.data_ptr(), None if quant else c.data_ptr(), q.data_ptr() if quant else None,
        qs.data_ptr() if quant else None, m, e, n, k, swiglu, tile_rows, torch.cuda.current_stream(gpu).cuda_stream))
    torch.cuda.synchronize(gpu)
    return (q, qs) if quant else c


# rows per expert around 32, 64 and 128 and several tiles; two, three, four and more stages; K % 512 of 1, 7, 8, 9 and 15 blocks
@pytest.mark.parametrize("rows,n,k", [([3, 0, 31, 33], 64, 512), ([1], 32, 544), ([64, 65, 0, 127], 96, 736), ([129, 5], 160, 768),
                                      ([32, 200, 1, 70], 128, 800), ([40, 130, 0, 300], 192, 992), ([17] * 20, 352, 1024),
                                      ([2] * 70, 64, 1312), ([66, 0, 140], 224, 2880), ([5] * 40 + [90], 512, 1792)])
@pytest.mark.parametrize("tile_rows", [32, 64, 128])
def test_stream_matches_oracle_and_its_own_fused_forms(gpu, rows, n, k, tile_rows):
    e, m = len(rows), sum(rows)
    ro = np.concatenate([[0], np.cumsum(rows)]).astype(np.int32)
    a, a_s = H.mx_operand(m, k, seed=m + k)
    b, b_s = H.mx_operand(e * 2 * n, k, seed=n + k, std=0.05)
    b, b_s = b.reshape(e, 2 * n, k // 2), b_s.reshape(e, 2 * n, k // 32)
    ops = [H.to_dev(t, gpu) for t in (a, a_s, b, b_s)]
    dro = torch.from_numpy(ro).to(gpu)
    plain = H.bits(_stream(gpu, ops, dro, 2 * n, tile_rows, 0, False))
    fused = _stream(gpu, ops, dro, n, tile_rows, 1, False)
    q, qs = _stream(gpu, ops, dro, n, tile_rows, 1, True)
    for x in range(e):
        r0, r1 = int(ro[x]), int(ro[x + 1])
        if r1 > r0:
            H.assert_mx_close(plain[r0:r1], a[r0:r1], a_s[r0:r1], b[x], b_s[x])
            ok, rep = orc.check_swiglu_bf16(H.bits(fused[r0:r1]), a[r0:r1], a_s[r0:r1], b[x], b_s[x])
            assert ok, (x, rep)
    want_q, want_s = quantize_mxfp4(fused)
    assert torch.equal(q, want_q) and torch.equal(qs, want_s)


# chunks of two pairs of scale rows: items of two, three, five, six and nine stages, several to a workgroup, so that short chunks (one
# stage, two stages) follow each other in the slots; scale bytes differ in every block, so a piece of another pair or row shows
@pytest.mark.parametrize("k", [512, 672, 1056, 1536, 2144])
@pytest.mark.parametrize("tile_rows", [32, 64, 128])
def test_stream_scale_chunks_over_several_tiles(gpu, k, tile_rows):
    e, n = 90, 384   # three n-tiles: 270 and more tiles on 256 compute units
    rows = [1 + 7 * x % 40 for x in range(e)]
    m = sum(rows)
    ro = np.concatenate([[0], np.cumsum(rows)]).astype(np.int32)
    rng = np.random.default_rng(k)
    a, a_s = H.mx_operand(m, k, seed=k)
    b, b_s = H.mx_operand(e * n, k, seed=k + 1, std=0.05)
    a_s = (a_s.astype(np.int32) + rng.integers(-3, 4, size=a_s.shape)).clip(1, 254).astype(np.uint8)
    b_s = (b_s.astype(np.int32) + rng.integers(-3, 4, size=b_s.shape)).clip(1, 254).astype(np.uint8)
    b, b_s = b.reshape(e, n, k // 2), b_s.reshape(e, n, k // 32)
    ops = [H.to_dev(t, gpu) for t in (a, a_s, b, b_s)]
    dro = torch.from_numpy(ro).to(gpu)
    c = H.bits(_stream(gpu, ops, dro, n, tile_rows | 0x1000, 0, False))   # (the form for weights from HBM)
    assert np.array_equal(c, H.bits(_stream(gpu, ops, dro, n, tile_rows, 0, False)))
    for x in (0, 38, e - 1):
        r0, r1 = int(ro[x]), int(ro[x + 1])
        H.assert_mx_close(c[r0:r1], a[r0:r1], a_s[r0:r1], b[x], b_s[x])
    for x in range(0, e, 7):   # the narrow-tile kernel adds up in this order
        r0, r1 = int(ro[x]), int(ro[x + 1])
        assert np.array_equal(c[r0:r1], H.run_mx(gpu, a[r0:r1], a_s[r0:r1], b[x], b_s[x], variant=NARROW)), x


# chunks without the form by lines on K of two stages and a tail, around 64 MB of weights
@pytest.mark.parametrize("k,n", [(672, 2240), (672, 2216), (992, 1504)])
@pytest.mark.parametrize("tile_rows", [32, 64, 128])
def test_stream_scale_chunks_by_the_weights_size(gpu, k, n, tile_rows):
    e = 90
    ro = np.arange(e + 1, dtype=np.int32) * 3
    gen = torch.Generator(device=gpu)
    gen.manual_seed(k + n)
    a, b = (torch.randint(0, 256, (*s, k // 2), generator=gen, device=gpu, dtype=torch.uint8) for s in ((3 * e,), (e, n)))
    a_s, b_s = (torch.randint(118, 130, (*s, k // 32), generator=gen, device=gpu, dtype=torch.uint8) for s in ((3 * e,), (e, n)))
    c = H.bits(_stream(gpu, [a, a_s, b, b_s], torch.from_numpy(ro).to(gpu), n, tile_rows | CHUNKS, 0, False))
    for x in range(0, e, 8):
        r = slice(3 * x, 3 * x + 3)
        want = H.run_mx(gpu, *(t.cpu().numpy() for t in (a[r], a_s[r], b[x], b_s[x])), variant=NARROW)
        assert np.array_equal(c[r], want), x


# two (one chunk), five (chunks of four and one in turn, the tightest use of the slots, with and without a tail), eight and nine stages;
# 270 tiles and more
@pytest.mark.parametrize("k", [512, 1120, 1280, 2048, 2304])
@pytest.mark.parametrize("tile_rows", [32, 128])
def test_stream_scale_chunks_and_pairs_give_the_same_bits_in_every_form(gpu, k, tile_rows):
    e, n = 90, 192
    ro = torch.arange(e + 1, dtype=torch.int32, device=gpu) * 5
    gen = torch.Generator(device=gpu)
    gen.manual_seed(k)
    a, b = (torch.randint(0, 256, (*s, k // 2), generator=gen, device=gpu, dtype=torch.uint8) for s in ((5 * e,), (e, 2 * n)))
    a_s, b_s = (torch.randint(118, 130, (*s, k // 32), generator=gen, device=gpu, dtype=torch.uint8) for s in ((5 * e,), (e, 2 * n)))
    for cols, swiglu, quant in ((2 * n, 0, False), (n, 1, False), (n, 1, True)):
        want = _stream(gpu, (a, a_s, b, b_s), ro, cols, tile_rows | PAIRS, swiglu, quant)
        for flags in (CHUNKS, BY_LINES, BY_LINES | PAIRS):   # (by lines: where rows do not all start at one)
            got = _stream(gpu, (a, a_s, b, b_s), ro, cols, tile_rows | flags, swiglu, quant)
            for x, y in zip(want, got) if quant else ((want, got),):
                assert torch.equal(x.view(torch.uint8), y.view(torch.uint8)), flags


# weights of 64 MB and more on both sides of the rule: rows at lines K = 1536 | 1792, by lines K = 1056 | 1568 (32 rows a tile), 2080 (128)
@pytest.mark.parametrize("k,n", [(1536, 4400), (1792, 3776), (1056, 6368), (1568, 4288), (2080, 3232)])
@pytest.mark.parametrize("tile_rows", [32, 128])
def test_stream_scale_rows_by_rule(gpu, k, n, tile_rows):
    e = 20
    ro = torch.arange(e + 1, dtype=torch.int32, device=gpu) * 3
    gen = torch.Generator(device=gpu)
    gen.manual_seed(k)
    a, b = (torch.randint(0, 256, (*s, k // 2), generator=gen, device=gpu, dtype=torch.uint8) for s in ((3 * e,), (e, n)))
    a_s, b_s = (torch.randint(118, 130, (*s, k // 32), generator=gen, device=gpu, dtype=torch.uint8) for s in ((3 * e,), (e, n)))
    assert b.numel() >= 64 << 20
    got = [_stream(gpu, (a, a_s, b, b_s), ro, n, tile_rows | flags, 0, False).view(torch.int16) for flags in (0, CHUNKS, PAIRS)]
    assert torch.equal(got[0], got[1]) and torch.equal(got[0], got[2])
    want = H.run_mx(gpu, *(t.cpu().numpy() for t in (a[-3:], a_s[-3:], b[-1], b_s[-1])), variant=NARROW)
    assert np.array_equal(H.bits(got[0][-3:].view(torch.bfloat16)), want)


# every offset of a row from its line (K / 32 mod 8), last stages that end in front of, at and behind a line's end, two to nine stages
@pytest.mark.parametrize("rows,n,k", [([3, 0, 31, 33], 64, 544), ([1, 64], 32, 576), ([64, 65, 0, 127], 96, 736), ([129, 5], 160, 768),
                                      ([32, 200, 1, 70], 128, 800), ([40, 130, 0, 300], 192, 992), ([17] * 20, 352, 1184),
                                      ([2] * 70, 64, 1312), ([66, 0, 140], 224, 2208), ([5] * 40 + [90], 96, 1056)])
@pytest.mark.parametrize("tile_rows", [32, 64, 128])
@pytest.mark.parametrize("off", [0, 16, 80])
def test_stream_by_lines_gives_the_same_bits(gpu, rows, n, k, tile_rows, off):
    """Rows loaded by whole cache lines: the same sums in the same order; `off`: operands that start 16 bytes behind each other's lines."""
    e, m = len(rows), sum(rows)
    ro = torch.from_numpy(np.concatenate([[0], np.cumsum(rows)]).astype(np.int32)).to(gpu)
    rng = np.random.default_rng(k + off)

    def behind(shape, at):
        t = torch.empty(int(np.prod(shape)) + at, dtype=torch.uint8, device=gpu)
        t[at:] = torch.from_numpy(rng.integers(0, 256, size=int(np.prod(shape)), dtype=np.uint8)).to(gpu)
        return t[at:].reshape(shape)

    a, b = behind((m, k // 2), off), behind((e, 2 * n, k // 2), 2 * off)
    a_s, b_s = (torch.from_numpy(rng.integers(118, 132, size=s, dtype=np.uint8)).to(gpu) for s in ((m, k // 32), (e, 2 * n, k // 32)))
    ops = (a, a_s, b, b_s)
    for cols, swiglu, quant in ((2 * n, 0, False), (n, 1, False), (n, 1, True)):
        want = _stream(gpu, ops, ro, cols, tile_rows, swiglu, quant)
        got = _stream(gpu, ops, ro, cols, tile_rows | 0x1000, swiglu, quant)
        for x, y in zip(want, got) if quant else ((want, got),):
            assert torch.equal(x.view(torch.uint8), y.view(torch.uint8))


def test_stream_walks_a_table_of_more_than_256_experts(gpu):
    n, k, e = 64, 736, 300
    rows = np.zeros(e, dtype=np.int64)
    rows[[0, 7, 255, 256, 299]] = [5, 40, 129, 1, 33]
    ro = np.concatenate([[0], np.cumsum(rows)]).astype(np.int32)
    a, a_s = H.mx_operand(int(ro[-1]), k, seed=1)
    b, b_s = H.mx_operand(e * n, k, seed=2, std=0.05)
    b, b_s = b.reshape(e, n, k // 2), b_s.reshape(e, n, k // 32)
    ops = [H.to_dev(t, gpu) for t in (a, a_s, b, b_s)]
    for tile_rows in (32, 128):
        c = H.bits(_stream(gpu, ops, torch.from_numpy(ro).to(gpu), n, tile_rows, 0, False))
        for x in np.nonzero(rows)[0]:
            H.assert_mx_close(c[ro[x]:ro[x + 1]], a[ro[x]:ro[x + 1]], a_s[ro[x]:ro[x + 1]], b[x], b_s[x])


@pytest.mark.parametrize("m,n,k", [(1, 5, 512), (33, 130, 544), (65, 200, 1248), (128, 300, 2880), (200, 128, 1536)])
@pytest.mark.parametrize("tile_rows", [32, 64, 128])
def test_stream_split_k(gpu, m, n, k, tile_rows):
    """K in slices of one to three pairs of stages, the tail with the last one; unit scales make the sums exact."""
    rng = np.random.default_rng(m + k)
    a = rng.integers(0, 256, size=(m, k // 2), dtype=np.uint8)
    b = rng.integers(0, 256, size=(n, k // 2), dtype=np.uint8)
    a_s, b_s = (rng.integers(118, 132, size=(r, k // 32), dtype=np.uint8) for r in (m, n))
    one_a, one_b = np.full_like(a_s, 127), np.full_like(b_s, 127)
    exact = orc.f64_to_bf16_bits(orc.gemm_mxfp4_fp64(a, one_a, b, one_b))
    for slice_pairs in range(1, min(3, k // 512) + 1):
        slices = -(-(k // 512) // slice_pairs)
        for sa, sb in ((a_s, b_s), (one_a, one_b)):
            ws = torch.full((slices * m * n,), float("nan"), dtype=torch.float32, device=gpu)
            out = torch.full((m, n), float("nan"), dtype=torch.bfloat16, device=gpu)
            da, dsa, db, dsb = (H.to_dev(t, gpu) for t in (a, sa, b, sb))
            _lib.check(_lib.load().ave_fp4_debug_gemm_mxfp4_stream_splitk(
                da.data_ptr(), dsa.data_ptr(), db.data_ptr(), dsb.data_ptr(), out.data_ptr(), m, n, k, ws.data_ptr(), ws.numel() * 4,
                tile_rows, slice_pairs, torch.cuda.current_stream(gpu).cuda_stream))
            torch.cuda.synchronize(gpu)
            if sa is one_a:
                assert np.array_equal(H.bits(out), exact)
            else:
                H.assert_mx_close(H.bits(out), a, sa, b, sb)


@pytest.mark.parametrize("m,n,k", [(1, 512, 8192), (20, 1536, 4992), (48, 512, 7168), (100, 256, 3776), (200, 128, 2880)])
def test_swiglu_forms_on_few_weight_rows(gpu, m, n, k):
    """Shapes whose K is cut over idle compute units: the fused quantiser gives the quantised bf16 result, within tolerance."""
    a, a_s = H.mx_operand(m, k, seed=m)
    b, b_s = H.mx_operand(2 * n, k, seed=n, std=0.05)
    ops = [H.to_dev(t, gpu) for t in (a, a_s, b, b_s)]
    with torch.cuda.device(gpu):
        split = [_lib.load().ave_fp4_gemm_mxfp4_swiglu_workspace_bytes(m, n, k, quant) for quant in (0, 1)]
    c = gemm_mxfp4_swiglu_transposed_b(*ops)
    ok, rep = orc.check_swiglu_bf16(H.bits(c), a, a_s, b, b_s)
    assert ok, rep
    q, qs = gemm_mxfp4_swiglu_quant_transposed_b(*ops)
    want_q, want_s = quantize_mxfp4(c)
    if split[0] == split[1]:
        assert torch.equal(q, want_q) and torch.equal(qs, want_s)
    codes, scales = q.cpu().numpy(), qs.cpu().numpy()
    assert np.mean(codes != want_q.cpu().numpy()) < 1e-3 and np.mean(scales != want_s.cpu().numpy()) < 1e-3
    padded = gemm_mxfp4_swiglu_quant_transposed_b(*ops, n_pad=n + 64)
    assert torch.equal(padded[0][:, :n // 2], q) and torch.equal(padded[1][:, :n // 32], qs)
    assert not padded[0][:, n // 2:].any() and not padded[1][:, n // 32:].any()


@pytest.mark.parametrize("m,n,k", [(1, 512, 8192), (3, 1024, 2816), (4, 1408, 5376), (8, 1024, 7680), (18, 1536, 3584), (25, 3936, 6912),
                                   (32, 64, 2080), (16, 1024, 1024), (65, 512, 4096), (130, 256, 7200)])
def test_swiglu_quant_is_the_quantised_swiglu_result(gpu, m, n, k):
    """Up to 32 rows and above 64 the fused quantiser's codes and scales are those of the two calls, bit for bit, whatever the forms do
    about compute units that few weight rows leave idle; with padded rows as well."""
    a, a_s = H.mx_operand(m, k, seed=m + n)
    b, b_s = H.mx_operand(2 * n, k, seed=n + k, std=0.05)
    ops = [H.to_dev(t, gpu) for t in (a, a_s, b, b_s)]
    want_q, want_s = quantize_mxfp4(gemm_mxfp4_swiglu_transposed_b(*ops))
    q, qs = gemm_mxfp4_swiglu_quant_transposed_b(*ops)
    assert torch.equal(q, want_q) and torch.equal(qs, want_s)
    q, qs = gemm_mxfp4_swiglu_quant_transposed_b(*ops, n_pad=n + 96)
    assert torch.equal(q[:, :n // 2], want_q) and torch.equal(qs[:, :n // 32], want_s)
    assert not q[:, n // 2:].any() and not qs[:, n // 32:].any()


@pytest.mark.parametrize("off", [1, 2, 4])
def test_swiglu_of_k_slices_into_a_result_at_any_element(gpu, off):
    """A result that starts 2, 4 or 8 bytes behind a 16-byte boundary (a view into a larger tensor): the same bits, and nothing beside it."""
    m, n, k = 100, 256, 3776
    ops = [H.to_dev(t, gpu) for t in (*H.mx_operand(m, k, seed=m), *H.mx_operand(2 * n, k, seed=n, std=0.05))]
    with torch.cuda.device(gpu):
        assert _lib.load().ave_fp4_gemm_mxfp4_swiglu_workspace_bytes(m, n, k, 0) > 0
    want = gemm_mxfp4_swiglu_transposed_b(*ops)
    buffer = torch.full((m * n + 16,), 7.0, dtype=torch.bfloat16, device=gpu)
    out = buffer[off:off + m * n].view(m, n)
    assert gemm_mxfp4_swiglu_transposed_b(*ops, out) is out and out.data_ptr() % 16 == 2 * off
    assert torch.equal(out.view(torch.int16), want.view(torch.int16))
    assert (buffer[:off] == 7).all() and (buffer[off + m * n:] == 7).all()


def test_swiglu_of_k_slices_is_cut_alike_whatever_the_result_address(gpu):
    """Scales over 2^24, so that the order of the sums shows in the bits: a result at an odd element is still made of the same K slices."""
    m, n, k = 100, 256, 3776
    rng = np.random.default_rng(5)
    ops = [torch.from_numpy(rng.integers(lo, hi, size=s, dtype=np.uint8)).to(gpu)
           for lo, hi, s in ((0, 256, (m, k // 2)), (108, 132, (m, k // 32)), (0, 256, (2 * n, k // 2)), (100, 124, (2 * n, k // 32)))]
    with torch.cuda.device(gpu):
        assert _lib.load().ave_fp4_gemm_mxfp4_swiglu_workspace_bytes(m, n, k, 0) > 0
    want = gemm_mxfp4_swiglu_transposed_b(*ops)
    out = torch.empty(m * n + 1, dtype=torch.bfloat16, device=gpu)[1:].view(m, n)
    gemm_mxfp4_swiglu_transposed_b(*ops, out)
    assert torch.equal(out.view(torch.int16), want.view(torch.int16))


# 260 tiles of 32 rows on 256 compute units (one round of 64-row tiles), 520 (one round of 128), few enough to stay; an average above 18 rows;
# one expert a little taller than a tile; rows loaded by lines; more experts than a table in registers
@pytest.mark.parametrize("rows,n,k", [([0, 128, 0, 0, 0, 0, 0, 0], 8320, 544), ([0, 0, 0, 0, 0, 128, 0, 0], 16640, 512),
                                      ([128, 0, 0, 0, 0, 0, 0, 0], 512, 736), ([9, 47, 24, 16, 12, 8, 7, 5], 4096, 1024),
                                      ([3, 300, 0, 1, 4, 0, 33, 11], 8320, 544), ([33] + [1] * 70, 512, 800),
                                      ([0, 0, 130, 0, 5, 0, 0, 0], 16640, 1312), ([200] + [1] * 299, 4224, 544)])
def test_uneven_tables_give_the_bits_of_every_tile_height(gpu, rows, n, k):
    """The height of the tiles follows the experts' table; an output's sum does not."""
    e, m = len(rows), sum(rows)
    ro = torch.from_numpy(np.concatenate([[0], np.cumsum(rows)]).astype(np.int32)).to(gpu)
    g = torch.Generator(device=gpu).manual_seed(m + n + k)
    a, b = (torch.randint(0, 256, s, dtype=torch.uint8, device=gpu, generator=g) for s in ((m, k // 2), (e, n, k // 2)))
    a_s, b_s = (torch.randint(110, 132, s, dtype=torch.uint8, device=gpu, generator=g) for s in ((m, k // 32), (e, n, k // 32)))
    ops = (a, a_s, b, b_s)
    got = [(grouped_gemm_mxfp4_transposed_b(*ops, ro),), (grouped_gemm_mxfp4_swiglu_transposed_b(*ops, ro),),
           grouped_gemm_mxfp4_swiglu_quant_transposed_b(*ops, ro)]
    for tile_rows in (32, 64, 128):
        want = [(_stream(gpu, ops, ro, n, tile_rows, 0, False),), (_stream(gpu, ops, ro, n // 2, tile_rows, 1, False),),
                _stream(gpu, ops, ro, n // 2, tile_rows, 1, True)]
        for form, (xs, ys) in enumerate(zip(got, want)):
            for x, y in zip(xs, ys):
                assert torch.equal(x.view(torch.uint8), y.view(torch.uint8)), (tile_rows, form)


# one tile and many, ragged rows and columns; two stages, an odd number of them and K % 512 of 1, 7, 8, 9 and 15 blocks
@pytest.mark.parametrize("m,n,k", [(1, 32, 512), (33, 96, 544), (64, 160, 736), (65, 32, 768), (127, 224, 800), (128, 64, 992), (129, 352, 1248),
                                   (200, 64, 2880), (300, 8224, 512)])
@pytest.mark.parametrize("tile_rows", [32, 64, 128])
def test_stream_one_matrix_with_k_in_one_piece(gpu, m, n, k, tile_rows):
    """The forms that shape-based dispatch takes without slices: plain, SwiGLU, SwiGLU + quantiser."""
    a, a_s = H.mx_operand(m, k, seed=m + k)
    b, b_s = H.mx_operand(2 * n, k, seed=n + k, std=0.05)
    ops = [H.to_dev(t, gpu) for t in (a, a_s, b, b_s)]

    def run(cols, swiglu, quant):
        c = torch.full((m, cols), float("nan"), dtype=torch.bfloat16, device=gpu)
        q = torch.full((m, cols // 2), 0xEE, dtype=torch.uint8, device=gpu)
        qs = torch.full((m, cols // 32), 0xEE, dtype=torch.uint8, device=gpu)
        _lib.check(_lib.load().ave_fp4_debug_gemm_mxfp4_stream(
            *(t.data_ptr() for t in ops), None if quant else c.data_ptr(), q.data_ptr() if quant else None,
            qs.data_ptr() if quant else None, m, cols, k, swiglu, tile_rows, torch.cuda.current_stream(gpu).cuda_stream))
        torch.cuda.synchronize(gpu)
        return (q, qs) if quant else c

    H.assert_mx_close(H.bits(run(2 * n, 0, False)), a, a_s, b, b_s)
    H.assert_mx_close(H.bits(run(2 * n - 3, 0, False)), a, a_s, b[:-3], b_s[:-3])
    fused = run(n, 1, False)
    ok, rep = orc.check_swiglu_bf16(H.bits(fused), a, a_s, b, b_s)
    assert ok, rep
    want_q, want_s = quantize_mxfp4(fused)
    q, qs = run(n, 1, True)
    assert torch.equal(q, want_q) and torch.equal(qs, want_s)


@pytest.mark.parametrize("m,n,k", [(100, 256, 3776), (65, 512, 4096), (130, 256, 7200), (48, 512, 7168)])
def test_swiglu_forms_whose_k_is_cut(gpu, m, n, k):
    """Shapes that are planned in slices (asserted, for a device of 256 compute units): both fused forms against the oracle."""
    lib = _lib.load()
    if torch.cuda.get_device_properties(gpu).multi_processor_count != 256:
        pytest.skip("planned for 256 compute units")
    with torch.cuda.device(gpu):
        split = [lib.ave_fp4_gemm_mxfp4_swiglu_workspace_bytes(m, n, k, quant) for quant in (0, 1)]
    for bytes_ in split:
        assert bytes_ > 0 and bytes_ % (m * 2 * n * 4) == 0 and bytes_ // (m * 2 * n * 4) > 1
    a, a_s = H.mx_operand(m, k, seed=m)
    b, b_s = H.mx_operand(2 * n, k, seed=n, std=0.05)
    ops = [H.to_dev(t, gpu) for t in (a, a_s, b, b_s)]
    c = gemm_mxfp4_swiglu_transposed_b(*ops)
    ok, rep = orc.check_swiglu_bf16(H.bits(c), a, a_s, b, b_s)
    assert ok, rep
    q, qs = gemm_mxfp4_swiglu_quant_transposed_b(*ops)
    want_q, want_s = quantize_mxfp4(c)
    assert np.mean(q.cpu().numpy() != want_q.cpu().numpy()) < 1e-3 and np.mean(qs.cpu().numpy() != want_s.cpu().numpy()) < 1e-3
