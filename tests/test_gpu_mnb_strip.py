"""The strip kernel of the MatMulNBits projections (from 3 rows on) at the edges of its tiles, against the fp64 oracle: one
and two rows around each count of 16-row tiles, a column count that no tile count divides, K of one half, an odd number
of halves and more groups than waves, every weight format; rows that keep their bits whatever M is; operands whose
alignment sends the call to the general kernels."""
import os
import sys

import numpy as np
import pytest

import hybrid_attention as ha

sys.path.insert(0, os.path.join(os.path.dirname(os.path.abspath(__file__)), "..", "oracle"))
import mnb_oracle as mo  # noqa: E402

pytestmark = pytest.mark.gpu
# max |err| / max |ref|: weights rounded to f16 once (2^-11 each, averaging over K) and an f16 output (2^-11)
TOL = 2e-3


def _weights(N, K, bits, group, asym, seed):
    rng = np.random.default_rng(seed)
    words = rng.integers(0, 2 ** 32, (N, K // 32, mo.words_per_block(bits)), dtype=np.uint64).astype(np.uint32)
    sc = (0.005 + 0.01 * rng.random((N, K // group))).astype(np.float16)
    bi = ((rng.random((N, K // group)) - 0.5) * 0.1).astype(np.float16) if asym else None
    return words, sc, bi


def _dev(x):
    import torch
    return torch.from_numpy(x.view(np.int32) if x.dtype == np.uint32 else x).to("cuda:0")


@pytest.mark.parametrize("N,K,bits,group,asym", [
    (16, 64, 4, 32, False), (1040, 192, 4, 32, True), (2064, 2112, 4, 64, False), (4112, 1152, 4, 64, True),
    (12304, 128, 4, 32, False), (1040, 192, 3, 32, False), (528, 2176, 3, 64, True), (1040, 1088, 2, 32, True),
    (16, 128, 2, 64, False)])
def test_tile_edges(N, K, bits, group, asym):
    import torch
    words, sc, bi = _weights(N, K, bits, group, asym, N + K + bits)
    W = mo.dequant(words, sc, N, K, bits, group, asym, bi)
    q, s, b = _dev(words), _dev(sc), _dev(bi) if asym else None
    w = ha.MnbWeight(N, K, q, s, b, bits=bits, group=group, asym=asym)
    a = ((np.random.default_rng(1).random((385, K)) - 0.5) * 2).astype(np.float16)
    ad, ref = _dev(a), mo.matmul(a, W)
    full = None
    for M in (256, 3, 15, 16, 17, 32, 33, 49, 65, 81, 97, 113, 129, 193, 257, 384, 385):
        y = torch.full((M + 1, N), 7.0, dtype=torch.float16, device="cuda:0")
        w.forward(M, ad, y)
        torch.cuda.synchronize()
        g = y.cpu().numpy()
        assert mo.rel_err(g[:M].astype(np.float64), ref[:M]) < TOL, M
        assert (g[M] == 7.0).all(), "row past M written (M = %d)" % M
        if full is None:
            full = g
        elif M < 256 and K % 64 == 0 and (group == 32 or K % 128 == 0):
            assert np.array_equal(g[:M].view(np.uint16), full[:M].view(np.uint16)), "bits of a row depend on M = %d" % M
    w.close()


@pytest.mark.parametrize("N,K,group,asym", [
    (4160, 192, 32, False), (4112, 448, 32, True), (3008, 1024, 64, False), (8256, 128, 64, True), (5120, 64, 32, False),
    (3008, 384, 64, True), (2208, 384, 32, True), (4256, 384, 64, False), (4256, 2048, 32, True), (2208, 2048, 64, True)])
def test_many_rows(N, K, group, asym):
    # more rows than the strip kernel is the faster for: the tile kernel, at edges of its tiles in both directions (rows just
    # over and under a multiple of 128 and 256; last column tiles of 32, 64, 160, 192 and 256 columns, so that some waves have
    # none, while the up to 64 columns past a multiple of 256 of 4112, 4160 and 8256 go to the strip kernel) and of its
    # six-tile K loop; rows keep their bits whatever M is
    import torch
    words, sc, bi = _weights(N, K, 4, group, asym, N + K)
    W = mo.dequant(words, sc, N, K, 4, group, asym, bi)
    q, s, b = _dev(words), _dev(sc), _dev(bi) if asym else None
    w = ha.MnbWeight(N, K, q, s, b, bits=4, group=group, asym=asym)
    a = ((np.random.default_rng(3).random((2050, K)) - 0.5) * 2).astype(np.float16)
    ad, ref, full = _dev(a), mo.matmul(a, W), None
    for M in (2050, 1025, 1151, 1409):
        y = torch.full((M + 1, N), 7.0, dtype=torch.float16, device="cuda:0")
        w.forward(M, ad, y)
        torch.cuda.synchronize()
        g = y.cpu().numpy()
        assert mo.rel_err(g[:M].astype(np.float64), ref[:M]) < TOL, M
        assert (g[M] == 7.0).all(), "row past M written (M = %d)" % M
        full = g if full is None else full
        assert np.array_equal(g[:M].view(np.uint16), full[:M].view(np.uint16)), "bits of a row depend on M = %d" % M
    w.close()


@pytest.mark.parametrize("N,K,bits,group,asym,Ms", [
    (33040, 128, 4, 32, True, [64, 129, 200]),   # beyond 12800 columns: strip, then tiles
    (33040, 128, 4, 64, False, [129, 256]),
    (151952, 64, 3, 32, False, [3, 64, 200, 384]),  # strip, then the GEMM
    (151952, 64, 2, 32, True, [300, 385]),
    (49168, 1088, 4, 32, False, [1, 2]),         # one row: four columns a wave; two rows: strip
    (8208, 1088, 3, 32, True, [1, 2]), (8208, 1152, 2, 64, False, [1, 2]),
    (8176, 1088, 4, 32, False, [1, 2]), (4112, 2080, 4, 32, True, [1, 2]), (8208, 2080, 3, 32, False, [1, 2])])
def test_lines_of_the_rule(N, K, bits, group, asym, Ms):
    # either side of the lines at which a call goes to another kernel (mnb_plan.h)
    import torch
    words, sc, bi = _weights(N, K, bits, group, asym, N + K + bits)
    W = mo.dequant(words, sc, N, K, bits, group, asym, bi)
    q, s, b = _dev(words), _dev(sc), _dev(bi) if asym else None
    w = ha.MnbWeight(N, K, q, s, b, bits=bits, group=group, asym=asym)
    a = ((np.random.default_rng(4).random((max(Ms), K)) - 0.5) * 2).astype(np.float16)
    ad, ref = _dev(a), mo.matmul(a, W)
    for M in Ms:
        y = torch.full((M + 1, N), 7.0, dtype=torch.float16, device="cuda:0")
        w.forward(M, ad, y)
        torch.cuda.synchronize()
        g = y.cpu().numpy()
        assert mo.rel_err(g[:M].astype(np.float64), ref[:M]) < TOL, M
        assert (g[M] == 7.0).all(), "row past M written (M = %d)" % M
    w.close()


@pytest.mark.parametrize("bits,off_q,off_s,group,asym,M", [
    (4, 4, 0, 32, False, 40), (4, 0, 2, 32, False, 40), (3, 4, 2, 32, False, 40), (4, 4, 2, 32, True, 1), (4, 4, 0, 32, True, 200),
    (4, 4, 2, 64, False, 200), (4, 0, 2, 64, True, 500), (2, 4, 2, 64, True, 200)])
def test_unaligned_operands(bits, off_q, off_s, group, asym, M):
    import torch
    N, K = 272, 256
    words, sc, bi = _weights(N, K, bits, group, asym, bits + off_q)
    qb = torch.zeros(words.size + 4, dtype=torch.int32, device="cuda:0")
    sb = torch.zeros(sc.size + 4, dtype=torch.float16, device="cuda:0")
    qb[off_q // 4:off_q // 4 + words.size] = _dev(words).reshape(-1)
    sb[off_s // 2:off_s // 2 + sc.size] = _dev(sc).reshape(-1)
    bb = torch.zeros(sc.size + 4, dtype=torch.float16, device="cuda:0")
    if asym:
        bb[off_s // 2:off_s // 2 + sc.size] = _dev(bi).reshape(-1)
    w = ha.MnbWeight(N, K, qb.data_ptr() + off_q, sb.data_ptr() + off_s, bb.data_ptr() + off_s if asym else None, bits=bits,
                     group=group, asym=asym)
    a = ((np.random.default_rng(2).random((M, K)) - 0.5) * 2).astype(np.float16)
    y = torch.empty(M, N, dtype=torch.float16, device="cuda:0")
    w.forward(M, _dev(a), y)
    torch.cuda.synchronize()
    assert mo.rel_err(y.double().cpu().numpy(), mo.matmul(a, mo.dequant(words, sc, N, K, bits, group, asym, bi))) < TOL
    w.close()
