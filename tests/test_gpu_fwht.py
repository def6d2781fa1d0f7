"""The Walsh-Hadamard rotation at every block size, ragged block counts and alignments, against the fp64 oracle, and bit for
bit between the two kernels (the same butterflies in the same order): an aligned array and a copy two bytes off."""
import os
import sys

import numpy as np
import pytest

import hybrid_attention as ha

sys.path.insert(0, os.path.join(os.path.dirname(os.path.abspath(__file__)), "..", "oracle"))
import mnb_oracle as mo  # noqa: E402

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [2, 32, 64, 128, 256, 512, 1024, 2048, 4096, 8192])
@pytest.mark.parametrize("blocks", [1, 3, 35])
def test_block_sizes(n, blocks):
    import torch
    x = np.random.default_rng(n + blocks).normal(size=(blocks, n)).astype(np.float16)
    xd = torch.from_numpy(x).to("cuda:0").reshape(-1)
    off = torch.zeros(x.size + 3, dtype=torch.float16, device="cuda:0")
    off[1:1 + x.size] = xd
    ha.fwht(xd, x.size, n)
    ha.fwht(off.data_ptr() + 2, x.size, n)
    torch.cuda.synchronize()
    ref = mo.fwht(x.astype(np.float64), n)
    # f32 butterflies, one rounding to f16 (2^-11 of each value)
    assert mo.rel_err(xd.double().cpu().numpy().reshape(blocks, n), ref) < 6e-4
    assert torch.equal(off[1:1 + x.size], xd)
    assert float(off[0]) == 0 and float(off[-2]) == 0 and float(off[-1]) == 0
