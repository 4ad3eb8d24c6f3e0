"""The activation on columns >= act_from (mx_gemm_bf16_act_from, mx_gemm_reduce_act_from): the same bits as two products over
the row slices of W, the first without and the second with the activation, in every kind of tile."""
import pytest
import torch

import strix_halo_maxx_amd.ops as ops
from strix_halo_maxx_amd import _lib

pytestmark = pytest.mark.gpu
BF = torch.bfloat16


# act_from: within a tile, on a tile's edge, in the last columns; whole and ragged tiles
@pytest.mark.parametrize("M,N,K,f", [(32, 448, 1024, 192), (300, 520, 904, 516), (1, 64, 256, 4), (129, 512, 512, 256)])
def test_act_from_equals_two_products(dev, M, N, K, f):
    g = torch.Generator().manual_seed(M + N)
    x = torch.randn(M, K, generator=g).to(BF).to(dev)
    w = (torch.randn(N, K, generator=g) * 0.02).to(BF)
    b = (torch.randn(N, generator=g) * 0.02).to(BF)
    whole, lo, hi = ops.MxLin(w, b), ops.MxLin(w[:f], b[:f]), ops.MxLin(w[f:], b[f:])
    for cfg in ((0, 1), (0, 2), (7, 1), (8, 1), (15, 1), (17, 1), (19, 1), (22, 1), (23, 1), (25, 1), (22, -2), (19, -2)):
        if abs(cfg[1]) > lo.Kw // 64:
            continue
        for act in ("tanh", "erf"):
            print(f"act_from={f} {M}x{N}x{K} cfg={cfg} {act}", flush=True)
            for l in (whole, lo, hi):
                l.cfgs[M] = cfg
            y = whole(x, act=act, act_from=f).cpu()
            assert torch.equal(y[:, :f], lo(x).cpu()) and torch.equal(y[:, f:], hi(x, act=act).cpu()), (cfg, act)


def test_act_from_refusals(dev):
    x = torch.zeros(8, 64, dtype=BF, device=dev)
    lin = ops.MxLin(torch.zeros(64, 64, dtype=BF), None)
    with pytest.raises(ValueError):
        lin(x, act="glu", act_from=8)
    with pytest.raises(ValueError):
        lin(x, act="tanh", act_from=8, act_cols=4)
    with pytest.raises(_lib.MxError):
        lin(x, act="tanh", act_from=-4)
    for cfg in ((7, 1), (22, -1)):
        lin.cfgs[8] = cfg
        with pytest.raises(_lib.MxError):
            lin(x, act="tanh", act_from=5)
