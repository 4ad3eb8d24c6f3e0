"""The one-tile-per-CU GEMM (tile configs 17, 19, 27, and 5 for partials) against the 128 x 128 tile (config 7) on the same
inputs: the same k order and roundings, so the same bits, for every epilogue and at the edges of its tiles and steps, with
nothing written past a row's end or below the last row (128 guard rows: a whole tile)."""
import pytest
import torch

import strix_halo_maxx_amd.ops as ops

pytestmark = pytest.mark.gpu
BF = torch.bfloat16


# one row and one k-step; fewer k-steps than ring slots, a ragged last step (136 = 2.1); the last tile a row / 8 columns
# wide; whole tiles; the tower's fc1
@pytest.mark.parametrize("M,N,K", [(1, 16, 64), (129, 264, 136), (300, 200, 904), (256, 768, 1152), (729, 4304, 1152)])
@pytest.mark.parametrize("cfg", [17, 19, 27])
def test_mid_tiles_equal_the_small_one(dev, cfg, M, N, K):
    g = torch.Generator().manual_seed(M + N + K)
    x = torch.randn(M, K, generator=g).to(BF).to(dev)
    w = (torch.randn(N, K, generator=g) * 0.02).to(BF)
    b = (torch.randn(N, generator=g) * 0.02).to(BF)
    r = torch.randn(M, N, generator=g).to(BF).to(dev)
    r3 = torch.randn(3, N + 8, generator=g).to(BF).to(dev)[:, :N]
    for bias in (b, None):
        lin = ops.MxLin(w, bias)
        for kw in (dict(), dict(gelu=True), dict(act="erf"), dict(gelu=True, act_cols=100), dict(act="erf", act_cols=N),
                   dict(res=r), dict(gelu=True, res=r), dict(act="erf", act_cols=36, res=r3 if M % 3 == 0 else r),
                   dict(act="glu")):
            print(f"mid cfg={cfg} {M}x{N}x{K} bias={bias is not None} {[k for k in kw]}", flush=True)
            No = N // 2 if kw.get("act") == "glu" else N
            got = []
            for c in (7, cfg):
                lin.cfgs[M] = (c, 1)
                y = torch.full((M + 128, No + 8), 7.0, device=dev, dtype=BF)  # longer and more rows than the output
                lin(x, out=y[:M, :No], **kw)
                got.append(y.cpu())
            assert torch.equal(got[0], got[1]), kw
            assert torch.all(got[1][M:] == 7.0) and torch.all(got[1][:, No:] == 7.0), kw


@pytest.mark.parametrize("M,N,K", [(1, 12, 200), (129, 268, 904), (730, 2048, 1024)])
@pytest.mark.parametrize("cfg", [5, 19, 27])
def test_mid_partials_equal_the_small_ones(dev, cfg, M, N, K):
    """Raw split-K partials in rows longer than N: the same bits as config 7's, nothing written past or below the rows."""
    g = torch.Generator().manual_seed(M + N)
    x = torch.randn(M, K, generator=g).to(BF).to(dev)
    lin = ops.MxLin((torch.randn(N, K, generator=g) * 0.02).to(BF), None)
    x2 = ops._rows(x, lin.K)
    for sp in (1, 2, 4):
        if sp > lin.Kw // 64:
            continue
        print(f"mid partial cfg={cfg} {M}x{N}x{K} splits={sp}", flush=True)
        out = []
        for c in (7, cfg):
            P = torch.full((sp, M + 128, N + 4), 7.0, device=dev)
            assert ops._partial(lin, c, sp, x2, P[:, :M, :N], M) == 0
            out.append(P.cpu())
        assert torch.equal(out[0], out[1])
        assert torch.all(out[1][:, M:] == 7.0) and torch.all(out[1][:, :, N:] == 7.0)


def test_mid_tiles_take_what_the_config_took(dev):
    """Calls outside the kernel's alignment (N % 8, rows of C 8-byte aligned) still run."""
    g = torch.Generator().manual_seed(3)
    for M, N, K in ((300, 1220, 1000), (64, 64, 64), (130, 132, 192)):
        x = torch.randn(M, K, generator=g).to(BF).to(dev)
        lin = ops.MxLin((torch.randn(N, K, generator=g) * 0.02).to(BF), None)
        out = []
        for c in (7, 17, 19, 27):
            lin.cfgs[M] = (c, 1)
            y = torch.full((M, N + 4), 7.0, device=dev, dtype=BF)
            lin(x, out=y[:, :N])
            out.append(y.cpu())
        assert all(torch.equal(out[0], o) for o in out[1:])


# (config, M, N, K): config 0's tile (one workgroup per CU, deep K), the 128 x 192 tile (176 .. 256 of them)
@pytest.mark.parametrize("cfg,M,N,K", [(19, 130, 132, 2056), (19, 300, 1220, 2504), (27, 1700, 2308, 200), (27, 32700, 132, 72)])
def test_mid_tiles_unaligned_grids(dev, cfg, M, N, K):
    g = torch.Generator().manual_seed(M)
    x = torch.randn(M, K, generator=g).to(BF).to(dev)
    lin = ops.MxLin((torch.randn(N, K, generator=g) * 0.02).to(BF), torch.randn(N, generator=g) * 0.02)
    r = torch.randn(M, N, generator=g).to(BF).to(dev)
    for kw in (dict(), dict(gelu=True), dict(res=r)):
        out = []
        for c in (7, cfg):
            lin.cfgs[M] = (c, 1)
            y = torch.full((M + 128, N + 8), 7.0, device=dev, dtype=BF)
            lin(x, out=y[:M, :N], **kw)
            out.append(y)
        print(f"unaligned cfg={cfg} {M}x{N}x{K} {[k for k in kw]}", flush=True)
        assert torch.equal(out[0], out[1]) and torch.all(out[1][M:] == 7.0) and torch.all(out[1][:, N:] == 7.0)
