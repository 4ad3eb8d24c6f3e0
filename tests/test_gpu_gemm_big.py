"""The persistent 256-row GEMM (tile configs 15 and 25) against the 128 x 128 tile (config 7) on the same inputs: the same
k order and roundings, so the same bits, for every epilogue and at the edges of its tiles and steps, with nothing written
past a row's end or below the last row (256 guard rows: a whole tile)."""
import pytest
import torch

import strix_halo_maxx_amd.ops as ops

pytestmark = pytest.mark.gpu
BF = torch.bfloat16


# one row; the last tile a row / 8 columns wide; an odd number of k-steps (904 = 14.1, 320 = 5); the fewest steps (256);
# whole tiles; more than one tile per CU with an odd last one (300 tiles of 256 columns, 600 of 192)
@pytest.mark.parametrize("M,N,K", [(1, 16, 256), (257, 272, 904), (300, 200, 320), (512, 768, 1152), (76699, 208, 256)])
@pytest.mark.parametrize("cfg", [15, 25])
def test_big_tiles_equal_the_small_one(dev, cfg, M, N, K):
    g = torch.Generator().manual_seed(M + N + K)
    x = torch.randn(M, K, generator=g).to(BF).to(dev)
    w = (torch.randn(N, K, generator=g) * 0.02).to(BF)
    b = (torch.randn(N, generator=g) * 0.02).to(BF)
    r = torch.randn(M, N, generator=g).to(BF).to(dev)
    r7 = torch.randn(7, N + 8, generator=g).to(BF).to(dev)[:, :N]
    for bias in (b, None):
        lin = ops.MxLin(w, bias)
        for kw in (dict(), dict(gelu=True), dict(act="erf"), dict(gelu=True, act_cols=100), dict(act="erf", act_cols=N),
                   dict(res=r), dict(gelu=True, res=r), dict(act="erf", act_cols=36, res=r7) if M % 7 == 0 else dict(res=r),
                   dict(act="glu")):
            print(f"big cfg={cfg} {M}x{N}x{K} bias={bias is not None} {[k for k in kw]}", flush=True)
            No = N // 2 if kw.get("act") == "glu" else N
            got = []
            for c in (7, cfg):
                lin.cfgs[M] = (c, 1)
                y = torch.full((M + 256, No + 8), 7.0, device=dev, dtype=BF)  # longer and more rows than the output
                lin(x, out=y[:M, :No], **kw)
                got.append(y.cpu())
            assert torch.equal(got[0], got[1]), kw
            assert torch.all(got[1][M:] == 7.0) and torch.all(got[1][:, No:] == 7.0), kw


def test_big_tiles_take_what_the_config_took(dev):
    """Calls outside the persistent kernel's alignment or depth (N % 8, rows of C 8-byte aligned, one k-step) still run."""
    g = torch.Generator().manual_seed(3)
    for M, N, K in ((300, 1220, 1000), (64, 64, 64), (130, 132, 192)):
        x = torch.randn(M, K, generator=g).to(BF).to(dev)
        lin = ops.MxLin((torch.randn(N, K, generator=g) * 0.02).to(BF), None)
        out = []
        for c in (7, 15, 25):
            lin.cfgs[M] = (c, 1)
            y = torch.full((M, N + 4), 7.0, device=dev, dtype=BF)
            lin(x, out=y[:, :N])
            out.append(y.cpu())
        assert torch.equal(out[0], out[1]) and torch.equal(out[0], out[2])


@pytest.mark.parametrize("M,N,cfg", [(40900, 132, 15), (49100, 132, 25), (8200, 1036, 15), (8200, 1036, 25)])
def test_big_tiles_unaligned_large_grids(dev, M, N, cfg):
    """The same calls where the 8-wave tile of the config's size fills the chip (from 9 M outputs of whole tiles)."""
    g = torch.Generator().manual_seed(M)
    x = torch.randn(M, 136, generator=g).to(BF).to(dev)
    lin = ops.MxLin((torch.randn(N, 136, generator=g) * 0.02).to(BF), torch.randn(N, generator=g) * 0.02)
    r = torch.randn(M, N, generator=g).to(BF).to(dev)
    for kw in (dict(), dict(gelu=True), dict(res=r)):
        out = []
        for c in (7, cfg):
            lin.cfgs[M] = (c, 1)
            y = torch.full((M + 256, N + 8), 7.0, device=dev, dtype=BF)
            lin(x, out=y[:M, :N], **kw)
            out.append(y)
        print(f"unaligned cfg={cfg} {M}x{N} {[k for k in kw]}", flush=True)
        assert torch.equal(out[0], out[1]) and torch.all(out[1][M:] == 7.0) and torch.all(out[1][:, N:] == 7.0)


# 313 row tiles (the last of 129 rows) x 5 column tiles of 256 or 7 of 192 (the last of 144 / 16 columns): 6 to 9 tiles per
# workgroup of 256 CUs, so the bias rows' ring of 4 comes round and every tile's loads run into the next one's; 5 steps of
# 64 (the odd step is followed by one of zeros) and 6
@pytest.mark.parametrize("K", [320, 384])
@pytest.mark.parametrize("cfg", [15, 25])
def test_big_tiles_many_per_workgroup(dev, cfg, K):
    M, N = 80001, 1168
    g = torch.Generator(device=dev).manual_seed(K)
    x = torch.randn(M, K, generator=g, device=dev).to(BF)
    lin = ops.MxLin((torch.randn(N, K, generator=g, device=dev) * 0.02).to(BF), torch.randn(N, generator=g, device=dev))
    r = torch.randn(M, N, generator=g, device=dev).to(BF)
    for kw in (dict(), dict(gelu=True), dict(res=r), dict(act="glu")):
        No = N // 2 if kw.get("act") == "glu" else N
        out = []
        for c in (7, cfg):
            lin.cfgs[M] = (c, 1)
            y = torch.full((M + 256, No + 8), 7.0, device=dev, dtype=BF)
            lin(x, out=y[:M, :No], **kw)
            out.append(y)
        print(f"big cfg={cfg} {M}x{N}x{K} {[k for k in kw]}", flush=True)
        assert torch.equal(out[0], out[1]) and torch.all(out[1][M:] == 7.0) and torch.all(out[1][:, No:] == 7.0), kw
