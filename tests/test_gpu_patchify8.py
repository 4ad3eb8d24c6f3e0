"""patchify's 16-byte form (rows of whole aligned chunks) against its element form (any other row stride), the same bits."""
import pytest
import torch

import strix_halo_maxx_amd.ops as ops

pytestmark = pytest.mark.gpu


# chunks that straddle (ky, kx) rows, channels and the end of K (3 P^2 = 588, 192, 147, 3, 27); one patch; more images than the
# grid has rows; below the size where the form is taken
@pytest.mark.parametrize("B,S,P", [(3, 378, 14), (40, 256, 8), (80, 35, 7), (2000, 6, 1), (70000, 3, 3), (1, 35, 7)])
@pytest.mark.parametrize("mode", [0, 1])
def test_chunks_equal_elements(dev, B, S, P, mode):
    g = torch.Generator().manual_seed(S)
    img = torch.randint(0, 256, (B, S, S, 3), generator=g, dtype=torch.uint8).to(dev)
    K = 3 * P * P
    one = ops.patchify(img, P, mode=mode, ldo=(K + 7) // 8 * 8 + 3).cpu()  # odd rows: the element form
    for ldo in ((K + 7) // 8 * 8, (K + 7) // 8 * 8 + 24):
        print(f"patchify {B}x{S} P={P} mode={mode} ldo={ldo}", flush=True)
        y = ops.patchify(img, P, mode=mode, ldo=ldo).cpu()
        assert torch.equal(y[..., :K], one[..., :K]) and torch.count_nonzero(y[..., K:]) == 0
