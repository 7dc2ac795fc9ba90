"""The fused layout's packing (ft_hip_pack_experts_fused) byte for byte against
its definition, from both row layouts, at sizes that do not fill a workgroup's
64 rows or 16 blocks, with experts that lie apart in the source."""
import numpy as np
import pytest
import torch

import ft_hip

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def rows(d, q, layout):
    """[n][nb] f16 scales and [n][nb][16] bytes as q4_0 or q4r rows."""
    n, nb = d.shape
    db = d.view(np.uint8).reshape(n, nb, 2)
    if layout == ft_hip.LAYOUT_Q4_0:
        return np.concatenate([db, q], axis=2).reshape(n, nb * 18)
    so = (nb * 2 + 15) // 16 * 16
    out = np.zeros((n, so + nb * 16), np.uint8)
    out[:, :nb * 2] = db.reshape(n, -1)
    out[:, so:] = q.reshape(n, -1)
    return out


def tiles(d, q, r):
    """Tiles of r rows: [nb][r] scales, then [nb][r][16] bytes."""
    n, nb = d.shape
    parts = []
    for t in range(0, n, r):
        parts.append(np.ascontiguousarray(d[t:t + r].T).view(np.uint8).ravel())
        parts.append(np.ascontiguousarray(q[t:t + r].transpose(1, 0, 2)).ravel())
    return np.concatenate(parts)


@pytest.mark.parametrize("layout", [ft_hip.LAYOUT_Q4_0, ft_hip.LAYOUT_Q4R])
@pytest.mark.parametrize("hidden,inter,n,gap", [(32, 32, 1, 0), (96, 544, 3, 16), (512, 96, 2, 32), (2816, 704, 2, 0)])
def test_pack_is_the_fused_layout(gemv, hidden, inter, n, gap, layout):
    rng = np.random.default_rng(hidden + inter)
    src, want = [], []
    for _ in range(n):
        gd, gq = rng.standard_normal((2 * inter, hidden // 32)).astype(np.float16), rng.integers(
            0, 256, (2 * inter, hidden // 32, 16), dtype=np.uint8)
        dd, dq = rng.standard_normal((hidden, inter // 32)).astype(np.float16), rng.integers(
            0, 256, (hidden, inter // 32, 16), dtype=np.uint8)
        src.append(np.concatenate([rows(gd, gq, layout).ravel(), rows(dd, dq, layout).ravel(), np.zeros(gap, np.uint8)]))
        order = np.concatenate([np.r_[j:j + 32, inter + j:inter + j + 32] for j in range(0, inter, 32)])
        want.append(np.concatenate([tiles(gd[order], gq[order], 64), tiles(dd, dq, 16)]))
    eb = len(src[0])
    pad = -eb % 16 if layout == ft_hip.LAYOUT_Q4R else 0  # q4r experts lie 16-byte aligned
    flat = torch.from_numpy(np.concatenate([np.pad(s, (0, pad)) for s in src])).to(DEV)
    dst = torch.zeros(n * gemv.fused_expert_bytes(hidden, inter), dtype=torch.uint8, device=DEV)
    gemv.pack_experts_fused(flat, layout, eb + pad, dst, n, hidden, inter)
    torch.cuda.synchronize()
    assert np.array_equal(dst.cpu().numpy(), np.concatenate(want))
