"""Column abs-max and top-k channel selection on the GPU against the oracle
(lrq_colmax / lrq_topk; the channel split of config 3).  Ties, k = 1 and k = hidden, and
both column abs-max kernels (16-byte rows and the 4-byte fallback) are covered."""

import numpy as np
import pytest
import torch

import oracle as O
from parity import bits16

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("hidden,k,levels", [
    (4096, 41, 0),       # config 3: distinct values
    (4096, 41, 6),       # heavy ties: six distinct values
    (5000, 1, 3),
    (5000, 5000, 0),     # k = hidden
    (1000, 999, 2),
    (37000, 1024, 50),   # near the LDS limit, many ties
])
def test_topk_matches_oracle(pkg, dev, hidden, k, levels):
    print(f"[topk] hidden={hidden} k={k} levels={levels}", flush=True)
    g = torch.Generator().manual_seed(hidden + k)
    if levels:
        cm = torch.randint(0, levels, (hidden,), generator=g).to(torch.float32) * 0.25
    else:
        cm = torch.rand(hidden, generator=g, dtype=torch.float32) * 3.0
    idx = pkg.topk_channels(cm.to(dev), k)
    torch.cuda.synchronize()
    ref = O.topk_channels(cm.numpy(), k)
    assert np.array_equal(idx.cpu().numpy(), ref)


@pytest.mark.parametrize("rows,hidden", [(129, 2048), (37, 1030), (1000, 4096)])
def test_colmax_matches_oracle(pkg, dev, rows, hidden):
    print(f"[colmax] rows={rows} hidden={hidden}", flush=True)
    x = pkg.inputs.activation(rows, hidden, n_outlier=3, outlier_scale=30.0, seed=rows)
    cm = pkg.column_absmax(x.to(dev))
    torch.cuda.synchronize()
    ref = O.colmax_abs(bits16(x))
    assert np.array_equal(cm.cpu().numpy().view(np.uint32), ref.view(np.uint32))


@pytest.mark.parametrize("k,hidden,rows", [(1, 64, 1), (41, 4096, 300), (257, 512, 16400), (700, 16000, 64),
                                           (50, 40000, 3), (60, 50000, 70)])
def test_outlier_index_is_sanitized(pkg, dev, k, hidden, rows):
    """The device-held channel list: -1 for entries out of range and for repeats of an earlier entry,
    their side columns zeroed and no other (one and several workgroups, the LDS tables up to and past
    their limit)."""
    g = torch.Generator().manual_seed(k)
    idx = torch.randint(-3, hidden + 3, (k,), generator=g, dtype=torch.int32)
    idx[k // 2:] = idx[: k - k // 2].clone()  # repeats
    seen, want = set(), []
    for c in idx.tolist():
        want.append(c if 0 <= c < hidden and c not in seen else -1)
        seen.add(c)
    side = torch.ones((rows, k), dtype=torch.float16, device=dev)
    out = pkg.api._sanitize_index(idx.to(dev), hidden, side)
    assert out.tolist() == want
    drop = torch.tensor(want) < 0
    assert not side[:, drop.to(dev)].any()
    if hidden <= 40000:
        assert (side[:, ~drop.to(dev)] == 1).all()
