"""GPU parity of the product-codebook fits (sva_amd.codebooks) with the
oracle's restatement of the reference's k-means
(experiments/sva_pq_lookup_test.py:66-106, experiments/sva_supervised_coarse_pq_test.py:88-131).

The centroid update is bit-exact with the oracle on the same labels (cell
sums in ascending row order, plain and weighted, empty cells kept).  Whole
fits from the same initial centroids match the oracle's fit; a label can
only differ where two centroids are equally near within rounding (the
assignment's own rule, tested in test_gpu_write.py), so centroids are
compared to 1e-5 and most must be bit-identical.  The seeded default
initialisation is deterministic on the device.
"""

from __future__ import annotations


import numpy as np
import pytest
import torch

import oracle

pytestmark = pytest.mark.gpu


def _data(seed, H=3, N=3000, R=64):
    rng = np.random.default_rng(seed)
    return rng, rng.standard_normal((H, N, R)).astype(np.float32)


@pytest.mark.parametrize("weighted", [False, True])
def test_centroid_update_bit_exact(device, weighted):
    from sva_amd import inverted, kernels
    from sva_amd._lib import lib, ptr, stream_handle

    rng, x = _data(3 + weighted)
    H, N, R = x.shape
    S, C = 2, 64
    sub = R // S
    cent = rng.standard_normal((H, S, C, sub)).astype(np.float32)
    cent[:, :, -3:] += 50.0  # far away: empty cells, which keep their centroid
    w = (rng.random((H, N)) + 0.05).astype(np.float32) if weighted else None
    xt = torch.from_numpy(x).to(device)
    ct = torch.from_numpy(cent).to(device)
    eye = torch.eye(R, device=device).expand(H, R, R).contiguous()
    codes = torch.empty(H, N, S, device=device, dtype=torch.uint8)
    kernels.write_encode(xt, eye, ct, torch.empty_like(xt), codes)
    post = inverted.build_postings(codes, N, C)
    nxt = torch.empty_like(ct)
    wt = torch.from_numpy(w).to(device) if weighted else None
    assert lib().sva_centroid_update(ptr(xt), xt.stride(0), N, H, R, S, C, ptr(wt), ptr(post.offsets),
                                     ptr(post.ids), ptr(ct), ptr(nxt), stream_handle(device)) == 0
    got = nxt.cpu().numpy()
    labels = codes.cpu().numpy().astype(np.int64)
    for h in range(H):
        for s in range(S):
            want = oracle.kmeans_update(x[h, :, s * sub:(s + 1) * sub], labels[h, :, s], cent[h, s],
                                        None if w is None else w[h])
            np.testing.assert_array_equal(got[h, s].view(np.uint32), want.view(np.uint32), err_msg=f"{h} {s}")
    np.testing.assert_array_equal(got[:, :, -3:], cent[:, :, -3:])


@pytest.mark.parametrize("weighted,S,C", [(False, 2, 64), (True, 4, 16)])
def test_fit_matches_oracle(device, weighted, S, C):
    from sva_amd import codebooks

    rng, x = _data(11 + C)
    H, N, R = x.shape
    sub = R // S
    init = np.stack([np.stack([x[h, rng.choice(N, C, replace=False), s * sub:(s + 1) * sub] for s in range(S)])
                     for h in range(H)])
    w = (rng.random((H, N)) * 3).astype(np.float32) if weighted else None
    t = lambda a: torch.from_numpy(a).to(device)  # noqa: E731
    if weighted:
        got = codebooks.fit_weighted_product_codebooks(t(x), t(w), S, C, 4, seed=0, initial=t(init))
    else:
        got = codebooks.fit_product_codebooks(t(x), S, C, 4, seed=0, initial=t(init))
    got = got.cpu().numpy()
    want = oracle.kmeans_fit(x, S, 4, init, w)
    assert got.shape == want.shape == (H, S, C, sub)
    np.testing.assert_allclose(got, want, rtol=1e-5, atol=1e-5)
    same = np.all(got.view(np.uint32) == want.view(np.uint32), axis=-1)
    assert same.mean() >= 0.95, f"only {same.mean():.3f} of the centroids are bit-identical"


def test_default_initialisation_is_seeded(device):
    from sva_amd import codebooks

    _, x = _data(5, H=2, N=600)
    xt = torch.from_numpy(x).to(device)
    a = codebooks.fit_product_codebooks(xt, 2, 256, 2, seed=7)
    b = codebooks.fit_product_codebooks(xt, 2, 256, 2, seed=7)
    assert a.shape == (2, 2, 256, 32)
    assert torch.equal(a, b)
    small = codebooks.fit_product_codebooks(xt[:, :100], 2, 256, 1, seed=7)
    assert small.shape == (2, 2, 100, 32)  # min(codewords, rows) as the reference


@pytest.mark.parametrize("N,C,code_dtype", [(1, 1, torch.uint8), (63, 5, torch.uint8), (1024, 256, torch.uint8),
                                            (1025, 3, torch.int16), (16385, 1024, torch.int32), (40001, 200, torch.uint8)])
def test_postings_wave_ranges(device, N, C, code_dtype):
    """Rows that leave waves of the build empty, partial or with several rounds: cells in ascending key order."""
    from sva_amd import inverted

    g = torch.Generator(device=device).manual_seed(N + C)
    codes = torch.randint(0, C, (2, N + 3, 2), device=device, generator=g).to(code_dtype)
    post = inverted.build_postings(codes, N, C)
    for h in range(2):
        for s in range(2):
            c = codes[h, :N, s].long()
            counts = torch.bincount(c, minlength=C)
            assert torch.equal(post.ids[h, s, :N].long(), torch.sort(c, stable=True).indices)
            assert torch.equal(post.offsets[h, s, 1:].long(), counts.cumsum(0)) and int(post.offsets[h, s, 0]) == 0
            assert int(post.max_count[h, s]) == int(counts.max())


@pytest.mark.parametrize("weighted", [False, True])
def test_centroid_update_cell_sizes(device, weighted):
    """Cells of none to 49 members (batches of 16 with every remainder): sums in ascending key order, bit for bit."""
    from sva_amd._lib import check, lib, ptr, stream_handle

    C, sub = 50, 8
    labels = torch.repeat_interleave(torch.arange(C), torch.arange(C))
    labels = labels[torch.randperm(len(labels), generator=torch.Generator().manual_seed(1))]
    n = len(labels)
    g = torch.Generator().manual_seed(2)
    x, w, prev = torch.randn(1, n, sub, generator=g), torch.rand(1, n, generator=g) + 0.1, torch.randn(1, 1, C, sub, generator=g)
    from sva_amd import inverted

    post = inverted.build_postings(labels.to(device, torch.uint8)[None, :, None].contiguous(), n, C)
    xd, wd, pd, nxt = x.to(device), w.to(device), prev.to(device), torch.empty(1, 1, C, sub, device=device)
    check(lib().sva_centroid_update(ptr(xd), xd.stride(0), n, 1, sub, 1, C, ptr(wd) if weighted else None,
                                    ptr(post.offsets), ptr(post.ids), ptr(pd), ptr(nxt), stream_handle(xd.device)), "update")
    rows = x[0] * w[0][:, None] if weighted else x[0]
    total = torch.zeros(C, sub).index_add_(0, labels, rows)
    count = torch.zeros(C).index_add_(0, labels, w[0]) if weighted else torch.bincount(labels, minlength=C).float()
    want = torch.where(count[:, None] > 0, total / count.clamp_min(1e-30)[:, None], prev[0, 0])
    assert torch.equal(nxt[0, 0].cpu(), want)
