"""knn_points rows of float 3-D points by the cell grid: sorted rows must be the
reference-order forward's rows as the module's sort leaves them, bit for bit
(rows with equal distances are replayed), over shapes, orders and extremes."""
import numpy as np
import pytest
import torch

from tests.test_knn_feat_gpu import _sorted_by_module

pytestmark = pytest.mark.gpu


def _cloud(kind, g, N, P):
    x = torch.randn(N, P, 3, generator=g)
    if kind == "sphere":
        x = x / x.norm(dim=-1, keepdim=True)
    elif kind == "plane":  # one axis without extent
        x[..., 1] = 0.25
    elif kind == "line":
        x[..., 1:] = torch.tensor([1.0, -2.0])
    elif kind == "blobs":  # two dense parts far apart, and outliers
        x = 0.01 * x + 5 * (torch.rand(N, P, 1, generator=g) < 0.5)
        x[:, :: max(1, P // 3)] *= 300
    elif kind == "offset":
        x = x * torch.tensor([1e-3, 1.0, 1e3]) + 1e4
    return x


# reference and query counts at the edges of the register-held setups (4096,
# 16384) and above, and on both sides of the choice between the grid and brute
# force; K at the edges of the slots' registers (16, 32)
@pytest.mark.parametrize("P1,P2,K", [
    (1, 1, 1), (15, 2, 3), (17, 40, 4), (64, 33, 32), (65, 257, 5), (255, 1024, 8), (257, 500, 9),
    (1000, 2048, 16), (4096, 4097, 17), (4097, 4096, 3), (700, 16384, 16), (16390, 300, 12),
    (300, 17001, 32), (2000, 5000, 1), (900, 33000, 7),
])
@pytest.mark.parametrize("kind", ["normal", "sphere", "plane", "line", "blobs", "offset"])
@pytest.mark.parametrize("norm", [2, 1])
def test_near_rows_match_the_reference_order(tpo, dev, P1, P2, K, kind, norm):
    g = torch.Generator().manual_seed(P1 + 7 * P2 + K)
    N = 3
    p2 = _cloud(kind, g, N, P2)
    p1 = _cloud(kind, g, N, P1)
    p1[1] *= 4  # queries outside the references' box
    l1 = torch.tensor([P1, max(1, P1 // 2), P1])
    l2 = torch.tensor([P2, max(1, (2 * P2) // 3), max(1, P2 // 50)])
    a, b, la, lb = p1.to(dev), p2.to(dev), l1.to(dev), l2.to(dev)
    if K == 1:  # (the raw forward takes the grid too: against float64 ties aside, the formula)
        i, d = tpo.knn_points(a, b, la, lb, K=1, norm=norm)
        for n in range(N):
            q, r = p1[n, : l1[n]].numpy(), p2[n, : l2[n]].numpy()
            for at in range(0, len(q), 256):
                e = q[at:at + 256, None] - r[None]
                e = np.abs(e.astype(np.float64)).sum(2) if norm == 1 else (e.astype(np.float64) ** 2).sum(2)
                got = d[n, at:at + 256, 0].cpu().numpy()[: len(e)]
                assert np.allclose(got, e.min(1), rtol=1e-6, atol=1e-30)
                pick = np.take_along_axis(e, i[n, at:at + 256].cpu().numpy()[: len(e)], 1)[:, 0]
                assert np.allclose(pick, e.min(1), rtol=1e-6, atol=1e-30)
        return
    ri, rd = torch.ops.torch_point_ops_knn.knn_forward(a, b, la, lb, norm, K, 0)
    ei, ed = _sorted_by_module(ri, rd, lb, K)
    for rep in range(2):
        si, sd = tpo.knn_points(a, b, la, lb, K=K, norm=norm, version=0)
        assert torch.equal(sd, ed)
        assert torch.equal(si, ei)


def _takes_rows(N, P1, P2, D, K):
    """Whether knn_points selects rows by distance for these sizes."""
    import ctypes

    from torch_point_ops import _native

    I = ctypes.c_int64
    L = ctypes.CDLL(_native.HIP_LIB)
    f = L.tpo_knn_rows_workspace_size, L.tpo_knn_workspace_size
    for g in f:
        g.argtypes, g.restype = [ctypes.c_int, I, I, I, I, I, ctypes.c_int], I
    return f[0](0, N, P1, P2, D, K, 2) > f[1](0, N, P1, P2, D, K, 2)


# a wave searches four queries and a workgroup 16; clouds shorter than a row's
# K, empty ones, and queries in row order (more of them than references)
@pytest.mark.parametrize("P1,P2,K", [(1, 512, 3), (3, 600, 16), (4, 512, 2), (5, 700, 8), (15, 513, 9),
                                     (16, 512, 17), (17, 640, 32), (31, 900, 1), (2100, 1800, 12),
                                     (700, 600, 5), (33, 2500, 24)])
@pytest.mark.parametrize("kind", ["normal", "blobs"])
def test_near_rows_of_few_queries_and_short_lengths(tpo, O, dev, P1, P2, K, kind):
    g = torch.Generator().manual_seed(P1 + 7 * P2 + K)
    N = 7
    assert _takes_rows(N, P1, P2, 3, K)
    p1, p2 = _cloud(kind, g, N, P1), _cloud(kind, g, N, P2)
    l1 = torch.tensor([P1, P1, P1, max(1, P1 - 1), P1, P1, 0])
    l2 = torch.tensor([P2, K + 1, K, max(0, K - 1), 1, 0, P2])
    a, b, la, lb = p1.to(dev), p2.to(dev), l1.to(dev), l2.to(dev)
    si, sd = tpo.knn_points(a, b, la, lb, K=K, version=0)
    if K == 1:
        ei, ed = O.knn_fwd(p1.numpy(), p2.numpy(), l1.numpy(), l2.numpy(), K=1, version=0)
        assert np.array_equal(si.cpu().numpy(), ei) and np.array_equal(sd.cpu().numpy(), ed)
        return
    ri, rd = torch.ops.torch_point_ops_knn.knn_forward(a, b, la, lb, 2, K, 0)
    ei, ed = _sorted_by_module(ri, rd, lb, K)
    assert torch.equal(sd, ed) and torch.equal(si, ei)


# rows with equal distances replayed one by one, and too many for that: lists in
# the queries' order (P1 <= P2) and from row order, to the grid's lane-a-row
# kernel (2048 references and more) and to brute force
@pytest.mark.parametrize("N,P1,P2,K", [(2, 5000, 6000, 16), (3, 3001, 3001, 3), (2, 5001, 2500, 8),
                                       (4, 1999, 700, 20), (3, 2600, 900, 5), (2, 8000, 1023, 32),
                                       (40, 130, 520, 16), (1, 3000, 40000, 4)])
@pytest.mark.parametrize("tied", [0.0, 0.02, 0.3, 1.0])
def test_near_rows_of_clouds_with_repeated_points(tpo, dev, N, P1, P2, K, tied):
    g = torch.Generator().manual_seed(P1 + P2 + K)
    assert _takes_rows(N, P1, P2, 3, K)
    p1, p2 = torch.randn(N, P1, 3, generator=g), torch.randn(N, P2, 3, generator=g)
    m = int(P2 * tied)
    p2[:, :m] = p2[:, torch.randint(0, max(1, m // 2), (m,), generator=g)]
    p2 = p2[:, torch.randperm(P2, generator=g)].contiguous()
    if tied == 1.0:  # a lattice as well
        p1, p2 = (p1 * 4).round() / 4, (p2 * 4).round() / 4
    l1 = torch.full((N,), P1)
    l1[-1] = P1 - 7
    l2 = torch.full((N,), P2)
    l2[0] = P2 - P2 // 3
    a, b, la, lb = p1.to(dev), p2.to(dev), l1.to(dev), l2.to(dev)
    for norm in (2, 1):
        si, sd = tpo.knn_points(a, b, la, lb, K=K, norm=norm, version=0)
        ri, rd = torch.ops.torch_point_ops_knn.knn_forward(a, b, la, lb, norm, K, 0)
        ei, ed = _sorted_by_module(ri, rd, lb, K)
        assert torch.equal(sd, ed) and torch.equal(si, ei)


@pytest.mark.parametrize("case", ["few_ties", "lattice", "nonfinite_query", "nonfinite_cloud", "nan_of_ones",
                                  "huge", "short", "one_point"])
@pytest.mark.parametrize("P2,K", [(1500, 16), (6000, 5)])
def test_near_rows_replayed_and_edge_values(tpo, dev, case, P2, K):
    g = torch.Generator().manual_seed(len(case) + P2)
    N, P1 = 3, 1200
    p1, p2 = torch.randn(N, P1, 3, generator=g), torch.randn(N, P2, 3, generator=g)
    l1, l2 = torch.tensor([P1, P1, 500]), torch.tensor([P2, 1100, P2])
    if case == "few_ties":
        p2[:, 700:710] = p2[:, 100:110]
        p1[:, :10] = p2[:, 100:110] + 1e-3
    elif case == "lattice":  # every row tied: more than the replay takes
        p1 = torch.randint(0, 8, (N, P1, 3), generator=g).float()
        p2 = torch.randint(0, 8, (N, P2, 3), generator=g).float()
    elif case == "nonfinite_query":
        p1[0, 3, 2] = float("nan")
        p1[1, 4, 0] = float("inf")
    elif case == "nonfinite_cloud":
        p2[0, 5, 1] = float("inf")
        p2[1, 7, 1] = float("nan")
        p2[2, 0, 0] = float("nan")
    elif case == "nan_of_ones":  # every bit set, with either sign (a difference flips it)
        for bits, at in ((-1, 0), (0x7FFFFFFF, 1)):
            p2.view(torch.int32)[1, 40 + at:60:2] = bits
            p2.view(torch.int32)[1, 3 + at, 1] = bits
            p2.view(torch.int32)[1, 700 + at] = bits
    elif case == "huge":
        p2[0, ::3] *= 1e25
        p1[1] *= 1e30
    elif case == "short":
        l2 = torch.tensor([K - 1, 0, 3])
    else:
        p2[:] = p2[:, :1]
    a, b, la, lb = p1.to(dev), p2.to(dev), l1.to(dev), l2.to(dev)
    for version in (-1, 0):
        for norm in (1, 2):
            si, sd = tpo.knn_points(a, b, la, lb, K=K, norm=norm, version=version)
            ri, rd = torch.ops.torch_point_ops_knn.knn_forward(a, b, la, lb, norm, K, version)
            ei, ed = _sorted_by_module(ri, rd, lb, K)
            assert torch.equal(sd.isnan(), ed.isnan())
            assert torch.equal(torch.nan_to_num(sd), torch.nan_to_num(ed))
            assert torch.equal(si, ei)


@pytest.mark.parametrize("P2", [3, 500, 5000])
def test_single_nearest_takes_the_lower_index(tpo, O, dev, P2):
    g = torch.Generator().manual_seed(P2)
    p2 = torch.randint(0, 6, (2, P2, 3), generator=g).float()  # many equal points
    p1 = torch.randint(0, 6, (2, 300, 3), generator=g).float()
    p1[0, 7, 1] = float("nan")
    l1, l2 = torch.tensor([300, 90]), torch.tensor([P2, 0])
    for norm in (1, 2):
        for version in (-1, 0):
            i, d = tpo.knn_points(p1.to(dev), p2.to(dev), l1.to(dev), l2.to(dev), K=1, norm=norm,
                                  version=version)
            ei, ed = O.knn_fwd(p1.numpy(), p2.numpy(), l1.numpy(), l2.numpy(), K=1, norm=norm,
                               version=version)
            assert np.array_equal(i.cpu().numpy(), ei)
            assert np.array_equal(d.cpu().numpy(), ed, equal_nan=True)
