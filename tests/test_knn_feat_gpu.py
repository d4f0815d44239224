"""knn_points rows of float points with many dimensions: candidates from the
matrix cores by an exact bound, equal distances replayed.  Every row must be
the reference-order forward's row as the module's sort leaves it, bit for bit."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


def _sorted_by_module(idxs, dists, lengths2, K):
    # knn_points' sort after the forward (reference knn/__init__.py:111-131)
    pad = (lengths2[:, None] <= torch.arange(K, device=dists.device)[None])[:, None].expand_as(dists)
    ds, order = dists.masked_fill(pad, float("inf")).sort(dim=2)
    return idxs.gather(2, order), ds.masked_fill(pad, 0.0)


def _check(tpo, dev, p1, p2, l1, l2, K):
    a, b, la, lb = p1.to(dev), p2.to(dev), l1.to(dev), l2.to(dev)
    for version in (-1, 0):
        si, sd = tpo.knn_points(a, b, la, lb, K=K, version=version)
        ri, rd = torch.ops.torch_point_ops_knn.knn_forward(a, b, la, lb, 2, K, version)
        ei, ed = _sorted_by_module(ri, rd, lb, K)
        assert torch.equal(sd.isnan(), ed.isnan())
        assert torch.equal(torch.nan_to_num(sd), torch.nan_to_num(ed))
        assert torch.equal(si, ei)


# widths at the edges of the 16-wide k-steps with six more entries for the
# norms, and not multiples of 4; reference counts at the edges of the tiles
# (32), of the fine groups (up to 32 tiles, made odd: 992 and 993 references)
# and of several tiles a group (over 128 tiles: 4064 and 4096)
@pytest.mark.parametrize("D,P1,P2,K", [
    (4, 70, 1, 3), (9, 64, 31, 5), (10, 65, 33, 20), (11, 130, 192, 32), (26, 63, 193, 32),
    (27, 200, 255, 16), (35, 333, 992, 20), (42, 1, 993, 2), (58, 128, 1024, 10),
    (64, 500, 2048, 20), (9, 70, 4064, 32), (20, 70, 4096, 31), (74, 96, 3000, 32),
    (90, 33, 5000, 5), (106, 40, 700, 8),
    (122, 64, 4128, 31), (128, 257, 9001, 16), (64, 30, 33000, 32), (16, 700, 4095, 12),
])
@pytest.mark.parametrize("case", ["normal", "offset", "self"])
def test_feature_rows_match_the_reference_order(tpo, dev, D, P1, P2, K, case):
    g = torch.Generator().manual_seed(D * P2 + K)
    N = 2
    p2 = torch.randn(N, P2, D, generator=g)
    p1 = torch.randn(N, P1, D, generator=g)
    if case == "offset":  # far from the origin, widths of very different sizes
        scale = 2.0 ** torch.randint(-6, 7, (D,), generator=g)
        p1, p2 = (p1 * scale + 50).float(), (p2 * scale + 50).float()
    if case == "self":
        p1 = p2[:, torch.randint(0, P2, (P1,), generator=g)].contiguous()
    l1 = torch.tensor([P1, max(1, P1 - 5)])
    l2 = torch.tensor([P2, max(1, (2 * P2) // 3)])
    _check(tpo, dev, p1, p2, l1, l2, K)


# lengths at the edges of the clouds that are listed whole (32 + 2 K) and of a
# row's list (128), alone and in the mostly empty tiles of a longer cloud, where
# few more than K groups hold a reference
@pytest.mark.parametrize("P2", [0, 352, 1056, 9001])
@pytest.mark.parametrize("D,K", [(16, 5), (64, 16), (9, 31), (35, 32)])
def test_feature_rows_of_short_lengths(tpo, dev, D, K, P2):
    g = torch.Generator().manual_seed(D + P2)
    l2 = torch.tensor([1, K - 1, K, K + 1, 31 + 2 * K, 32 + 2 * K, 33 + 2 * K, 127, 128, 129, 130, 0])
    N, P1, P2 = len(l2), 70, P2 or 130
    p1, p2 = torch.randn(N, P1, D, generator=g), torch.randn(N, P2, D, generator=g)
    p2[:, 3] = p2[:, 9]
    l1 = torch.full((N,), P1)
    l1[2], l1[-2] = 64, 33
    _check(tpo, dev, p1, p2, l1, l2, K)


# every row tied or not finite, more of them than are replayed: left to the
# lane-a-row kernel, and (64 and 128 dimensions, few queries, long clouds) to
# the kernels that slice the references
@pytest.mark.parametrize("N,P1,P2,D,K", [(3, 4003, 300, 9, 5), (2, 9000, 170, 4, 12), (1, 1500, 4000, 64, 8),
                                         (2, 1100, 3000, 128, 20)])
@pytest.mark.parametrize("case", ["lattice", "one_nan"])
def test_feature_rows_too_many_to_replay(tpo, dev, N, P1, P2, D, K, case):
    g = torch.Generator().manual_seed(P1 + D)
    p1, p2 = torch.randn(N, P1, D, generator=g), torch.randn(N, P2, D, generator=g)
    if case == "lattice":
        p1, p2 = (p1 > 0.5).float(), (p2 > 0.5).float()
    else:
        p2[0, P2 - 2, 1] = float("nan")
    l1, l2 = torch.full((N,), P1), torch.full((N,), P2)
    l1[-1] = P1 - 3
    l2[-1] = P2 - 1
    _check(tpo, dev, p1, p2, l1, l2, K)


@pytest.mark.parametrize("case", ["few_ties", "all_ties", "runs", "nonfinite_query",
                                  "nonfinite_cloud", "nan_of_ones", "huge", "tiny", "short", "far_cloud"])
@pytest.mark.parametrize("D,K", [(64, 20), (9, 5)])
def test_feature_rows_replayed_and_edge_values(tpo, dev, case, D, K):
    g = torch.Generator().manual_seed(len(case) + D)
    N, P1, P2 = 3, 900, 1500
    p1 = torch.randn(N, P1, D, generator=g)
    p2 = torch.randn(N, P2, D, generator=g)
    l1, l2 = torch.tensor([P1, P1, 500]), torch.tensor([P2, 1100, P2])
    if case == "few_ties":  # copies of a few references, queries beside them
        p2[:, 700:710] = p2[:, 100:110]
        p1[:, :10] = p2[:, 100:110] + 1e-3
    elif case == "all_ties":  # every row: more than the replay takes
        p1 = torch.randint(0, 2, (N, P1, D), generator=g).float()
        p2 = torch.randint(0, 2, (N, P2, D), generator=g).float()
    elif case == "runs":  # all neighbours of a query next to each other in the cloud
        c = torch.randn(N, P2 // 50, 1, D, generator=g) * 10
        p2 = (c + 0.1 * torch.randn(N, P2 // 50, 50, D, generator=g)).reshape(N, P2, D)
        p1 = (c[:, torch.randint(0, P2 // 50, (P1,), generator=g), 0]
              + 0.1 * torch.randn(N, P1, D, generator=g))
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
    elif case == "huge":  # distances that overflow to infinity
        p2[0, ::3] *= 1e25
        p1[1] *= 1e30
    elif case == "tiny":
        p1, p2 = p1 * 1e-22, p2 * 1e-22
    elif case == "short":
        l2 = torch.tensor([K - 1, 0, 3])
    else:
        p1 = p1 + 1e4
    _check(tpo, dev, p1, p2, l1, l2, K)


@pytest.mark.parametrize("D,P2", [(4, 3), (16, 500), (64, 2100)])
def test_single_nearest_takes_the_lower_index(tpo, O, dev, D, P2):
    g = torch.Generator().manual_seed(P2)
    p2 = torch.randint(0, 3, (2, P2, D), generator=g).float()  # many equal rows
    p1 = torch.randint(0, 3, (2, 150, D), generator=g).float()
    l1, l2 = torch.tensor([150, 90]), torch.tensor([P2, 0])
    for version in (-1, 0):
        i, d = tpo.knn_points(p1.to(dev), p2.to(dev), l1.to(dev), l2.to(dev), K=1, version=version)
        ei, ed = O.knn_fwd(p1.numpy(), p2.numpy(), l1.numpy(), l2.numpy(), K=1, version=version)
        assert np.array_equal(i.cpu().numpy(), ei) and np.array_equal(d.cpu().numpy(), ed)


@pytest.mark.parametrize("D", [3, 9, 64])
def test_rows_of_views_off_16_bytes(tpo, dev, D):
    """Clouds that start 4 bytes past a 16-byte boundary."""
    g = torch.Generator().manual_seed(D)
    P1, P2, K = 70, 700, 9
    a = torch.randn(2 * P1 * D + 1, generator=g).to(dev)[1:].view(2, P1, D)
    b = torch.randn(2 * P2 * D + 1, generator=g).to(dev)[1:].view(2, P2, D)
    b[:, 5] = b[:, 6]  # equal distances: replayed rows
    l1, l2 = torch.tensor([P1, 33], device=dev), torch.tensor([P2, 500], device=dev)
    ri, rd = torch.ops.torch_point_ops_knn.knn_forward(a, b, l1, l2, 2, K, 0)
    ei, ed = _sorted_by_module(ri, rd, l2, K)
    si, sd = tpo.knn_points(a, b, l1, l2, K=K, version=0)
    assert torch.equal(si, ei) and torch.equal(sd, ed)


def test_rows_captured_in_a_graph(tpo, dev):
    """knn_points (both row paths, ties among the rows), sampling and the
    gathers' gradients replayed from a graph on new inputs, with eager work
    between the replays."""
    g = torch.Generator().manual_seed(8)

    def draw():
        p = torch.randn(2, 900, 3, generator=g).round(decimals=1)
        f = torch.randn(2, 300, 40, generator=g).round(decimals=0)
        w = torch.randn(2, 900, 8, 3, generator=g)
        return p.to(dev), f.to(dev), w.to(dev)

    s_p, s_f, s_w = draw()
    lens = torch.tensor([900, 700], device=dev)

    def step(p, f, w):
        q = p.detach().requires_grad_(True)
        i, d = tpo.knn_points(p, p, lens, lens, K=8)
        nn = tpo.knn_gather(q, i, lens)
        (gq,) = torch.autograd.grad(nn, (q,), w)
        fi, fd = tpo.knn_points(f, f, K=5)
        s = tpo.furthest_point_sampling(p, 40)
        return i, d, gq, fi, fd, s

    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        for _ in range(2):
            step(s_p, s_f, s_w)
    torch.cuda.current_stream().wait_stream(side)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        got = step(s_p, s_f, s_w)
    for _ in range(4):
        p, f, w = draw()
        want = [t.clone() for t in step(p, f, w)]
        s_p.copy_(p), s_f.copy_(f), s_w.copy_(w)
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        for a, b in zip(got, want):
            assert torch.equal(a, b)
