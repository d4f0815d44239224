"""The work that programs have this package do, as cases that can be timed and checked.

Each case is one call (or one training step) through the public entry points: Chamfer
distance, k nearest neighbours, furthest point sampling, feature gathering and the earth
mover's distance, from the smallest call to the benchmark's sizes, in the data types and
directions that are used.  Run it from the repository's root: the package is taken from
the torch-point-ops_amd folder of the working folder.
"""
import os
import sys

_PKG = os.path.abspath("torch-point-ops_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

import torch  # noqa: E402

import torch_point_ops as tpo  # noqa: E402

DTYPES = {"f32": torch.float32, "f16": torch.float16, "bf16": torch.bfloat16}
SIZE = {"f32": 4, "f16": 2, "bf16": 2}


def listed():
    return [
        # one small pair of clouds: an evaluation loop's latency
        {"name": "chamfer_1x128", "op": "chamfer", "B": 1, "N": 128, "M": 128, "dtype": "f32",
         "cloud": "uniform", "mode": "forward"},
        # the headline training step: loss and gradients of a reconstructed batch
        {"name": "chamfer_train_32x8192", "op": "chamfer", "B": 32, "N": 8192, "M": 8192,
         "dtype": "f32", "cloud": "mixture", "mode": "train"},
        # mixed precision, a sparse prediction against a dense target, no round sizes
        {"name": "chamfer_train_f16_8x5000x12345", "op": "chamfer", "B": 8, "N": 5000, "M": 12345,
         "dtype": "f16", "cloud": "mixture", "mode": "train"},
        # neighbourhoods of ordinary clouds: grouping in a point network's layer
        {"name": "knn_16x2048_k16", "op": "knn", "B": 16, "P1": 2048, "P2": 2048, "D": 3, "K": 16,
         "dtype": "f32", "cloud": "normal", "ragged": False, "mode": "forward"},
        # scans of different lengths, padded, with neighbours and gradients
        {"name": "knn_train_8x16384_k16", "op": "knn", "B": 8, "P1": 16384, "P2": 16384, "D": 3,
         "K": 16, "dtype": "f32", "cloud": "sphere", "ragged": True, "mode": "train"},
        # upsampling: three nearest of a sparse level for every point of the dense one
        {"name": "knn_8x16384x1024_k3", "op": "knn", "B": 8, "P1": 16384, "P2": 1024, "D": 3,
         "K": 3, "dtype": "f32", "cloud": "sphere", "ragged": False, "mode": "forward"},
        # a neighbour graph in feature space: every point's nearest in its own cloud
        {"name": "knn_features_8x2048x64_k20", "op": "knn", "B": 8, "P1": 2048, "P2": 2048,
         "D": 64, "K": 20, "dtype": "f32", "cloud": "self", "ragged": False, "mode": "forward"},
        # retrieval among bfloat16 descriptors
        {"name": "knn_bf16_4x4096x65536x128_k32", "op": "knn", "B": 4, "P1": 4096, "P2": 65536,
         "D": 128, "K": 32, "dtype": "bf16", "cloud": "unit", "ragged": False, "mode": "forward"},
        # centroids of ordinary clouds
        {"name": "fps_16x2048_128", "op": "fps", "B": 16, "N": 2048, "S": 128, "dtype": "f32"},
        # centroids of large scans
        {"name": "fps_16x65536_4096", "op": "fps", "B": 16, "N": 65536, "S": 4096,
         "dtype": "f32"},
        # features at the centroids, and their gradients
        {"name": "gather_train_16x64x65536_4096", "op": "gather", "B": 16, "C": 64, "N": 65536,
         "S": 4096, "dtype": "f32"},
        # a matching loss: cost and gradients
        {"name": "emd_train_16x2048", "op": "emd", "B": 16, "N": 2048, "M": 2048, "dtype": "f32",
         "mode": "train"},
    ]


def _size(rng, lo, hi):
    """A size of [lo, hi], spread over its logarithm; every other one a multiple of 64."""
    n = int(round(lo * (hi / lo) ** rng.random()))
    if rng.random() < 0.5 and n >= 64:
        n -= n % 64
    return max(lo, min(hi, n))


def draw(rng):
    op = rng.choice(["chamfer", "chamfer", "knn", "knn", "features", "fps", "gather", "emd"])
    if op == "chamfer":
        c = {"op": op, "B": _size(rng, 1, 32), "N": _size(rng, 128, 16384),
             "M": _size(rng, 128, 16384), "dtype": rng.choice(["f32", "f32", "f16"]),
             "cloud": rng.choice(["mixture", "uniform"]),
             "mode": rng.choice(["forward", "train"])}
        while c["B"] * (c["N"] + c["M"]) > 32 * 16384:
            c["B"] -= 1
        return c
    if op == "knn":
        c = {"op": op, "B": _size(rng, 1, 16), "P1": _size(rng, 256, 16384),
             "P2": _size(rng, 256, 16384), "D": 3, "K": rng.choice([1, 3, 5, 8, 12, 16, 20, 32]),
             "dtype": rng.choice(["f32", "f32", "f32", "f16"]),
             "cloud": rng.choice(["sphere", "normal"]), "ragged": rng.random() < 0.3,
             "mode": rng.choice(["forward", "forward", "train"])}
        while c["B"] * c["P1"] * c["P2"] > 8 * 16384 * 16384:
            c["B"] -= 1
        return c
    if op == "features":
        c = {"op": "knn", "B": _size(rng, 1, 16), "P1": _size(rng, 256, 4096), "P2": 0,
             "D": rng.choice([9, 16, 32, 35, 64, 64, 96, 128]), "K": rng.choice([5, 10, 16, 20, 32]),
             "dtype": rng.choice(["f32", "f32", "bf16"]), "cloud": rng.choice(["self", "unit"]),
             "ragged": rng.random() < 0.2, "mode": "forward"}
        c["P2"] = c["P1"] if c["cloud"] == "self" else _size(rng, 256, 16384)
        while c["B"] > 1 and c["B"] * c["P1"] * c["P2"] * c["D"] > 2 ** 31:
            c["B"] -= 1
        return c
    if op == "fps":
        n = _size(rng, 1024, 65536)
        return {"op": op, "B": _size(rng, 1, 16), "N": n, "S": max(16, n // rng.choice([4, 8, 16])) if n < 16384
                else n // 16, "dtype": rng.choice(["f32", "f32", "f16"])}
    if op == "gather":
        n = _size(rng, 1024, 65536)
        return {"op": op, "B": _size(rng, 1, 16), "C": _size(rng, 3, 64), "N": n,
                "S": max(16, n // rng.choice([2, 4, 16])), "dtype": rng.choice(["f32", "f32", "f16"])}
    return {"op": "emd", "B": _size(rng, 1, 16), "N": _size(rng, 128, 2048), "M": _size(rng, 128, 2048),
            "dtype": "f32", "mode": rng.choice(["forward", "train"])}


def _rand(g, *shape):
    return torch.rand(*shape, generator=g, device=g.device)


def _randn(g, *shape):
    return torch.randn(*shape, generator=g, device=g.device)


def _mixture(g, B, N):
    """Clouds of eight Gaussian parts of width 0.1 in [-1, 1]^3."""
    centres = _rand(g, B, 8, 3) * 2 - 1
    part = torch.randint(0, 8, (B, N, 1), generator=g, device=g.device)
    return torch.gather(centres, 1, part.expand(-1, -1, 3)) + 0.1 * _randn(g, B, N, 3)


def _sphere(g, B, N):
    """A scanned surface: the unit sphere with radial noise."""
    d = _randn(g, B, N, 3)
    return d / d.norm(dim=-1, keepdim=True) * (1 + 0.02 * _randn(g, B, N, 1))


def _of_width(g, P, cloud, D):
    """Rows of features: of length one, or as a layer leaves them (correlated, not centred)."""
    if cloud == "unit":
        x = _randn(g, *P, D)
        return x / x.norm(dim=-1, keepdim=True)
    mix = _randn(g, P[0], D, D) / D ** 0.5
    return torch.bmm(_randn(g, *P, D), mix).add_(0.5).clamp_(min=-0.2)


def _lengths(g, B, P):
    return torch.randint((P + 1) // 2, P + 1, (B,), generator=g, device=g.device)


def prepare(case, seed):
    g = torch.Generator("cuda").manual_seed(seed)
    t, B, op = DTYPES[case["dtype"]], case["B"], case["op"]
    s = {"case": case}
    if op == "chamfer":
        N, M = case["N"], case["M"]
        if case["cloud"] == "uniform":
            a, b = _rand(g, B, N, 3), _rand(g, B, M, 3)
        else:  # a reconstruction of the same shape, a little off
            a = _mixture(g, B, N)
            pick = torch.randint(0, N, (B, M, 1), generator=g, device="cuda").expand(-1, -1, 3)
            b = torch.gather(a, 1, pick) + 0.01 * _randn(g, B, M, 3)
        s["a"], s["b"] = a.to(t), b.to(t)
        if case["mode"] == "train":
            s["a"].requires_grad_(True)
            s["b"].requires_grad_(True)
            s["loss"] = tpo.ChamferDistance("mean")
    elif op == "knn":
        P1, P2, D, cloud = case["P1"], case["P2"], case["D"], case["cloud"]
        if cloud == "sphere":
            p1, p2 = _sphere(g, B, P1), _sphere(g, B, P2)
        elif cloud == "normal":
            p1, p2 = _randn(g, B, P1, 3), _randn(g, B, P2, 3)
        else:
            p1 = _of_width(g, (B, P1), cloud, D)
            p2 = p1 if cloud == "self" else _of_width(g, (B, P2), cloud, D)
        s["p1"] = p1.to(t)
        s["p2"] = s["p1"] if cloud == "self" else p2.to(t)
        s["l1"] = _lengths(g, B, P1) if case["ragged"] else None
        s["l2"] = (s["l1"] if cloud == "self" else _lengths(g, B, P2)) if case["ragged"] else None
        s["knn"] = tpo.KNearestNeighbors(K=case["K"], return_nn=D == 3)
        if case["mode"] == "train":
            s["p1"].requires_grad_(True)
            s["p2"].requires_grad_(True)
            s["g_dists"] = _randn(g, B, P1, case["K"]).to(t)
            s["g_nn"] = _randn(g, B, P1, case["K"], 3).to(t)
            if case["ragged"]:  # a loss leaves out the padding
                row = torch.arange(P1, device="cuda")[None, :, None] < s["l1"][:, None, None]
                s["g_dists"] *= row
                s["g_nn"] *= row[..., None]
    elif op == "fps":
        N = case["N"]
        blob = N // 10  # a room with one dense object in it
        p = torch.cat([_rand(g, B, N - blob, 3) * 2 - 1,
                       _rand(g, B, 1, 3) * 2 - 1 + 0.05 * _randn(g, B, blob, 3)], 1)
        order = torch.argsort(_rand(g, B, N), 1)[..., None].expand(-1, -1, 3)
        s["points"] = torch.gather(p, 1, order).to(t)
    elif op == "gather":
        N, S = case["N"], case["S"]
        s["points"] = _randn(g, B, case["C"], N).to(t).requires_grad_(True)
        s["idx"] = torch.argsort(_rand(g, B, N), 1)[:, :S].contiguous()  # distinct, as sampling gives
        s["g_out"] = _randn(g, B, case["C"], S).to(t)
    else:
        s["a"], s["b"] = _randn(g, B, case["N"], 3).to(t), _randn(g, B, case["M"], 3).to(t)
        if case["mode"] == "train":
            s["a"].requires_grad_(True)
            s["b"].requires_grad_(True)
            s["loss"] = tpo.EarthMoverDistance()
    return s


def run(s):
    case = s["case"]
    op, train = case["op"], case.get("mode") == "train"
    if op == "chamfer" or op == "emd":
        if not train:
            f = tpo.chamfer_distance if op == "chamfer" else tpo.earth_movers_distance
            return f(s["a"], s["b"])
        loss = s["loss"](s["a"], s["b"])
        return (loss, *torch.autograd.grad(loss, (s["a"], s["b"])))
    if op == "knn":
        out = s["knn"](s["p1"], s["p2"], s["l1"], s["l2"])
        if not train:
            return out
        idxs, dists, nn = out
        return (idxs, dists, nn, *torch.autograd.grad((dists, nn), (s["p1"], s["p2"]),
                                                      (s["g_dists"], s["g_nn"])))
    if op == "fps":
        return tpo.farthest_point_sample_and_gather(s["points"], case["S"])
    out = tpo.gather_points(s["points"], s["idx"])
    return (out, *torch.autograd.grad(out, s["points"], s["g_out"]))


def work(case):
    z, B, op = SIZE[case["dtype"]], case["B"], case["op"]
    train = case.get("mode") == "train"
    if op == "chamfer":  # one distance a point is the least that has to be computed
        points = B * (case["N"] + case["M"])
        return {"bytes": points * z * (3 + (3 if train else 1)), "flops": points * 9}
    if op == "knn":
        P1, P2, D, K = case["P1"], case["P2"], case["D"], case["K"]
        rows = B * P1 * K
        pts = B * P1 * D + (0 if case["cloud"] == "self" else B * P2 * D)
        n = pts * z + rows * (8 + z)
        if D == 3:
            n += rows * 3 * z  # the neighbours themselves
        if train:
            n += rows * 4 * z + pts * z
        # a grid leaves few pairs in three dimensions; in many the products are needed
        return {"bytes": n, "flops": rows * 9 if D == 3 else 2 * D * B * P1 * P2}
    if op == "fps":  # every point against one sample at least, and every sample
        return {"bytes": B * (case["N"] * 3 * z + case["S"] * (8 + 3 * z)),
                "flops": 10 * B * (case["N"] + case["S"])}
    if op == "gather":
        C, N, S = case["C"], case["N"], case["S"]
        return {"bytes": B * (S * 8 + C * S * z * 3 + C * N * z), "flops": 0}
    # ten levels: a distance, an exponential a level and three weighted sums a level
    pairs = B * case["N"] * case["M"]
    pts = 3 * z * B * (case["N"] + case["M"])
    return {"bytes": pts * (2 if train else 1) + B * z, "flops": pairs * (8 + 10 * (1 + 6))}


def tolerance(case):
    op, f16, train = case["op"], case["dtype"] == "f16", case.get("mode") == "train"
    if op == "chamfer":
        # distances are the formula's own roundings; gradients are sums in any order
        return ({"rel": 2e-3, "max": 2e-1} if f16 else {"rel": 1e-6, "max": 2e-5}) if train else "exact"
    if op == "knn":
        if case["dtype"] == "bf16":  # sums of products in any order, rounded to bf16
            return {"rel": 4e-3, "max": 2e-2, "differ": 5e-3}
        return ({"rel": 2e-3, "max": 2e-1} if f16 else {"rel": 1e-6, "max": 2e-5}) if train else "exact"
    if op == "emd":
        return {"rel": 2.5e-4, "max": 2e-2}
    return "exact"


def _sq(a, b):
    """(b, n, m) squared distances of (b, n, 3) and (b, m, 3), in float64."""
    return sum((a[:, :, None, d] - b[:, None, :, d]).square_() for d in range(3))


def _nearest(a, b):
    """Squared distance and index of every point's nearest in the other cloud."""
    d, i = [], []
    step = max(1, 2 ** 26 // (a.shape[0] * b.shape[1]))
    for at in range(0, a.shape[1], step):
        m = _sq(a[:, at:at + step], b).min(2)
        d.append(m.values)
        i.append(m.indices)
    return torch.cat(d, 1), torch.cat(i, 1)


def _rows(x, i):
    return torch.gather(x, 1, i[..., None].expand(-1, -1, x.shape[2]))


def _exact_chamfer(s, train):
    a, b = s["a"].detach().double(), s["b"].detach().double()
    (d1, i1), (d2, i2) = _nearest(a, b), _nearest(b, a)
    if not train:
        return d1, d2
    loss = d1.mean() + d2.mean()
    if s["a"].dtype == torch.float16:  # which point is nearest is a matter of rounding there
        return loss, None, None
    t1 = 2 * (a - _rows(b, i1)) / d1.numel()
    t2 = 2 * (b - _rows(a, i2)) / d2.numel()
    ga = t1.scatter_add(1, i2[..., None].expand(-1, -1, 3), -t2)
    gb = t2.scatter_add(1, i1[..., None].expand(-1, -1, 3), -t1)
    return loss, ga, gb


def _exact_knn(s, case, train):
    p1, p2 = s["p1"].detach().double(), s["p2"].detach().double()
    (B, P1, D), P2, K = p1.shape, p2.shape[1], case["K"]
    l1 = s["l1"] if s["l1"] is not None else torch.full((B,), P1, device="cuda")
    l2 = s["l2"] if s["l2"] is not None else torch.full((B,), P2, device="cuda")
    past = torch.arange(P2, device="cuda")[None, None] >= l2[:, None, None]
    step = max(1, 2 ** 25 // (B * P2))
    dists = []
    for at in range(0, P1, step):
        d = 0
        for k in range(D):
            d = d + (p1[:, at:at + step, None, k] - p2[:, None, :, k]).square_()
        dists.append(d.masked_fill_(past, float("inf")).topk(min(K, P2), 2, largest=False, sorted=True))
    i = torch.cat([d.indices for d in dists], 1)
    d = torch.cat([d.values for d in dists], 1)
    if i.shape[2] < K:
        return None
    row = torch.arange(P1, device="cuda")[None, :, None] < l1[:, None, None]
    d = d * row
    if case["D"] != 3:
        return None, d
    if not train:
        return None, d, None
    if case["dtype"] == "f16":
        return None, d, None, None, None
    i = i * row
    g = 2 * s["g_dists"].double()[..., None] * row[..., None]
    flat = i.reshape(B, P1 * K, 1).expand(-1, -1, 3)
    diff = p1[:, :, None] - torch.gather(p2, 1, flat).reshape(B, P1, K, 3)
    back = torch.zeros_like(p2).scatter_add(1, flat, (s["g_nn"].double() - g * diff).reshape(B, P1 * K, 3))
    return None, d, None, (g * diff).sum(2), back


def _exact_emd(s, train):
    a, b = s["a"].detach().double(), s["b"].detach().double()
    (B, N, _), M = a.shape, b.shape[1]
    d = _sq(a, b)
    eps = float(torch.tensor(1e-9, dtype=torch.float32))
    left = torch.full((B, N, 1), max(1.0, M / N), dtype=torch.float64, device="cuda")
    right = torch.full((B, 1, M), max(1.0, N / M), dtype=torch.float64, device="cuda")
    match = torch.zeros_like(d)
    for level in [-4.0 ** j for j in range(7, -2, -1)] + [0.0]:
        w = torch.exp(level * d)
        share = left / ((w * right).sum(2, keepdim=True) + 2 * eps)
        taken = (w * share).sum(1, keepdim=True) * right
        given = torch.clamp(right / (taken + eps), max=1) * right
        right = torch.clamp(right - taken, min=0)
        w *= share
        w *= given
        match += w
        left = torch.clamp(left - w.sum(2, keepdim=True), min=0)
    cost = (d * match).sum((1, 2)) / N
    if not train:
        return cost
    c = 2.0 / (N * B)
    ga = c * (a * match.sum(2)[..., None] - torch.bmm(match, b))
    gb = c * (b * match.sum(1)[..., None] - torch.bmm(match.transpose(1, 2).contiguous(), a))
    return cost.mean(), ga, gb


def exact(case, seed):
    op, train = case["op"], case.get("mode") == "train"
    if op == "fps":  # indices and copies
        return None
    s = prepare(case, seed)
    if op == "chamfer":
        return _exact_chamfer(s, train)
    if op == "knn":
        return _exact_knn(s, case, train)
    if op == "emd":
        return _exact_emd(s, train)
    idx = s["idx"][:, None].expand(-1, case["C"], -1)
    x, g = s["points"].detach().double(), s["g_out"].double()
    return torch.gather(x, 2, idx), torch.zeros_like(x).scatter_add(2, idx, g)
