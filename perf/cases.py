"""Performance cases of the framework's public entry points.

listed() names twelve calls a program makes through hiperml_amd: SGEMV and
skinny SGEMM on device buffers (row-major, transposed, odd sizes, beta), the
host-pointer call of the reference's apps, dense SGEMM in plain FP32 and in
split precision, a batch of uneven skinny problems replayed as one graph, and
the k-means assignment.  draw() gives further sizes, layouts, precisions and
betas of the same ranges.  prepare() makes what such a program holds before
the call, run() is one call, work() the bytes and operations the call cannot
do without, exact() the same result in 64 bits.
"""
import math
import random

import numpy as np
import torch

import hiperml_amd as hml

DEV = "cuda"


def listed():
    return [
        # One small layer or update step: the call's own latency, not its bytes.
        dict(name="gemv_small", op="gemv", m=1000, n=300, trans=False, beta=0.0),
        # The large square product y = A x of the headline sweep, 1 GiB of A.
        dict(name="gemv_square", op="gemv", m=16384, n=16384, trans=False, beta=0.0),
        # y = A^T x of a tall panel: column sums over a million observations.
        dict(name="gemv_tall_t", op="gemv", m=1048576, n=64, trans=True, beta=0.0),
        # The reference app's flow: host arrays in, result copied back, all of it counted.
        dict(name="gemm_host", op="host", m=2048, n=16, k=2048, beta=0.0),
        # The headline sweep's widest memory- / FP32-balanced shape.
        dict(name="gemm_skinny", op="gemm", m=8192, n=64, k=8192, order="row", ta=False, tb=False,
             beta=0.0),
        # A million rows by a few dozen features (the extents the reference's
        # online tuning runs over: M = 10^6, K <= 96, N <= 96): projection of a
        # tall data set, where C is as large as A.
        dict(name="gemm_tall", op="gemm", m=1000000, n=32, k=48, order="row", ta=False, tb=False,
             beta=0.0),
        # Gradient-like A^T B with odd extents, accumulated into C.
        dict(name="gemm_trans_odd", op="gemm", m=5003, n=24, k=9001, order="row", ta=True, tb=False,
             beta=0.5),
        # An ordinary dense product through the general call: FP32 tiles, odd extents.
        dict(name="gemm_dense", op="gemm", m=3001, n=2047, k=2500, order="row", ta=False, tb=False,
             beta=0.0),
        # Large dense product at FP32-level error on the 16-bit matrix cores.
        dict(name="dense_f16x3", op="dense", m=8192, n=8192, k=8192, precision="f16x3",
             loguniform=False, ta=False, tb=False, beta=0.0),
        # Outer-product-like dense update (short K), writes as large as its products.
        dict(name="dense_bf16x3_k256", op="dense", m=8192, n=8192, k=256, precision="bf16x3",
             loguniform=True, ta=False, tb=False, beta=0.0),
        # 512 uneven skinny problems in one captured launch, replayed.
        dict(name="grouped_512", op="grouped", count=512, shapes=0),
        # Assignment step of one Lloyd iteration over 16M points.
        dict(name="kmeans", op="kmeans", rows=1 << 24, dims=32, clusters=64),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """One more case: each kind of call above over its whole range."""
    op = rng.choice(["gemv", "gemv", "gemm", "gemm", "gemm", "tall", "square", "dense", "dense",
                     "grouped", "kmeans", "kmeans", "host"])
    beta = rng.choice([0.0, 0.0, 0.0, 0.5, 1.0])
    if op == "gemv":
        while True:
            m, n = _log(rng, 128, 1 << 20), _log(rng, 32, 16384)
            if 1 << 16 <= m * n <= 1 << 28:
                return dict(op="gemv", m=m, n=n, trans=rng.random() < 0.5, beta=beta)
    if op == "gemm":
        while True:
            m, k, n = _log(rng, 256, 65536), _log(rng, 64, 16384), rng.randint(2, 128)
            if m * k <= 1 << 27:
                return dict(op="gemm", m=m, n=n, k=k, order=rng.choice(["row", "row", "col"]),
                            ta=rng.random() < 0.4, tb=rng.random() < 0.3, beta=beta)
    if op == "tall":
        return dict(op="gemm", m=_log(rng, 100000, 1000000), n=rng.randint(8, 96),
                    k=rng.randint(2, 96), order="row", ta=False, tb=False, beta=beta)
    if op == "square":
        return dict(op="gemm", m=_log(rng, 512, 6000), n=_log(rng, 512, 6000),
                    k=_log(rng, 256, 4096), order="row", ta=rng.random() < 0.3,
                    tb=rng.random() < 0.3, beta=beta)
    if op == "dense":
        return dict(op="dense", m=_log(rng, 1024, 8192), n=_log(rng, 1024, 8192),
                    k=_log(rng, 128, 8192),
                    precision=rng.choice(["fp32", "bf16x3", "bf16x6", "f16x3", "f16x3"]),
                    loguniform=rng.random() < 0.5, ta=rng.random() < 0.3, tb=rng.random() < 0.3,
                    beta=beta)
    if op == "grouped":
        return dict(op="grouped", count=_log(rng, 16, 320), shapes=rng.randint(1, 1 << 20))
    if op == "kmeans":
        while True:
            rows, dims, cl = _log(rng, 1 << 15, 1 << 24), rng.randint(4, 64), _log(rng, 4, 512)
            if rows * dims * cl <= 1 << 36:
                return dict(op="kmeans", rows=rows, dims=dims, clusters=cl)
    return dict(op="host", m=_log(rng, 256, 16384), n=rng.randint(1, 64), k=_log(rng, 64, 2048),
                beta=beta)


def _group_shapes(case):
    """(M, N, K) per problem: M log-uniform [64, 65536], K log-uniform [64, 4096], N 1..64."""
    rng = random.Random(case["shapes"])
    return [(_log(rng, 64, 65536), rng.randint(1, 64), _log(rng, 64, 4096))
            for _ in range(case["count"])]


def _up64(n):
    return -(-n // 64) * 64


def _uniform(g, *shape):
    return torch.empty(shape, device=DEV).uniform_(-1.0, 1.0, generator=g)


def _loguniform(g, *shape):
    """Magnitudes log-uniform in [1e-3, 1e3], random sign."""
    t = torch.empty(shape, device=DEV).uniform_(-math.log(1e3), math.log(1e3), generator=g).exp_()
    s = torch.empty(shape, device=DEV).uniform_(-1.0, 1.0, generator=g)
    return t.copysign_(s)


def _stored(order, trans, rows, cols):
    """Extents (as a C-contiguous tensor) of op(X) = rows x cols stored in `order`."""
    return (cols, rows) if trans != (order == "col") else (rows, cols)


def prepare(case, seed):
    op = case["op"]
    s = dict(case=case)
    if op == "host":
        rng = np.random.default_rng(seed)
        m, n, k = case["m"], case["n"], case["k"]
        s["a"] = rng.uniform(-1.0, 1.0, (m, k)).astype(np.float32)
        s["b"] = rng.uniform(-1.0, 1.0, (k, n)).astype(np.float32)
        s["c"] = rng.uniform(-1.0, 1.0, (m, n)).astype(np.float32)
        return s
    g = torch.Generator(device=DEV).manual_seed(seed)
    if op == "gemv":
        m, n = case["m"], case["n"]
        s["a"] = _uniform(g, m, n)
        s["x"] = _uniform(g, m if case["trans"] else n)
        s["y"] = _uniform(g, n if case["trans"] else m)
    elif op in ("gemm", "dense"):
        m, n, k, order = case["m"], case["n"], case["k"], case.get("order", "row")
        fill = _loguniform if case.get("loguniform") else _uniform
        s["a"] = fill(g, *_stored(order, case["ta"], m, k))
        s["b"] = fill(g, *_stored(order, case["tb"], k, n))
        s["c"] = fill(g, *_stored(order, False, m, n))
    elif op == "grouped":
        shapes = _group_shapes(case)
        s["a"] = _uniform(g, sum(_up64(m * k) for m, n, k in shapes))
        s["b"] = _uniform(g, sum(_up64(k * n) for m, n, k in shapes))
        s["c"] = torch.zeros(sum(_up64(m * n) for m, n, k in shapes), device=DEV)
        problems, a, b, c = [], s["a"].data_ptr(), s["b"].data_ptr(), s["c"].data_ptr()
        for m, n, k in shapes:
            problems.append((m, n, k, a, b, c))
            a += 4 * _up64(m * k)
            b += 4 * _up64(k * n)
            c += 4 * _up64(m * n)
        s["plan"] = hml.GroupedPlan(problems)
    elif op == "kmeans":
        r, d, cl = case["rows"], case["dims"], case["clusters"]
        centres = _uniform(g, cl, d)
        pick = torch.randint(0, cl, (r,), device=DEV, generator=g, dtype=torch.int32)
        rows = torch.empty(r, d, device=DEV).normal_(0.0, 0.25, generator=g)
        for at in range(0, r, 1 << 21):
            rows[at:at + (1 << 21)] += centres[pick[at:at + (1 << 21)]]
        # centroids a few Lloyd steps in: near the true centres, not on them
        s["rows"] = rows
        s["ctrds"] = centres + torch.empty(cl, d, device=DEV).normal_(0.0, 0.02, generator=g)
        s["assign"] = torch.zeros(r, dtype=torch.int32, device=DEV)
    else:
        raise ValueError(op)
    return s


def run(s):
    case = s["case"]
    op = case["op"]
    if op == "host":
        return hml.sgemm(s["c"], s["a"], s["b"], 1.0, case["beta"])
    if op == "grouped":
        s["plan"].run(graph=True, stream=torch.cuda.current_stream().cuda_stream)
        return s["c"]
    stream = torch.cuda.current_stream().cuda_stream
    if op == "gemv":
        hml.sgemv_ex(case["m"], case["n"], s["a"].data_ptr(), s["x"].data_ptr(), s["y"].data_ptr(),
                     1.0, case["beta"], trans=case["trans"], stream=stream)
        return s["y"]
    if op == "gemm":
        hml.sgemm_ex(case["m"], case["n"], case["k"], s["a"].data_ptr(), s["b"].data_ptr(),
                     s["c"].data_ptr(), 1.0, case["beta"], order=case["order"], transA=case["ta"],
                     transB=case["tb"], stream=stream)
        return s["c"]
    if op == "dense":
        hml.sgemm_dense(case["m"], case["n"], case["k"], s["a"].data_ptr(), s["b"].data_ptr(),
                        s["c"].data_ptr(), 1.0, case["beta"], precision=case["precision"],
                        transA=case["ta"], transB=case["tb"], stream=stream)
        return s["c"]
    hml.kmeans_assign(s["rows"].data_ptr(), s["ctrds"].data_ptr(), s["assign"].data_ptr(),
                      case["rows"], case["dims"], case["clusters"], stream=stream)
    return s["assign"]


def work(case):
    op = case["op"]
    if op == "grouped":
        shapes = _group_shapes(case)
        return {"bytes": sum(4.0 * (m * k + k * n + m * n) for m, n, k in shapes),
                "flops": sum(2.0 * m * n * k for m, n, k in shapes)}
    if op == "kmeans":
        r, d, cl = case["rows"], case["dims"], case["clusters"]
        return {"bytes": 4.0 * (r * d + cl * d + r), "flops": 2.0 * r * d * cl}
    m, n = case["m"], case["n"]
    reads_c = 1 if case["beta"] != 0.0 or op == "host" else 0
    if op == "gemv":
        out = n if case["trans"] else m
        return {"bytes": 4.0 * (m * n + m + n + reads_c * out), "flops": 2.0 * m * n}
    k = case["k"]
    return {"bytes": 4.0 * (m * k + k * n + (1 + reads_c) * m * n), "flops": 2.0 * m * n * k}


def exact(case, seed):
    op = case["op"]
    if op == "kmeans":
        return None  # whole numbers
    s = prepare(case, seed)
    if op == "host":
        return case["beta"] * s["c"].astype(np.float64) + s["a"].astype(np.float64) @ s["b"].astype(np.float64)
    if op == "grouped":
        out = torch.zeros(s["c"].numel(), dtype=torch.float64, device=DEV)
        a = b = c = 0
        for m, n, k in _group_shapes(case):
            out[c:c + m * n] = (s["a"][a:a + m * k].view(m, k).double()
                                @ s["b"][b:b + k * n].view(k, n).double()).reshape(-1)
            a += _up64(m * k)
            b += _up64(k * n)
            c += _up64(m * n)
        return out
    a = s["a"].double()
    if op == "gemv":
        return (a.t() if case["trans"] else a) @ s["x"].double() + case["beta"] * s["y"].double()
    b, order = s["b"].double(), case.get("order", "row")
    at = a.t() if case["ta"] != (order == "col") else a
    bt = b.t() if case["tb"] != (order == "col") else b
    c = at @ bt
    if order == "col":
        c = c.t().contiguous()
    return c + case["beta"] * s["c"].double() if case["beta"] != 0.0 else c
