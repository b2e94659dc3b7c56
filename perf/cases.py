"""Performance cases of the BLAS path: the calls a program makes through the
Python entry points (mtm, mtv, vtm, dot_prod, outer_prod, transpose, grouped
plans, the live server), at the sizes of the repository's benchmark, sweeps
and tests.

listed() names twelve of them, draw() gives more of the same ranges; a case is
a dict of plain values.  prepare() makes what a program holds before the call
(operands on the GPU, a grouped plan, an open server), run() makes one call,
exact() gives the same outputs from torch's FP64 operations and work() the
bytes and operations that the call cannot do without.
"""
import math

import numpy as np
import torch

from __graft_entry__ import load_package

omb = load_package()

MODES = {"plain": omb.PLAIN_F32, "bf16": omb.SPLIT_BF16, "fp16": omb.SPLIT_FP16}


def listed():
    return [
        # An inner product at the top of the reference dot driver's sweep
        # (2 .. 2^20), odd length: latency and two dependent reductions.
        {"name": "dot_1m", "op": "dot", "n": 1000003},
        # One small ragged product as the size sweep and the test suites make
        # them, column-major like the reference's default: launch latency.
        {"name": "mtm_small_ragged", "op": "mtm", "mode": "plain", "M": 200, "N": 150, "K": 301,
         "a": "col", "b": "col", "c": "col", "pad": 0},
        # The ordinary product: 1024^3 row-major, the benchmark's configuration 1.
        {"name": "mtm_1024", "op": "mtm", "mode": "plain", "M": 1024, "N": 1024, "K": 1024,
         "a": "row", "b": "row", "c": "row", "pad": 0},
        # The full-size plain product of the benchmark.
        {"name": "mtm_8192", "op": "mtm", "mode": "plain", "M": 8192, "N": 8192, "K": 8192,
         "a": "row", "b": "row", "c": "row", "pad": 0},
        # The benchmark's headline: 8192^3 as 6 split-BF16 products.
        {"name": "mtm_8192_bf16", "op": "mtm", "mode": "bf16", "M": 8192, "N": 8192, "K": 8192,
         "a": "row", "b": "row", "c": "row", "pad": 0},
        # A mid-size ragged product in the scaled split-FP16 mode, A B^T
        # (B column-major).
        {"name": "mtm_ragged_fp16", "op": "mtm", "mode": "fp16", "M": 2500, "N": 3001, "K": 1777,
         "a": "row", "b": "col", "c": "row", "pad": 0},
        # The benchmark's matrix-vector product, row-major.
        {"name": "mtv_16384", "op": "mtv", "M": 16384, "N": 16384, "a": "row", "pad": 0},
        # The transposed direction, c += A^T b, odd extents.
        {"name": "vtm_ragged", "op": "vtm", "M": 6001, "N": 9003, "a": "row", "pad": 0},
        # Rank-1 update inside the reference outer driver's sweep (.. 16382).
        {"name": "outer_ragged", "op": "outer", "M": 10007, "N": 8191, "c": "row", "pad": 0},
        # Out-of-place transpose of a row-major matrix, odd extents.
        {"name": "transpose_ragged", "op": "transpose", "M": 8001, "N": 12007, "a": "row",
         "c": "row", "pad": 0},
        # The benchmark's grouped batch: 4096 GEMMs (extents log-uniform on
        # [16, 512]) and 4096 GEMVs (on [64, 4096]) in one launch.
        {"name": "grouped_4096", "op": "grouped", "mode": "plain", "gemms": 4096, "gemvs": 4096,
         "gemm_hi": 512, "gemv_hi": 4096, "shapes": 3},
        # The serving mix (half GEMM, 0.3 GEMV, 0.2 dot, split-BF16) as one
        # burst through the live server: submit all, wait for all.
        {"name": "serve_burst", "op": "serve", "mode": "bf16", "count": 192, "shapes": 4},
    ]


def _log_int(rng, lo, hi):
    return max(lo, min(hi, int(math.exp(rng.uniform(math.log(lo), math.log(hi + 1))))))


def draw(rng):
    order = lambda: rng.choice(["row", "col"])  # noqa: E731
    pad = lambda: rng.choice([0, 0, 0, 4, 5])  # noqa: E731
    op = rng.choice(["mtm", "mtm", "mtm", "mtm", "mtv", "vtm", "dot", "outer", "transpose",
                     "grouped", "serve"])
    if op == "mtm":
        return {"op": op, "mode": rng.choice(["plain", "plain", "bf16", "fp16"]),
                "M": _log_int(rng, 32, 6144), "N": _log_int(rng, 32, 6144),
                "K": _log_int(rng, 32, 6144), "a": order(), "b": order(), "c": order(),
                "pad": pad()}
    if op in ("mtv", "vtm"):
        return {"op": op, "M": _log_int(rng, 64, 16384), "N": _log_int(rng, 64, 16384),
                "a": order(), "pad": pad()}
    if op == "dot":
        return {"op": op, "n": _log_int(rng, 1 << 10, 1 << 28)}
    if op == "outer":
        return {"op": op, "M": _log_int(rng, 32, 16382), "N": _log_int(rng, 32, 16382),
                "c": order(), "pad": pad()}
    if op == "transpose":
        return {"op": op, "M": _log_int(rng, 32, 16384), "N": _log_int(rng, 32, 16384),
                "a": order(), "c": order(), "pad": pad()}
    if op == "grouped":
        return {"op": op, "mode": rng.choice(["plain", "plain", "bf16", "fp16"]),
                "gemms": _log_int(rng, 64, 2048), "gemvs": _log_int(rng, 64, 2048),
                "gemm_hi": 512, "gemv_hi": 4096, "shapes": rng.randrange(1 << 20)}
    return {"op": op, "mode": rng.choice(["plain", "bf16"]), "count": _log_int(rng, 32, 160),
            "shapes": rng.randrange(1 << 20)}


# ------------------------------------------------------------------ inputs --
def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(seed)


def _uniform(n, gen):
    """n floats uniform on [-1, 1), the distribution of every configuration."""
    return torch.rand(n, dtype=torch.float32, device="cuda", generator=gen).mul_(2.0).sub_(1.0)


def _matrix(rows, cols, order, pad, gen):
    """A rows x cols matrix in row- or column-major order; pad > 0: a view
    whose leading dimension is that much larger than its extent."""
    if order == "row":
        return _uniform(rows * (cols + pad), gen).view(rows, cols + pad)[:, :cols]
    return _uniform(cols * (rows + pad), gen).view(cols, rows + pad)[:, :rows].t()


def _mtm_operands(case, seed):
    g = _gen(seed)
    return (_matrix(case["M"], case["K"], case["a"], case["pad"], g),
            _matrix(case["K"], case["N"], case["b"], case["pad"], g),
            _matrix(case["M"], case["N"], case["c"], case["pad"], g))


def _vec_operands(case, seed):
    """A and b, c of mtv (c: M) or vtm (c: N)."""
    g = _gen(seed)
    a = _matrix(case["M"], case["N"], case["a"], case["pad"], g)
    nb, nc = (case["N"], case["M"]) if case["op"] == "mtv" else (case["M"], case["N"])
    return a, _uniform(nb, g), _uniform(nc, g)


def _outer_operands(case, seed):
    g = _gen(seed)
    return (_uniform(case["M"], g), _uniform(case["N"], g),
            _matrix(case["M"], case["N"], case["c"], case["pad"], g))


def _grouped_shapes(case):
    rng = np.random.default_rng(case["shapes"])
    gs = np.stack([omb.log_uniform_ints(rng, 16, case["gemm_hi"], case["gemms"])
                   for _ in range(3)], 1)
    vs = np.stack([omb.log_uniform_ints(rng, 64, case["gemv_hi"], case["gemvs"])
                   for _ in range(2)], 1)
    return [tuple(map(int, r)) for r in gs], [tuple(map(int, r)) for r in vs]


def _pools(sizes_in, sizes_out, seed):
    """One pool of inputs and one of outputs, with every operand's offset in
    floats (each on a 256-byte boundary)."""
    def offsets(sizes):
        padded = np.asarray([-(-s // 64) * 64 for s in sizes], dtype=np.int64)
        return [int(v) for v in np.cumsum(padded) - padded], int(padded.sum())
    oin, nin = offsets(sizes_in)
    oout, nout = offsets(sizes_out)
    pin = _uniform(nin, _gen(seed))
    pout = torch.zeros(nout, dtype=torch.float32, device="cuda")
    return pin, oin, pout, oout


def _grouped_operands(case, seed):
    gs, vs = _grouped_shapes(case)
    sin = [s for m, n, k in gs for s in (m * k, k * n)] + [s for m, n in vs for s in (m * n, n)]
    sout = [m * n for m, n, k in gs] + [m for m, n in vs]
    return (gs, vs) + _pools(sin, sout, seed)


def _serve_trace(case):
    return [(k, m, n, kk) for k, m, n, kk, _ in
            omb.serving_trace(case["count"], 1.0, seed=case["shapes"])]


def _serve_operands(case, seed):
    reqs = _serve_trace(case)
    sin, sout = [], []
    for kind, m, n, k in reqs:
        if kind == omb.REQ_GEMM:
            sin += [m * k, k * n]
            sout.append(m * n)
        elif kind == omb.REQ_GEMV:
            sin += [m * n, n]
            sout.append(m)
        else:
            sin += [n, n]
            sout.append(1)
    return (reqs,) + _pools(sin, sout, seed)


# -------------------------------------------------------------- the passes --
def prepare(case, seed):
    op = case["op"]
    if op == "mtm":
        a, b, c = _mtm_operands(case, seed)
        return {"op": op, "a": a, "b": b, "c": c, "mode": MODES[case["mode"]]}
    if op in ("mtv", "vtm"):
        a, b, c = _vec_operands(case, seed)
        return {"op": op, "a": a, "b": b, "c": c}
    if op == "dot":
        g = _gen(seed)
        return {"op": op, "a": _uniform(case["n"], g), "b": _uniform(case["n"], g),
                "c": torch.zeros(1, device="cuda")}
    if op == "outer":
        a, b, c = _outer_operands(case, seed)
        return {"op": op, "a": a, "b": b, "c": c}
    if op == "transpose":
        a = _matrix(case["M"], case["N"], case["a"], case["pad"], _gen(seed))
        c = _matrix(case["N"], case["M"], case["c"], case["pad"], _gen(seed + 1)).zero_()
        return {"op": op, "a": a, "c": c}
    if op == "grouped":
        gs, vs, pin, oin, pout, oout = _grouped_operands(case, seed)
        i, o = pin.data_ptr(), pout.data_ptr()
        gemms = [(m, n, k, i + 4 * oin[2 * q], k, i + 4 * oin[2 * q + 1], n, o + 4 * oout[q], n,
                  1.0, 0.0) for q, (m, n, k) in enumerate(gs)]
        g = len(gs)
        gemvs = [(m, n, i + 4 * oin[2 * (g + q)], n, i + 4 * oin[2 * (g + q) + 1],
                  o + 4 * oout[g + q], 1.0, 0.0) for q, (m, n) in enumerate(vs)]
        return {"op": op, "in": pin, "out": pout,
                "plan": omb.GroupPlan(gemms, gemvs, MODES[case["mode"]])}
    reqs, pin, oin, pout, oout = _serve_operands(case, seed)
    i, o = pin.data_ptr(), pout.data_ptr()
    requests = [omb.Request(kind, MODES[case["mode"]], m, n, k, 0.0, i + 4 * oin[2 * q],
                            i + 4 * oin[2 * q + 1], o + 4 * oout[q], 0)
                for q, (kind, m, n, k) in enumerate(reqs)]
    most = max(omb.serve_request_bytes(r) for r in requests)
    torch.cuda.synchronize()  # the server's streams do not wait for torch's
    return {"op": op, "in": pin, "out": pout, "requests": requests,
            "server": omb.Server(slots=8, max_request_bytes=max(most, 1 << 20), spin_poll=False)}


def run(state):
    op = state["op"]
    if op == "mtm":
        omb.mtm(state["c"], state["a"], state["b"], mode=state["mode"])()
        return state["c"]
    if op == "mtv":
        omb.mtv(state["c"], state["a"], state["b"])()
        return state["c"]
    if op == "vtm":
        omb.vtm(state["c"], state["a"], state["b"])()
        return state["c"]
    if op == "dot":
        omb.dot_prod(state["c"], state["a"], state["b"])()
        return state["c"]
    if op == "outer":
        omb.outer_prod(state["c"], state["a"], state["b"])()
        return state["c"]
    if op == "transpose":
        omb.transpose(state["c"], state["a"])()
        return state["c"]
    if op == "grouped":
        state["plan"].launch()
        return state["out"]
    server = state["server"]
    for t in [server.submit(r) for r in state["requests"]]:
        res = server.wait(t)
        if res["status"] != omb.OK:
            raise RuntimeError("request refused: status %d" % res["status"])
    return state["out"]


def exact(case, seed):
    op = case["op"]
    if op == "mtm":
        a, b, c = _mtm_operands(case, seed)
        return c.double() + a.double() @ b.double()
    if op in ("mtv", "vtm"):
        a, b, c = _vec_operands(case, seed)
        # column-major A: mtv accumulates; row-major A: vtm does
        add = (case["a"] == "col") == (op == "mtv")
        p = (a if op == "mtv" else a.t()).double() @ b.double()
        return c.double() + p if add else p
    if op == "dot":
        g = _gen(seed)
        a, b = _uniform(case["n"], g), _uniform(case["n"], g)
        return (a.double() * b.double()).sum().view(1)
    if op == "outer":
        a, b, c = _outer_operands(case, seed)
        return c.double() + torch.outer(a.double(), b.double())
    if op == "transpose":
        return _matrix(case["M"], case["N"], case["a"], case["pad"], _gen(seed)).double().t()
    if op == "grouped":
        gs, vs, pin, oin, pout, oout = _grouped_operands(case, seed)
        items = [(m, n, k) for m, n, k in gs] + [(m, 1, n) for m, n in vs]
    else:
        reqs, pin, oin, pout, oout = _serve_operands(case, seed)
        items = [(m, n, k) if kind == omb.REQ_GEMM else
                 ((m, 1, n) if kind == omb.REQ_GEMV else (1, 1, n)) for kind, m, n, k in reqs]
    out = torch.zeros(pout.numel(), dtype=torch.float64, device="cuda")
    for q, (m, n, k) in enumerate(items):
        a = pin[oin[2 * q]:oin[2 * q] + m * k].view(m, k).double()
        b = pin[oin[2 * q + 1]:oin[2 * q + 1] + k * n].view(k, n).double()
        out[oout[q]:oout[q] + m * n] = (a @ b).reshape(-1)
    return out


def work(case):
    """Inputs read once, outputs written once (and read first where the call
    accumulates); one multiply and one add per product."""
    op = case["op"]
    if op == "mtm":
        m, n, k = case["M"], case["N"], case["K"]
        return {"bytes": 4.0 * (m * k + k * n + 2 * m * n), "flops": 2.0 * m * n * k}
    if op in ("mtv", "vtm"):
        m, n = case["M"], case["N"]
        out = m if op == "mtv" else n
        add = (case["a"] == "col") == (op == "mtv")
        return {"bytes": 4.0 * (m * n + m + n + (out if add else 0)), "flops": 2.0 * m * n}
    if op == "dot":
        return {"bytes": 8.0 * case["n"] + 4.0, "flops": 2.0 * case["n"]}
    if op == "outer":
        m, n = case["M"], case["N"]
        return {"bytes": 8.0 * m * n + 4.0 * (m + n), "flops": 2.0 * m * n}
    if op == "transpose":
        return {"bytes": 8.0 * case["M"] * case["N"], "flops": 0.0}
    if op == "grouped":
        gs, vs = _grouped_shapes(case)
        kinds = [(omb.REQ_GEMM, m, n, k) for m, n, k in gs] + [(omb.REQ_GEMV, m, n, 0) for m, n in vs]
    else:
        kinds = _serve_trace(case)
    return {"bytes": float(sum(omb.request_bytes(*r) for r in kinds)),
            "flops": float(sum(omb.request_flop(*r) for r in kinds))}
