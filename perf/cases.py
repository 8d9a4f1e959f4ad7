"""The workloads this engine's speed is measured on.

A user of the engine either hands it a circuit (`qflex.simulate`) or calls
its primitives through `qflex_amd.capi`: pairwise contractions read in the
tensors' stored index orders, plain matrix products, index permutations,
matrix-vector closings, grouped products of many slices, and the cost
model's training step and scoring.  Each family is one `op` below.

Tensors are complex64 torch tensors on the GPU; the C-ABI takes their
addresses.  Every state of this process shares one context, as one program
does.
"""
import math

import numpy as np
import torch

from qflex_amd import capi, circuits

_CTX = None


def _context():
    global _CTX
    if _CTX is None:
        _CTX = capi.Context(0)
    return _CTX


class _Buffer:
    """A torch tensor as the capi's device buffer."""

    def __init__(self, tensor):
        self.tensor = tensor
        self.ptr = tensor.data_ptr()
        self.nbytes = tensor.numel() * tensor.element_size()


def listed():
    return [
        # One amplitude of a small rectangular circuit: the smallest call a
        # user makes, all parsing, network build and launch latency.
        {"name": "amplitude_4x4_d16", "op": "simulate", "rows": 4, "cols": 4, "depth": 16,
         "open": 0, "ordering": "snake", "precision": "fp32"},
        # The benchmark workload: 7x7, depth 1+32+1, 256 slices, 64 amplitudes.
        {"name": "amplitudes_7x7_d32", "op": "simulate", "rows": 7, "cols": 7, "depth": 32,
         "open": 6, "ordering": "corner", "precision": "split_fp16"},
        # The merge of two patches over three bonds of 16: the largest
        # single contraction of the 7x7 job.
        {"name": "merge_patches", "op": "contract", "precision": "split_fp16", "m": 4096,
         "n": 4096, "k": 4096, "inner": "k"},
        # A patch grown by one interior site (two bonds contracted, two new).
        {"name": "expand_site", "op": "contract", "precision": "split_fp16", "m": 65536,
         "n": 256, "k": 256, "inner": "m"},
        # The same growth in the engine's default precision, on a smaller patch.
        {"name": "expand_site_fp32", "op": "contract", "precision": "fp32", "m": 16384, "n": 256,
         "k": 256, "inner": "m"},
        # A patch grown by a boundary site (one bond contracted, one new).
        {"name": "expand_boundary", "op": "contract", "precision": "split_fp16", "m": 1 << 20,
         "n": 16, "k": 16, "inner": "m"},
        # A product whose dimensions are no powers of two (cuts restricted to
        # some of their values), odd in every dimension.
        {"name": "product_odd", "op": "product", "precision": "split_fp16", "m": 6145, "n": 515,
         "k": 333},
        # Reorder of a 2^25-element bond-16 tensor (256 MiB).
        {"name": "reorder_bond16", "op": "reorder", "dims": "16,16,2,16,16,16,16",
         "perm": "3,0,6,2,5,1,4"},
        # Reorder with axes narrowed to some of a cut's values.
        {"name": "reorder_narrowed", "op": "reorder", "dims": "16,11,16,3,16,16,5",
         "perm": "4,1,6,0,3,2,5"},
        # A patch closed by a tensor with no other open index.
        {"name": "close_vector", "op": "vector", "trans": 1, "m": 4096, "k": 4096},
        # The same step of many slices, uneven sizes, in one call.
        {"name": "grouped_slices", "op": "grouped", "precision": "split_fp16", "count": 192,
         "m": 512, "n": 128, "k": 64},
        # One training step of the cost model (its default minibatch).
        {"name": "cost_model_step", "op": "train", "batch": 512},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    op = rng.choice(["simulate", "contract", "contract", "product", "product", "reorder",
                     "reorder", "vector", "grouped", "train", "score"])
    if op == "simulate":
        return {"op": op, "rows": rng.randint(3, 6), "cols": rng.randint(3, 5),
                "depth": rng.choice([8, 16, 17, 23, 24, 32]), "open": rng.randint(0, 3),
                "ordering": "snake", "precision": rng.choice(["fp32", "split_fp16",
                                                              "split_bf16x3"])}
    if op == "contract":
        while True:
            m, n, k = (1 << rng.randint(4, 20), 1 << rng.randint(2, 12), 1 << rng.randint(2, 12))
            if 2 ** 16 <= m * n * k <= 2 ** 36 and max(m * k, k * n, m * n) <= 2 ** 26:
                return {"op": op, "precision": rng.choice(["fp32", "split_fp16", "split_fp16",
                                                           "split_bf16x3"]),
                        "m": m, "n": n, "k": k, "inner": rng.choice(["m", "k"])}
    if op == "product":
        while True:
            m, n, k = _log(rng, 16, 65536), _log(rng, 2, 4096), _log(rng, 2, 4096)
            if 2 ** 14 <= m * n * k <= 2 ** 34 and max(m * k, k * n, m * n) <= 2 ** 25:
                return {"op": op, "precision": rng.choice(["fp32", "split_fp16", "split_fp16",
                                                           "split_bf16x3"]),
                        "m": m, "n": n, "k": k}
    if op == "reorder":
        narrowed = rng.random() < 0.5
        target = rng.uniform(12, 25)
        dims = []
        while sum(math.log2(d) for d in dims) < target:
            dims.append(rng.choice([2, 3, 4, 5, 7, 8, 11, 16] if narrowed else [2, 4, 8, 16]))
        while sum(math.log2(d) for d in dims) > 25.5:
            dims.pop()
        perm = list(range(len(dims)))
        while perm == sorted(perm):
            rng.shuffle(perm)
        return {"op": op, "dims": ",".join(map(str, dims)), "perm": ",".join(map(str, perm))}
    if op == "vector":
        while True:
            m, k = _log(rng, 16, 1 << 20), _log(rng, 4, 65536)
            if 2 ** 12 <= m * k <= 2 ** 26:
                return {"op": op, "trans": rng.randint(0, 1), "m": m, "k": k}
    if op == "grouped":
        return {"op": op, "precision": rng.choice(["split_fp16", "split_bf16x3", "fp32"]),
                "count": _log(rng, 8, 256), "m": _log(rng, 64, 1024), "n": _log(rng, 2, 256),
                "k": _log(rng, 2, 256)}
    if op == "train":
        return {"op": op, "batch": _log(rng, 32, 4096)}
    return {"op": op, "batch": _log(rng, 16, 65536)}


# ------------------------------------------------------------------ inputs

def _generator(seed, salt=0):
    return torch.Generator(device="cuda").manual_seed(1000003 * int(seed) + salt)


def _complex(gen, *shape):
    return torch.view_as_complex(torch.randn(*shape, 2, device="cuda", generator=gen))


def _digits(size):
    """A power of two as bond dimensions of 16 after one smaller remainder."""
    dims = []
    while size > 1:
        dims.insert(0, min(size, 16))
        size //= dims[0]
    return dims or [1]


def _layout(case):
    """Stored orders of a contraction: dims of A and B and, for each matrix
    dimension, its tensor axes (most significant first).  A is a patch whose
    contracted bonds lie between its other ones, the innermost axis on the
    side `inner` names; B is a site or patch stored (common, right)."""
    left = [("l", i, d) for i, d in enumerate(_digits(case["m"]))]
    common = [("c", i, d) for i, d in enumerate(_digits(case["k"]))]
    right = [("r", i, d) for i, d in enumerate(_digits(case["n"]))]
    last = left.pop() if case["inner"] == "m" else common.pop()
    a_axes = []
    l, c = list(left), list(common)
    while l or c:
        if l:
            a_axes.append(l.pop())
        if c:
            a_axes.append(c.pop(0))
    a_axes.append(last)
    (left if case["inner"] == "m" else common).append(last)
    b_axes = common[::-1] + right
    find = lambda axes, group: [axes.index(x) for x in group]
    return ([x[2] for x in a_axes], find(a_axes, left), find(a_axes, common),
            [x[2] for x in b_axes], find(b_axes, common), find(b_axes, right))


def _group_shapes(case):
    return [(max(1, case["m"] >> (i % 3)), case["n"], case["k"] * (1 + i % 2))
            for i in range(case["count"])]


def _group_offsets(case):
    """Element offsets of each product's A, B and C in one buffer per operand,
    each product starting at an even element (16 bytes)."""
    at, out = [0, 0, 0], []
    for m, n, k in _group_shapes(case):
        out.append(tuple(at))
        for j, size in enumerate((m * k, k * n, m * n)):
            at[j] += size + size % 2
    return out, at


def _circuit(case, seed):
    return circuits.random_circuit(case["rows"], case["cols"], case["depth"], int(seed))


def _region(case):
    last = case["rows"] - 1
    return [(last, j) for j in range(case["open"])]


def _final_state(case, seed):
    if case["ordering"] == "corner":
        return ""
    rng = np.random.default_rng(int(seed) + 17)
    bits = [str(b) for b in rng.integers(0, 2, case["rows"] * case["cols"])]
    for i, j in _region(case):
        bits[i * case["cols"] + j] = "x"
    return "".join(bits)


def _options(case, seed):
    rows, cols = case["rows"], case["cols"]
    order = (circuits.corner_inward_7x7() if case["ordering"] == "corner"
             else circuits.snake_ordering(rows, cols, final_region=_region(case)))
    return {"circuit": _circuit(case, seed).splitlines(), "ordering": order.splitlines(),
            "grid": circuits.grid_text(rows, cols).splitlines(),
            "initial_state": "0" * (rows * cols), "final_state": _final_state(case, seed),
            "memory_limit": "200GB", "precision": case["precision"]}


def _network(case, seed):
    """Parameters, features, targets and Adam moments some steps into training."""
    gen = _generator(seed)
    n_in, hid = capi.MLP_IN, capi.MLP_HIDDEN
    rand = lambda *s: torch.randn(*s, device="cuda", generator=gen)
    params = torch.cat([(rand(n_in, hid) * math.sqrt(2 / n_in)).reshape(-1), 0.1 * rand(hid),
                        (rand(hid, hid) * math.sqrt(2 / hid)).reshape(-1), 0.1 * rand(hid),
                        rand(hid) * math.sqrt(1 / hid), 0.1 * rand(1)])
    X = rand(case["batch"], n_in)
    target = torch.tanh(X[:, :8].sum(1) / 3) + 0.1 * rand(case["batch"])
    m = 0.01 * rand(capi.MLP_PARAMS)
    v = (0.01 * rand(capi.MLP_PARAMS)) ** 2 + 1e-5
    return params, X, target, m, v


_ADAM = {"step": 101, "lr": 1e-3, "beta1": 0.9, "beta2": 0.999, "eps": 1e-8}


def prepare(case, seed):
    op = case["op"]
    state = {"op": op}
    if op == "simulate":
        from qflex_amd import qflex
        state.update(simulate=qflex.simulate, options=_options(case, seed))
        return state
    state["ctx"] = _context()
    gen = _generator(seed)
    empty = lambda *s, dtype=torch.complex64: torch.zeros(*s, dtype=dtype, device="cuda")
    if op == "contract":
        a_dims, a_left, a_common, b_dims, b_common, b_right = _layout(case)
        state["precision"] = capi.PRECISIONS[case["precision"]]
        state["A"], state["B"] = (_Buffer(_complex(gen, *d)) for d in (a_dims, b_dims))
        state["maps"] = (capi.index_map(a_dims, a_left), capi.index_map(a_dims, a_common),
                         capi.index_map(b_dims, b_common), capi.index_map(b_dims, b_right))
        state["a_reorder"], state["b_reorder"] = ((a_dims, a_left + a_common),
                                                  (b_dims, b_common + b_right))
        # the engine's general buffers, for forms that are reordered first
        state["A2"], state["B2"] = (_Buffer(empty(math.prod(d))) for d in (a_dims, b_dims))
        state["shape"] = (case["m"], case["n"], case["k"])
        state["C"] = _Buffer(empty(case["m"], case["n"]))
    elif op == "product":
        m, n, k = case["m"], case["n"], case["k"]
        state.update(precision=capi.PRECISIONS[case["precision"]], shape=(m, n, k),
                     A=_Buffer(_complex(gen, m, k)), B=_Buffer(_complex(gen, k, n)),
                     C=_Buffer(empty(m, n)))
    elif op == "reorder":
        dims, perm = ([int(x) for x in case[key].split(",")] for key in ("dims", "perm"))
        state.update(dims=dims, perm=perm, src=_Buffer(_complex(gen, *dims)),
                     dst=_Buffer(empty(*[dims[p] for p in perm])))
    elif op == "vector":
        m, k, t = case["m"], case["k"], case["trans"]
        state.update(trans=t, m=m, k=k, A=_Buffer(_complex(gen, m, k)),
                     x=_Buffer(_complex(gen, m if t else k)), y=_Buffer(empty(k if t else m)))
    elif op == "grouped":
        offsets, sizes = _group_offsets(case)
        flat = [_complex(gen, sizes[0]), _complex(gen, sizes[1]), empty(sizes[2])]
        state.update(precision=capi.PRECISIONS[case["precision"]], C=_Buffer(flat[2]), problems=[
            (m, n, k, _Buffer(flat[0][a:]), _Buffer(flat[1][b:]), _Buffer(flat[2][c:]))
            for (m, n, k), (a, b, c) in zip(_group_shapes(case), offsets)])
    else:
        params, X, target, m, v = (_Buffer(t) for t in _network(case, seed))
        real = lambda *s: _Buffer(empty(*s, dtype=torch.float32))
        state.update(batch=case["batch"], params=params, X=X, target=target, m=m, v=v,
                     step=_ADAM["step"], grads=real(capi.MLP_PARAMS), loss=real(1),
                     y=real(case["batch"]))
    torch.cuda.synchronize()
    return state


# -------------------------------------------------------------------- pass

def run(state):
    op = state["op"]
    if op == "simulate":
        pairs = state["simulate"](state["options"])
        # sums of complex64 contractions: single precision is what they hold
        return np.array([a for _, a in sorted(pairs, key=lambda p: p[0])], dtype=np.complex64)
    ctx = state["ctx"]
    if op == "contract":
        prec, A, B, C = state["precision"], state["A"], state["B"], state["C"]
        ar, ac, br, bc = state["maps"]
        if not ctx.cgemm_mapped(prec, A, ar, ac, B, br, bc, C):
            ctx.reorder(A, state["A2"], *state["a_reorder"])
            ctx.reorder(B, state["B2"], *state["b_reorder"])
            ctx.cgemm(prec, *state["shape"], state["A2"], state["B2"], C)
        return C.tensor
    if op == "product":
        ctx.cgemm(state["precision"], *state["shape"], state["A"], state["B"], state["C"])
        return state["C"].tensor
    if op == "reorder":
        ctx.reorder(state["src"], state["dst"], state["dims"], state["perm"])
        return state["dst"].tensor
    if op == "vector":
        ctx.cgemv(state["trans"], state["m"], state["k"], state["A"], state["x"], state["y"])
        return state["y"].tensor
    if op == "grouped":
        ctx.cgemm_grouped(state["precision"], state["problems"])
        return state["C"].tensor
    if op == "score":
        ctx.mlp_forward(state["batch"], state["X"], state["params"], state["y"])
        return state["y"].tensor
    ctx.mlp_backward(state["batch"], state["X"], state["target"], state["params"],
                     state["grads"], state["loss"])
    ctx.mlp_adam(state["params"], state["grads"], state["m"], state["v"], state["step"],
                 _ADAM["lr"], _ADAM["beta1"], _ADAM["beta2"], _ADAM["eps"])
    state["step"] += 1
    return {key: state[key].tensor for key in ("params", "grads", "loss", "m", "v")}


# -------------------------------------------------------------------- work

def _product_work(m, n, k):
    return {"bytes": 8 * (m * k + k * n + m * n), "flops": 8 * m * n * k}


def work(case):
    op = case["op"]
    if op == "simulate":
        from qflex_amd import qflex
        steps = qflex.plan(_options(case, 0))["steps"]
        return {"bytes": 16 << case["open"],
                "flops": sum(8 * s["m"] * s["n"] * s["k"] * s["multiplicity"] for s in steps)}
    if op in ("contract", "product"):
        return _product_work(case["m"], case["n"], case["k"])
    if op == "reorder":
        return {"bytes": 16 * math.prod(int(x) for x in case["dims"].split(",")), "flops": 0}
    if op == "vector":
        m, k = case["m"], case["k"]
        return {"bytes": 8 * (m * k + m + k), "flops": 8 * m * k}
    if op == "grouped":
        each = [_product_work(*s) for s in _group_shapes(case)]
        return {key: sum(w[key] for w in each) for key in ("bytes", "flops")}
    n_in, hid, b = capi.MLP_IN, capi.MLP_HIDDEN, case["batch"]
    forward = 2 * b * (n_in * hid + hid * hid + hid)
    if op == "score":
        return {"bytes": 4 * (b * n_in + b + capi.MLP_PARAMS), "flops": forward}
    # backward: the gradients of every layer's weights and of both hidden layers' outputs
    return {"bytes": 4 * (b * n_in + b + 7 * capi.MLP_PARAMS),
            "flops": 2 * forward + 2 * b * (hid * hid + hid)}


# ------------------------------------------------------------------- exact

def _state_vector(text, n):
    """Textbook gates applied one by one to |0...0>, complex128 on the GPU."""
    one = torch.eye(2, dtype=torch.complex128)
    x = torch.tensor([[0, 1], [1, 0]], dtype=torch.complex128)
    y = torch.tensor([[0, -1j], [1j, 0]], dtype=torch.complex128)
    root = lambda p: 0.5 * (1 + 1j) * one + 0.5 * (1 - 1j) * p
    gates = {"h": torch.tensor([[1, 1], [1, -1]], dtype=torch.complex128) / math.sqrt(2),
             "t": torch.diag(torch.tensor([1, complex(math.cos(math.pi / 4),
                                                       math.sin(math.pi / 4))],
                                          dtype=torch.complex128)),
             "x_1_2": root(x), "y_1_2": root(y)}
    psi = torch.zeros(1 << n, dtype=torch.complex128, device="cuda")
    psi[0] = 1
    for line in text.splitlines()[1:]:
        _, gate, *qubits = line.split()
        q = [int(v) for v in qubits]
        if gate == "cz":
            a, b = sorted(q)
            psi.view(1 << a, 2, 1 << (b - a - 1), 2, -1)[:, 1, :, 1] *= -1
        else:
            u = gates[gate].tolist()
            v = psi.view(1 << q[0], 2, -1)
            psi = torch.stack([u[0][0] * v[:, 0] + u[0][1] * v[:, 1],
                               u[1][0] * v[:, 0] + u[1][1] * v[:, 1]], dim=1).reshape(-1)
    return psi


def exact(case, seed):
    op = case["op"]
    wide = lambda t: t.to(torch.complex128)
    if op == "simulate":
        n = case["rows"] * case["cols"]
        if n > 25:
            return None
        psi = _state_vector(_circuit(case, seed), n)
        index = [0]
        for c in _final_state(case, seed):
            index = [2 * i + b for i in index for b in ((0, 1) if c == "x" else (int(c),))]
        return psi[torch.tensor(index, device="cuda")].cpu().numpy()
    gen = _generator(seed)
    if op == "contract":
        a_dims, a_left, a_common, b_dims, b_common, b_right = _layout(case)
        a, b = _complex(gen, *a_dims), _complex(gen, *b_dims)
        return (wide(a.permute(a_left + a_common).reshape(case["m"], case["k"]))
                @ wide(b.permute(b_common + b_right).reshape(case["k"], case["n"])))
    if op == "product":
        a, b = _complex(gen, case["m"], case["k"]), _complex(gen, case["k"], case["n"])
        return wide(a) @ wide(b)
    if op == "reorder":
        dims, perm = ([int(x) for x in case[key].split(",")] for key in ("dims", "perm"))
        return wide(_complex(gen, *dims).permute(perm).contiguous())
    if op == "vector":
        m, k, t = case["m"], case["k"], case["trans"]
        a, x = wide(_complex(gen, m, k)), wide(_complex(gen, m if t else k))
        return x @ a if t else a @ x
    if op == "grouped":
        offsets, sizes = _group_offsets(case)
        flat_a, flat_b = wide(_complex(gen, sizes[0])), wide(_complex(gen, sizes[1]))
        out = torch.zeros(sizes[2], dtype=torch.complex128, device="cuda")
        for (m, n, k), (a, b, c) in zip(_group_shapes(case), offsets):
            out[c:c + m * n] = (flat_a[a:a + m * k].view(m, k)
                                @ flat_b[b:b + k * n].view(k, n)).reshape(-1)
        return out
    params, X, target, m, v = (t.double() for t in _network(case, seed))
    n_in, hid = capi.MLP_IN, capi.MLP_HIDDEN
    p = params.clone().requires_grad_(op == "train")
    w1, b1, w2, b2, w3, b3 = p.split([n_in * hid, hid, hid * hid, hid, hid, 1])
    h1 = torch.relu(X @ w1.view(n_in, hid) + b1)
    h2 = torch.relu(h1 @ w2.view(hid, hid) + b2)
    y = h2 @ w3 + b3
    if op == "score":
        return y
    loss = ((y - target) ** 2).mean()
    loss.backward()
    g, step = p.grad, _ADAM["step"]
    m = _ADAM["beta1"] * m + (1 - _ADAM["beta1"]) * g
    v = _ADAM["beta2"] * v + (1 - _ADAM["beta2"]) * g * g
    denom = (v / (1 - _ADAM["beta2"] ** step)).sqrt() + _ADAM["eps"]
    params = params - _ADAM["lr"] * (m / (1 - _ADAM["beta1"] ** step)) / denom
    return {"params": params, "grads": g, "loss": loss.detach().reshape(1), "m": m, "v": v}
