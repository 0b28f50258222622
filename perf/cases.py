"""What a user of this framework has it do, as cases that can be timed: the two executors D = A (B C) through the
bindings, on matrices from a small grid to a power-law graph of two million nodes, and graph-convolution layers and
two-layer models, forward and backward, through the torch operators.

    listed()            the cases
    draw(rng)           one more case of the same ranges
    prepare(case, seed) the operands and the schedule a program keeps, on the GPU
    run(state)          one pass, and everything it computes
    work(case)          the bytes and operations one pass cannot do without
    tolerance(case)     how far another correct implementation may be off
"""
import importlib
import math

import torch

tf = importlib.import_module("tile-fusion_amd")
importlib.import_module("tile-fusion_amd.torch_ops")

# kind      what one pass is
# gemm_spmm   D = A (B C), A sparse, B and C dense: tf.gemm_spmm on resident operands
# spmm_spmm   D = A (A C), the two-hop product: tf.spmm_spmm on resident operands
# layer       one graph-convolution layer, forward and backward for features and weights (sw_gcn.fusedGeMMSpMM_vt_ro)
# train       two layers with a ReLU between, forward and backward for both weights (sw_gcn.fusedGCN)
# infer       the same two layers without gradients
#
# pattern   a, b and c are its sizes
# grid2d      5-point Laplacian on a x b points
# grid3d      7-point Laplacian on a x b x c points
# box3d       27-point stencil on a x b x c points, rows scaled to sum 1
# band        a rows of b entries at random places in a band of c columns
# er          Erdos-Renyi graph with self-loops, a nodes of mean degree b, symmetric-normalised
# rmat        R-MAT graph of 2^a nodes and b edges per node, symmetrised, row-normalised


def _case(name, kind, pattern, a, b=0, c=0, K=0, H=0, N=0):
    d = {"kind": kind, "pattern": pattern, "a": a, "b": b, "c": c, "K": K, "H": H, "N": N}
    return dict(d, name=name) if name else d


def listed():
    return [
        # a small system in an iteration: latency
        _case("grid2d_small", "gemm_spmm", "grid2d", 64, 64, K=64, N=64),
        # a banded matrix times a block of vectors, twice
        _case("band_two_hops", "spmm_spmm", "band", 65536, 16, 32, N=128),
        # an unstructured graph, an odd number of vectors
        _case("graph_two_hops", "spmm_spmm", "er", 50001, 12, N=100),
        # stencils on 3D grids: the large sparse-sparse products, narrow and wide rows
        _case("grid3d_two_hops", "spmm_spmm", "grid3d", 128, 128, 128, N=64),
        _case("box3d_two_hops", "spmm_spmm", "box3d", 96, 96, 96, N=64),
        # layers without gradients straight through the executor: wide features to a narrower layer, a reordered
        # (banded) graph, and a large power-law graph
        _case("er_layer", "gemm_spmm", "er", 200000, 10, K=256, N=128),
        _case("band_layer", "gemm_spmm", "band", 262144, 16, 32, K=128, N=128),
        _case("powerlaw_layer", "gemm_spmm", "rmat", 21, 8, K=128, N=128),
        # a hidden layer in training
        _case("layer_fwd_bwd", "layer", "er", 100000, 10, K=128, N=64),
        # full-batch training of a two-layer classifier: raw feature widths and class counts are what a dataset has
        _case("small_model_training", "train", "er", 3000, 8, K=500, H=32, N=7),
        _case("model_training", "train", "rmat", 17, 8, K=300, H=64, N=40),
        # ... and its inference on a larger graph
        _case("model_inference", "infer", "rmat", 18, 8, K=128, H=128, N=40),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _width(rng, lo, hi):
    """A layer width: half of them multiples of 32, as hidden layers are, half any number."""
    w = _log(rng, lo, hi)
    return w if rng.random() < 0.5 else max(32, (w + 16) // 32 * 32)


def draw(rng):
    kind = rng.choice(["gemm_spmm", "gemm_spmm", "spmm_spmm", "spmm_spmm", "layer", "train", "infer"])
    if kind == "spmm_spmm":
        pattern = rng.choice(["grid2d", "grid3d", "box3d", "band", "er"])
    elif kind == "gemm_spmm":
        pattern = rng.choice(["grid2d", "band", "er", "rmat"])
    else:
        pattern = rng.choice(["er", "rmat"])
    executor = kind in ("gemm_spmm", "spmm_spmm")
    if pattern == "grid2d":
        a, b, c = _log(rng, 48, 1024), _log(rng, 48, 1024), 0
    elif pattern == "grid3d":
        a, b, c = (_log(rng, 20, 128) for _ in range(3))
    elif pattern == "box3d":
        a, b, c = (_log(rng, 16, 96) for _ in range(3))
    elif pattern == "band":
        c = rng.choice([16, 32, 48, 64])
        a, b = _log(rng, 4000, 300000), rng.randint(4, min(24, c // 2))
    elif pattern == "er":
        a, b, c = _log(rng, 2000, 200000), rng.randint(4, 16), 0
    else:
        a, b, c = rng.randint(12, 20 if executor else 18), rng.randint(4, 10), 0
    N = _width(rng, 16, 128) if executor or kind == "layer" else _log(rng, 4, 128)
    K = 0 if kind == "spmm_spmm" else _width(rng, 16, 300 if executor else 512)
    H = _width(rng, 16, 128) if kind in ("train", "infer") else 0
    return _case(None, kind, pattern, a, b, c, K=K, H=H, N=N)


# ---- patterns, made on the GPU: (rows, crow, col, val) with sorted int32 columns and fp32 values ----------------

def _from_keys(n, key):
    """CSR row pointers and columns of the sorted, distinct keys row * n + column."""
    row = torch.div(key, n, rounding_mode="floor")
    crow = torch.zeros(n + 1, dtype=torch.int64, device=key.device)
    crow[1:] = torch.bincount(row, minlength=n).cumsum(0)
    return row, crow.int(), (key - row * n).int()


def _stencil(sizes, reach, values):
    """All neighbours that `reach` accepts of the offsets (x, y, z) in {-1, 0, 1}, x fastest."""
    nx, ny, nz = (list(sizes) + [1, 1])[:3]
    n = nx * ny * nz
    i = torch.arange(n, device="cuda", dtype=torch.int64)
    x, y, z = i % nx, (i // nx) % ny, i // (nx * ny)
    offs = [(dx, dy, dz) for dz in (-1, 0, 1) for dy in (-1, 0, 1) for dx in (-1, 0, 1) if reach(abs(dx) + abs(dy) + abs(dz))]
    offs = [o for o in offs if (ny > 1 or o[1] == 0) and (nz > 1 or o[2] == 0)]
    there = torch.stack([(x + dx >= 0) & (x + dx < nx) & (y + dy >= 0) & (y + dy < ny) & (z + dz >= 0) & (z + dz < nz)
                         for dx, dy, dz in offs], 1)
    step = torch.tensor([dx + nx * (dy + ny * dz) for dx, dy, dz in offs], device="cuda")
    col = (i[:, None] + step[None, :])[there].int()
    count = there.sum(1)
    crow = torch.zeros(n + 1, dtype=torch.int64, device="cuda")
    crow[1:] = count.cumsum(0)
    if values is None:  # rows of sum 1
        val = (1.0 / count.float())[:, None].expand(n, len(offs))[there]
    else:
        on, off = values
        val = torch.tensor([on if o == (0, 0, 0) else off for o in offs], device="cuda").float()[None, :].expand(n, len(offs))[there]
    return n, crow.int(), col, val.contiguous()


def _pattern(case, g):
    kind, a, b, c = case["pattern"], case["a"], case["b"], case["c"]
    if kind == "grid2d":
        return _stencil((a, b), lambda d: d <= 1, (4.0, -1.0))
    if kind == "grid3d":
        return _stencil((a, b, c), lambda d: d <= 1, (6.0, -1.0))
    if kind == "box3d":
        return _stencil((a, b, c), lambda d: True, None)
    if kind == "band":
        key = torch.rand(a, c, generator=g, device="cuda")
        col = torch.arange(a, device="cuda")[:, None] + torch.arange(-(c // 2), c - c // 2, device="cuda")[None, :]
        key[(col < 0) | (col >= a)] = 2.0
        pick = key.topk(b, dim=1, largest=False).indices.sort(dim=1).values
        col = col.gather(1, pick).reshape(-1).int()
        val = torch.rand(a * b, generator=g, device="cuda") * 2 - 1
        return a, (torch.arange(a + 1, device="cuda") * b).int(), col, val
    if kind == "er":
        n, m = a, a * b // 2
        u = torch.randint(n, (m,), generator=g, device="cuda")
        v = torch.randint(n, (m,), generator=g, device="cuda")
        own = torch.arange(n, device="cuda")
        row, crow, col = _from_keys(n, torch.cat([u * n + v, v * n + u, own * (n + 1)]).unique())
        d = (crow[1:] - crow[:-1]).float().rsqrt()
        return n, crow, col, d[row] * d[col.long()]
    n, m = 1 << a, b << a
    u = torch.zeros(m, dtype=torch.int64, device="cuda")
    v = torch.zeros(m, dtype=torch.int64, device="cuda")
    for _ in range(a):  # quadrants of probability 0.57, 0.19, 0.19, 0.05
        r = torch.rand(m, generator=g, device="cuda")
        u = u * 2 + (r >= 0.76)
        v = v * 2 + (((r >= 0.57) & (r < 0.76)) | (r >= 0.95))
    row, crow, col = _from_keys(n, torch.cat([u * n + v, v * n + u]).unique())
    return n, crow, col, (1.0 / (crow[1:] - crow[:-1]).clamp(min=1).float())[row]


def _uniform(g, rows, cols, lo, hi):
    return torch.rand(rows, cols, generator=g, device="cuda") * (hi - lo) + lo


def _weight(g, out_dim, in_dim):
    lim = math.sqrt(6.0 / (in_dim + out_dim))
    return _uniform(g, out_dim, in_dim, -lim, lim)


class _Executor:
    """Operands of an executor call: the matrix uploaded once, the dense operands and the result in device memory."""

    def __init__(self, case, n, crow, col, val, g):
        K, N = case["K"], case["N"]
        self.A = tf.CsrMatrix(n, n, crow.cpu().numpy(), col.cpu().numpy(), val.cpu().numpy()).to_device()
        self.keep = [_uniform(g, K or n, N, -1.0, 1.0), torch.zeros(n, N, device="cuda")]
        self.D = self.keep[1]
        if K:
            self.keep.append(_uniform(g, n, K, 0.0, 1.0))
            self.schedule = tf.inspector(self.A, op=tf.OP_GEMM_SPMM, N=N, K=K)
        else:
            self.schedule = tf.inspector(self.A, op=tf.OP_SPMM_SPMM, N=N, inner=self.A)
        self.dense = [tf.DenseMatrix.wrap_device(t.shape[0], t.shape[1], t.data_ptr()) for t in self.keep]

    def run(self):
        if len(self.dense) == 3:
            tf.gemm_spmm(self.A, self.dense[2], self.dense[0], self.dense[1], self.schedule)
        else:
            tf.spmm_spmm(self.A, self.A, self.dense[0], self.dense[1], self.schedule)
        return self.D


class _Layer:
    """A hidden layer in training: features and weights want gradients."""

    def __init__(self, case, n, crow, col, val, g):
        K, N = case["K"], case["N"]
        self.adj = torch.sparse_csr_tensor(crow, col, val, size=(n, n))
        self.x = _uniform(g, n, K, 0.0, 1.0).requires_grad_()
        self.w = _weight(g, N, K).requires_grad_()
        self.grad = _uniform(g, n, N, -1.0, 1.0)
        self.schedule = torch.ops.sw_gcn.inspect_vt_ro(self.adj, K, N, 500000, 16)

    def run(self):
        out = torch.ops.sw_gcn.fusedGeMMSpMM_vt_ro(self.adj, self.x, self.w, self.schedule, 16, 0)
        gx, gw = torch.autograd.grad(out, (self.x, self.w), self.grad)
        return out.detach(), gx, gw


class _Model:
    """A two-layer classifier: training (gradients of both weights) or inference."""

    def __init__(self, case, n, crow, col, val, g):
        K, H, N = case["K"], case["H"], case["N"]
        self.adj = torch.sparse_csr_tensor(crow, col, val, size=(n, n))
        self.x = _uniform(g, n, K, 0.0, 1.0)
        self.train = case["kind"] == "train"
        self.w1 = _weight(g, H, K).requires_grad_(self.train)
        self.w2 = _weight(g, N, H).requires_grad_(self.train)
        self.grad = _uniform(g, n, N, -1.0, 1.0) if self.train else None
        torch.ops.sw_gcn.inspect_vt_ro(self.adj, K, H, 500000, 16)
        torch.ops.sw_gcn.inspect_vt_ro(self.adj, H, N, 500000, 16)

    def run(self):
        out = torch.ops.sw_gcn.fusedGCN(self.adj, self.x, self.w1, self.w2, 16)
        if not self.train:
            return out
        g1, g2 = torch.autograd.grad(out, (self.w1, self.w2), self.grad)
        return out.detach(), g1, g2


def prepare(case, seed):
    g = torch.Generator(device="cuda").manual_seed(int(seed))
    n, crow, col, val = _pattern(case, g)
    kind = {"gemm_spmm": _Executor, "spmm_spmm": _Executor, "layer": _Layer}.get(case["kind"], _Model)
    return kind(case, n, crow, col, val, g)


def run(state):
    return state.run()


def _rows_and_entries(case):
    """Rows and stored entries (for the random graphs: the expected number, nearly)."""
    kind, a, b, c = case["pattern"], case["a"], case["b"], case["c"]
    if kind == "grid2d":
        return a * b, 5 * a * b - 2 * (a + b)
    if kind == "grid3d":
        return a * b * c, 7 * a * b * c - 2 * (a * b + b * c + a * c)
    if kind == "box3d":
        return a * b * c, (3 * a - 2) * (3 * b - 2) * (3 * c - 2)
    if kind == "band":
        return a, a * b
    if kind == "er":
        return a, a * (b + 1)
    return 1 << a, int(1.9 * (b << a))


def work(case):
    M, nnz = _rows_and_entries(case)
    K, H, N = case["K"], case["H"], case["N"]
    sparse = 8 * nnz + 4 * (M + 1)
    if case["kind"] == "spmm_spmm":
        return {"bytes": sparse + 8 * M * N, "flops": 4 * nnz * N}
    if case["kind"] == "gemm_spmm":
        return {"bytes": sparse + 4 * (M * K + K * N + M * N), "flops": 2 * M * K * N + 2 * nnz * N}
    if case["kind"] == "layer":  # the adjacency is its own transpose or is read a second time, once here
        return {"bytes": sparse + 4 * (2 * M * K + 2 * K * N + 2 * M * N), "flops": 6 * M * K * N + 4 * nnz * N}
    fwd = 2 * M * K * H + 2 * M * H * N + 2 * nnz * (H + N)
    if case["kind"] == "infer":
        return {"bytes": sparse + 4 * (M * K + K * H + H * N + M * N), "flops": fwd}
    return {"bytes": sparse + 4 * (M * K + 2 * K * H + 2 * H * N + 2 * M * N),
            "flops": fwd + 2 * M * K * H + 4 * M * H * N + 2 * nnz * (H + N)}


def tolerance(case):
    if case["kind"] == "train":
        # fp32 sums, and the ReLU's derivative: of some million hidden values one or two lie within their rounding error
        # of zero, where another order of the sums flips a whole row's share of a gradient
        return {"rel": 1e-3}
    return {"rel": 1e-5, "max": 1e-4}
