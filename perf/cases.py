"""Performance cases of the public sparse operations on one GPU.

Each case is one call (or one forward + backward step) that a program makes
through `trnsparse_amd`: the block-sparse product, CSR SpMV / SpMM, the
Schwarz-screened product and block-sparse attention, at the smallest,
ordinary and largest sizes they are used at, with sizes off the tiles among
them. Inputs are seeded and made on the GPU; `exact` restates every result in
float64 with plain torch.
"""

import math

import torch

import trnsparse_amd as ts

DEV = "cuda"
DTYPES = {"f32": torch.float32, "bf16": torch.bfloat16}


def listed():
    return [
        # A small block-sparse layer, or one step of a solver on a small
        # blocked operator: 8 x 8 blocks, where latency counts.
        {"name": "bsr_small", "op": "bsr", "dtype": "f32", "b": 128, "m": 1024, "n": 1024, "density": 0.3, "cols": 256,
         "train": False},
        # The blocked operator at scale: 16384^2, a tenth of the 128-blocks,
        # against 512 vectors in fp32.
        {"name": "bsr_large", "op": "bsr", "dtype": "f32", "b": 128, "m": 16384, "n": 16384, "density": 0.1,
         "cols": 512, "train": False},
        # A training step of a large block-sparse layer in bf16: the product,
        # the gradient of the stored blocks and of the dense operand.
        {"name": "bsr_train_bf16", "op": "bsr", "dtype": "bf16", "b": 128, "m": 16384, "n": 16384, "density": 0.1,
         "cols": 512, "train": True},
        # The same step with fine blocks and dimensions that are whole in
        # neither the blocks nor the vector width.
        {"name": "bsr_train_b32", "op": "bsr", "dtype": "f32", "b": 32, "m": 6000, "n": 5010, "density": 0.1,
         "cols": 201, "train": True},
        # An iterative method's product on a large general sparse matrix
        # (a mesh or a graph of a million nodes), reused from step to step.
        {"name": "spmv_large", "op": "spmv", "m": 1 << 20, "n": 1 << 20, "mean": 16, "dist": "poisson", "index": "i64"},
        # One layer of a graph network: node features times the adjacency
        # matrix, and the gradients of its weights and of the features.
        {"name": "spmm_train", "op": "spmm", "m": 150001, "n": 150001, "mean": 16, "dist": "poisson", "index": "i64",
         "cols": 64, "train": True},
        # A screened exchange-like build over a large basis.
        {"name": "screened_large", "op": "screened", "n": 4096, "cols": 4096, "train": False},
        # The same with gradients on a basis of an odd size.
        {"name": "screened_train_odd", "op": "screened", "n": 1111, "cols": 1111, "train": True},
        # A training step of long-context attention with a local window and
        # global blocks: the largest of the attention calls.
        {"name": "attn_train_bf16", "op": "attn", "dtype": "bf16", "heads": 32, "seq": 8192, "d": 128, "window": 4,
         "globals": 2, "train": True},
        # The same for a smaller network with 64-wide heads.
        {"name": "attn_train_bf16_d64", "op": "attn", "dtype": "bf16", "heads": 16, "seq": 4096, "d": 64, "window": 4,
         "globals": 2, "train": True},
        # And in fp32, the reference's own data type.
        {"name": "attn_train_f32", "op": "attn", "dtype": "f32", "heads": 8, "seq": 4096, "d": 64, "window": 4,
         "globals": 2, "train": True},
        # The forward call on one short sequence with few heads: 72 pairs of
        # a head and a query block, fewer than the chip's compute units.
        {"name": "attn_fwd_small", "op": "attn", "dtype": "bf16", "heads": 8, "seq": 1152, "d": 128, "window": 4,
         "globals": 2, "train": False},
    ]


def _log_int(rng, low, high):
    return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))


def draw(rng):
    """One more case of the ranges above; sizes spread over their logarithm,
    with the total work bounded by the listed cases'."""
    op = rng.choice(["bsr", "bsr", "bsr", "spmv", "spmm", "screened", "attn", "attn", "attn"])
    train = rng.random() < 0.6
    while True:
        if op == "bsr":
            b = rng.choice([16, 32, 64, 128, 128, 128])
            top = 16384 if b == 128 else 8192
            c = {"op": op, "dtype": rng.choice(["f32", "bf16"]), "b": b, "m": _log_int(rng, 512, top),
                 "n": _log_int(rng, 512, top), "density": round(rng.uniform(0.05, 0.4), 3),
                 "cols": _log_int(rng, 16, 512), "train": train}
            if work(c)["flops"] > 8.0e10:
                continue
            return c
        if op in ("spmv", "spmm"):
            c = {"op": op, "m": _log_int(rng, 1 << 11, 1 << 20 if op == "spmv" else 1 << 18), "n": 0,
                 "mean": rng.randint(4, 32), "dist": rng.choice(["poisson", "poisson", "zipf"]),
                 "index": rng.choice(["i64", "i64", "i32"])}
            c["n"] = c["m"] if rng.random() < 0.7 else _log_int(rng, 1 << 11, 1 << 18)
            if op == "spmm":
                c["cols"] = _log_int(rng, 2, 128)
                c["train"] = train
            if c["m"] * c["mean"] * c.get("cols", 1) > (1 << 24 if op == "spmv" else 1 << 27):
                continue
            return c
        if op == "screened":
            c = {"op": op, "n": _log_int(rng, 200, 4096), "cols": 0, "train": train}
            c["cols"] = c["n"] if rng.random() < 0.6 else _log_int(rng, 32, 4096)
            if work(c)["flops"] > 1.3e11:
                continue
            return c
        c = {"op": op, "dtype": rng.choice(["bf16", "bf16", "f32"]), "heads": _log_int(rng, 1, 32),
             "seq": 128 * _log_int(rng, 2, 64) - rng.choice([0, 0, 0, 37]), "d": rng.choice([64, 128]),
             "window": rng.randint(2, 8), "globals": rng.randint(1, 3), "train": train}
        if work(c)["flops"] > (3.4e11 if c["dtype"] == "bf16" else 6.0e10):
            continue
        return c


# ------------------------------------------------------------------- inputs


def _gen(seed, device=DEV):
    return torch.Generator(device=device).manual_seed(seed)


def _block_grid(c):
    b = c["b"]
    return -(-c["m"] // b), -(-c["n"] // b)


def _block_count(c):
    mb, nb = _block_grid(c)
    return max(1, round(c["density"] * mb * nb))


def _bsr_pattern(c, seed):
    """Row pointers and columns of a pattern with a band and uniform blocks off it."""
    mb, nb = _block_grid(c)
    i, j = torch.arange(mb)[:, None], torch.arange(nb)[None, :]
    score = torch.rand(mb, nb, generator=_gen(seed, "cpu"))
    score[(i * nb // mb - j).abs() <= 1] += 1.0  # the band goes first
    keep = torch.zeros(mb * nb, dtype=torch.bool)
    keep[score.flatten().topk(_block_count(c)).indices] = True
    keep = keep.view(mb, nb)
    ptrs = torch.zeros(mb + 1, dtype=torch.long)
    ptrs[1:] = keep.sum(1).cumsum(0)
    return ptrs, keep.nonzero()[:, 1].contiguous()


def _csr(c, seed):
    """Row lengths are the case's own (the same for every seed, so that the
    number of entries is too); columns, values and operands are the seed's."""
    g, shape = _gen(seed), _gen(c["m"] + c["mean"])
    m, n = c["m"], c["n"]
    if c["dist"] == "poisson":
        lens = torch.poisson(torch.full((m,), float(c["mean"]), device=DEV), generator=shape).long()
        lens = lens.clamp(1, min(64, n))
    else:  # a power law of exponent 1.5 up to 4096, as degrees of a graph
        u = torch.rand(m, device=DEV, generator=shape, dtype=torch.float64)
        lens = (1.0 - u).pow(-2.0).clamp(1, 4096)
        lens = (lens * c["mean"] / lens.mean()).round().long().clamp(1, min(4096, n // 2))
    ptrs = torch.zeros(m + 1, dtype=torch.long, device=DEV)
    ptrs[1:] = lens.cumsum(0)
    # columns of a row distinct and ascending: one in each of as many equal stretches
    nnz = int(ptrs[-1])
    L = torch.repeat_interleave(lens, lens)
    j = torch.arange(nnz, device=DEV) - torch.repeat_interleave(ptrs[:-1], lens)
    low, high = j * n // L, (j + 1) * n // L
    u = torch.rand(nnz, device=DEV, generator=g, dtype=torch.float64)
    cols = low + (u * (high - low)).long()
    values = torch.randn(nnz, device=DEV, generator=g)
    it = torch.int32 if c["index"] == "i32" else torch.int64
    return values, cols.to(it), ptrs.to(it), g


def _attn_mask(c):
    t = -(-c["seq"] // 128)
    i, j = torch.arange(t)[:, None], torch.arange(t)[None, :]
    return ((j <= i) & (j > i - c["window"])) | (j < c["globals"])


def prepare(case, seed):
    """Inputs made from the seed, with the matrix or mask object that the
    program keeps; operands that get a gradient are leaves."""
    c, train = case, case.get("train", False)
    if c["op"] == "bsr":
        g = _gen(seed)
        dt = DTYPES[c["dtype"]]
        ptrs, cols = _bsr_pattern(c, seed)
        blocks = torch.randn(cols.numel(), c["b"], c["b"], device=DEV, generator=g).to(dt)
        # an aligned matrix would hold zeros past its edge: so does this one
        em, en = c["m"] % c["b"], c["n"] % c["b"]
        mb, nb = _block_grid(c)
        rows = torch.repeat_interleave(torch.arange(mb), ptrs.diff())
        if em:
            blocks[(rows == mb - 1).to(DEV), em:, :] = 0
        if en:
            blocks[(cols == nb - 1).to(DEV), :, en:] = 0
        B = torch.randn(c["n"], c["cols"], device=DEV, generator=g).to(dt)
        s = {"B": B.requires_grad_(train)}
        s["A"] = ts.BSRMatrix(blocks=blocks.requires_grad_(train), block_col_indices=cols.to(DEV),
                              block_row_ptrs=ptrs.to(DEV), shape=(c["m"], c["n"]), block_size=c["b"])
        if train:
            s["G"] = torch.randn(c["m"], c["cols"], device=DEV, generator=g).to(dt)
    elif c["op"] in ("spmv", "spmm"):
        values, cols, ptrs, g = _csr(c, seed)
        s = {"A": ts.CSRMatrix(values=values.requires_grad_(train), col_indices=cols, row_ptrs=ptrs,
                               shape=(c["m"], c["n"]))}
        if c["op"] == "spmv":
            s["x"] = torch.randn(c["n"], device=DEV, generator=g)
        else:
            s["x"] = torch.randn(c["n"], c["cols"], device=DEV, generator=g).requires_grad_(train)
            if train:
                s["G"] = torch.randn(c["m"], c["cols"], device=DEV, generator=g)
    elif c["op"] == "screened":
        g = _gen(seed)
        n = c["n"]
        diag = torch.pow(10.0, torch.rand(n, device=DEV, generator=g, dtype=torch.float64) * 14.0 - 14.0).float()
        i = torch.arange(n, device=DEV, dtype=torch.float32)
        A = torch.exp(-(i[:, None] - i[None, :]).abs() / 256.0)
        A *= torch.rand(n, n, device=DEV, generator=g) * 0.5 + 0.5
        A *= torch.where(torch.rand(n, n, device=DEV, generator=g) < 0.5, -1.0, 1.0)
        B = torch.randn(n, c["cols"], device=DEV, generator=g)
        s = {"A": A.requires_grad_(train), "diag": diag, "B": B.requires_grad_(train), "threshold": 1e-20}
        if train:
            s["G"] = torch.randn(n, c["cols"], device=DEV, generator=g)
    else:
        g = _gen(seed)
        dt = DTYPES[c["dtype"]]
        shape = (c["heads"], c["seq"], c["d"])
        Q, K, V = (torch.randn(shape, device=DEV, generator=g).to(dt).requires_grad_(train) for _ in range(3))
        keep = _attn_mask(c)
        ptrs = torch.zeros(keep.shape[0] + 1, dtype=torch.long)
        ptrs[1:] = keep.sum(1).cumsum(0)
        cols = keep.nonzero()[:, 1].contiguous()
        mask = ts.BSRMatrix(blocks=torch.ones(cols.numel(), 128, 128, device=DEV), block_col_indices=cols.to(DEV),
                            block_row_ptrs=ptrs.to(DEV), shape=(128 * keep.shape[0], 128 * keep.shape[1]),
                            block_size=128)
        s = {"Q": Q, "K": K, "V": V, "mask": mask}
        if train:
            s["G"] = torch.randn(shape, device=DEV, generator=g).to(dt)
    s["op"] = c["op"]
    return s


# --------------------------------------------------------------------- work


def run(state):
    s = state
    if s["op"] == "bsr":
        out, leaves = ts.bsr_spmm(s["A"], s["B"]), (s["A"].blocks, s["B"])
    elif s["op"] == "spmv":
        return ts.spmv(s["A"], s["x"])
    elif s["op"] == "spmm":
        out, leaves = ts.spmm(s["A"], s["x"]), (s["A"].values, s["x"])
    elif s["op"] == "screened":
        out, leaves = ts.screened_spmm(s["A"], s["diag"], s["B"], s["threshold"]), (s["A"], s["B"])
    else:
        out = ts.block_sparse_attention_tiled(s["Q"], s["K"], s["V"], s["mask"])
        leaves = (s["Q"], s["K"], s["V"])
    if "G" not in s:
        return out
    return (out.detach(),) + torch.autograd.grad(out, leaves, s["G"])


def work(case):
    c, steps = case, 3 if case.get("train") else 1  # a product and its two gradients
    if c["op"] == "bsr":
        size = 4 if c["dtype"] == "f32" else 2
        blocks = _block_count(c) * c["b"] ** 2
        io = blocks + (c["m"] + c["n"]) * c["cols"]  # blocks, B and the result
        return {"bytes": size * (io * 2 + (c["m"] * c["cols"]) if c.get("train") else io),
                "flops": 2 * blocks * c["cols"] * steps}
    if c["op"] in ("spmv", "spmm"):
        nnz, idx, k = c["m"] * c["mean"], 8 if c["index"] == "i64" else 4, c.get("cols", 1)
        io = 4 * nnz + 4 * (c["m"] + c["n"]) * k
        structure = idx * (nnz + c["m"] + 1)
        return {"bytes": structure + (2 * io + 4 * c["m"] * k if c.get("train") else io), "flops": 2 * nnz * k * steps}
    if c["op"] == "screened":
        n, k = c["n"], c["cols"]
        io = 4 * (n * n + n + 2 * n * k)
        return {"bytes": 2 * io + 4 * n * k if c.get("train") else io, "flops": 2 * n * n * k * steps}
    size = 4 if c["dtype"] == "f32" else 2
    pairs = int(_attn_mask(c)[: c["seq"] // 128].sum()) * 128 * 128
    # forward: scores and output; backward: scores, dP, dV, dK, dQ
    return {"bytes": size * c["heads"] * c["seq"] * c["d"] * (8 if c.get("train") else 4),
            "flops": 2 * c["heads"] * pairs * c["d"] * (7 if c.get("train") else 2)}


def tolerance(case):
    """About four times the distance from `exact`: 1.1e-6 at most in fp32
    (4096-term sums), 1.7e-3 for products and 2.4e-3 for attention in bf16
    (results, probabilities and their gradients each rounded to 8 bits)."""
    if case.get("dtype") == "bf16":
        return {"rel": 0.007, "max": 0.03} if case["op"] == "bsr" else {"rel": 0.01, "max": 0.1}
    return {"rel": 4e-6, "max": 1e-4}


# -------------------------------------------------------------------- exact


def exact(case, seed):
    """What `run` returns, from the same inputs in float64."""
    c, s = case, prepare(case, seed)
    s = {k: v.detach() if isinstance(v, torch.Tensor) else v for k, v in s.items()}
    train = "G" in s
    with torch.no_grad():
        if c["op"] == "bsr":
            A, b = s["A"], c["b"]
            mb, nb = _block_grid(c)
            rows = torch.repeat_interleave(torch.arange(mb, device=DEV), A.block_row_ptrs.diff())
            dense = torch.zeros(mb, nb, b, b, dtype=torch.float64, device=DEV)
            dense[rows, A.block_col_indices] = A.blocks.detach().double()
            dense = dense.transpose(1, 2).reshape(mb * b, nb * b)[: c["m"], : c["n"]]
            B = s["B"].double()
            out = dense @ B
            if not train:
                return out
            G = s["G"].double()
            dB = dense.t() @ G
            Gp = torch.zeros(mb * b, c["cols"], dtype=torch.float64, device=DEV)
            Bp = torch.zeros(nb * b, c["cols"], dtype=torch.float64, device=DEV)
            Gp[: c["m"]], Bp[: c["n"]] = G, B
            dA = (Gp @ Bp.t()).view(mb, b, nb, b).transpose(1, 2)[rows, A.block_col_indices]
            return out, dA, dB
        if c["op"] in ("spmv", "spmm"):
            A = s["A"]
            cols, x, v = A.col_indices.long(), s["x"].double(), A.values.detach().double()
            rows = torch.repeat_interleave(torch.arange(c["m"], device=DEV), A.row_ptrs.long().diff())
            k = c.get("cols", 1)
            out = torch.zeros((c["m"], k), dtype=torch.float64, device=DEV)
            dx = torch.zeros((c["n"], k), dtype=torch.float64, device=DEV)
            dv = torch.zeros_like(v)
            x = x.view(-1, k)
            step = max(1, (1 << 27) // k)
            for at in range(0, v.numel(), step):
                p = slice(at, at + step)
                out.index_add_(0, rows[p], v[p, None] * x[cols[p]])
                if train:
                    Gr = s["G"].double()[rows[p]]
                    dv[p] = (Gr * x[cols[p]]).sum(1)
                    dx.index_add_(0, cols[p], v[p, None] * Gr)
            return (out, dv, dx) if train else out.view(-1) if c["op"] == "spmv" else out
        if c["op"] == "screened":
            q = s["diag"].abs().sqrt()
            keep = (q[:, None] * q[None, :]) > math.sqrt(s["threshold"])  # the mask is defined in diag's type
            A, B = s["A"].double() * keep, s["B"].double()
            out = A @ B
            if not train:
                return out
            G = s["G"].double()
            return out, (G @ B.t()) * keep, A.t() @ G
        S, d, scale = c["seq"], c["d"], c["d"] ** -0.5
        whole = S // 128 * 128  # rows past the last whole block have no output
        seen = _attn_mask(c).to(DEV).repeat_interleave(128, 0).repeat_interleave(128, 1)[:whole, :S]
        res = [torch.zeros(s["Q"].shape, dtype=torch.float64, device=DEV) for _ in range(4 if train else 1)]
        for h in range(c["heads"]):
            Q, K, V = (s[k][h].double() for k in ("Q", "K", "V"))
            Q = Q[:whole]
            P = (Q @ K.t() * scale).masked_fill_(~seen, -math.inf).softmax(1)
            res[0][h, :whole] = P @ V
            if train:
                dO = s["G"][h, :whole].double()
                dP = dO @ V.t()
                dS = P * (dP - (dP * P).sum(1, keepdim=True)) * scale
                res[1][h, :whole], res[2][h], res[3][h] = dS @ K, dS.t() @ Q, P.t() @ dO
        return tuple(res) if train else res[0]
