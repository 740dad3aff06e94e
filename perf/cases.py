"""What is timed when this framework's speed is looked at: the products that its users call.

A case is a dict of plain values. `call` names the public entry point:

  gemm    spla::gemm, a local product of any operand form
  ssb     spla::pgemm_ssb, C <- alpha op(A) B + beta C with op = T or C, long reduction
  ssbtr   spla::pgemm_ssbtr, the same for one triangle of C
  sbs     spla::pgemm_sbs, C <- alpha A B + beta C with tall A and C
  batch   the block products of one ring step, planned once and executed many times

`type` is the BLAS letter of the element type (s, d, c, z), `mode` the arithmetic of double
products (fp64, split: INT8 residues, auto), `where` the memory of the operands, `pad` what the
leading dimensions have on top of the rows they need and `row`, `col` the offset of C inside its
distributed matrix. Matrices are column-major: a torch tensor of shape (columns, leading
dimension).
"""

import functools
import math
import random

import torch

import spla_amd as spla

TYPES = {"s": torch.float32, "d": torch.float64, "c": torch.complex64, "z": torch.complex128}
WIDE = {"s": torch.float64, "d": torch.float64, "c": torch.complex128, "z": torch.complex128}
OPS = {"N": spla.Operation.NONE, "T": spla.Operation.TRANSPOSE,
       "C": spla.Operation.CONJ_TRANSPOSE}
MODES = {"fp64": spla.GemmMode.FP64, "split": spla.GemmMode.SPLIT_INT8,
         "auto": spla.GemmMode.AUTO}
# the guaranteed normwise bound that the split products are planned for (bench.py)
TOLERANCE = 1e-13
ALPHA = {"s": 1.5, "d": 1.5, "c": 1.0 + 0.5j, "z": 1.0 + 0.5j}


def _case(call, type, m, n, k, **more):
    case = {"call": call, "type": type, "m": m, "n": n, "k": k, "opA": "C", "opB": "N",
            "mode": "fp64", "where": "device", "beta": 0.0, "pad": 0, "row": 0, "col": 0}
    if call in ("gemm", "sbs"):
        case["opA"] = "N"
    elif type in "sd":
        case["opA"] = "T"
    case.update(more)
    return case


def listed():
    return [
        # the reference's unit-test grid: a small local product, where the call itself is what costs
        _case("gemm", "d", 13, 32, 263, name="gemm_d_small", beta=0.5, pad=5),
        # overlap of two sets of 256 states: the benchmark's smallest distributed product
        _case("ssb", "z", 256, 256, 4096, name="ssb_z_256"),
        # one triangle of an ordinary overlap matrix with ragged sizes, placed inside a larger C
        _case("ssbtr", "z", 700, 700, 30011, name="ssbtr_z_700", beta=0.5, pad=3, row=2, col=2,
              fill="L"),
        # few states over very many grid points: bound by reading A and B
        _case("ssb", "z", 16, 16, 8000000, name="ssb_z_16"),
        # the headline product: overlap of 2048 states over 2e5 plane waves, FP64 kernels
        _case("ssb", "z", 2048, 2048, 200000, name="ssb_z_2048", beta=0.5),
        # the same in split precision
        _case("ssb", "z", 2048, 2048, 200000, name="ssb_z_2048_split", beta=0.5, mode="split"),
        # real states of very uneven magnitudes, the library choosing the arithmetic
        _case("ssb", "d", 1000, 1000, 100000, name="ssb_d_1000_auto", mode="auto", spread=10),
        # the headline product in single precision
        _case("ssb", "c", 2048, 2048, 200000, name="ssb_c_2048"),
        # the same kind of product from pinned host memory, staged through the device
        _case("ssb", "z", 1024, 1024, 20000, name="ssb_z_1024_host", beta=0.5, where="host"),
        # rotation of a few real states over many grid points
        _case("sbs", "d", 100003, 260, 260, name="sbs_d_260", beta=0.5),
        # rotation of 4096 complex states: the largest product of the benchmark
        _case("sbs", "z", 100000, 4096, 4096, name="sbs_z_4096"),
        # one ring step: uneven blocks of an overlap matrix in one launch
        _case("batch", "z", 512, 512, 65536, name="batch_z_128", blocks=128, sizes=5),
    ]


def _between(rng, low, high):
    """A whole number, uniform over its logarithm."""
    return min(high, max(low, int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))))


def draw(rng):
    kind = rng.choice(("gemm", "ssb", "ssb", "ssbtr", "ssb_long", "split", "split", "single",
                       "host", "sbs", "sbs", "batch"))
    beta = rng.choice((0.0, 0.5))
    pad = rng.choice((0, 0, 1, 6))
    if kind == "gemm":
        t = rng.choice("sdcz")
        ops = "NTC" if t in "cz" else "NT"
        return _case("gemm", t, _between(rng, 1, 2000), _between(rng, 1, 2000),
                     _between(rng, 1, 4000), opA=rng.choice(ops), opB=rng.choice(ops), beta=beta,
                     pad=pad)
    if kind == "ssb":
        t = rng.choice("ddzzz")
        return _case("ssb", t, _between(rng, 48, 2048), _between(rng, 48, 2048),
                     _between(rng, 4096, 200000), beta=beta, pad=pad)
    if kind == "ssbtr":
        m = _between(rng, 200, 2048)
        return _case("ssbtr", rng.choice("dz"), m, m, _between(rng, 4096, 100000), beta=beta,
                     pad=pad, row=2, col=2, fill=rng.choice("LU"))
    if kind == "ssb_long":
        return _case("ssb", rng.choice("dz"), _between(rng, 1, 32), _between(rng, 1, 32),
                     _between(rng, 100000, 8000000), beta=beta, pad=pad)
    if kind == "split":
        return _case("ssb", rng.choice("dz"), _between(rng, 400, 2048), _between(rng, 400, 2048),
                     _between(rng, 10000, 200000), beta=beta, pad=pad,
                     mode=rng.choice(("split", "auto")), spread=rng.choice((0, 10)))
    if kind == "single":
        return _case("ssb", rng.choice("sc"), _between(rng, 48, 2048), _between(rng, 48, 2048),
                     _between(rng, 4096, 200000), beta=beta, pad=pad)
    if kind == "host":
        return _case("ssb", rng.choice("dz"), _between(rng, 128, 1024), _between(rng, 128, 1024),
                     _between(rng, 4096, 20000), beta=beta, where="host")
    if kind == "sbs":
        return _case("sbs", rng.choice("dzz"), _between(rng, 5000, 100000),
                     _between(rng, 64, 2048), _between(rng, 64, 2048), beta=beta, pad=pad)
    return _case("batch", rng.choice("dz"), 512, 512, 65536, blocks=_between(rng, 16, 128),
                 sizes=rng.randrange(1 << 20))


@functools.lru_cache(maxsize=None)
def _context(mode):
    """A program keeps one context for all its products."""
    ctx = spla.Context(spla.ProcessingUnit.GPU)
    ctx.set_gemm_mode(MODES[mode])
    ctx.set_split_tolerance(TOLERANCE)
    return ctx


@functools.lru_cache(maxsize=None)
def _distribution():
    return spla.MatrixDistribution.create_blacs_block_cyclic(spla.MPI_COMM_SELF, "R", 1, 1, 256,
                                                             256)


def _shapes(case):
    """Stored (columns, rows) of A, B and C."""
    m, n, k = case["m"], case["n"], case["k"]
    a = (k, m) if case["opA"] == "N" else (m, k)
    b = (n, k) if case["opB"] == "N" else (k, n)
    return a, b, (n + case["col"], m + case["row"])


def _block_sizes(case):
    """(m, n, k) of a ring step's blocks: uniform over their logarithms."""
    rng = random.Random(case["sizes"])
    return [(_between(rng, 32, case["m"]), _between(rng, 32, case["n"]),
             _between(rng, 4096, case["k"])) for _ in range(case["blocks"])]


def _uniform(shape, dtype, gen, spread=0):
    """Components uniform in [-1, 1), times 2^e with e in [-spread, spread]."""
    real = torch.float32 if dtype in (torch.float32, torch.complex64) else torch.float64
    x = torch.empty((*shape, 2) if dtype.is_complex else shape, dtype=real, device="cuda")
    x.uniform_(-1.0, 1.0, generator=gen)
    if spread:
        x.mul_(torch.exp2(torch.randint(-spread, spread + 1, x.shape, device="cuda",
                                        generator=gen).to(real)))
    return torch.view_as_complex(x) if dtype.is_complex else x


def _operands(case, seed):
    gen = torch.Generator(device="cuda")
    gen.manual_seed(seed)
    dtype = TYPES[case["type"]]
    if case["call"] == "batch":
        blocks = []
        sizes = _block_sizes(case)
        total = [sum(x) for x in zip(*((m * k, n * k, m * n) for m, n, k in sizes))]
        flat = [_uniform((t,), dtype, gen) for t in total]
        flat[2].zero_()
        at = [0, 0, 0]
        for m, n, k in sizes:
            part = []
            for i, (cols, rows) in enumerate(((m, k), (n, k), (n, m))):
                part.append(flat[i][at[i]:at[i] + cols * rows].view(cols, rows))
                at[i] += cols * rows
            blocks.append(part)
        return flat, blocks
    return [_uniform((cols, rows + case["pad"]), dtype, gen, case.get("spread", 0) if i < 2 else 0)
            for i, (cols, rows) in enumerate(_shapes(case))], None


def prepare(case, seed):
    arrays, blocks = _operands(case, seed)
    state = {"case": case, "ctx": _context(case["mode"]), "A": arrays[0], "B": arrays[1],
             "C": arrays[2]}
    if blocks is not None:
        specs = [dict(m=C.shape[1], n=C.shape[0], k=A.shape[1], A=A.data_ptr(), lda=A.shape[1],
                      B=B.data_ptr(), ldb=B.shape[1], C=C.data_ptr(), ldc=C.shape[1])
                 for A, B, C in blocks]
        state["batch"] = spla.Batch(state["ctx"], specs, ALPHA[case["type"]], 0.0,
                                    complex_=case["type"] == "z", opA=OPS[case["opA"]])
    elif case["where"] == "host":
        for name in "ABC":
            x = state[name]
            state[name] = torch.empty(x.shape, dtype=x.dtype, pin_memory=True).copy_(x)
    return state


def run(state):
    case, ctx = state["case"], state["ctx"]
    if case["call"] == "batch":
        state["batch"].execute()
        return state["C"]
    A, B, C = state["A"], state["B"], state["C"]
    lda, ldb, ldc = A.shape[1], B.shape[1], C.shape[1]
    m, n, k, alpha, beta = case["m"], case["n"], case["k"], ALPHA[case["type"]], case["beta"]
    if case["call"] == "gemm":
        spla.gemm(OPS[case["opA"]], OPS[case["opB"]], m, n, k, alpha, A, lda, B, ldb, beta, C,
                  ldc, ctx)
    elif case["call"] == "sbs":
        spla.pgemm_sbs(m, n, k, alpha, A, lda, B, ldb, 0, 0, _distribution(), beta, C, ldc, ctx)
    elif case["call"] == "ssb":
        spla.pgemm_ssb(m, n, k, OPS[case["opA"]], alpha, A, lda, B, ldb, beta, C, ldc,
                       case["row"], case["col"], _distribution(), ctx)
    else:
        fill = spla.FillMode.LOWER if case["fill"] == "L" else spla.FillMode.UPPER
        spla.pgemm_ssbtr(m, n, k, OPS[case["opA"]], alpha, A, lda, B, ldb, beta, C, ldc,
                         case["row"], case["col"], fill, _distribution(), ctx)
        return _triangle(case, C)
    return C


def _triangle(case, C):
    """The triangle that pgemm_ssbtr defines: the rest of C may or may not be computed."""
    return torch.triu(C) if case["fill"] == "L" else torch.tril(C)


def work(case):
    size = torch.empty(0, dtype=TYPES[case["type"]]).element_size()
    per = 8 if case["type"] in "cz" else 2
    sizes = _block_sizes(case) if case["call"] == "batch" else [(case["m"], case["n"], case["k"])]
    total = flops = 0.0
    for m, n, k in sizes:
        c = m * (n + 1) / 2 if case["call"] == "ssbtr" else m * n
        total += size * (m + n) * k
        total += size * c * (2 if case["beta"] else 1)
        flops += per * c * k
    return {"bytes": total, "flops": flops}


def exact(case, seed):
    arrays, blocks = _operands(case, seed)
    wide, alpha = WIDE[case["type"]], ALPHA[case["type"]]

    def product(A, B, opA, opB, m, n, k):
        # column-major: a stored (columns, rows) tensor is the transposed matrix
        A, B = A[:, :(m if opA == "N" else k)].to(wide), B[:, :(k if opB == "N" else n)].to(wide)
        a = A.T if opA == "N" else (A.conj() if opA == "C" else A)
        b = B.T if opB == "N" else (B.conj() if opB == "C" else B)
        return alpha * torch.matmul(a, b)

    if blocks is not None:
        return torch.cat([product(A, B, case["opA"], "N", C.shape[1], C.shape[0], A.shape[1])
                          .T.reshape(-1) for A, B, C in blocks])
    m, n, r, c = case["m"], case["n"], case["row"], case["col"]
    C = arrays[2].to(wide)
    C[c:c + n, r:r + m] = case["beta"] * C[c:c + n, r:r + m] + product(
        arrays[0], arrays[1], case["opA"], case["opB"], m, n, case["k"]).T
    C = _triangle(case, C) if case["call"] == "ssbtr" else C
    return C.cpu() if case["where"] == "host" else C
