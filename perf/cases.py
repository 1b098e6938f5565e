"""What the library is measured on: every transfer pattern through its public entry point, at the sizes of the benchmark
configurations, at ordinary and at small ones.

A case names a pattern ("kind") and its sizes.  Every call uses the entry point's default variant, the one a program gets
that does not choose a buffering idiom itself.  Inputs come from the library's own seeded generators: uniform [-1, 1)
floats, normal bf16 values, uniform element indices of which one in ten repeats a recent one.
"""
import math

import torch

from cudadma_amd import examples, workloads

RECORD = workloads.REC_FLOATS            # floats of a 128-byte record
TILE = workloads.RECS_PER_TILE           # records per gathered or scattered tile
COPY_TILE = workloads.SEQ_TILE_BYTES
PAD = 2 * workloads.STENCIL_RADIUS       # ghost cells per dimension, both stencils

# largest sizes: those of the benchmark
MOST_COPY_TILES = (1 << 30) // COPY_TILE
MOST_RECORDS = 32 << 20                  # a table of 4 GiB
MOST_INDICES = 32 << 20
MOST_SIDE = 16384
MOST_GRID = 512
MOST_PRODUCTS = 4096 ** 3
MOST_CELLS_2D = 960 * 160 * 200


def listed():
    return [
        # the headline of the benchmark: a matrix that no cache holds
        {"name": "transpose_16384", "kind": "transpose", "n": 16384},
        # an ordinary matrix, 33 tiles a side: the tiles divide by neither the compute units nor a power of two
        {"name": "transpose_2112", "kind": "transpose", "n": 2112},
        # a staging copy of the size that the read-bandwidth program uses
        {"name": "copy_64MiB", "kind": "copy", "tiles": 4096},
        # table lookups with a reduction over 32 records, as embedding bags do: the benchmark's table and index list
        {"name": "gather_rowsum_32Mi", "kind": "gather_rowsum", "records": 4 << 20, "indices": 32 << 20},
        # a small batch of table lookups: the call itself counts
        {"name": "gather_copy_160", "kind": "gather_copy", "records": 65536, "indices": 160},
        # a permutation of a 512 MiB table, the reverse of the gather
        {"name": "scatter_4Mi", "kind": "scatter", "records": 4 << 20, "indices": 4 << 20},
        # one sweep of a wave-equation solver: the benchmark's grid
        {"name": "halo_512", "kind": "halo", "nx": 512, "ny": 512, "nz": 512},
        # the same sweep on a grid of an ordinary subdomain, not a cube
        {"name": "halo_192x256x130", "kind": "halo", "nx": 192, "ny": 256, "nz": 130},
        # the benchmark's product
        {"name": "gemm_4096", "kind": "gemm", "m": 4096, "n": 4096, "k": 4096},
        # an ordinary product with odd numbers of tiles in every dimension
        {"name": "gemm_1408x2176x1920", "kind": "gemm", "m": 1408, "n": 2176, "k": 1920},
        # matrix times vector, as in the sgemv program
        {"name": "sgemv_4096", "kind": "sgemv", "n": 4096, "m": 4096},
        # cross average over the slices of a volume of two components: the volume of the stencil program
        {"name": "stencil2d_960x160x200", "kind": "stencil2d", "dimx": 960, "dimy": 160, "dimz": 200, "full_cross": False},
    ]


def _spread(rng, lo, hi, step=1):
    """A multiple of `step` in [lo, hi], spread over the logarithm."""
    v = math.exp(rng.uniform(math.log(lo), math.log(hi)))
    return max(lo, min(hi, int(round(v / step)) * step))


def draw(rng):
    kind = rng.choice(("transpose", "copy", "gather_rowsum", "gather_copy", "scatter", "halo", "gemm", "sgemv", "stencil2d"))
    if kind == "transpose":
        return {"kind": kind, "n": _spread(rng, 64, MOST_SIDE, 64)}
    if kind == "copy":
        return {"kind": kind, "tiles": _spread(rng, 1, MOST_COPY_TILES)}
    if kind in ("gather_rowsum", "gather_copy"):
        most = MOST_INDICES // 2 if kind == "gather_rowsum" else MOST_INDICES // 4
        return {"kind": kind, "records": _spread(rng, 1024, MOST_RECORDS), "indices": _spread(rng, TILE, most, TILE)}
    if kind == "scatter":
        records = _spread(rng, 1024, MOST_RECORDS // 4)
        return {"kind": kind, "records": records, "indices": _spread(rng, TILE, records // TILE * TILE, TILE)}
    if kind == "halo":
        return {"kind": kind, "nx": _spread(rng, 32, MOST_GRID, 32), "ny": _spread(rng, 32, MOST_GRID, 32),
                "nz": _spread(rng, 4, MOST_GRID)}
    if kind == "gemm":
        m, n = _spread(rng, 128, 8192, 128), _spread(rng, 128, 8192, 128)
        return {"kind": kind, "m": m, "n": n, "k": _spread(rng, 128, min(8192, MOST_PRODUCTS // (m * n) // 128 * 128), 128)}
    if kind == "sgemv":
        return {"kind": kind, "n": _spread(rng, 128, 16384), "m": _spread(rng, 32, 16384, 32)}
    dimx, dimy = _spread(rng, 32, 1024, 32), _spread(rng, 4, 512, 4)
    return {"kind": kind, "dimx": dimx, "dimy": dimy, "dimz": _spread(rng, 2, max(2, min(256, MOST_CELLS_2D // (dimx * dimy)))),
            "full_cross": rng.random() < 0.5}


def _uniform(shape, seed):
    return workloads.fill_uniform(torch.empty(shape, dtype=torch.float32, device="cuda"), seed)


def _normal(shape, seed):
    return workloads.fill_normal_bf16(torch.empty(shape, dtype=torch.bfloat16, device="cuda"), seed)


def _out(*shape):
    return torch.zeros(shape, dtype=torch.float32, device="cuda")


def _leading(n):
    return (n + 127) // 128 * 128          # columns start on whole groups of 128 rows, which the staged matrix needs


def prepare(case, seed):
    s = 4 * seed
    kind = case["kind"]
    if kind == "transpose":
        n = case["n"]
        args = (_uniform((n, n), s), _out(n, n))
    elif kind == "copy":
        floats = case["tiles"] * COPY_TILE // 4
        args = (_uniform((floats,), s), _out(floats))
    elif kind in ("gather_rowsum", "gather_copy"):
        table = _uniform((case["records"], RECORD), s)
        idx = workloads.fill_indices(torch.empty(case["indices"], dtype=torch.int32, device="cuda"), case["records"], s + 1)
        args = (table, idx, _out(case["indices"] // (TILE if kind == "gather_rowsum" else 1), RECORD))
    elif kind == "scatter":
        g = torch.Generator(device="cuda").manual_seed(s + 1)
        idx = torch.randperm(case["records"], generator=g, device="cuda", dtype=torch.int32)[:case["indices"]].contiguous()
        args = (_uniform((case["indices"], RECORD), s), idx, _out(case["records"], RECORD))
    elif kind == "halo":
        nx, ny, nz = case["nx"], case["ny"], case["nz"]
        args = (_uniform((nz + PAD, ny + PAD, nx + PAD), s), _out(nz, ny, nx))
    elif kind == "gemm":
        m, n, k = case["m"], case["n"], case["k"]
        args = (_normal((m, k), s), _normal((k, n), s + 1), _out(m, n))
    elif kind == "sgemv":
        n, m = case["n"], case["m"]
        args = (1.25, _uniform((m, _leading(n)), s), _uniform((m,), s + 1), _out(n), n)
    else:
        shape = (case["dimz"] + PAD, case["dimy"] + PAD, case["dimx"] + PAD, 2)
        args = (_uniform(shape, s), _out(*shape))
    return {"case": case, "args": args}


def run(state):
    kind, args = state["case"]["kind"], state["args"]
    if kind == "transpose":
        return workloads.strided_transpose(*args)
    if kind == "copy":
        return workloads.sequential_copy(*args)
    if kind == "gather_rowsum":
        return workloads.gather_rowsum(*args)
    if kind == "gather_copy":
        return workloads.gather_copy(*args)
    if kind == "scatter":
        return workloads.scatter_copy(*args)
    if kind == "halo":
        return workloads.halo_stencil(*args)
    if kind == "gemm":
        return workloads.gemm_bf16(*args)
    if kind == "sgemv":
        return examples.sgemv(*args)
    return examples.stencil2d(*args, full_cross=state["case"]["full_cross"])


def work(case):
    kind = case["kind"]
    if kind == "transpose":
        return {"bytes": 8 * case["n"] ** 2, "flops": 0}
    if kind == "copy":
        return {"bytes": 2 * case["tiles"] * COPY_TILE, "flops": 0}
    if kind in ("gather_rowsum", "gather_copy"):
        r, i = case["records"], case["indices"]
        touched = -r * math.expm1(-0.9 * i / r)          # different records among i uniform draws, one in ten a repeat
        rows = i // TILE if kind == "gather_rowsum" else i
        return {"bytes": int(4 * i + 4 * RECORD * (touched + rows)), "flops": RECORD * (i - rows) if kind == "gather_rowsum" else 0}
    if kind == "scatter":
        return {"bytes": (4 + 8 * RECORD) * case["indices"], "flops": 0}
    if kind == "halo":
        nx, ny, nz = case["nx"], case["ny"], case["nz"]
        # the padded corner columns are never read: one centre block and a slab of four planes on every face
        read = nx * ny * nz + PAD * (nx * ny + ny * nz + nx * nz)
        return {"bytes": 4 * (read + nx * ny * nz), "flops": 29 * nx * ny * nz}
    if kind == "gemm":
        m, n, k = case["m"], case["n"], case["k"]
        return {"bytes": 2 * (m * k + k * n) + 4 * m * n, "flops": 2 * m * n * k}
    if kind == "sgemv":
        n, m = case["n"], case["m"]
        return {"bytes": 4 * (n * m + n + m), "flops": 2 * n * m}
    dimx, dimy, dimz = case["dimx"], case["dimy"], case["dimz"]
    reach = PAD if case["full_cross"] else PAD - 2       # three or four neighbours on each arm
    return {"bytes": 8 * dimz * (2 * dimx * dimy + reach * (dimx + dimy)), "flops": 2 * dimz * dimx * dimy * (2 * reach + 2)}


def tolerance(case):
    """Bytes that are only moved are exact.  Sums in 32 bits: about four times what the same sums in 64 bits differ by
    (measured, relative in the 2-norm and largest: products 5.7e-7 and 4e-6 at k = 8192, matrix times vector 2.3e-6 and 1.1e-5
    at m = 16384, row sums and stencils up to 1.1e-7 and 5.8e-7)."""
    kind = case["kind"]
    if kind in ("transpose", "copy", "gather_copy", "scatter"):
        return "exact"
    if kind == "gemm":
        return {"rel": 2.5e-6, "max": 1.6e-5}
    if kind == "sgemv":
        return {"rel": 1e-5, "max": 5e-5}
    return {"rel": 5e-7, "max": 2.5e-6}
