"""Workloads of the framework as its users run them, for timing and comparison.

A reconstruction builds a system matrix for the measured channels of a scan,
attaches the transposed copy and runs MLEM iterations on it; a dynamic series
runs several frames on one matrix, usually stored in 16 bits; a training
program differentiates the projector; and a caller of the reference's own
interface builds a chunk of the matrix as CSR and multiplies with it.  The
cases are those calls, on the repository's scanners (two heads of 5x5 or 13x13
segments), grids (16^3 of 3 mm, 52^3 of 1 mm, 104^3 of 0.5 mm) and ray counts,
over scans of few or many angles, and on odd sizes in between.

A scan's data are Poisson counts of the line integrals of a seeded phantom
(ellipsoids on a round background) along the channels' centre lines, in closed
form; `rows` consecutive channels with counts are the measured ones.
"""
from __future__ import annotations

import math

import numpy as np
import torch

from epetreco_amd.api import OP_N, OP_T, VAL_BF16, VAL_F16, VAL_F32, Context
from epetreco_amd.geometry import MeasurementSetup, VoxelGrid
from epetreco_amd.projector import poisson_nll

STORAGE = {"f32": VAL_F32, "bf16": VAL_BF16, "f16": VAL_F16}
SEGMENT = (0.020, 0.004, 0.004)      # segment edges (x depth, y, z), metres
HEAD = 0.230                         # segment centres at x = -/+ HEAD


def _scan(name, kind, segments, angles, nx, ny, nz, voxel_um, rays, rows, **more):
    return {"name": name, "kind": kind, "segments": segments, "angles": angles, "nx": nx,
            "ny": ny, "nz": nz, "voxel_um": voxel_um, "rays": rays, "rows": rows, **more}


def listed():
    return [
        # the operator of the small scanner, rebuilt by a program that varies its geometry:
        # a few thousand short rows, where launches and allocations count
        _scan("build_small", "build", 5, 18, 16, 16, 16, 3000, 8, 11250),
        # the operator of one chunk of a full scan's measured channels (13x13 segments, 52^3)
        _scan("build_52", "build", 13, 180, 52, 52, 52, 1000, 64, 40000),
        # plain reconstruction on the small scanner: every kernel is a few microseconds
        _scan("mlem_small", "mlem", 5, 18, 16, 16, 16, 3000, 8, 9001, frames=1, storage="f32",
              iterations=10, graph=False),
        # plain FP32 reconstruction at 52^3, the largest listed case: a third of the full
        # scan's angles, the matrix resident in HBM, iterations replayed as a graph
        _scan("mlem_52", "mlem", 13, 60, 52, 52, 52, 1000, 64, 1100000, frames=1, storage="f32",
              iterations=4, graph=True),
        # a short dynamic series on the small scanner
        _scan("frames_small", "mlem", 5, 18, 16, 16, 16, 3000, 8, 9001, frames=5, storage="f32",
              iterations=10, graph=True),
        # the headline dynamic series: 32 frames, BF16 values with a row scale, 52^3
        _scan("frames_52_bf16", "mlem", 13, 24, 52, 52, 52, 1000, 64, 445000, frames=32,
              storage="bf16", iterations=2, graph=True),
        # an odd number of frames in the storage that meets the accuracy bar, a shorter scan
        _scan("frames_52_f16", "mlem", 13, 8, 52, 52, 52, 1000, 64, 150001, frames=13,
              storage="f16", iterations=3, graph=True),
        # the fine grid: 104^3 voxels, 32 rays, 8 frames of FP16 values
        _scan("frames_104_f16", "mlem", 13, 6, 104, 104, 104, 500, 32, 99000, frames=8,
              storage="f16", iterations=2, graph=True),
        # gradient of the Poisson loss through the projector (small scanner, 52^3, no
        # transposed copy): one step of a training program
        _scan("project_52", "project", 5, 18, 52, 52, 52, 1000, 8, 11250, frames=1,
              transposed=False),
        # the same for a batch of four images of a short 52^3 scan, transposed copy attached
        _scan("project_frames", "project", 13, 3, 52, 52, 52, 1000, 64, 50000, frames=4,
              transposed=True),
        # a whole reconstruction from the measured channels and counts: matrix, transposed
        # copy, sensitivity, 20 iterations (what the `reco` driver does once per scan)
        _scan("reco_52", "reco", 13, 6, 52, 52, 52, 1000, 64, 100000, iterations=20, graph=True),
        # the reference's own interface: one chunk as COO sorted to ECSR, forward and back
        # projection with the general CSR product
        _scan("chunk_52", "chunk", 13, 180, 52, 52, 52, 1000, 64, 2001),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """A case of the same kinds with other sizes: any scanner, grid and ray count between the
    listed ones, odd ones among them."""
    kind = rng.choice(["build", "mlem", "mlem", "frames", "frames", "frames", "project", "reco",
                       "chunk"])
    segments = rng.choice([5, 7, 9, 11, 13])
    # voxels per edge, drawn edge by edge about one size; the grid covers 48..52 mm
    n = _log(rng, 16, 104 if kind == "frames" else 64)
    nx, ny, nz = (max(12, int(n * rng.uniform(0.85, 1.0))) for _ in range(3))
    voxel_um = int(round(rng.uniform(48000.0, 52000.0) / n))
    rays = _log(rng, 5, 64)
    per_row = entries_per_row(voxel_um * 1e-6, rays)
    # entries: small scans to those of the listed cases of each kind
    lo, hi = {"build": (1e5, 3e7), "mlem": (1e5, 4e8), "frames": (1e5, 2e8),
              "project": (1e5, 4e7), "reco": (1e5, 8e7), "chunk": (1e5, 2e6)}[kind]
    rows = max(64, int(_log(rng, lo, hi) / per_row))
    per_angle = segments ** 4
    rows = min(rows, int(0.6 * 180 * per_angle))
    angles = min(180, max(1, -(-rows * 10 // (6 * per_angle))))
    case = _scan("", "mlem" if kind == "frames" else kind, segments, angles, nx, ny, nz, voxel_um,
                 rays, rows)
    del case["name"]
    if kind in ("mlem", "frames"):
        # single-frame scans stay FP32 mostly; series are mostly stored in 16 bits
        case["frames"] = 1 if kind == "mlem" else _log(rng, 2, 40)
        case["storage"] = rng.choice(["f32", "f32", "f16"] if kind == "mlem"
                                     else ["f32", "bf16", "f16"])
        case["iterations"] = rng.randint(2, 6)
        case["graph"] = rng.random() < 0.7
    elif kind == "project":
        case["frames"] = rng.choice([1, 1, 2, 3, 4, 7, 8])
        case["transposed"] = rng.random() < 0.5
    elif kind == "reco":
        case["iterations"] = rng.randint(5, 20)
        case["graph"] = True
    return case


# ------------------------------------------------------------------ inputs
def _geometry(case):
    seg = case["segments"]
    # a scan's angles are spread over the same circle, whatever their number (the small
    # scanner's over half of it)
    setup = MeasurementSetup(-HEAD, HEAD, case["angles"], seg, seg, seg, seg,
                             (180.0 if seg == 5 else 360.0) / case["angles"], *SEGMENT)
    d = case["voxel_um"] * 1e-6
    n = (case["nx"], case["ny"], case["nz"])
    grid = VoxelGrid(*(-0.5 * k * d for k in n), d, d, d, *n)
    return setup, grid


def _centre_lines(setup, ids):
    """Centres of both segments of every channel (two n x 3 FP64 tensors)."""
    p1 = setup.n1y
    p2 = p1 * setup.n1z
    p3 = p2 * setup.n0y
    p4 = p3 * setup.n0z
    th = (ids // p4).double() * (math.pi * setup.da / 180.0)
    t = ids % p4
    iz0, iy0 = t // p3, (t % p3) // p2
    iz1, iy1 = (t % p2) // p1, t % p1
    ends = []
    for px, iz, iy, nz, ny in ((setup.pos0x, iz0, iy0, setup.n0z, setup.n0y),
                               (setup.pos1x, iz1, iy1, setup.n1z, setup.n1y)):
        py = (iy.double() - 0.5 * (ny - 1)) * setup.segy
        pz = (iz.double() - 0.5 * (nz - 1)) * setup.segz
        ends.append(torch.stack([torch.cos(th) * px + torch.sin(th) * pz, py,
                                 -torch.sin(th) * px + torch.cos(th) * pz], 1))
    return ends


def _line_integrals(setup, grid, frames, seed):
    """Activity along every channel's centre line, (channels, frames): an ellipsoid that fills
    most of the grid, and six smaller ones that fade at their own rates."""
    rng = np.random.default_rng(seed)
    half = 0.46 * grid.dx * min(grid.nx, grid.ny, grid.nz)     # metres, inside the grid
    ids = torch.arange(setup.nchannels, device="cuda")
    p, q = _centre_lines(setup, ids)
    d = q - p
    length = d.norm(dim=1)

    def chord(centre, inv):      # length inside {|(x - centre) inv| <= 1}
        a = d * inv
        b = (p - centre) * inv
        A, B, C = (a * a).sum(1), (a * b).sum(1), (b * b).sum(1) - 1.0
        return 2.0 * torch.sqrt(torch.clamp(B * B - A * C, min=0.0)) / A * length

    def vec(v):
        return torch.tensor(list(v), dtype=torch.float64, device="cuda")

    fade = np.arange(frames)
    out = 0.05 * chord(vec((0, 0, 0)), vec((1 / half,) * 3))[:, None].repeat(1, frames)
    for _ in range(6):
        c = chord(half * vec(rng.uniform(-0.45, 0.45, 3)), 1.0 / (half * vec(rng.uniform(0.1, 0.55, 3))))
        act = rng.uniform(0.1, 1.0) * np.exp(-fade / rng.uniform(5.0, 50.0))
        out += c[:, None] * vec(act)[None, :]
    return out


def _counts(case, setup, grid, seed):
    """(channel ids of the `rows` measured channels, ascending; their counts, rows x frames)."""
    F, rows = case.get("frames", 1), case["rows"]
    gen = torch.Generator(device="cuda").manual_seed(seed)
    rate = _line_integrals(setup, grid, F, seed)
    # about three counts per channel and frame, as a scan of 1e7 counts has
    y = torch.poisson((rate * (3.0 / rate.mean(0))).float(), generator=gen)
    ids = torch.nonzero(y.sum(1) > 0)[:, 0]
    if ids.numel() < rows:       # the channels with the highest rates then
        ids = torch.topk(rate.sum(1), rows).indices.sort().values
    start = int(torch.randint(ids.numel() - rows + 1, (1,), generator=gen, device="cuda"))
    ids = ids[start:start + rows]
    return ids.to(torch.int32), y[ids].contiguous()


class State:
    pass


def prepare(case, seed):
    st = State()
    st.case = case
    setup, grid = _geometry(case)
    kind = case["kind"]
    st.ctx = Context(0)
    st.ctx.set_geometry(setup, grid, nrays=case["rays"], seed=seed)
    st.rows, st.y = _counts(case, setup, grid, seed)
    V = grid.nvoxels
    gen = torch.Generator(device="cuda").manual_seed(seed + 1)
    if kind in ("mlem", "project"):
        st.A = st.ctx.sm_build(st.rows)
        if case.get("storage", "f32") != "f32":
            A32 = st.A
            st.A = A32.convert(STORAGE[case["storage"]])
            A32.close()
    if kind == "mlem":
        F = case["frames"]
        st.s = st.A.colsum_f64().float()
        st.A.attach_transpose()
        st.x0 = torch.full((V,) if F == 1 else (V, F), 1.0 / V, device="cuda")
        if F == 1:
            st.y = st.y[:, 0].contiguous()
        # the first iteration builds the plans that the matrix keeps
        st.ctx.mlem(st.A, st.y, st.s, st.x0.clone(), 1, use_graph=case["graph"])
    elif kind == "project":
        F = case["frames"]
        if case["transposed"]:
            st.A.attach_transpose()
        shape = (V,) if F == 1 else (V, F)
        st.x = (torch.rand(shape, generator=gen, device="cuda") + 0.5).requires_grad_(True)
        if F == 1:
            st.y = st.y[:, 0].contiguous()
        torch.autograd.grad(poisson_nll(st.A, st.x, st.y), st.x)   # builds the plans
    elif kind == "reco":
        st.y = st.y[:, 0].contiguous()
        st.x0 = torch.full((V,), 1.0 / V, device="cuda")
    elif kind == "chunk":
        st.y = st.y[:, 0].contiguous()
        st.x = torch.rand(V, generator=gen, device="cuda") + 0.5
        st.capacity = int(case["rows"] * _candidates(grid))
    else:
        st.capacity = int(case["rows"] * min(V, 2.0 * entries_per_row(grid.dx, case["rays"]) + 64))
    if kind in ("build", "chunk"):
        # where the program collects the entries, zeros past the last one
        st.col = torch.zeros(st.capacity, dtype=torch.int32, device="cuda")
        st.val = torch.zeros(st.capacity, dtype=torch.float32, device="cuda")
    return st


def _candidates(grid):
    """A bound on the candidate voxels of one channel: a tube of the candidate radius (half the
    diagonals of a segment and of a voxel, 10.5 mm and more) over the grid's space diagonal."""
    d = grid.dx
    radius = 0.5 * (math.sqrt(sum(e * e for e in SEGMENT)) + math.sqrt(3.0) * d)
    diag = d * math.sqrt(grid.nx ** 2 + grid.ny ** 2 + grid.nz ** 2)
    return min(grid.nvoxels, math.pi * (radius + d) ** 2 * (diag + 2 * radius) / d ** 3)


# ------------------------------------------------------------------ the calls
def run(st):
    case = st.case
    kind = case["kind"]
    if kind == "build":
        A = st.ctx.sm_build(st.rows)
        rowptr, col, val, _ = A.to_torch()
        A.close()
        st.col[:A.nnz] = col
        st.val[:A.nnz] = val
        return {"rowptr": rowptr, "col": st.col, "val": st.val}
    if kind == "mlem":
        x = st.x0.clone()
        loglik, _ = st.ctx.mlem(st.A, st.y, st.s, x, case["iterations"], use_graph=case["graph"])
        # log-likelihoods of FP32 projections, kept to FP32
        return {"x": x, "loglik": loglik.astype(np.float32)}
    if kind == "project":
        loss = poisson_nll(st.A, st.x, st.y)
        (g,) = torch.autograd.grad(loss, st.x)
        return {"loss": loss.detach(), "grad": g}
    if kind == "reco":
        A = st.ctx.sm_build(st.rows)
        s = A.colsum_f64()
        A.attach_transpose()
        x = st.x0.clone()
        loglik, _ = st.ctx.mlem(A, st.y, s.float(), x, case["iterations"], use_graph=case["graph"])
        A.close()
        return {"x": x, "s": s, "loglik": loglik.astype(np.float32)}
    if kind == "chunk":
        ctx, m, n = st.ctx, case["rows"], st.x.numel()
        rowptr, col, val, nnz = ctx.systemMatrixCalculation(st.rows, ctx.setup.nchannels, st.capacity)
        yhat = ctx.csrmv(OP_N, m, n, 1.0, val, rowptr, col, st.x, 0.0, torch.zeros_like(st.y))
        e = ctx.divides(torch.empty_like(yhat), st.y, yhat)
        c = ctx.csrmv(OP_T, m, n, 1.0, val, rowptr, col, e, 0.0, torch.zeros_like(st.x))
        st.col[:nnz] = col
        st.val[:nnz] = val
        return {"rowptr": rowptr, "col": st.col, "val": st.val, "yhat": yhat, "c": c}
    raise ValueError(kind)


# ------------------------------------------------------------------ what it takes
def entries_per_row(d, rays):
    """Mean voxels that a channel's `rays` lines cross, voxel edge d (metres): about 57 mm of
    lines in a tube 3 mm wide; 57, 406, 916 and 3,031 entries per row measured on the
    repository's four workloads, 58, 371, 899 and 2,794 here."""
    k = ((0.003 + d) / d) ** 2
    return 0.057 / d * k * (1.0 - math.exp(-rays * 1.05 / k))


def work(case):
    """Matrix entries (value and int32 column) once per product, the row pointers, and the
    vectors; two operations per entry and frame."""
    V = case["nx"] * case["ny"] * case["nz"]
    d = case["voxel_um"] * 1e-6
    m, kind = case["rows"], case["kind"]
    nnz = m * entries_per_row(d, case["rays"])
    F = case.get("frames", 1)
    vb = 4 if case.get("storage", "f32") == "f32" else 2
    product = nnz * (vb + 4) + 8 * (m + 1) + 4 * F * (m + V)
    iteration = 2 * product + F * (8 * m + 16 * V)
    # a ray meets about 1.5 voxels per voxel edge of its way; 30 operations for each
    generate = {"bytes": nnz * 8 + 8 * m, "flops": m * case["rays"] * 1.5 * 0.057 / d * 30}
    if kind == "build":
        return generate
    if kind == "mlem":
        k = case["iterations"]
        return {"bytes": k * iteration, "flops": k * 4.0 * nnz * F}
    if kind == "project":
        return {"bytes": 2 * product, "flops": 4.0 * nnz * F}
    if kind == "reco":
        k = case["iterations"]
        return {"bytes": generate["bytes"] + 2 * nnz * 8 + k * iteration,
                "flops": generate["flops"] + k * 4.0 * nnz}
    # chunk: all candidates are kept; one (row, column, value) triplet written, then sorted
    # (read and written once), and two products
    grid = _geometry(case)[1]
    cand = m * 0.35 * _candidates(grid)
    return {"bytes": cand * (12 + 24 + 2 * 8) + 8 * m, "flops": generate["flops"] + cand * (30 + 4)}


# ------------------------------------------------------------------ 64-bit values
CHUNK = 1 << 25    # entries times frames held at once


def _csr(A):
    """A's stored operator: row pointers, columns, FP64 values of a range of entries."""
    rowptr, col, val, scale = A.to_torch()
    row = torch.repeat_interleave(torch.arange(A.m, device="cuda", dtype=torch.int32),
                                  rowptr[1:] - rowptr[:-1])

    def value(a, b):
        v = val[a:b]
        if A.value_type == VAL_F32:
            return v.double()
        v = v.view(torch.bfloat16 if A.value_type == VAL_BF16 else torch.float16).double()
        return v * scale[row[a:b]].double()

    return row, col, value


def _times(csr, m, X):
    row, col, value = csr
    Y = torch.zeros(m, X.shape[1], dtype=torch.float64, device="cuda")
    step = CHUNK // X.shape[1]
    for a in range(0, col.numel(), step):
        b = min(col.numel(), a + step)
        Y.index_add_(0, row[a:b], value(a, b)[:, None] * X[col[a:b]])
    return Y


def _times_t(csr, n, E):
    row, col, value = csr
    C = torch.zeros(n, E.shape[1], dtype=torch.float64, device="cuda")
    step = CHUNK // E.shape[1]
    for a in range(0, col.numel(), step):
        b = min(col.numel(), a + step)
        C.index_add_(0, col[a:b], value(a, b)[:, None] * E[row[a:b]])
    return C


def _mlem64(csr, m, y, s, x, iterations):
    ll = []
    s = s / s.sum()
    for _ in range(iterations):
        yhat = _times(csr, m, x)
        hit = yhat > 0
        safe = torch.where(hit, yhat, torch.ones_like(yhat))
        ll.append(torch.where(hit, y * torch.log(safe) - yhat, torch.zeros_like(y)).sum(0))
        c = _times_t(csr, x.shape[0], torch.where(hit, y / safe, torch.zeros_like(y)))
        x = x * c / torch.where(s == 0, torch.ones_like(s), s)[:, None]
        x = x / x.sum(0)
    return x, torch.stack(ll)


def _philox(c0, c1, c2, key):
    """Philox4x32-10 on int64 tensors, counters (c0, c1, c2, 0): four words."""
    m32 = 0xFFFFFFFF

    def mul(a, b):      # 32 x 32 -> (high, low)
        lo = a * (b & 0xFFFF)
        hi = a * (b >> 16) + (lo >> 16)
        return hi >> 16, ((hi << 16) | (lo & 0xFFFF)) & m32

    c = [c0, c1, torch.full_like(c0, c2), torch.zeros_like(c0)]
    k0, k1 = key & m32, (key >> 32) & m32
    for _ in range(10):
        h0, l0 = mul(c[0], 0xD2511F53)
        h1, l1 = mul(c[2], 0xCD9E8D57)
        c = [h1 ^ c[1] ^ k0, l1, h0 ^ c[3] ^ k1, l0]
        k0, k1 = (k0 + 0x9E3779B9) & m32, (k1 + 0xBB67AE85) & m32
    return c


def _values64(setup, grid, rays, seed, channel, col):
    """Mean length of each channel's rays inside each voxel."""
    out = torch.empty(col.numel(), dtype=torch.float64, device="cuda")
    for a in range(0, col.numel(), 1 << 22):
        ch, v = channel[a:a + (1 << 22)].long(), col[a:a + (1 << 22)].long()
        p4 = setup.n1y * setup.n1z * setup.n0y * setup.n0z
        th = (ch // p4).double() * (math.pi * setup.da / 180.0)
        sn, cs = torch.sin(th), torch.cos(th)
        c0, c1 = _centre_lines(setup, ch)
        box = [(v // (grid.ny * grid.nz), grid.ox, grid.dx), (v // grid.nz % grid.ny, grid.oy, grid.dy),
               (v % grid.nz, grid.oz, grid.dz)]
        acc = torch.zeros(ch.numel(), dtype=torch.float64, device="cuda")
        for r in range(rays):
            u = _philox(torch.full_like(ch, r), ch, 0, seed) + _philox(torch.full_like(ch, r), ch, 1, seed)
            u = [((w >> 8) | 1).double() * 2.0 ** -24 - 0.5 for w in u[:6]]
            ends = []
            for c, (a0, a1, a2) in ((c0, u[:3]), (c1, u[3:])):
                a0, a1, a2 = a0 * setup.segx, a1 * setup.segy, a2 * setup.segz
                ends.append((c[:, 0] + cs * a0 + sn * a2, c[:, 1] + a1, c[:, 2] - sn * a0 + cs * a2))
            lo = torch.full_like(acc, -1e30)
            hi = torch.full_like(acc, 1e30)
            sq = torch.zeros_like(acc)
            for (i, o, d), p, q in zip(box, *ends):
                den = q - p
                t0 = (o + i.double() * d - p) / den
                t1 = (o + (i + 1).double() * d - p) / den
                lo = torch.maximum(lo, torch.minimum(t0, t1))
                hi = torch.minimum(hi, torch.maximum(t0, t1))
                sq += den * den
            acc += torch.clamp(hi - lo, min=0.0) * torch.sqrt(sq)
        out[a:a + (1 << 22)] = acc / rays
    return out


def exact(case, seed):
    """The outputs in 64 bits.  The operator is the one the call was given (its entries as
    stored); the entries of a newly built one are recomputed from the rays."""
    kind, m = case["kind"], case["rows"]
    nnz = m * entries_per_row(case["voxel_um"] * 1e-6, case["rays"])
    if nnz * case.get("frames", 1) * case.get("iterations", 1) > 3e10 or \
            (kind == "build" and nnz * case["rays"] > 4e9):
        return None      # about 20 seconds
    st = prepare(case, seed)
    if kind == "build":
        A = st.ctx.sm_build(st.rows)
        row, col, _ = _csr(A)
        val = torch.zeros(st.capacity, dtype=torch.float64, device="cuda")
        val[:A.nnz] = _values64(st.ctx.setup, st.ctx.grid, case["rays"], seed, st.rows[row.long()], col)
        return {"rowptr": None, "col": None, "val": val}
    if kind in ("mlem", "reco"):
        F = case.get("frames", 1)
        A = st.A if kind == "mlem" else st.ctx.sm_build(st.rows)
        csr = _csr(A)
        s = _times_t(csr, A.n, torch.ones(m, 1, dtype=torch.float64, device="cuda"))[:, 0]
        s_in = s.float().double()       # the sensitivity is handed over in FP32
        x, ll = _mlem64(csr, m, st.y.double().reshape(m, F), s_in, st.x0.double().reshape(-1, F),
                        case["iterations"])
        out = {"x": x.reshape(st.x0.shape), "loglik": ll}
        return {**out, "s": s} if kind == "reco" else out
    if kind == "project":
        csr = _csr(st.A)
        X = st.x.detach().double().reshape(st.A.n, -1)
        y = st.y.double().reshape(m, -1)
        yhat = _times(csr, m, X)
        loss = (yhat - y * torch.log(yhat + 1e-8)).sum()
        g = _times_t(csr, st.A.n, 1.0 - y / (yhat + 1e-8))
        return {"loss": loss, "grad": g.reshape(st.x.shape)}
    if kind == "chunk":
        got = run(st)
        rowptr = got["rowptr"].long()
        nnz = int(rowptr[-1])
        col, val = got["col"][:nnz], got["val"]
        row = torch.repeat_interleave(torch.arange(m, device="cuda", dtype=torch.int32),
                                      rowptr[1:] - rowptr[:-1])
        csr = (row, col, lambda a, b: val[a:b].double())
        yhat = _times(csr, m, st.x.double()[:, None])
        c = _times_t(csr, st.x.numel(), st.y.double()[:, None] / yhat)
        return {"rowptr": None, "col": None, "val": None, "yhat": yhat[:, 0], "c": c[:, 0]}
    return None
