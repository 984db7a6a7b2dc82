"""Performance cases of the single-rank 3D transforms: what a user's program has this library do.

A case names one transform (or convolution, reshape, mixed-size batch), its box, element type and
orders.  listed() holds one case of each use, draw() more of the same ranges; prepare() makes the
plan and the arrays a program keeps, run() is one pass through the Python binding, exact() the same
result in 64 bits from torch.fft, cosine sums through FFTs, or DFT matrices.
"""
import math

import torch

import heffte_amd as heffte

REAL = {"c64": torch.float32, "c128": torch.float64, "f32": torch.float32, "f64": torch.float64}
COMPLEX = {"c64": torch.complex64, "c128": torch.complex128, "f32": torch.complex64, "f64": torch.complex128}
WIDTH = {"c64": 8, "c128": 16, "f32": 4, "f64": 8}

# sides of the mixed-size batches (the 17 smooth lengths of the benchmark's batch)
MIXED_SIDES = [16, 20, 24, 27, 28, 32, 40, 45, 48, 56, 63, 64, 80, 96, 105, 112, 128]
ORDERS = ["012", "021", "102", "120", "201", "210"]


def _fft(name, use, nx, ny, nz, dtype, out_order="012", in_order="012", batch=1, passes="pair", scaling="full", axis=0):
    return {"name": name, "use": use, "nx": nx, "ny": ny, "nz": nz, "dtype": dtype, "in_order": in_order,
            "out_order": out_order, "batch": batch, "passes": passes, "scaling": scaling, "axis": axis,
            "form": "fp32"}


def listed():
    return [
        # the smallest calls: one small box, where launches and host work are all there is
        _fft("c2c_32", "c2c", 32, 32, 32, "c64", passes="forward", scaling="none"),
        # grid of a plane-wave code: 7-smooth sides near 100, complex<double>, potential applied
        # between forward and backward
        _fft("c2c_grid", "c2c", 90, 100, 108, "c128"),
        # many equal boxes in one call (bands or right-hand sides of such a code)
        _fft("c2c_many", "c2c", 48, 60, 72, "c64", batch=40),
        # the headline transform
        _fft("c2c_512", "c2c", 512, 512, 512, "c64", out_order="120", scaling="symmetric"),
        # a large box with smooth sides that are no powers of two, transposed output
        _fft("c2c_large", "c2c", 384, 400, 320, "c128", out_order="210", scaling="none", passes="forward"),
        # real data of a turbulence or particle-mesh code: the large power-of-two box ...
        _fft("r2c_large", "r2c", 1024, 1024, 512, "f32"),
        # ... and a middle one with odd sides, halved along another axis
        _fft("r2c_odd", "r2c", 225, 180, 147, "f64", in_order="102", out_order="102", axis=1),
        # cosine transforms of a Poisson solver
        _fft("cos_256", "cos", 256, 256, 256, "f64"),
        # sine transforms on a ragged grid, in single precision
        _fft("sin_ragged", "sin", 150, 127, 96, "f32", out_order="120"),
        # 1000 boxes of mixed sizes in one batch
        {"name": "mixed_batch", "use": "mixed", "count": 1000, "small": 0.0, "dtype": "c64", "sides_seed": 4},
        # circular convolution of two fields
        _fft("convolve_mid", "convolve", 256, 240, 250, "c64", out_order="210"),
        # a reshape alone
        _fft("reshape", "reshape", 300, 500, 400, "c64", out_order="210"),
    ]


def _smooth(n):
    for p in (2, 3, 5, 7):
        while n % p == 0:
            n //= p
    return n == 1


def draw(rng):
    use = rng.choices(["c2c", "r2c", "cos", "sin", "cos1", "convolve", "reshape", "mixed"],
                      [38, 18, 7, 5, 4, 8, 8, 12])[0]
    if use == "mixed":
        return {"use": use, "count": int(2 ** rng.uniform(4, 9.5)), "small": rng.choice([0.0, 0.0, 0.2]),
                "dtype": rng.choice(["c64", "c64", "c128"]), "sides_seed": rng.randrange(10 ** 6)}
    volume = 2 ** rng.uniform(12, 23.5)
    sides = []
    for d in range(3):
        want = volume ** (1 / 3) * 2 ** rng.uniform(-0.7, 0.7)
        n = max(4, round(want))
        kind = rng.random()
        if kind < 0.2:  # a power of two
            n = 2 ** max(2, round(math.log2(want)))
        elif kind < 0.85:  # a 7-smooth length
            while not _smooth(n):
                n += 1
        elif n > 200:  # any length, primes among them
            n = rng.randint(64, 200)
        sides.append(n)
    if use == "reshape":
        dtype = rng.choice(["f32", "f64", "c64", "c128"])
    elif use in ("c2c", "convolve"):
        dtype = rng.choice(["c64", "c64", "c128"])
    else:
        dtype = rng.choice(["f32", "f64"])
    form = "fp32"
    if use == "c2c" and dtype == "c64" and rng.random() < 0.1:
        # the split-precision form of the 512-point passes
        form, sides[rng.randrange(3)] = "split_fp16", 512
    count = sides[0] * sides[1] * sides[2]
    batch = 1 if rng.random() < 0.8 else max(1, int(2 ** rng.uniform(1, 6) * min(1.0, 2 ** 18 / count)))
    in_order = rng.choice(ORDERS) if rng.random() < 0.3 else "012"
    out_order = rng.choice(ORDERS) if rng.random() < 0.5 else in_order
    return {"use": use, "nx": sides[0], "ny": sides[1], "nz": sides[2], "dtype": dtype, "in_order": in_order,
            "out_order": out_order, "batch": batch, "passes": rng.choice(["pair", "forward"]),
            "scaling": rng.choice(["full", "full", "symmetric"]), "axis": rng.randrange(3),
            "form": form}


# ------------------------------------------------------------------ sizes

def _box(case, order):
    return heffte.box3d([0, 0, 0], [case["nx"] - 1, case["ny"] - 1, case["nz"] - 1], [int(c) for c in order])


def _mixed_sizes(case):
    g = torch.Generator()
    g.manual_seed(case["sides_seed"])
    small = torch.rand(case["count"], generator=g).tolist()
    pick = torch.randint(0, len(MIXED_SIDES), (case["count"], 3), generator=g).tolist()
    odd = torch.randint(1, 41, (case["count"], 3), generator=g).tolist()
    return [tuple(o) if s < case["small"] else tuple(MIXED_SIDES[i] for i in p)
            for s, p, o in zip(small, pick, odd)]


def _half(case):
    n = [case["nx"], case["ny"], case["nz"]]
    n[case["axis"]] = n[case["axis"]] // 2 + 1
    return n[0] * n[1] * n[2]


def work(case):
    w = WIDTH[case["dtype"]]
    if case["use"] == "mixed":
        sizes = _mixed_sizes(case)
        total = sum(a * b * c for a, b, c in sizes)
        flops = sum(5.0 * a * b * c * math.log2(max(2, a * b * c)) for a, b, c in sizes)
        return {"bytes": 2.0 * 2 * w * total, "flops": 2 * flops}
    n = case["nx"] * case["ny"] * case["nz"]
    moved, flops = 2.0 * w * n, 5.0 * n * math.log2(n)
    if case["use"] == "reshape":
        flops = 0.0
    elif case["use"] == "r2c":
        moved, flops = float(w * n + 2 * w * _half(case)), flops / 2
    elif case["use"] in ("cos", "sin", "cos1"):
        flops /= 2
    elif case["use"] == "convolve":
        moved, flops = 3.0 * w * n, 3 * flops + 6.0 * n
    times = case["batch"] * (2 if case["passes"] == "pair" and case["use"] not in ("reshape", "convolve") else 1)
    return {"bytes": moved * times, "flops": flops * times}


def tolerance(case):
    if case["use"] == "reshape":
        return "exact"
    # four times the largest error measured against exact(): 3.5e-7 in single and 7e-16 in double precision
    return {"rel": 1.4e-6 if case["dtype"] in ("c64", "f32") else 2.8e-15}


# ------------------------------------------------------------------ inputs

def _values(shape, dtype, seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    return torch.randn(shape, dtype=dtype, device="cuda", generator=g)


def _input(case, seed):
    """The input arrays: flat, stored in the case's input order, transforms of a batch back to back."""
    if case["use"] == "mixed":
        return [_values(sum(a * b * c for a, b, c in _mixed_sizes(case)), COMPLEX[case["dtype"]], seed)]
    n = case["batch"] * case["nx"] * case["ny"] * case["nz"]
    real = case["dtype"] in ("f32", "f64")
    x = _values(n, REAL[case["dtype"]] if real else COMPLEX[case["dtype"]], seed)
    return [x, _values(n, x.dtype, seed + 7919)] if case["use"] == "convolve" else [x]


def prepare(case, seed):
    arrays = _input(case, seed)
    x = arrays[0]
    if case["use"] == "mixed":
        return {"case": case, "plan": heffte.batch_plan(_mixed_sizes(case)), "x": x, "y": torch.empty_like(x),
                "z": torch.empty_like(x)}
    inbox, outbox = _box(case, case["in_order"]), _box(case, case["out_order"])
    state = {"case": case, "x": x, "y": torch.empty_like(x), "z": torch.empty_like(x),
             "scaling": getattr(heffte.scale, case["scaling"]), "inbox": inbox}
    if case["use"] == "reshape":
        return state
    mi355 = heffte.backend.mi355
    work_type = COMPLEX[case["dtype"]]
    if case["use"] in ("c2c", "convolve"):
        plan = heffte.fft3d(mi355, inbox, outbox)
        plan.set_precision(getattr(heffte.precision, case["form"]))
    elif case["use"] == "r2c":
        plan = heffte.fft3d_r2c(mi355, inbox, outbox.r2c(case["axis"]), case["axis"])
        state["y"] = torch.empty(case["batch"] * plan.size_outbox(), dtype=work_type, device="cuda")
    else:
        plan = heffte.rtransform(mi355, inbox, outbox, getattr(heffte.kind, case["use"]))
        work_type = REAL[case["dtype"]]
    state["plan"] = plan
    if case["use"] == "convolve":
        state["other"] = arrays[1]
        state["ws"] = torch.empty(case["batch"] * plan.size_convolve_workspace(), dtype=work_type, device="cuda")
    else:
        state["ws"] = torch.empty(max(1, case["batch"] * plan.size_workspace()), dtype=work_type, device="cuda")
    return state


def run(state):
    case, x, y, z = state["case"], state["x"], state["y"], state["z"]
    if case["use"] == "mixed":
        state["plan"].forward(x, y, heffte.scale.none)
        state["plan"].backward(y, z, heffte.scale.full)
        return [y, z]
    batch = case["batch"]
    if case["use"] == "reshape":
        heffte.reshape(state["inbox"], [int(c) for c in case["out_order"]], x, y, batch)
        return [y]
    plan, ws = state["plan"], state["ws"]
    if case["use"] == "convolve":
        plan.convolve(x, state["other"], y, ws, state["scaling"], batch)
        return [y]
    if case["passes"] == "forward":
        plan.forward_buffered(x, y, ws, state["scaling"], batch)
        return [y]
    symmetric = state["scaling"] == heffte.scale.symmetric
    plan.forward_buffered(x, y, ws, state["scaling"] if symmetric else heffte.scale.none, batch)
    plan.backward_buffered(y, z, ws, state["scaling"], batch)
    return [y, z]


# ------------------------------------------------------------------ the same in 64 bits

def _shape(case, order):
    n = [case["nx"], case["ny"], case["nz"]]
    return [case["batch"]] + [n[int(c)] for c in reversed(order)]


def _to_natural(x, case, order):
    """Flat array in box order `order` -> array indexed [batch, i0, i1, i2]."""
    a = x.reshape(_shape(case, order))
    at = {int(c): 3 - i for i, c in enumerate(order)}
    return a.permute(0, at[0], at[1], at[2])


def _to_flat(a, order):
    return a.permute(0, *[1 + int(c) for c in reversed(order)]).reshape(-1)


def _cosine(a, dim, kind):
    """DCT-II, DST-II or DCT-I (unnormalised) along dim through the FFT of an extended line."""
    n = a.shape[dim]
    a = a.movedim(dim, -1)
    k = torch.arange(n, device=a.device, dtype=torch.float64)
    if kind == "cos1":
        y = torch.fft.fft(torch.cat([a, a[..., 1:-1].flip(-1)], -1).to(torch.complex128))[..., :n].real
    else:
        if kind == "sin":
            a = a * (1 - 2 * (k % 2))
        y = torch.fft.fft(torch.cat([a, a.flip(-1)], -1).to(torch.complex128))[..., :n]
        y = (y * torch.exp(-0.5j * math.pi * k / n)).real
        if kind == "sin":
            y = y.flip(-1)
    return y.movedim(-1, dim)


def _mixed_exact(case, x):
    roots, out, at = {}, [], 0
    for a, b, c in _mixed_sizes(case):
        for n in (a, b, c):
            if n not in roots:
                j = torch.arange(n, dtype=torch.int64)
                roots[n] = torch.exp(-2j * math.pi * ((j[:, None] * j[None, :]) % n).to(torch.float64) / n).cuda()
        v = x[at:at + a * b * c].to(torch.complex128).reshape(c * b, a) @ roots[a]
        v = torch.matmul(roots[b], v.reshape(c, b, a)).reshape(c, b * a)
        out.append((roots[c] @ v).reshape(-1))
        at += a * b * c
    return torch.cat(out)


def exact(case, seed):
    arrays = _input(case, seed)
    x = arrays[0]
    if case["use"] == "mixed":
        return [_mixed_exact(case, x), x.to(torch.complex128)]
    a = _to_natural(x, case, case["in_order"])
    if case["use"] == "reshape":
        return [_to_flat(a, case["out_order"])]
    dims, count = (1, 2, 3), case["nx"] * case["ny"] * case["nz"]
    real = case["dtype"] in ("f32", "f64")
    a = a.to(torch.float64 if real else torch.complex128)
    if case["use"] == "convolve":
        b = _to_natural(arrays[1], case, case["in_order"]).to(torch.complex128)
        full = count if case["scaling"] == "full" else math.sqrt(count)
        y = torch.fft.ifftn(torch.fft.fftn(a, dim=dims) * torch.fft.fftn(b, dim=dims), dim=dims)
        return [_to_flat(y * (count / full), case["in_order"])]
    if case["use"] == "c2c":
        y, unit = torch.fft.fftn(a, dim=dims), 1.0 / count
    elif case["use"] == "r2c":
        at = 1 + case["axis"]
        y, unit = torch.fft.fftn(torch.fft.rfft(a, dim=at), dim=[d for d in dims if d != at]), 1.0 / count
    else:
        y = a
        for d in dims:
            y = _cosine(y, d, case["use"])
        unit = 1.0 / (64.0 * count)
        if case["use"] == "cos1":
            unit = 1.0 / (64.0 * (case["nx"] - 1) * (case["ny"] - 1) * (case["nz"] - 1))
    forward_only = case["passes"] == "forward"
    if case["scaling"] == "symmetric":
        y = y * math.sqrt(unit)
    elif case["scaling"] == "full" and forward_only:
        y = y * unit
    y = _to_flat(y, case["out_order"])
    return [y] if forward_only else [y, x.to(a.dtype)]
