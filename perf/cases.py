"""Performance cases of the DiaQ GPU path: what they run, on which inputs, and the exact results in 64 bits.

Every case goes through a public entry point (the diaq_gpu module, the C ABI, BatchedEvolution). listed() names the
cases, draw() gives more of the same ranges, prepare() makes what a program has in hand before the call, run() is one
pass, work() the bytes and operations it cannot do without, exact() its result from plain torch in 64 bits.
"""
import math
import random

import numpy as np
import torch

import diaq_amd  # noqa: F401  (registers diaq_gpu)
import diaq_gpu as d
from diaq_amd import capi, evolution

DEV = "cuda"


def listed():
    return [
        # y = H x for a small Hamiltonian: one short launch, where latency is all
        dict(name="spmv_tfim12", kind="spmv", matrix="tfim", n=12, times=1, precision="fp64", tuned=False),
        # y = A^4 x (a power iteration) in single precision, odd size, a band
        dict(name="power_band_f32", kind="spmv", matrix="band", rows=1000003, cols=1000003, diags=33, times=4,
             precision="fp32", tuned=False),
        # the largest single product: 2^24 rows, 64 diagonals spread over the whole matrix, planned by the tuner
        dict(name="spmv_random24", kind="spmv", matrix="random", rows=1 << 24, cols=1 << 24, diags=64, times=1,
             precision="fp64", tuned=True),
        # evolving one small state through many steps: hundreds of short Taylor terms
        dict(name="evolve_xxz10", kind="evolve", matrix="xxz", n=10, steps=20, m=18, dt=0.05, precision="fp64"),
        # the same for a state of a million amplitudes
        dict(name="evolve_xxz20", kind="evolve", matrix="xxz", n=20, steps=10, m=18, dt=0.05, precision="fp64"),
        # H H for a Pauli sum with complex entries and many diagonals, as a dense matrix
        dict(name="square_pauli11", kind="square", matrix="pauli", n=11, strings=16),
        # H H for the largest Hamiltonian whose square fits comfortably (727 diagonals, 11 GB), applied to a state
        dict(name="square_tfim20", kind="square", matrix="tfim", n=20),
        # the propagator exp(-i t H) of a dense matrix in device memory, back as a dense matrix: small
        dict(name="expm_tfim8", kind="expm", matrix="tfim", n=8, t=0.1),
        # and the size at which the propagator fills every diagonal of 4096 x 4096
        dict(name="expm_tfim12", kind="expm", matrix="tfim", n=12, t=0.1),
        # DIA times a block of 8 dense columns
        dict(name="spmm_c128", kind="spmm", rows=1 << 22, cols=1 << 22, diags=9, right=8, complex=True,
             layout="scattered"),
        # one first-order Trotter step of a 28-qubit chain on a resident state
        dict(name="trotter_tfim28", kind="trotter", n=28, dt=0.05, precision="fp64"),
        # 16 Hamiltonians x 8 states from the host, evolved to their own times as one batch, and back
        dict(name="batch_tfim10_15", kind="batch", jobs=16, n_min=10, n_max=15, states=8, t=1.0),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["spmv", "spmv", "evolve", "square", "expm", "spmm", "trotter", "batch"])
    if kind == "spmv":
        matrix = rng.choice(["tfim", "xxz", "band", "random"])
        c = dict(kind=kind, matrix=matrix, times=rng.choice([1, 1, 2, 5]), precision=rng.choice(["fp64", "fp32"]),
                 tuned=rng.random() < 0.3)
        if matrix in ("tfim", "xxz"):
            c["n"] = rng.randint(8, 22)
        else:
            c["rows"] = _log_int(rng, 1000, 8000000)
            c["cols"] = c["rows"] if c["times"] > 1 else max(1, int(c["rows"] * rng.uniform(0.6, 1.6)))
            c["diags"] = _log_int(rng, 3, 80)
        return c
    if kind == "evolve":
        n = rng.randint(6, 19)
        return dict(kind=kind, matrix=rng.choice(["tfim", "xxz"]), n=n, steps=rng.randint(1, 12 if n > 14 else 40),
                    m=rng.randint(8, 24), dt=rng.uniform(0.01, 0.06), precision=rng.choice(["fp64", "fp64", "fp32"]))
    if kind == "square":
        if rng.random() < 0.4:
            return dict(kind=kind, matrix="pauli", n=rng.randint(7, 12), strings=rng.randint(4, 24))
        return dict(kind=kind, matrix=rng.choice(["tfim", "xxz"]), n=rng.randint(8, 19))
    if kind == "expm":
        return dict(kind=kind, matrix=rng.choice(["tfim", "xxz"]), n=rng.randint(5, 11), t=rng.uniform(0.03, 0.3))
    if kind == "spmm":
        rows = _log_int(rng, 1000, 3000000)
        right = _log_int(rng, 1, 64)
        return dict(kind=kind, rows=rows, cols=max(1, int(rows * rng.uniform(0.7, 1.4))),
                    diags=min(_log_int(rng, 3, 60), rows // 4), right=max(1, min(right, 30000000 // rows)),
                    complex=rng.random() < 0.6, layout=rng.choice(["band", "scattered"]))
    if kind == "trotter":
        return dict(kind=kind, n=rng.randint(13, 27), dt=rng.uniform(0.01, 0.1),
                    precision=rng.choice(["fp64", "fp64", "fp32"]))
    n_min = rng.randint(6, 11)
    return dict(kind=kind, jobs=rng.randint(2, 14), n_min=n_min, n_max=n_min + rng.randint(0, 3),
                states=rng.choice([1, 4, 8]), t=rng.uniform(0.2, 1.0))


# ---------------------------------------------------------------------------------------------------------------------
# Hamiltonians as Pauli terms (coefficient, flip mask, phase mask). Couplings are multiples of 2^-10, so the matrix
# elements are exact in single precision too; the seed varies them by a few per cent.
# ---------------------------------------------------------------------------------------------------------------------
def _terms(case, seed, n=None):
    rng = random.Random(seed * 1000003 + 17)
    n = case["n"] if n is None else n

    def near(v):
        return v + rng.randint(-48, 48) / 1024.0

    out = []
    if case.get("matrix", "tfim") == "tfim":
        J, h = near(1.0), near(0.6875)
        out += [(-J, 0, 3 << i) for i in range(n - 1)]
        out += [(-h, 1 << i, 0) for i in range(n)]
    elif case["matrix"] == "xxz":
        Jxy, Jz = near(1.0), near(0.8125)
        for i in range(n - 1):
            out += [(Jxy, 3 << i, 0), (Jxy, 3 << i, 3 << i), (Jz, 0, 3 << i)]
        out += [(rng.randint(-1024, 1024) / 1024.0, 0, 1 << i) for i in range(n)]
    else:  # 2- to 4-local Pauli strings: which ones is the case's, the coefficients are the seed's
        pick = random.Random(n * 1009 + case["strings"])
        for _ in range(case["strings"]):
            x = z = 0
            for q in pick.sample(range(n), pick.randint(2, 4)):
                p = pick.choice("XYZ")
                x |= (1 << q) if p in "XY" else 0
                z |= (1 << q) if p in "YZ" else 0
            out.append((rng.randint(-2048, 2048) / 1024.0, x, z))
    return out


def _device_matrix(case, seed, n=None, precision="fp64"):
    t = _terms(case, seed, n)
    N = case["n"] if n is None else n
    return d.prune(d.pauli_sum_device(N, [x for _, x, _ in t], [z for _, _, z in t], [complex(c) for c, _, _ in t],
                                      precision))


def _factors(terms, n):
    """H as {flip mask x: f} with (H v)[r] = sum_x f_x[r] v[r ^ x], in 64 bits."""
    idx = torch.arange(1 << n, device=DEV, dtype=torch.int64)
    f = {}
    for c, x, z in terms:
        p = (idx ^ x) & z
        for s in (16, 8, 4, 2, 1):
            p = p ^ (p >> s)
        sign = 1.0 - 2.0 * (p & 1).to(torch.float64)
        phase = (1j) ** (bin(x & z).count("1") % 4)
        term = sign.to(torch.complex128) * (c * phase)
        f[x] = f[x] + term if x in f else term
    return idx, f


def _apply(idx, f, v):
    y = torch.zeros_like(v)
    for x, fx in f.items():
        fx = fx.to(v.dtype)
        y += (fx if v.dim() == 1 else fx[:, None]) * v[idx ^ x]
    return y


def _dense(terms, n):
    idx, f = _factors(terms, n)
    D = torch.zeros(1 << n, 1 << n, dtype=torch.complex128, device=DEV)
    for x, fx in f.items():
        D[idx, idx ^ x] = fx
    return D


def _offsets_of(terms, n):
    """The offsets of the diagonals that hold a nonzero (terms of one flip mask that cancel are left out)."""
    got = set()
    masks = {}
    for c, x, z in terms:
        masks.setdefault(x, []).append((c, z))
    for x, group in masks.items():
        bits = [k for k in range(n) if (x >> k) & 1]
        for s in range(1 << len(bits)):
            row = sum(1 << b for j, b in enumerate(bits) if (s >> j) & 1)  # the row's bits at the flipped places
            col = row ^ x
            if len(group) > 1:  # XX + YY cancels where the two bits are equal
                total = {}
                for c, z in group:
                    ph = (1j) ** (bin(x & z).count("1") % 4) * (-1) ** (bin(col & z & x).count("1") % 2)
                    total[z & ~x] = total.get(z & ~x, 0) + c * ph
                if all(abs(v) < 1e-15 for v in total.values()):
                    continue
            got.add(col - row)
    return sorted(got)


def _stored(rows, cols, offsets):
    return sum(max(0, min(rows + o if o < 0 else cols - o, rows, cols)) for o in offsets)


# ---------------------------------------------------------------------------------------------------------------------
# Generic diagonal matrices
# ---------------------------------------------------------------------------------------------------------------------
def _offsets(case):
    """A band around the main diagonal, or diagonals spread over the middle half of the offsets; the case's own."""
    rows, cols, k = case["rows"], case["cols"], case["diags"]
    if case.get("matrix") == "band" or case.get("layout") == "band":
        return [o for o in range(-(k // 2), k - k // 2) if -rows < o < cols]
    r = random.Random(rows * 31 + k)
    return sorted(r.sample(range(-(rows // 2), cols // 2 + 1), min(k, rows // 2)))


def _gen(seed, salt=0):
    return torch.Generator(device=DEV).manual_seed(seed * 7919 + salt)


def _randn(shape, dtype, g):
    return torch.randn(shape, dtype=dtype, device=DEV, generator=g)


def _state(n, seed):
    g = _gen(seed, 5)
    r, i = _randn(1 << n, torch.float64, g), _randn(1 << n, torch.float64, g)
    nrm = torch.sqrt((r * r).sum() + (i * i).sum())
    return r / nrm, i / nrm


def _dia_values(case, seed, dtype):
    """Packed values, diagonal after diagonal; scaled so that powers of the matrix stay of order one."""
    g = _gen(seed, 1)
    total = _stored(case["rows"], case["cols"], _offsets(case))
    s = 1.0 / math.sqrt(2.0 * case["diags"])
    re = _randn(total, dtype, g).mul_(s)
    return re, _randn(total, dtype, g).mul_(s)


class _Dia:
    """A dq_devmat filled from packed device arrays through the C ABI."""

    def __init__(self, case, seed, dtype):
        L = capi.lib()
        offs = _offsets(case)
        self.handle = capi.c_void_p()
        arr = (capi.c_int32 * len(offs))(*offs)
        capi.check(L.dq_devmat_zeros(case["rows"], case["cols"], len(offs), arr,
                                     capi.DQ_F32 if dtype == torch.float32 else capi.DQ_F64, self.handle))
        re, im = _dia_values(case, seed, dtype)
        capi.check(L.dq_devmat_set_packed_device(self.handle, re.data_ptr(), im.data_ptr(), 0))
        torch.cuda.synchronize()

    def __del__(self):
        capi.lib().dq_devmat_destroy(self.handle)


def _spmv_shape(case):
    if "n" in case:
        return 1 << case["n"], 1 << case["n"]
    return case["rows"], case["cols"]


def _spmv_x(case, seed, dtype):
    g = _gen(seed, 2)
    n = _spmv_shape(case)[1]
    return _randn(n, dtype, g), _randn(n, dtype, g)


def _dtype(case):
    return torch.float32 if case.get("precision") == "fp32" else torch.float64


# ---------------------------------------------------------------------------------------------------------------------
# The five functions' bodies by kind
# ---------------------------------------------------------------------------------------------------------------------
def prepare(case, seed):
    s = dict(case=case, kind=case["kind"], stream=torch.cuda.current_stream().cuda_stream)
    kind = case["kind"]
    if kind == "spmv":
        dt = _dtype(case)
        if "n" in case:
            s["A"] = _device_matrix(case, seed, precision=case["precision"])
        else:
            s["A"] = _Dia(case, seed, dt)
        s["x"] = _spmv_x(case, seed, dt)
        rows = _spmv_shape(case)[0]
        s["y"] = tuple(torch.empty(rows, dtype=dt, device=DEV) for _ in range(2))
        if case["times"] > 1:
            s["w"] = tuple(torch.empty(rows, dtype=dt, device=DEV) for _ in range(2))
        if case["tuned"]:
            capi.check(capi.lib().dq_spmv_tune(s["A"].handle, 3, s["stream"], None))
    elif kind == "evolve":
        s["H"] = _device_matrix(case, seed, precision=case["precision"])
        r, i = _state(case["n"], seed)
        s["psi"] = (r.to(_dtype(case)), i.to(_dtype(case)))
    elif kind == "square":
        s["H"] = _device_matrix(case, seed)
        if case["matrix"] == "pauli":
            s["D"] = torch.empty((1 << case["n"],) * 2, dtype=torch.complex128, device=DEV)
            return s
        s["x"] = _state(case["n"], seed)
        s["y"] = tuple(torch.empty(1 << case["n"], dtype=torch.float64, device=DEV) for _ in range(2))
    elif kind == "expm":
        s["D"] = _dense(_terms(case, seed), case["n"])
        s["U"] = torch.empty_like(s["D"])
    elif kind == "spmm":
        dt = torch.complex128 if case["complex"] else torch.float64
        g = _gen(seed, 3)
        offs = _offsets(case)
        s["off"] = torch.tensor(offs, dtype=torch.int64, device=DEV)
        s["vals"] = _randn((len(offs), case["rows"]), dt, g)
        s["B"] = _randn((case["cols"], case["right"]), dt, g)
        s["C"] = torch.empty((case["rows"], case["right"]), dtype=dt, device=DEV)
    elif kind == "trotter":
        zz, c, si = _trotter_angles(case, seed)
        n = case["n"]
        GZ = d.to_device(d.diaQMatrix.from_diagonals([4, 4], [0], [zz]), case["precision"])
        GX = d.to_device(d.diaQMatrix.from_diagonals([2, 2], [-1, 0, 1], [np.array([-1j * si]),
                                                                          np.array([c, c]) + 0j,
                                                                          np.array([-1j * si])]), case["precision"])
        s["plan"] = d.GatePlan(n, [(GZ, q) for q in range(n - 1)] + [(GX, q) for q in range(n)])
        r, i = _state(n, seed)
        s["psi"] = (r.to(_dtype(case)), i.to(_dtype(case)))
    else:
        jobs = _batch_jobs(case, seed)
        mats = [_device_matrix(dict(matrix="tfim"), sd, n=n) for n, sd, t in jobs]
        B = evolution.BatchedEvolution(mats, case["states"], "fp32")
        sched = [evolution.plain_rule(d.estimate_1norm(M), t, 1e-6) for M, (n, sd, t) in zip(mats, jobs)]
        B.set_schedule([t for _, _, t in jobs], [m for m, _ in sched], [q for _, q in sched])
        s["sizes"] = [1 << n for n, _, _ in jobs]
        s["states"] = [_batch_states(n, case["states"], sd) for n, sd, _ in jobs]
        for j, st in enumerate(s["states"]):
            B.set_states(j, st)
        B.tune()
        s["B"] = B
    return s


def run(s):
    kind, case = s["kind"], s["case"]
    if kind == "spmv":
        (xr, xi), (yr, yi) = s["x"], s["y"]
        if case["times"] > 1:
            wr, wi = s["w"]
            capi.check(capi.lib().dq_spmv_ntimes_device(s["A"].handle, xr.data_ptr(), xi.data_ptr(), yr.data_ptr(),
                                                        yi.data_ptr(), case["times"], wr.data_ptr(), wi.data_ptr(),
                                                        s["stream"]))
        elif "n" in case:
            d.spmv_device(s["A"], xr.data_ptr(), xi.data_ptr(), yr.data_ptr(), yi.data_ptr(), s["stream"])
        else:
            capi.check(capi.lib().dq_spmv_device(s["A"].handle, xr.data_ptr(), xi.data_ptr(), yr.data_ptr(),
                                                 yi.data_ptr(), s["stream"]))
        return [yr, yi]
    if kind == "evolve":
        pr, pi = s["psi"]
        d.hamsim_device(s["H"], pr.data_ptr(), pi.data_ptr(), case["dt"] * case["steps"], case["steps"], case["m"],
                        s["stream"])
        return [pr, pi]
    if kind == "square":
        C = d.product(s["H"], s["H"])
        if "D" in s:
            d.to_dense_device(C, s["D"].data_ptr(), stream=s["stream"])
            return s["D"]
        (xr, xi), (yr, yi) = s["x"], s["y"]
        d.spmv_device(C, xr.data_ptr(), xi.data_ptr(), yr.data_ptr(), yi.data_ptr(), s["stream"])
        return [yr, yi]
    if kind == "expm":
        N = 1 << case["n"]
        H = d.from_dense_device(s["D"].data_ptr(), N, N, stream=s["stream"])
        d.to_dense_device(d.expm_negative(H, case["t"]), s["U"].data_ptr(), stream=s["stream"])
        return s["U"]
    if kind == "spmm":
        d.spmm_dia_device(s["off"].data_ptr(), s["vals"].data_ptr(), s["vals"].shape[0], case["rows"], case["cols"],
                          s["B"].data_ptr(), case["right"], s["C"].data_ptr(), case["complex"], s["stream"])
        return s["C"]
    if kind == "trotter":
        pr, pi = s["psi"]
        s["plan"].run(pr.data_ptr(), pi.data_ptr(), 1, s["stream"])
        return [pr, pi]
    B = s["B"]
    for j, st in enumerate(s["states"]):
        B.set_states(j, st)
    B.run(use_graph=True, renormalize=True, stream=s["stream"])
    return [B.get_states(j, N) for j, N in enumerate(s["sizes"])]


def _trotter_angles(case, seed):
    rng = random.Random(seed * 31 + 7)
    J, h = 1.0 + rng.uniform(-0.05, 0.05), 0.7 + rng.uniform(-0.05, 0.05)
    zz = np.exp(-1j * case["dt"] * J * np.array([1.0, -1.0, -1.0, 1.0]))
    c, si = math.cos(case["dt"] * h), math.sin(case["dt"] * h)
    if case["precision"] == "fp32":
        zz = zz.astype(np.complex64).astype(np.complex128)
        c, si = float(np.float32(c)), float(np.float32(si))
    return zz, c, si


def _batch_jobs(case, seed):
    """(qubits, the job's own seed, time): sizes in turn, times from t / jobs to t."""
    span = case["n_max"] - case["n_min"] + 1
    return [(case["n_min"] + j % span, seed * 64 + j, case["t"] * (j + 1) / case["jobs"]) for j in range(case["jobs"])]


def _batch_states(n, states, seed):
    rng = np.random.default_rng(seed)
    st = rng.standard_normal((states, 1 << n)) + 1j * rng.standard_normal((states, 1 << n))
    return st / np.linalg.norm(st, axis=1, keepdims=True)


def work(case):
    kind = case["kind"]
    b = 8 if case.get("precision") == "fp32" else 16  # bytes of a complex value
    if kind in ("spmv", "evolve", "square") and "n" in case:
        N = 1 << case["n"]
        offs = _offsets_of(_terms(case, 1), case["n"])
        S = _stored(N, N, offs)
    if kind == "spmv":
        rows, cols = _spmv_shape(case)
        if "n" not in case:
            S = _stored(rows, cols, _offsets(case))
        return dict(bytes=b * (S + rows + cols), flops=8 * S * case["times"])
    if kind == "evolve":
        return dict(bytes=b * (S + 2 * N), flops=8 * (S + N) * case["m"] * case["steps"])
    if kind == "square":
        pairs = {}
        for p in offs:
            for q in offs:
                if -N < p + q < N:
                    lo, hi = max(0, -p, -p - q), min(N, N - p, N - p - q)
                    pairs[p + q] = pairs.get(p + q, 0) + max(0, hi - lo)
        SC = _stored(N, N, list(pairs))
        if case["matrix"] == "pauli":
            return dict(bytes=16 * (S + 2 * SC + N * N), flops=8 * sum(pairs.values()))
        return dict(bytes=16 * (S + 2 * SC + 2 * N), flops=8 * (sum(pairs.values()) + SC))
    if kind == "expm":
        N = 1 << case["n"]
        S = _stored(N, N, _offsets_of(_terms(case, 1), case["n"]))
        return dict(bytes=2 * 16 * N * N, flops=8 * N * S * 14)  # 14 Taylor terms
    if kind == "spmm":
        v = 16 if case["complex"] else 8
        offs = _offsets(case)
        return dict(bytes=v * (len(offs) * case["rows"] + (case["rows"] + case["cols"]) * case["right"]),
                    flops=(8 if case["complex"] else 2) * _stored(case["rows"], case["cols"], offs) * case["right"])
    if kind == "trotter":
        N = 1 << case["n"]
        return dict(bytes=2 * b * N, flops=N * (6 * (case["n"] - 1) + 14 * case["n"]))
    by = fl = 0
    for n, sd, t in _batch_jobs(case, 1):
        N = 1 << n
        S = _stored(N, N, _offsets_of(_terms(dict(matrix="tfim"), sd, n), n))
        m, q = evolution.plain_rule((n - 1) * 1.0 + n * 0.6875, t, 1e-6)
        by += 8 * S + 2 * 16 * N * case["states"]
        fl += 8 * S * case["states"] * m * 2 ** q
    return dict(bytes=by, flops=fl)


def exact(case, seed):
    kind = case["kind"]
    if kind == "spmv":
        dt = _dtype(case)
        xr, xi = _spmv_x(case, seed, dt)
        v = torch.complex(xr.double(), xi.double())
        if "n" in case:
            idx, f = _factors(_terms(case, seed), case["n"])
            for _ in range(case["times"]):
                v = _apply(idx, f, v)
        else:
            re, im = _dia_values(case, seed, dt)
            rows, cols = case["rows"], case["cols"]
            for _ in range(case["times"]):
                y = torch.zeros(rows, dtype=torch.complex128, device=DEV)
                at = 0
                for o in _offsets(case):
                    ln = _stored(rows, cols, [o])
                    a = torch.complex(re[at:at + ln].double(), im[at:at + ln].double())
                    r0, c0 = max(0, -o), max(0, o)
                    y[r0:r0 + ln] += a * v[c0:c0 + ln]
                    at += ln
                v = y
        return [v.real.clone(), v.imag.clone()]
    if kind == "evolve":
        idx, f = _factors(_terms(case, seed), case["n"])
        r, i = (p.to(_dtype(case)).double() for p in _state(case["n"], seed))
        psi = torch.complex(r, i)
        norm = torch.linalg.vector_norm(psi)
        for _ in range(case["steps"]):
            term = psi
            for k in range(1, case["m"] + 1):
                term = _apply(idx, f, term) * (-1j * case["dt"] / k)
                psi = psi + term
        if case["precision"] == "fp32":  # the single-precision form renormalises
            psi = psi * (norm / torch.linalg.vector_norm(psi))
        return [psi.real.clone(), psi.imag.clone()]
    if kind == "square" and case["matrix"] == "pauli":
        D = _dense(_terms(case, seed), case["n"])
        return D @ D
    if kind == "square":
        idx, f = _factors(_terms(case, seed), case["n"])
        v = torch.complex(*_state(case["n"], seed))
        v = _apply(idx, f, _apply(idx, f, v))
        return [v.real.clone(), v.imag.clone()]
    if kind == "expm":
        return torch.linalg.matrix_exp(-1j * case["t"] * _dense(_terms(case, seed), case["n"]))
    if kind == "spmm":
        s = prepare(case, seed)
        rows, cols = case["rows"], case["cols"]
        C = torch.zeros_like(s["C"])
        for k, o in enumerate(_offsets(case)):
            r0, r1 = max(0, -o), min(rows, cols - o)
            if r1 > r0:
                C[r0:r1] += s["vals"][k, r0:r1, None] * s["B"][r0 + o:r1 + o]
        return C
    if kind == "trotter":
        zz, c, si = _trotter_angles(case, seed)
        n = case["n"]
        r, i = (p.to(_dtype(case)).double() for p in _state(n, seed))
        psi = torch.complex(r, i)
        z = torch.tensor(zz, device=DEV)
        for q in range(n - 1):
            psi.view(-1, 4, 1 << q).mul_(z[:, None])
        for q in range(n):
            v = psi.view(-1, 2, 1 << q)
            a, b = v[:, 0].clone(), v[:, 1].clone()
            v[:, 0] = c * a - 1j * si * b
            v[:, 1] = c * b - 1j * si * a
        return [psi.real.clone(), psi.imag.clone()]
    out = []
    for n, sd, t in _batch_jobs(case, seed):
        idx, f = _factors(_terms(dict(matrix="tfim"), sd, n), n)
        psi = torch.tensor(_batch_states(n, case["states"], sd).T.copy(), device=DEV)
        steps = max(1, math.ceil(t * 2 * n))
        for _ in range(steps):
            term = psi
            for k in range(1, 25):
                term = _apply(idx, f, term) * (-1j * t / steps / k)
                psi = psi + term
        out.append((psi / torch.linalg.vector_norm(psi, dim=0)).T.contiguous().cpu().numpy())
    return out
