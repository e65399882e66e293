"""The work whose speed is measured: what a user of the library has it do,
through its public entry points (include/hypjac.h, mirrored by gpujachx_amd).

    entry    "dev"      hypJacL2_dev on device-resident data
             "noalloc"  hypJacL2_dev_noalloc (no device allocation inside)
             "host"     hypJacL2 on host buffers (copies included)
             "level1"   one sweep driven by the caller through the level-1 layer
             "batch"    many independent problems in one persistent launch
    m, n     rows, columns; nplus positive signs of J first (n: an SVD)
    alg      the routine's bits (8: one inner sweep, 2: V, 1: sorted)
    matrix   "geom6"    U diag(10^(-6 i/(n-1))) V^T      (well conditioned SVD)
             "log12"    U diag(10^(-12 u)) V^T, u ~ U(0,1) (the headline class)
             "graded"   N(0,1) x column scales 10^U(-4,4)  (the HSVD class)
    fam      level-1 strategy family; form, width, fact, cap: the library's options
             (learned/split form, block width, factorization, sweep cap)

The library overwrites its input, so a pass first restores it from the
caller's own copy, as a program that keeps its matrix does.
"""
import ctypes
import os

import numpy as np
import torch

import gpujachx_amd as g
from gpujachx_amd import learned

os.environ.setdefault("HJ_QUIET", "1")
_NPROB = 384  # problems of the listed batch


def _case(name, entry, m, n, nplus, alg, matrix, fam="cycwor", form="plain", width=16, fact=0, cap=30,
          pad=0, count=1):
    return {"name": name, "entry": entry, "m": m, "n": n, "nplus": nplus, "alg": alg, "matrix": matrix,
            "fam": fam, "form": form, "width": width, "fact": fact, "cap": cap, "pad": pad, "count": count}


def listed():
    return [
        # the smallest call: two block pairs, where launches and host work are everything
        _case("svd_64", "dev", 64, 64, 64, 11, "geom6"),
        # a small SVD with V, the smallest benchmark configuration
        _case("svd_256", "dev", 256, 256, 256, 11, "geom6"),
        # a serving loop that may not allocate: tall, hyperbolic
        _case("hsvd_noalloc_512x128", "noalloc", 512, 128, 48, 11, "graded"),
        # a host program's whole call; an order (42 blocks) that only the modulus strategy has
        _case("hsvd_host_1344x672", "host", 1344, 672, 250, 11, "graded", fam="mmstep"),
        # a caller that drives the level-1 steps itself (the thin layer), J mixed in a block
        _case("level1_2048x1024", "level1", 2048, 1024, 500, 11, "graded"),
        # inner sweeps to convergence (not block oriented), unsorted, J = -I
        _case("inner_1024x512", "dev", 1024, 512, 0, 2, "graded", fam="rowcyc"),
        # the accuracy option: QR factorization of the pairs, Drmac's level 0
        _case("drmac_512x256", "dev", 512, 256, 256, 11, "graded", fact=2),
        # the middle-sized HSVD benchmark configuration
        _case("hsvd_4096x2048", "dev", 4096, 2048, 1024, 11, "graded"),
        # the learned + split form on the headline matrix class
        _case("learned_4096", "dev", 4096, 4096, 4096, 9, "log12", form="learned+split", cap=80),
        # 32-column blocks, V accumulated, a padded leading dimension
        _case("wide_4608x2048", "dev", 4608, 2048, 2048, 11, "log12", width=32, cap=80, pad=16),
        # the largest: the headline size, J mixed (staged sweeps)
        _case("hsvd_8192", "dev", 8192, 8192, 4096, 9, "graded"),
        # many small uneven (H)SVDs at once
        _case("batch_512", "batch", 0, 512, 0, 11, "graded", count=_NPROB),
    ]


def _log_uniform(rng, lo, hi):
    return int(round(lo * (hi / lo) ** rng.random()))


def draw(rng):
    """A case of the listed ones' ranges: any entry, sizes over the logarithm
    of its range (columns a multiple of 32, rows of 64: what the library
    takes), the strategy, signs, routine and options that go with them."""
    kind = rng.choice(["dev", "dev", "dev", "noalloc", "host", "level1", "inner", "qr", "learned", "wide",
                       "staged", "batch"])
    alg = rng.choice([8, 9, 10, 11, 11])
    if kind == "batch":
        return _draw_case("batch", 0, 32 * _log_uniform(rng, 4, 16), 0, alg, "graded",
                          count=_log_uniform(rng, 32, _NPROB))
    if kind == "learned":
        # at least 32000 visits a sweep: 4096 columns; sorted (unsorted, this
        # class takes several times the sweeps)
        n = 4096
        return _draw_case("dev", n, n, rng.choice([n // 2, rng.randrange(1, n)]), 9, "log12", cap=80,
                          form=rng.choice(["learned", "learned+split"]), pad=rng.choice([0, 16, 64]))
    if kind == "staged":
        n = 4096
        return _draw_case("dev", 512 * rng.randrange(11, 16), n, rng.choice([n, rng.randrange(1, n)]),
                          rng.choice([9, 11]), "graded", fam=rng.choice(["cycwor", "rowcyc"]))
    top = {"dev": 2048, "noalloc": 1024, "host": 1024, "level1": 2048, "inner": 1024, "qr": 320,
           "wide": 2048}[kind]
    n = 32 * _log_uniform(rng, 1 if kind not in ("wide", "qr") else 4, top // 32)
    fam = rng.choice(["mmstep", "BrentL"])
    if kind in ("wide", "level1") or rng.random() < 0.5:
        # a power of two, where the cyclic families exist (what a caller of
        # the level-1 layer stays with)
        n = 1 << max({"wide": 7, "level1": 6}.get(kind, 5), n.bit_length() - 1)
        fam = rng.choice(["cycwor", "cycwor", "rowcyc", "colcyc"] + (["mmstep"] if kind != "level1" else []))
    m = 64 * ((n + 63) // 64 + rng.randrange(0, max(12, n // 64 + 1)))
    if n > 1024:
        m = 512 * ((m + 511) // 512)
    nplus = rng.choice([n, n, 0, n // 2, rng.randrange(0, n + 1)])
    if kind == "qr":
        m = min(m, 64 * ((n + 63) // 64) + 128)
        return _draw_case("dev", m, n, nplus, alg, "graded", fam=fam, fact=rng.choice([1, 2]))
    if kind == "inner":
        return _draw_case("dev", m, n, nplus, rng.choice([0, 1, 2, 3]), "graded", fam=fam)
    matrix = rng.choice(["geom6", "graded"]) if nplus == n else "graded"
    if kind == "wide":
        return _draw_case("dev", m, n, nplus, alg, matrix, fam=fam, width=32, pad=rng.choice([0, 16]))
    return _draw_case(kind, m, n, nplus, alg, matrix, fam=fam, pad=rng.choice([0, 0, 2, 16]) if kind == "dev" else 0)


def _draw_case(entry, m, n, nplus, alg, matrix, **kw):
    c = _case("", entry, m, n, nplus, alg, matrix, **kw)
    del c["name"]
    return c


# ---------------------------------------------------------------------------
# Inputs

def _matrix(kind, m, n, gen):
    """n x m row-major on the GPU: the column-major m x n matrix."""
    f64 = dict(dtype=torch.float64, device="cuda", generator=gen)
    if kind == "graded":
        Gt = torch.randn(n, m, **f64)
        return Gt.mul_(torch.pow(10.0, torch.rand(n, 1, **f64) * 8.0 - 4.0))
    if kind == "geom6":
        s = torch.pow(10.0, -6.0 * torch.arange(n, dtype=torch.float64, device="cuda") / max(n - 1, 1))
    else:
        s = torch.pow(10.0, -12.0 * torch.rand(n, **f64))
    U = torch.linalg.qr(torch.randn(m, n, **f64))[0]
    V = torch.linalg.qr(torch.randn(n, n, **f64))[0]
    return torch.matmul(V * s, U.T).contiguous()


def _batch_shapes(case):
    """Uneven sizes up to case["n"] columns, half SVDs, half HSVDs."""
    rng = np.random.default_rng([case["n"], case["count"]])
    ns = 32 * rng.integers(2, case["n"] // 32 + 1, case["count"])
    ms = 64 * ((ns + 63) // 64) * rng.integers(1, 3, case["count"])
    hyp = rng.uniform(size=case["count"]) < 0.5
    return [(int(m), int(n), int(n) // 2 if h else int(n)) for m, n, h in zip(ms, ns, hyp)]


def _batch_matrices(case, seed):
    gen = torch.Generator(device="cuda").manual_seed(seed)
    shapes = _batch_shapes(case)
    flat = torch.randn(sum(m * n for m, n, _ in shapes), dtype=torch.float64, device="cuda", generator=gen)
    at = 0
    for m, n, _ in shapes:
        # column scales 10^U(-3,3)
        sc = torch.rand(n, 1, dtype=torch.float64, device="cuda", generator=gen) * 6.0 - 3.0
        flat[at:at + m * n].view(n, m).mul_(torch.pow(10.0, sc))
        at += m * n
    return shapes, flat


_active = None


def _configure(case):
    """The process-wide options of the library for this case."""
    global _active
    key = tuple(sorted((k, v) for k, v in case.items() if k != "name"))
    if key == _active:
        return
    g.configureGPU(0)
    if case["entry"] != "batch":
        g.init_strats_builtin("cycwor", 32, case["fam"], case["n"] // 16)
    g.set_max_sweeps(case["cap"])
    g.lib().hj_set_block_width(case["width"])
    g.set_factorization(case["fact"])
    bits = (g.FORM_LEARNED_SKIP if "learned" in case["form"] else 0) | (
        g.FORM_SPLIT_GRAM if "split" in case["form"] else 0)
    if bits & g.FORM_LEARNED_SKIP:
        learned.enable(form=bits)
    else:
        g.set_form(bits)
    _active = key


def prepare(case, seed):
    _configure(case)
    if case["entry"] == "batch":
        return _prepare_batch(case, seed)
    m, n, ld = case["m"], case["n"], case["m"] + case["pad"]
    gen = torch.Generator(device="cuda").manual_seed(seed)
    Gt = _matrix(case["matrix"], m, n, gen)
    full = bool(case["alg"] & 2)
    st = {"case": case, "ld": ld, "sw": ctypes.c_uint(0), "s": ctypes.c_ulonglong(0), "b": ctypes.c_ulonglong(0)}
    if case["entry"] == "host":
        st["G0"] = np.ascontiguousarray(Gt.cpu().numpy())
        st["G"] = np.empty((n, ld))
        st["V"] = np.empty((n, n)) if full else None
        st["D"] = np.empty(n)
        return st
    st["G0"] = Gt
    st["G"] = torch.empty(n, ld, dtype=torch.float64, device="cuda")[:, :m]
    st["V"] = torch.empty(n, n, dtype=torch.float64, device="cuda") if full else None
    st["D"] = torch.empty(n, dtype=torch.float64, device="cuda")
    if case["entry"] == "level1":
        st["cvg"] = torch.zeros(1, dtype=torch.int64, device="cuda")
        st["fn"] = _level1(case)
    return st


def _prepare_batch(case, seed):
    shapes, flat = _batch_matrices(case, seed)
    full = bool(case["alg"] & 2)
    st = {"case": case, "G0": flat, "G": torch.empty_like(flat),
          "V": torch.empty(sum(n * n for _, n, _ in shapes), dtype=torch.float64, device="cuda") if full else None,
          "D": torch.empty(sum(n for _, n, _ in shapes), dtype=torch.float64, device="cuda")}
    descs, og, ov, od = [], 0, 0, 0
    for m, n, nplus in shapes:
        descs.append(g.BatchDesc(case["alg"], m, n, nplus, m, n if full else 0, st["G"].data_ptr() + 8 * og,
                                 st["V"].data_ptr() + 8 * ov if full else None, st["D"].data_ptr() + 8 * od))
        og, ov, od = og + m * n, ov + n * n, od + n
    st["batch"] = g.Batch(descs)  # the plan a serving program keeps
    return st


def _level1(case):
    L = g.lib()
    u, vp = ctypes.c_uint, ctypes.c_void_p
    L.initSymbols.argtypes = [vp, vp, vp, u, u, u, u, u]
    L.initSymbols.restype = None
    L.initV.argtypes = [vp, u, u, u]
    L.initV.restype = None
    definite = case["nplus"] in (0, case["n"])
    fn = getattr(L, ("def" if definite else "hyp") + "JacL1" + ("s" if case["alg"] & 1 else "")
                 + ("v" if case["alg"] & 2 else ""))
    fn.argtypes = [u, ctypes.c_int if definite else u]
    fn.restype = None
    return fn


# ---------------------------------------------------------------------------
# One pass

def run(st):
    case = st["case"]
    _configure(case)
    return {"dev": _run_dev, "noalloc": _run_dev, "host": _run_host, "level1": _run_level1,
            "batch": _run_batch}[case["entry"]](st, case)


def _outputs(st, **more):
    out = {"G": st["G"], "D": st["D"], **more}
    if st["V"] is not None:
        out["V"] = st["V"]
    return out


def _ptr(t):
    return t.data_ptr() if t is not None else None


def _run_dev(st, case):
    n, V = case["n"], st["V"]
    st["G"].copy_(st["G0"])
    fn = g.lib().hypJacL2_dev if case["entry"] == "dev" else g.lib().hypJacL2_dev_noalloc
    rc = fn(case["alg"], case["m"], n, case["nplus"], st["G"].data_ptr(), st["ld"], _ptr(V),
            n if V is not None else 0, st["D"].data_ptr(), ctypes.byref(st["sw"]), ctypes.byref(st["s"]),
            ctypes.byref(st["b"]), None, torch.cuda.current_stream().cuda_stream)
    if rc:
        raise RuntimeError("%s returned %d" % (case["entry"], rc))
    return _outputs(st, sweeps=st["sw"].value, rot_s=st["s"].value, rot_b=st["b"].value)


def _run_host(st, case):
    n, V = case["n"], st["V"]
    np.copyto(st["G"], st["G0"])
    pd = ctypes.POINTER(ctypes.c_double)
    rc = g.lib().hypJacL2(case["alg"], case["m"], n, case["nplus"], st["G"].ctypes.data_as(pd), st["ld"],
                          V.ctypes.data_as(pd) if V is not None else None, n if V is not None else 0,
                          st["D"].ctypes.data_as(pd), ctypes.byref(st["sw"]), ctypes.byref(st["s"]),
                          ctypes.byref(st["b"]), None)
    if rc:
        raise RuntimeError("hypJacL2 returned %d" % rc)
    return _outputs(st, sweeps=st["sw"].value, rot_s=st["s"].value, rot_b=st["b"].value)


def _run_level1(st, case):
    L, n, V, fn = g.lib(), case["n"], st["V"], st["fn"]
    st["G"].copy_(st["G0"])
    st["cvg"].zero_()
    L.initSymbols(st["G"].data_ptr(), _ptr(V), st["cvg"].data_ptr(), case["m"], n, st["ld"],
                  n if V is not None else 0, 1)
    if V is not None:
        L.initV(V.data_ptr(), 0, n, n)
    nplus = case["nplus"]
    sign = nplus if 0 < nplus < n else (1 if nplus else -1)
    for step in range(ctypes.c_uint.in_dll(L, "STRAT1_STEPS").value):
        fn(step, sign)
    out = {"G": st["G"], "cvg": st["cvg"]}
    if V is not None:
        out["V"] = V
    return out


def _run_batch(st, case):
    st["G"].copy_(st["G0"])
    st["batch"].run(torch.cuda.current_stream().cuda_stream)
    r = st["batch"].results()
    return _outputs(st, sweeps=r["sweeps"].astype(np.int64), rot_s=r["rot_s"].astype(np.int64),
                    rot_b=r["rot_b"].astype(np.int64))


# ---------------------------------------------------------------------------
# What a pass cannot do without, and what it has to give

def work(case):
    """G read, U written, V and D written, and the flops of one sweep of the
    method (Gram and update of every pair of 32 columns): the least that any
    run does."""
    full = bool(case["alg"] & 2)
    shapes = _batch_shapes(case) if case["entry"] == "batch" else [(case["m"], case["n"], 0)]
    by = sum(8.0 * (2.0 * m * n + (n * n if full else 0) + n) for m, n, _ in shapes)
    fl = sum(2048.0 * (2.0 * m + (n if full else 0)) * (n / 16.0) * (n / 16.0 - 1.0) / 2.0 for m, n, _ in shapes)
    return {"bytes": by, "flops": fl}


def _exact_d(Gt, nplus):
    """The diagonal of J Sigma^2 in descending order: for J = +-I the squared
    singular values, else the nonzero eigenvalues of G J G^T (those of the
    R J R^T of G^T = Q R's triangle)."""
    n = Gt.shape[0]
    J = np.ones(n)
    J[nplus:] = -1.0
    if nplus in (0, n):
        w = np.linalg.eigvalsh(Gt @ Gt.T)
        return (w if nplus else -w[::-1])[::-1].copy()
    # G = Q R, so G J G^T has the eigenvalues of R J R^T
    R = np.linalg.qr(Gt.T, mode="r")
    return np.linalg.eigvalsh((R * J) @ R.T)[::-1].copy()


def exact(case, seed):
    """D of the sorted routines, which leave it in descending order; U and V
    are unique only up to signs, and one sweep ends nowhere."""
    if case["entry"] == "level1" or not case["alg"] & 1 or case["n"] > 2048:
        return None
    if case["entry"] == "batch":
        shapes, flat = _batch_matrices(case, seed)
        flat, ds, at = flat.cpu().numpy(), [], 0
        for m, n, nplus in shapes:
            ds.append(_exact_d(flat[at:at + m * n].reshape(n, m), nplus))
            at += m * n
        D = np.concatenate(ds)
    else:
        gen = torch.Generator(device="cuda").manual_seed(seed)
        D = _exact_d(_matrix(case["matrix"], case["m"], case["n"], gen).cpu().numpy(), case["nplus"])
    none = {"G": None, "D": D, "sweeps": None, "rot_s": None, "rot_b": None}
    if case["alg"] & 2:
        none["V"] = None
    return none
