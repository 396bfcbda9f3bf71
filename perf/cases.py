"""The work a user of this framework has it do, as cases that can be timed.

Five kinds of pass, each through the public Python binding of libgfc:

  fix     a configuration resident in HBM is gauge-fixed and measured, and G is
          taken to the host (Job.restore_config, fix, plaquette, observables,
          download_gauge): the product path, re-run for another set of
          parameters on the same lattice
  host    a host array is uploaded, reunitarized, measured, fixed, measured
          again, and U and G are downloaded: the drop-in sequence on arrays
  measure reunitarization, plaquettes and residues of a resident
          configuration, or of one streamed from a file first
  trace   the residue after every half-sweep (convergence studies)
  serve   several lattices submitted together to the batching server

Lattice sizes are those of the tests and the benchmark; configurations are
gauge-rotated smooth SU(3) links, in FP32 as stored files mostly are, with the
spread eps of the link matrices that the benchmark and the serving mix use.
"""
import math
import os
import sys
import tempfile

import numpy as np
import torch

sys.path.insert(0, os.path.abspath("gaugefix-coulomb_amd"))
import gfc  # noqa: E402

BIG = 1 << 22          # lattices above this are synthesised in HBM by the framework
EXACT_MOST = 1.6e8     # site half-sweeps that `exact` runs in torch


def _case(name, kind, ns, nt, precision="fp64", tol=1e-16, est=1000, reunit=10, omega=1.95,
          hits=2, proxy="e2", eps=0.35, max_sweeps=100000, retire=False, sweeps=1085, count=0,
          source="hbm"):
    """`sweeps`: half-sweeps the fix takes (about), for work() alone."""
    c = dict(kind=kind, ns=ns, nt=nt, precision=precision, tol=tol, est=est, reunit=reunit,
             omega=omega, hits=hits, proxy=proxy, eps=eps, max_sweeps=max_sweeps, retire=retire,
             sweeps=sweeps, count=count, source=source)
    if name:
        c["name"] = name
    return c


def listed():
    return [
        # the smallest lattice people test a new setup on; launches and latency
        _case("fix_8x16", "fix", 8, 16, eps=0.25),
        # an odd size (a timeslice is no whole number of tiles), the theta proxy,
        # one hit, a milder overrelaxation, the dense check schedule
        _case("fix_14x28_theta", "fix", 14, 28, tol=1e-10, est=0, reunit=250, omega=1.7, hits=1,
              proxy="theta", eps=0.3, sweeps=560),
        # the command line's sequence on a small production lattice
        _case("host_16x32", "host", 16, 32, eps=0.3),
        # a convergence study: the residue after each half-sweep
        _case("trace_16x32", "trace", 16, 32, tol=1e-300, est=100000000, eps=0.3,
              max_sweeps=100, sweeps=100),
        # a burst of the serving mix (16^3 x 32 to 32^3 x 64, both precisions)
        _case("serve_mix", "serve", 16, 32, "mixed", count=6, eps=0.3),
        # ordinary production sizes, fixed in mixed and in double precision
        _case("fix_20x40_mixed", "fix", 20, 40, "mixed", eps=0.3),
        _case("fix_32x64", "fix", 32, 64, eps=0.35),
        # a configuration file looked over: loaded, reunitarized, measured
        _case("measure_file_32x64", "measure", 32, 64, source="file", sweeps=0),
        # the headline workload, in both precisions
        _case("fix_48x96", "fix", 48, 96),
        _case("fix_48x96_mixed", "fix", 48, 96, "mixed"),
        # its configuration reunitarized and measured in place
        _case("measure_48x96", "measure", 48, 96, sweeps=0),
        # the largest lattice of the benchmark, fixed loosely with timeslices
        # retired as they converge
        _case("fix_64x128_retire", "fix", 64, 128, "mixed", tol=1e-13, est=0, retire=True,
              sweeps=500),
    ]


def draw(rng):
    def even(lo, hi, step=2):
        """An even size spread over its logarithm."""
        return max(lo, min(hi, step * round(math.exp(rng.uniform(math.log(lo), math.log(hi))) / step)))

    kind = rng.choice(["fix"] * 6 + ["host", "measure", "trace", "serve"])
    if kind == "serve":
        return _case("", "serve", rng.choice([8, 12, 16]), rng.choice([16, 24, 32]), "mixed",
                     count=rng.randint(2, 6), eps=round(rng.uniform(0.2, 0.4), 3))
    if kind == "trace":
        n = rng.randint(20, 100)
        return _case("", "trace", even(4, 24), even(4, 48), tol=1e-300, est=100000000,
                     reunit=rng.choice([7, 10, 50]), omega=round(rng.uniform(1.5, 1.95), 3),
                     eps=round(rng.uniform(0.2, 0.4), 3), max_sweeps=n, sweeps=n)
    if kind == "measure":
        return _case("", "measure", even(8, 48), even(8, 96), eps=round(rng.uniform(0.2, 0.4), 3),
                     sweeps=0)
    if kind == "host":
        return _case("", "host", even(6, 20), even(6, 40), rng.choice(["fp64", "mixed"]),
                     eps=round(rng.uniform(0.2, 0.4), 3))
    retire = rng.random() < 0.2
    ns = even(8, 56, 8) if retire else even(6, 56)
    nt = even(6, min(112, 2 * ns + 8))
    precision = rng.choice(["fp64", "mixed"])
    if rng.random() < 0.5:  # to convergence on the reference's schedule
        return _case("", "fix", ns, nt, precision, tol=rng.choice([1e-16, 1e-14, 1e-12]),
                     reunit=rng.choice([10, 50, 250]), eps=round(rng.uniform(0.2, 0.4), 3),
                     proxy=rng.choice(["e2", "theta"]), retire=retire)
    n = rng.randint(60, 400)  # stopped after a number of half-sweeps
    return _case("", "fix", ns, nt, precision, tol=1e-300, est=100000000,
                 reunit=rng.choice([5, 10, 250]), omega=round(rng.uniform(1.5, 1.95), 3),
                 hits=rng.randint(1, 3), eps=round(rng.uniform(0.2, 0.4), 3), max_sweeps=n,
                 retire=retire, sweeps=n)


# ---------------------------------------------------------------------------
# SU(3) fields in torch: complex matrices as (3, 3, ...) with the sites last.

def _mul(a, b):
    return (a[:, :, None] * b[None]).sum(1)


def _dag(a):
    return a.transpose(0, 1).conj()


def _cross(a, b):
    """conj(a x b) of two rows."""
    return torch.stack([a[1] * b[2] - a[2] * b[1], a[2] * b[0] - a[0] * b[2],
                        a[0] * b[1] - a[1] * b[0]]).conj()


def _unit(r):
    return r / r.abs().square().sum(0).sqrt()


def _project(m):
    """The reference's projectSU3: row 0 and the cross product normalised."""
    r0 = _unit(m[0])
    r2 = _unit(_cross(r0, m[1]))
    return torch.stack([r0, _cross(r2, r0), r2])


def _smooth(ns, nt, eps, seed):
    """U_mu(n) = g(n) X_mu(n) g(n + mu)^dagger with X within eps of 1 and g Haar-random, as a
    host array (V, 4, 3, 3) in FP32."""
    gen = torch.Generator(device="cuda")
    gen.manual_seed(seed * 1000003 + ns * 131 + nt)
    shape = (nt, ns, ns, ns)

    def normal(*s):
        z = torch.randn(*s, 2, generator=gen, device="cuda", dtype=torch.float64)
        return torch.view_as_complex(z)

    z = normal(3, 3, *shape)
    r0 = _unit(z[0])
    r1 = _unit(z[1] - (r0.conj() * z[1]).sum(0) * r0)
    g = torch.stack([r0, r1, _cross(r0, r1)])
    del z
    one = torch.eye(3, device="cuda", dtype=torch.complex128).reshape(3, 3, 1, 1, 1, 1)
    U = torch.empty(*shape, 4, 3, 3, device="cuda", dtype=torch.complex64)
    for mu in range(4):
        h = normal(3, 3, *shape) * math.sqrt(0.5)
        h = h + _dag(h)
        x = _project(one + 1j * eps * h * 0.7)
        u = _mul(_mul(g, x), _dag(g.roll(-1, 2 + mu)))
        U[..., mu, :, :] = u.permute(2, 3, 4, 5, 0, 1).to(torch.complex64)
    return U.reshape(-1, 4, 3, 3)


def _links(case, seed):
    return _smooth(case["ns"], case["nt"], case["eps"], seed)


def _params(case):
    return gfc.Params(tolerance=case["tol"],
                      gfix_proxy=gfc.PROXY_THETA if case["proxy"] == "theta" else gfc.PROXY_E2,
                      max_sweeps_to_fix=case["max_sweeps"],
                      estimate_sweeps_to_gf_progress=case["est"],
                      sweeps_to_reunitarization=case["reunit"], omega_OR=case["omega"],
                      hits=case["hits"])


def _options(case):
    return gfc.Options(precision=gfc.PREC_MIXED if case["precision"] == "mixed" else gfc.PREC_FP64,
                       retire_slices=int(case["retire"]))


def _volume(case):
    return case["ns"] ** 3 * case["nt"]


# The requests of a serve case, from the size and precision it names up.
def _requests(case):
    out = []
    for k in range(case["count"]):
        c = dict(case)
        c["ns"] = case["ns"] * (1, 1, 2, 1, 1.5, 1)[k % 6]
        c["nt"] = case["nt"] * (1, 1, 2, 1, 1.5, 1)[k % 6]
        c["ns"], c["nt"] = 2 * int(c["ns"] // 2), 2 * int(c["nt"] // 2)
        c["precision"] = "fp64" if k % 6 == 3 else "mixed"
        c["tol"] = 1e-16 if k % 2 == 0 else 1e-14
        out.append(c)
    return out


def prepare(case, seed):
    state = {"case": case, "ctx": gfc.Context(0)}
    if case["kind"] == "serve":
        reqs = _requests(case)
        state["inputs"] = [(gfc.Geometry(c["ns"], c["nt"]), _links(c, seed + 17 * k).cpu().numpy(),
                            _params(c), _options(c)) for k, c in enumerate(reqs)]
        state["server"] = gfc.Server(state["ctx"], max_jobs=8, keep_results=True)
        return state
    geom = gfc.Geometry(case["ns"], case["nt"])
    state.update(geom=geom, params=_params(case), options=_options(case))
    state["job"] = job = gfc.Job(state["ctx"], geom, state["options"].precision)
    if case["source"] == "file":
        state["folder"] = tempfile.TemporaryDirectory()
        state["path"] = os.path.join(state["folder"].name, "config")
        _links(case, seed).cpu().numpy().tofile(state["path"])
        return state
    if _volume(case) > BIG:
        job.generate_smooth(seed, case["eps"])
    elif case["kind"] == "host":
        state["U"] = _links(case, seed).cpu().numpy()
        return state
    else:
        job.upload_config(_links(case, seed).cpu().numpy())
    if case["kind"] != "measure":
        job.reunitarize()
        job.save_config()
    return state


def _after(job):
    """What the command line measures after a fix, and G.  (The residue itself, some 1e-17 of
    rounding and of how far the last sweeps went, is no number to compare.)"""
    return {"plaquette": np.array(job.plaquette()), "F": np.array(job.observables()[2]),
            "G": job.download_gauge()}


def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "serve":
        server = state["server"]
        ids = [server.submit_config(g, U, p, o) for g, U, p, o in state["inputs"]]
        server.drain()
        out = []
        for rid, (g, _, _, _) in zip(ids, state["inputs"]):
            out.append(server.result_gauge(rid, g))
            server.release(rid)
        return out
    job = state["job"]
    if kind == "measure":
        if case["source"] == "file":
            job.load_config(state["path"], 4, False)
        job.reunitarize()
        return {"plaquette": np.array(job.plaquette()), "observables": np.array(job.observables())}
    if kind == "host":
        job.upload_config(state["U"])
        job.reunitarize()
        before = np.array(job.plaquette())
        job.fix(state["params"], state["options"])
        return {"before": before, **_after(job), "U": job.download_config()}
    job.restore_config()
    if kind == "trace":
        _, _, trace = job.fix(state["params"], state["options"], trace_len=case["max_sweeps"])
        return {"trace": trace, "G": job.download_gauge()}
    job.fix(state["params"], state["options"])
    return _after(job)


# ---------------------------------------------------------------------------
# What a pass cannot do without.  A half-sweep reads, for all sites, two of the
# three spatial links (the third can be gauged away) and G, and writes G on one
# parity, each matrix as the 8 real numbers of SU(3); a fix also reads the
# configuration and writes G and the fixed configuration.  Operations per site
# update: six complex matrix products and sums, one more for w, the hits and
# the projection.

def _fix_work(case, sweeps, f32_share):
    V = _volume(case)
    real = 8 * (1 - f32_share) + 4 * f32_share
    half = V * 8 * (2 + 1 + 0.5) * real
    flops = V / 2 * (6 * 216 + 198 + 3 * case["hits"] * 110 + 300)
    return {"bytes": V * (576 + 576 + 144) + sweeps * half, "flops": sweeps * flops}


def work(case):
    V = _volume(case)
    kind = case["kind"]
    if kind == "serve":
        parts = [_fix_work(c, 1085, 0.0 if c["precision"] == "fp64" else 0.7)
                 for c in _requests(case)]
        return {k: sum(p[k] for p in parts) for k in ("bytes", "flops")}
    if kind == "measure":
        return {"bytes": V * (288 + 1152 if case["source"] == "file" else 1152),
                "flops": V * (4 * 110 + 6 * 2 * 198 + 300)}
    w = _fix_work(case, case["sweeps"], 0.7 if case["precision"] == "mixed" else 0.0)
    if kind == "host":
        w["bytes"] += V * 288  # the FP32 input; U and G written are counted above
    if kind == "trace":
        w["bytes"] += case["sweeps"] * V * 8 * 3 * 8
    return w


def tolerance(case):
    if case["kind"] == "serve" or case["precision"] == "mixed":
        # G keeps the rounding of the single-precision phase in the directions
        # that do not change the gauge condition (a rotation per timeslice):
        # 1e-6 to 1e-5 against double precision, by lattice size
        return {"rel": 1e-4, "max": 1e-3}
    # rounding carried through up to a thousand overrelaxed half-sweeps: 5e-15
    # to 1.5e-13 in G, 2e-16 to 2e-15 in the sums
    return {"rel": 1e-12, "max": 1e-11}


# ---------------------------------------------------------------------------
# The same results in plain torch, in double precision.

def _obs(U):
    """e2, theta, F of U (4 x (3, 3, t, z, y, x), mu = T, Z, Y, X)."""
    V = U[1][0, 0].numel()
    D = sum((U[m] - _dag(U[m])) - (U[m] - _dag(U[m])).roll(1, 2 + m) for m in (1, 2, 3))
    eye = torch.eye(3, device=D.device, dtype=D.dtype).reshape(3, 3, 1, 1, 1, 1)
    D = D - (D[0, 0] + D[1, 1] + D[2, 2]) / 3 * eye
    A = -0.5j * D
    c = [A[0, 1].real + A[1, 0].real, A[1, 0].imag - A[0, 1].imag, A[0, 0].real - A[1, 1].real,
         A[0, 2].real + A[2, 0].real, A[2, 0].imag - A[0, 2].imag,
         A[1, 2].real + A[2, 1].real, A[2, 1].imag - A[1, 2].imag,
         (A[0, 0].real + A[1, 1].real - 2 * A[2, 2].real) / math.sqrt(3)]
    e2 = sum(float(x.square().sum()) for x in c) / V
    theta = float(A.abs().square().sum()) / (3 * V)
    F = sum(float((U[m][0, 0] + U[m][1, 1] + U[m][2, 2]).real.sum()) for m in (1, 2, 3)) / (9 * V)
    return e2, theta, F


def _plaquette(U):
    out = []
    for planes in (((3, 2), (3, 1), (2, 1)), ((0, 1), (0, 2), (0, 3))):
        s = 0.0
        for m, n in planes:
            a = _mul(U[m], U[n].roll(-1, 2 + m))
            b = _mul(U[n], U[m].roll(-1, 2 + n))
            s += float((a * b.conj()).sum().real) / 3
        out.append(s / (3 * U[0][0, 0].numel()))
    return tuple(out)


def _transform(U0, G):
    return [_mul(_mul(G, U0[m]), _dag(G.roll(-1, 2 + m))) if m else U0[0] for m in range(4)]


def _local(w, hits, omega):
    g = torch.zeros_like(w)
    for k in range(3):
        g[k, k] = 1
    for _ in range(hits):
        for a, b in ((0, 1), (0, 2), (1, 2)):
            q = torch.stack([(w[a, a] + w[b, b]).real, -(w[a, b] + w[b, a]).imag,
                             -(w[a, b] - w[b, a]).real, -(w[a, a] - w[b, b]).imag])
            q = q / q.square().sum(0).sqrt()
            x0, x1, x2, x3 = q
            al, be = torch.complex(x0, x3), torch.complex(x2, x1)
            for m in (w, g):
                ra, rb = m[a].clone(), m[b].clone()
                m[a] = al * ra + be * rb
                m[b] = -be.conj() * ra + al.conj() * rb
    g = omega * g
    for k in range(3):
        g[k, k] += 1 - omega
    return _project(g)


def _fix(U0, case, trace=None):
    """gaugefixOverrelaxation in double precision, with G and the input kept apart."""
    omega = float(np.float32(case["omega"]))
    which = 1 if case["proxy"] == "theta" else 0
    shape = U0[1].shape[2:]
    at = sum(torch.arange(n, device="cuda").reshape([-1 if k == d else 1 for k in range(4)])
             for d, n in enumerate(shape))
    parity = (at & 1).to(torch.bool)
    G = torch.zeros_like(U0[1])
    for k in range(3):
        G[k, k] = 1
    res = _obs(_transform(U0, G))[which]

    def due_after(s, r):
        return s + 10 + int(case["est"] * (1 - math.log10(r) / math.log10(case["tol"])))

    due, s = due_after(0, res), 0
    while res > case["tol"]:
        W = sum(_mul(U0[m], _dag(G.roll(-1, 2 + m))) +
                _mul(_dag(U0[m].roll(1, 2 + m)), _dag(G.roll(1, 2 + m))) for m in (1, 2, 3))
        new = _mul(_local(_mul(G, W), case["hits"], omega), G)
        G = torch.where(parity if s & 1 else ~parity, new, G)
        s += 1
        if trace is not None:
            trace.append(_obs(_transform(U0, G))[which])
        if s == due:
            res = _obs(_transform(U0, G))[which]
            if res <= case["tol"]:
                break
            due = due_after(s, res)
        if s >= case["max_sweeps"]:
            return G
        if s % case["reunit"] == 0:
            G = _project(G)
    return _project(G)


def _field(case, seed):
    """The reunitarized input: 4 fields (3, 3, t, z, y, x)."""
    U = _links(case, seed).to(torch.complex128)
    U = U.reshape(case["nt"], case["ns"], case["ns"], case["ns"], 4, 3, 3)
    return [_project(U[..., m, :, :].permute(4, 5, 0, 1, 2, 3).contiguous()) for m in range(4)]


def _array(G):
    return G.permute(2, 3, 4, 5, 0, 1).reshape(-1, 3, 3).cpu().numpy()


def exact(case, seed):
    kind = case["kind"]
    if kind == "serve":
        return [_array(_fix(_field(c, seed + 17 * k), c)) if _volume(c) * 1085 < EXACT_MOST / 4 or
                (k == 0 and _volume(c) * 1085 < EXACT_MOST) else None
                for k, c in enumerate(_requests(case))]
    if _volume(case) > BIG or case["retire"] or _volume(case) * case["sweeps"] > EXACT_MOST:
        return None
    U = _field(case, seed)
    if kind == "measure":
        return {"plaquette": np.array(_plaquette(U)), "observables": np.array(_obs(U))}
    trace = [] if kind == "trace" else None
    G = _fix(U, case, trace)
    if kind == "trace":
        return {"trace": np.array(trace), "G": _array(G)}
    fixed = [_mul(_mul(G, U[m]), _dag(G.roll(-1, 2 + m))) for m in range(4)]
    out = {"plaquette": np.array(_plaquette(fixed)), "F": np.array(_obs(fixed)[2]), "G": _array(G)}
    if kind == "host":
        out["before"] = np.array(_plaquette(U))
        out["U"] = np.stack([_array(u) for u in fixed], axis=1)
    return out
