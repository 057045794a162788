"""Timed cases of the alpha transport: what programs built on this library have
it do, through its public entry points, over the range of sizes, meshes and
dictionary options that its tests and benchmark use.

Kinds of case
  run      the advection benchmark's time loop on fields resident in HBM
           (plicVof.H:37-42): Courant number, time step, flow factor,
           reconstruct, advect; `steps` of them from a given alpha.
  coupled  one alpha step of a two-phase solver whose fields live on the GPU
           (interPlicFoam's alphaEqnSubCycle.H): old alpha, phi and U handed
           over, `sub` reconstruct + advect steps, new alpha and rhoPhi out.
  batch    independent small cases advanced together, `steps` batch steps with
           each case's own time step.
  export   reconstruct and the PLIC polygons into the program's device buffers,
           as at every write time.

Meshes: "hex" N^3 hexahedra, "hexp" the same with interior vertices displaced
by 20 % (warped faces), "tet" N^3 cubes of six tetrahedra, "refined" N^3 with a
2:1 refined middle block (cells of up to 24 faces).

The starting alpha is the exact field of seeded ellipsoids or spheres after a
few steps of the case's own flow, so that it has the layers of nearly full and
nearly empty cells that a run has behind its interface.
"""
import ctypes as C
import functools

import numpy as np
import torch

import geometricvofext_amd as g
from geometricvofext_amd import cases as shapes_of
from geometricvofext_amd import harness

WARM_STEPS = 12
PERIOD = 6.0      # of the deformation's time factor (end time 3, reversing)
START = 0.4       # time at which a pass starts


def listed():
    return [
        # the smallest mesh of the batched workload on one handle: launches and latency
        case("run-hex16", kind="run", mesh="hex", N=16, steps=8),
        # odd size, warped faces, the library's default dictionary (10 bounding passes, clip)
        case("run-hex33p-defaults", kind="run", mesh="hexp", N=33, steps=6, bounds=10, clip=True),
        # the reference tutorial's own mesh and dictionary
        case("run-hex64", kind="run", mesh="hex", N=64, steps=4),
        # the headline workload: 128^3 perturbed hexahedra
        case("run-hex128p", kind="run", mesh="hexp", N=128, steps=4),
        # tetrahedra under solid-body rotation, 8 spheres
        case("run-tet28", kind="run", mesh="tet", N=28, steps=4, flow="rotation", shapes=8),
        # the reconstructed-distance-function normal
        case("run-hex48p-rdf", kind="run", mesh="hexp", N=48, steps=2, method="isoRDF"),
        # the learned normal
        case("run-hex64-learned", kind="run", mesh="hex", N=64, steps=4, method="learned"),
        # cells of up to 24 faces next to a refined block
        case("run-refined20", kind="run", mesh="refined", N=20, steps=2),
        # a solver's alpha step, two sub-cycles, the tutorials' snap and clip
        case("coupled-hex64", kind="coupled", mesh="hex", N=64, sub=2, snap=1e-12, clip=True),
        # a phase-change solver's step: sources, Gauss-gradient normal, odd size
        case("coupled-hex45p-sources", kind="coupled", mesh="hexp", N=45, sub=1, method="alphaGrad", sources=True),
        # many small cases in the same launches
        case("batch-12", kind="batch", mesh="hex", N=40, count=12, steps=6),
        # the interface written as polygons
        case("export-hex64", kind="export", mesh="hex", N=64),
    ]


def case(name=None, kind="run", mesh="hex", N=32, steps=1, sub=1, count=1, method="LS", bounds=3, snap=0.0,
         clip=False, flow="deformation", shapes=3, sources=False):
    c = dict(kind=kind, mesh=mesh, N=N, steps=steps, sub=sub, count=count, method=method, bounds=bounds, snap=snap,
             clip=clip, flow=flow, shapes=shapes, sources=sources)
    return dict(c, name=name) if name else c


# cells per N^3 of each mesh
CELLS = {"hex": 1.0, "hexp": 1.0, "tet": 6.0, "refined": 1.9}


def draw(rng):
    """One more case: sizes spread over their logarithm, every mesh, normal and dictionary option."""
    def size(lo, hi):
        return int(round(lo * (hi / lo) ** rng.random()))
    kind = rng.choices(["run", "coupled", "batch", "export"], [5, 3, 1, 1])[0]
    if kind == "batch":
        return case(kind=kind, mesh=rng.choice(["hex", "hexp"]), N=size(18, 44), count=rng.randint(4, 14),
                    steps=rng.randint(2, 6), bounds=3)
    mesh = rng.choices(["hex", "hexp", "tet", "refined"], [4, 4, 2, 1])[0]
    N = size(12, 96) if mesh in ("hex", "hexp") else (size(8, 30) if mesh == "tet" else size(8, 24))
    method = rng.choices(["LS", "isoRDF", "alphaGrad", "learned"], [5, 1, 1, 1])[0]
    if mesh != "hex" and method == "learned":
        method = "LS"
    if kind == "export":
        return case(kind=kind, mesh=mesh, N=N, method="LS", shapes=rng.randint(1, 8))
    snap, clip = rng.choice([(0.0, False), (0.0, True), (1e-12, True)])
    return case(kind=kind, mesh=mesh, N=N, steps=rng.randint(1, 4) if kind == "run" else 1,
                sub=rng.choice([1, 1, 2, 3]) if kind == "coupled" else 1, method=method,
                bounds=rng.choice([2, 3, 10]), snap=snap, clip=clip, flow=rng.choice(["deformation", "rotation"]),
                shapes=rng.randint(1, 8), sources=kind == "coupled" and rng.random() < 0.3)


# ---------------------------------------------------------------------------
@functools.lru_cache(maxsize=4)
def make_mesh(mesh, N):
    if mesh == "tet":
        return g.tet_box(N, perturb=0.1, seed=2)
    if mesh == "refined":
        return g.refined_hex_box(N)
    return g.hex_box(N, perturb=0.2 if mesh == "hexp" else 0.0, seed=1)


@functools.lru_cache(maxsize=1)
def normal_model():
    """A network trained as the benchmark trains it, on fewer samples."""
    m = g.NormalModel(seed=11)
    m.generate(1 << 16, seed=23, depth=4)
    m.train(epochs=20, batch=4096, lr0=3e-3, lr1=3e-5, seed=12)
    return m


def ok(rc):
    if rc != 0:
        raise RuntimeError(g.lib().svp_last_error().decode())


def solver_of(case, seed):
    """A handle with the case's dictionary, the seeded shapes as its alpha and its base flow uploaded."""
    s = g.SolveVofEqu(make_mesh(case["mesh"], case["N"]),
                      dict(orientationMethod=case["method"], nAlphaBounds=case["bounds"], snapTol=case["snap"],
                           clip=case["clip"], mixedCellTol=1e-8))
    if case["method"] == "learned":
        s.set_normal_model(normal_model())
    if case["shapes"] > 3:
        s.init_alpha(shapes_of.random_spheres(seed, n=case["shapes"]), max_depth=3)
    else:
        s.init_alpha(shapes_of.random_ellipsoids(seed, n=case["shapes"]), max_depth=3)
    if case["flow"] == "rotation":
        U, phi = s.rotation_field(shapes_of.rotation_omega(seed, 1.0), (0.5, 0.5, 0.5))
    else:
        U, phi = s.deformation_field()
    s.upload_base_flow(U, phi)
    s.scale_flow(1.0)
    return s, U, phi


def alpha_of(s):
    a = torch.empty(s.mesh.n_cells, dtype=torch.float64, device="cuda")
    ok(g.lib().svp_get_alpha(s.h, a.data_ptr(), g.SVP_DEVICE))
    s.synchronize()
    return a


def prepare(case, seed):
    if case["kind"] == "batch":
        return prepare_batch(case, seed)
    s, U, phi = solver_of(case, seed)
    dt = 0.5 / (0.5 * s.courant()[0])     # Courant number 0.5
    for _ in range(WARM_STEPS):
        s.reconstruct()
        s.advect(dt)
    st = dict(kind=case["kind"], s=s, dt=dt, steps=case["steps"], sub=case["sub"],
              period=0.0 if case["flow"] == "rotation" else PERIOD, alpha0=alpha_of(s))
    m = s.mesh
    if case["kind"] == "export":
        # the program's own buffers, large enough for any of its interfaces
        st["cap"] = (40 if case["mesh"] == "tet" else 16) * case["N"] ** 2
        st["cells"] = torch.zeros(st["cap"], dtype=torch.int32, device="cuda")
        st["offsets"] = torch.zeros(st["cap"] + 1, dtype=torch.int32, device="cuda")
        st["points"] = torch.zeros((8 * st["cap"], 3), dtype=torch.float64, device="cuda")
    st["alpha"] = torch.empty_like(st["alpha0"])
    st["flux"] = torch.empty(m.n_faces, dtype=torch.float64, device="cuda")
    if case["kind"] == "coupled":
        st["phi"] = torch.from_numpy(np.ascontiguousarray(phi)).cuda()
        st["U"] = torch.from_numpy(np.ascontiguousarray(U)).cuda()
        st["Ub"] = torch.zeros(3 * (m.n_faces - m.n_internal_faces), dtype=torch.float64, device="cuda")
        st["Sp"] = st["Su"] = None
        if case["sources"]:
            gen = torch.Generator(device="cuda").manual_seed(seed)
            st["Sp"] = -0.05 * torch.rand(m.n_cells, dtype=torch.float64, device="cuda", generator=gen)
            st["Su"] = 0.02 * torch.rand(m.n_cells, dtype=torch.float64, device="cuda", generator=gen)
    torch.cuda.synchronize()
    return st


def prepare_batch(case, seed):
    rng = np.random.default_rng(seed)
    solvers, alpha0, periods = [], [], []
    for k in range(case["count"]):
        # sizes spread over the workload's range 16 .. N, the same for every seed
        n = 16 + (7 * k + 3) % max(case["N"] - 15, 1)
        one = dict(case, N=n, shapes=1 + k % 3, flow="rotation" if k % 2 else "deformation")
        s, _, _ = solver_of(one, int(rng.integers(1 << 30)))
        dt = 0.5 / (0.5 * s.courant()[0])
        for _ in range(WARM_STEPS):
            s.reconstruct()
            s.advect(dt)
        solvers.append(s)
        alpha0.append(alpha_of(s))
        periods.append(0.0 if k % 2 else PERIOD)
    b = g.CaseBatch(solvers)
    torch.cuda.synchronize()
    return dict(kind="batch", batch=b, solvers=solvers, alpha0=alpha0, periods=periods, steps=case["steps"],
                alpha=[torch.empty_like(a) for a in alpha0])


def clock(dt):
    return harness.RunTime(end_time=10.0, delta_t=dt, write_interval=10.0, start_time=0.0, max_co=0.5,
                           max_alpha_co=0.5)


def run(st):
    return {"run": run_steps, "coupled": run_coupled, "batch": run_batch, "export": run_export}[st["kind"]](st)


def run_steps(st):
    s, L = st["s"], g.lib()
    rt = clock(st["dt"])
    rt.value = START
    ok(L.svp_set_alpha(s.h, st["alpha0"].data_ptr(), g.SVP_DEVICE))
    s.scale_flow(harness.u_factor(rt.value, rt.delta_t, st["period"]))
    for _ in range(st["steps"]):
        co, aco = s.courant()
        rt.set_delta_t(0.5 * co * rt.delta_t, 0.5 * aco * rt.delta_t)
        rt.increment()
        s.scale_flow(harness.u_factor(rt.value, rt.delta_t, st["period"]))
        s.reconstruct()
        s.advect(rt.delta_t)
    ok(L.svp_get_alpha(s.h, st["alpha"].data_ptr(), g.SVP_DEVICE))
    ok(L.svp_get_alpha_phi(s.h, st["flux"].data_ptr(), g.SVP_DEVICE))
    s.synchronize()
    return {"alpha": st["alpha"], "alphaPhi": st["flux"]}


def run_coupled(st):
    s, L = st["s"], g.lib()

    def p(t):
        return None if t is None else t.data_ptr()
    ok(L.svp_set_alpha(s.h, p(st["alpha0"]), g.SVP_DEVICE))
    ok(L.svp_set_flow(s.h, p(st["phi"]), p(st["U"]), p(st["Ub"]), g.SVP_DEVICE))
    ok(L.svp_advect_sub_cycles(s.h, st["dt"], st["sub"], p(st["Sp"]), p(st["Su"]), 1000.0, 1.0, p(st["flux"]),
                               g.SVP_DEVICE))
    ok(L.svp_get_alpha(s.h, p(st["alpha"]), g.SVP_DEVICE))
    s.synchronize()
    return {"alpha": st["alpha"], "rhoPhi": st["flux"]}


def run_batch(st):
    b, L, n = st["batch"], g.lib(), len(st["solvers"])
    for s, a in zip(st["solvers"], st["alpha0"]):
        ok(L.svp_set_alpha(s.h, a.data_ptr(), g.SVP_DEVICE))
    clocks = [clock(1e-3) for _ in range(n)]
    for rt in clocks:
        rt.value = START
    b.scale_flow([harness.u_factor(rt.value, rt.delta_t, p) for rt, p in zip(clocks, st["periods"])])
    for _ in range(st["steps"]):
        co, aco = b.courant()
        for k, rt in enumerate(clocks):
            rt.set_delta_t(0.5 * co[k] * rt.delta_t, 0.5 * aco[k] * rt.delta_t)
            rt.increment()
        b.scale_flow([harness.u_factor(rt.value, rt.delta_t, p) for rt, p in zip(clocks, st["periods"])])
        b.step([rt.delta_t for rt in clocks])
    for s, a in zip(st["solvers"], st["alpha"]):
        ok(L.svp_get_alpha(s.h, a.data_ptr(), g.SVP_DEVICE))
    st["solvers"][0].synchronize()
    return list(st["alpha"])


def run_export(st):
    s, L = st["s"], g.lib()
    nf, npt = C.c_int32(), C.c_int32()
    s.reconstruct()
    ok(L.svp_get_plic_surface(s.h, C.addressof(nf), C.addressof(npt), None, None, None, g.SVP_DEVICE))
    if nf.value > st["cap"] or npt.value > 8 * st["cap"]:
        raise RuntimeError("the program's polygon buffers are too small")
    ok(L.svp_get_plic_surface(s.h, C.addressof(nf), C.addressof(npt), st["cells"].data_ptr(), st["offsets"].data_ptr(),
                              st["points"].data_ptr(), g.SVP_DEVICE))
    return {"polygons": nf.value, "points": npt.value, "cells": st["cells"], "offsets": st["offsets"],
            "xyz": st["points"]}


# ---------------------------------------------------------------------------
def sizes(case, N):
    """(cells, faces, interface cells) of one mesh: faces about 3 per hexahedron and 2 per tetrahedron; interface
    cells from the area of the seeded shapes (radius about 0.11, smeared over one and a half layers)."""
    nc = CELLS[case["mesh"]] * N ** 3
    nf = (2.0 if case["mesh"] == "tet" else 3.0) * nc + 6.0 * N * N
    area = 4.0 * 3.14159 * 0.11 ** 2 * min(case["shapes"], 6)
    return nc, nf, 2.0 * area * N * N * (3.0 if case["mesh"] == "tet" else 1.0)


def work(case):
    """Per step: alpha, alpha_old and V per cell, phi, the owner and neighbour labels and dVf per face, and about
    0.5 kB per interface cell (plane placement and flux integrals: points, labels, normal, plane)."""
    if case["kind"] == "batch":
        meshes = [16 + (7 * k + 3) % max(case["N"] - 15, 1) for k in range(case["count"])]
    else:
        meshes = [case["N"]]
    nbytes = flops = 0.0
    for n in meshes:
        nc, nf, nic = sizes(case, n)
        steps = case["sub"] if case["kind"] == "coupled" else case["steps"]
        per_ic = 272.0 if case["mesh"] == "tet" else 512.0
        if case["kind"] == "export":
            nbytes += 8.0 * nc + per_ic * nic
            flops += 6.0e3 * nic
        else:
            nbytes += steps * (24.0 * nc + 24.0 * nf + per_ic * nic)
            flops += steps * (8.0e3 * nic + 4.0 * nf + 8.0 * nc)
    return {"bytes": nbytes, "flops": flops}


def exact(case, seed):
    """None: every output is a 64-bit result of the whole transport (cut geometry, root search, bounding walk), which
    has no independent plain restatement of this size; the outputs are FP64 throughout."""
    return None
