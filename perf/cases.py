"""The work that programs have this framework do, as timed cases: single steps of one instance, batched
steps, and a served request stream, through the public entry points of hobakv1_amd.lib.

A pass of a `step` or `batch` case sets the instances' states, advances each by one step and reads the
states back, which is what the reference-shaped solve() does and what a program that edits or
records every frame does.  A pass of a `serve` case submits a few step requests per session to the
continuous-batching scheduler and ticks it until all of them are done.
"""
import math

import numpy as np
import torch

from hobakv1_amd import lib, scenes

JACOBI, BLOCK = scenes.PRECOND_JACOBI, scenes.PRECOND_BLOCK_JACOBI


def _step(name, nx, ny, nz, precision="fp64", material="snh", precond="block", newton=1, form="position",
          pinned=True):
    return {"name": name, "kind": "step", "nx": nx, "ny": ny, "nz": nz, "precision": precision,
            "material": material, "precond": precond, "newton": newton, "form": form, "pinned": pinned}


def listed():
    return [
        # the smallest call: the two dozen vertices' worth of latency a toy scene or a unit test sees
        _step("step_4_fp64", 4, 4, 4),
        # an interactive single object with the reference's own preconditioner
        _step("step_10_jacobi_fp64", 10, 10, 10, precond="jacobi"),
        # the same object in the reduced-precision form
        _step("step_10_fp32", 10, 10, 10, precision="fp32"),
        # an odd-sized ARAP body on the BDF_1 integrator, up to three Newton iterations a step
        _step("step_17x9x23_arap_bdf_fp64", 17, 9, 23, material="arap", newton=3),
        # a body landing on a kinematic cube, on the velocity integrator (plane constraints)
        _step("drop_11x13x12_velocity_fp64", 11, 13, 12, form="velocity", pinned=False),
        # the 384,000-tet stretch scene, in the reference's arithmetic and in the reduced-precision form
        _step("step_40_fp64", 40, 40, 40),
        _step("step_40_fp32", 40, 40, 40, precision="fp32"),
        # one mesh whose matrix does not fit the caches, both forms
        _step("step_57x64x50_fp64", 57, 64, 50),
        _step("step_72x61x66_fp32", 72, 61, 66, precision="fp32"),
        # many independent instances of 4..24 cells per axis, stepped together
        {"name": "batch_48_fp64", "kind": "batch", "count": 48, "lo": 4, "hi": 24, "mix": 4,
         "precision": "fp64"},
        {"name": "batch_128_fp32", "kind": "batch", "count": 128, "lo": 4, "hi": 24, "mix": 4,
         "precision": "fp32"},
        # served sessions of very uneven size falling onto a penalty ground, two requests each
        {"name": "serve_24_fp32", "kind": "serve", "count": 24, "requests": 2, "mix": 5,
         "precision": "fp32"},
    ]


def draw(rng):
    """Any of the three kinds: single steps from about 400 to 400,000 tets with odd, uneven axes, batches
    of 2 to 64 small instances, and streams of 2 to 16 sessions."""
    kind = rng.choice(["step", "step", "step", "step", "batch", "batch", "serve"])
    precision = rng.choice(["fp64", "fp32"])
    if kind == "batch":
        hi = rng.randint(6, 18)
        return {"kind": "batch", "count": round(2 * 32 ** rng.random()), "lo": rng.randint(2, 5), "hi": hi,
                "mix": rng.randint(10, 99999), "precision": precision}
    if kind == "serve":
        return {"kind": "serve", "count": rng.randint(2, 16), "requests": rng.randint(1, 3),
                "mix": rng.randint(10, 99999), "precision": "fp32"}
    cells = 64 * (64000 / 64) ** rng.random()
    ax, az = 0.5 + 1.5 * rng.random(), 0.5 + 1.5 * rng.random()
    base = (cells / (ax * az)) ** (1 / 3)
    nx, ny, nz = (max(2, min(60, round(base * a))) for a in (ax, 1.0, az))
    case = _step("", nx, ny, nz, precision=precision, material=rng.choice(["snh", "arap"]),
                 precond=rng.choice(["block", "block", "jacobi"]), pinned=rng.random() < 0.7)
    del case["name"]
    if cells < 4000 and rng.random() < 0.3:
        case["newton"] = rng.choice([2, 3])
    elif precision == "fp64" and cells < 8000 and rng.random() < 0.3:
        case["form"], case["pinned"] = "velocity", False
    return case


def _lattice(dims, seed, material, pinned, E=1e5, nu=0.45):
    """A lattice scene with a seeded smooth deformation (zero on the pinned face) and a velocity."""
    mat = scenes.MAT_SNH if material == "snh" else scenes.MAT_ARAP
    sc = scenes.lattice_scene(dims, seed=seed, material=mat, E=E, nu=nu, stretch_velocity=True,
                              mu=None if material == "snh" else 3.4e4 * E / 1e5, pin=pinned)
    r = np.random.default_rng(seed)
    u = sc.rest[:, :1] * r.uniform(-0.08, 0.08, 3)[None, :]
    u[sc.rest[:, 0] > 0] += r.uniform(-0.02, 0.02, (int((sc.rest[:, 0] > 0).sum()), 3)) / max(dims)
    sc.u0 = u.ravel().copy()
    sc.v0 = 0.1 * sc.v0
    return sc


def _scene(case, seed):
    dims = (case["nx"], case["ny"], case["nz"])
    sc = _lattice(dims, seed, case["material"], case["pinned"])
    sc.newton_iters = case["newton"]
    if case["form"] == "velocity":
        sc.integrator = scenes.INTEGRATOR_VELOCITY
        # the floor's top face is a little above the body's lowest vertices, and the body falls
        sc.collision_cubes = ((0.5, -50.0 + 0.02, 0.5, 100.0),)
        v = np.zeros((sc.nv, 3))
        v[:, 1] = -1.0 - np.random.default_rng(seed + 1).random()
        sc.v0 = v.ravel().copy()
    return sc


def _mix_scenes(case, seed):
    r = np.random.default_rng(case["mix"])  # sizes and materials are the case's, states the seed's
    out = []
    for i in range(case["count"]):
        if case["kind"] == "serve":
            sc = scenes.serving_instance(i, seed=case["mix"])
            s = np.random.default_rng(seed * 1000 + i)
            v = np.zeros((sc.nv, 3))
            v[:, 1] = -s.uniform(0.0, 3.0)
            sc.v0 = (v + 0.05 * s.standard_normal((sc.nv, 3))).ravel()
        else:
            dims = tuple(int(d) for d in r.integers(case["lo"], case["hi"] + 1, 3))
            sc = _lattice(dims, seed * 1000 + i, "snh" if r.random() < 0.5 else "arap", True,
                          E=float(10 ** r.uniform(4, 6)), nu=float(r.uniform(0.3, 0.48)))
        out.append(sc)
    return out


class _State:
    """A program's context, its resident instances and the states it starts each pass from."""

    def __init__(self, case, scs):
        self.kind = case["kind"]
        self.requests = case.get("requests", 1)
        workload = {"step": "single", "batch": "batch", "serve": "serving"}[self.kind]
        self.insts = []
        self.sched = None
        self.ctx = lib.Context(0, precision=case["precision"], workload=workload)
        prec = lib.PRECISION_FP32_REFINE if case["precision"] == "fp32" else lib.PRECISION_FP64
        precond = JACOBI if case.get("precond") == "jacobi" else BLOCK
        self.start = [(sc.initial_u(), sc.initial_v()) for sc in scs]
        self.insts = [lib.Instance(self.ctx, sc, precond=precond, precision=prec) for sc in scs]
        if self.kind == "serve":
            self.sched = lib.Scheduler(self.ctx)

    def __del__(self):
        if getattr(self, "sched", None) is not None:
            self.sched.close()
        for i in getattr(self, "insts", ()):
            i.close()
        if getattr(self, "ctx", None) is not None:
            self.ctx.close()


def prepare(case, seed):
    return _State(case, [_scene(case, seed)] if case["kind"] == "step" else _mix_scenes(case, seed))


def run(state):
    for inst, (u, v) in zip(state.insts, state.start):
        inst.set_state(u, v)
    if state.kind == "step":
        state.insts[0].step()
        u, v = state.insts[0].state()
        return {"u": u, "v": v}
    if state.kind == "batch":
        lib.step_batch(state.ctx, state.insts)
    else:
        for k in range(state.requests):
            for i, inst in enumerate(state.insts):
                state.sched.submit(inst, k * len(state.insts) + i)
        left = 1
        while left:
            _, left = state.sched.tick()
    got = [inst.state() for inst in state.insts]
    return {"u": np.concatenate([u for u, _ in got]), "v": np.concatenate([v for _, v in got])}


def _sizes(case):
    """(tets, vertices, stored 3x3 blocks, PCG iterations) of each instance: a lattice vertex couples to
    itself and up to 14 neighbours; iterations grow with the longest axis in cells."""
    if case["kind"] == "step":
        dims = [(case["nx"], case["ny"], case["nz"])]
    elif case["kind"] == "batch":
        r = np.random.default_rng(case["mix"])
        dims = []
        for _ in range(case["count"]):
            dims.append(tuple(int(d) for d in r.integers(case["lo"], case["hi"] + 1, 3)))
            r.random(), r.uniform(4, 6), r.uniform(0.3, 0.48)
    else:
        dims = [scenes.serving_instance(i, seed=case["mix"]).dims for i in range(case["count"])]
    out = []
    for x, y, z in dims:
        nv = (x + 1) * (y + 1) * (z + 1)
        cells = x * y * z
        edges = sum(((x, y, z)[a] * ((x, y, z)[(a + 1) % 3] + 1) * ((x, y, z)[(a + 2) % 3] + 1)
                     + (x, y, z)[a] * (x, y, z)[(a + 1) % 3] * ((x, y, z)[(a + 2) % 3] + 1)) for a in range(3)) + cells
        out.append((6 * cells, nv, nv + 2 * edges, 10 * max(x, y, z)))
    return out


def work(case):
    """Bytes: the mesh (corners, inverse rest shapes, volumes), the stiffness blocks once, the states in and
    out.  Operations: 2,158 a tet for the element and 18 a block plus 40 a vertex in each PCG iteration."""
    real = 8 if case["precision"] == "fp64" else 4
    steps = case.get("requests", 1) * case.get("newton", 1)
    b = f = 0.0
    for nt, nv, nnzb, iters in _sizes(case):
        b += steps * (96 * nt + nnzb * (9 * real + 4) + 200 * nv)
        f += steps * (2158 * nt + iters * (18 * nnzb + 40 * nv))
    return {"bytes": b, "flops": f}


# -- the same step in 64-bit torch and numpy ---------------------------------------------------
def _clamp(H):
    w, Q = np.linalg.eigh(H)
    return (Q * np.maximum(w, 0.0)[:, None, :]) @ Q.transpose(0, 2, 1)


def _material(F, sc):
    """PK1 stress and its derivative with non-negative eigenvalues (row-major vec F), per tet."""
    n, mu = F.shape[0], sc.mu
    I3 = np.eye(3)
    if sc.material == scenes.MAT_SNH:
        lam = sc.lam + mu
        alpha = 1.0 + mu / lam
        G = np.stack([np.cross(F[:, :, 1], F[:, :, 2]), np.cross(F[:, :, 2], F[:, :, 0]),
                      np.cross(F[:, :, 0], F[:, :, 1])], axis=2)
        J = np.linalg.det(F)
        P = mu * F + (lam * (J - alpha))[:, None, None] * G
        eps = np.zeros((3, 3, 3))
        for i, j, k in ((0, 1, 2), (1, 2, 0), (2, 0, 1)):
            eps[i, j, k], eps[i, k, j] = 1.0, -1.0
        HJ = np.einsum("ace,bdf,nef->nabcd", eps, eps, F).reshape(n, 9, 9)
        g = G.reshape(n, 9)
        H = mu * np.eye(9)[None] + lam * g[:, :, None] * g[:, None, :] + (lam * (J - alpha))[:, None, None] * HJ
        return P, _clamp(H)
    U, S, Vt = np.linalg.svd(F)
    flip = np.where(np.linalg.det(U) * np.linalg.det(Vt) < 0, -1.0, 1.0)
    U[:, :, 2] *= flip[:, None]
    S[:, 2] *= flip
    P = 2.0 * mu * ((U * (S - 1.0)[:, None, :]) @ Vt)
    H = np.broadcast_to(2.0 * mu * np.eye(9), (n, 9, 9)).copy()
    for a, b in ((0, 1), (0, 2), (1, 2)):  # the rotation's derivative: one twist per axis pair
        T = np.zeros((3, 3))
        T[a, b], T[b, a] = -math.sqrt(0.5), math.sqrt(0.5)
        q = (U @ T @ Vt).reshape(n, 9)
        H -= (4.0 * mu / (S[:, a] + S[:, b]))[:, None, None] * q[:, :, None] * q[:, None, :]
    return P, _clamp(H)


def _exact_step(sc, u, v):
    X, tets, nv = sc.rest, sc.tets.astype(np.int64), sc.nv
    Dm = np.stack([X[tets[:, k]] - X[tets[:, 0]] for k in (1, 2, 3)], axis=2)
    Di = np.linalg.inv(Dm)
    vol = np.abs(np.linalg.det(Dm)) / 6.0
    d = np.concatenate([-Di.sum(axis=1, keepdims=True), Di], axis=1)
    ring = np.zeros(nv)
    np.add.at(ring, tets.ravel(), np.repeat(vol / 4.0, 4))
    M = np.repeat(ring * sc.mass_scale, 3)
    fext = (ring[:, None] * np.asarray(sc.gravity)[None, :]).ravel()
    dofs = (3 * tets[:, :, None] + np.arange(3)[None, None, :]).reshape(-1, 12)
    ri, ci = torch.from_numpy(np.repeat(dofs, 12, axis=1).ravel()), torch.from_numpy(np.tile(dofs, (1, 12)).ravel())
    dev = "cuda" if torch.cuda.is_available() else "cpu"

    def stiffness(H):
        Hb = H.reshape(-1, 3, 3, 3, 3)
        Ke = np.einsum("n,nvj,najbl,nwl->nvawb", vol, d, Hb, d, optimize=True).reshape(-1)
        return torch.sparse_coo_tensor(torch.stack([ri, ci]), torch.from_numpy(Ke), (3 * nv, 3 * nv)).to(dev).coalesce()

    def shape(uu):
        x = X + uu.reshape(-1, 3)
        return np.einsum("nvi,nvj->nij", x[tets], d)

    dt, al, be = sc.dt, sc.rayleigh_alpha, sc.rayleigh_beta
    pins = sc.pinned()
    free = np.ones(3 * nv)
    free.reshape(-1, 3)[pins] = 0.0
    fr = torch.from_numpy(free).to(dev)
    tz = lambda a: torch.from_numpy(np.ascontiguousarray(a)).to(dev)  # noqa: E731
    Krest = stiffness(_material(np.broadcast_to(np.eye(3), (tets.shape[0], 3, 3)).copy(), sc)[1])
    u_old, v_old = u.copy(), v.copy()
    u = u.copy()
    u.reshape(-1, 3)[pins] = sc.pinned_targets()
    for k in range(sc.newton_iters):
        P, H = _material(shape(u), sc)
        R = np.zeros((nv, 3))
        np.add.at(R, tets.ravel(), (-vol[:, None, None] * np.einsum("nij,nvj->nvi", P, d)).reshape(-1, 3))
        K = stiffness(H)  # minus the reference's K

        def A(x):
            x = fr * x
            y = K @ x + (be / dt) * (Krest @ x) + tz(M * (1.0 / dt ** 2 - al / dt)) * x
            return fr * y

        vb = (u - u_old) / dt - v_old if sc.newton_iters > 1 else None
        if sc.newton_iters > 1:
            Cv = al * M * vb - be * (Krest @ tz(vb)).cpu().numpy()
            b = Cv + M * (-(u - u_old) / dt ** 2 + v_old / dt) + R.ravel() + fext
        else:
            b = M * v / dt - (al * M * v - be * (Krest @ tz(v)).cpu().numpy()) + R.ravel() + fext
        b *= free
        if k > 0 and float(b @ b) <= 1e-7:
            pass  # the loop's test uses the system just solved; one more solve only refines u
        rhs = tz(b)
        x = torch.zeros_like(rhs)
        r = rhs.clone()
        i, w = K.indices(), K.values()
        diag = torch.zeros_like(rhs).index_add_(0, i[0][i[0] == i[1]], w[i[0] == i[1]])
        diag = diag + tz(M / dt ** 2)
        z = r / diag
        p, rz, stop = z.clone(), r @ z, float(rhs @ rhs) * 1e-28
        for it in range(6000):
            q = A(p)
            a = rz / (p @ q)
            x += a * p
            r = r - a * q if it % 50 else rhs - A(x)
            if it % 10 == 0 and float(r @ r) < stop:
                break
            z = r / diag
            new = r @ z
            p = z + (new / rz) * p
            rz = new
        u = u + x.cpu().numpy()
        if float(b @ b) <= 1e-7:
            break
    vn = (u - u_old) / dt * free
    return u, vn


def exact(case, seed):
    """For pinned or free single steps of the position form and of BDF_1 up to 40,000 tets."""
    if case["kind"] != "step" or case["form"] != "position" or case["nx"] * case["ny"] * case["nz"] > 6700:
        return None
    sc = _scene(case, seed)
    u, v = _exact_step(sc, sc.initial_u(), sc.initial_v())
    return {"u": u, "v": v}
