"""The work that a program of this library has it do, as cases that can be timed and checked.

A case names one path through the public entry points (`spg_amd.native`) and its sizes. The paths are the library's
solvers: the VBD step (cloth, solid, many objects, further energies, sweeps to a residual tolerance), the XPBD step,
the implicit Euler step, the rigid-body VBD step, and the learned start (its network's training, a substep from it).
A pass of a solver case is what a frame of a simulation does: advance the objects from a device checkpoint (so that
every pass does the same work) and read the new positions and velocities back.

`exact` restates each path in 64-bit torch: energies as functions of the stencil's positions, differentiated by
torch.func, in the solvers' own order (greedy colours by ascending index).
"""
import math

import numpy as np
import torch

from spg_amd import native, scenes

DT = scenes.DT
G = (0.0, -9.81, 0.0)
LEARNED_FIRST = 10  # sweeps of the substep before a learned one
SMOOTHING = 2
LEARNING_RATE = 2e-3


# ------------------------------------------------------------------------------------------------
# Cases
# ------------------------------------------------------------------------------------------------

def listed():
    return [
        # a small cloth stepped interactively: 40 dependent sweeps of 256 vertices, latency and launches
        {"name": "vbd_cloth_32", "path": "vbd", "mesh": "cloth", "n": 32, "iterations": 10, "substeps": 1},
        # the library's headline workload: a large cloth, 20 sweeps
        {"name": "vbd_cloth_512", "path": "vbd", "mesh": "cloth", "n": 512, "iterations": 20, "substeps": 1},
        # a large solid of Stable Neo-Hookean tetrahedra: 8 colours of uneven size
        {"name": "vbd_cube_64", "path": "vbd", "mesh": "cube", "n": 64, "iterations": 20, "substeps": 1},
        # many garments or training scenes advanced together, sides 16 to 128, each read back
        {"name": "vbd_batch_24", "path": "vbd", "mesh": "batch", "n": 24, "iterations": 15, "substeps": 1},
        # the further energies (Baraff-Witkin membrane and bending, continuum springs) on an odd-sided cloth
        {"name": "vbd_further_251", "path": "vbd", "mesh": "further", "n": 251, "iterations": 20, "substeps": 1},
        # sweeps until the FP64 force residual has fallen far enough, checked every fourth sweep
        {"name": "vbd_tolerance_256", "path": "tolerance", "mesh": "cloth", "n": 256, "iterations": 60, "rel_tol": 1e-4},
        # XPBD with many substeps on the large cloth: 22 stencil groups per substep
        {"name": "xpbd_cloth_512", "path": "xpbd", "mesh": "cloth", "n": 512, "substeps": 20},
        # XPBD on a small solid, odd-sided, as in a game
        {"name": "xpbd_cube_17", "path": "xpbd", "mesh": "cube", "n": 17, "substeps": 10},
        # implicit Euler with conjugate gradients (Baraff-Witkin) on a cloth
        {"name": "implicit_cloth_200", "path": "implicit", "mesh": "cloth", "n": 200},
        # a lattice of jointed rigid boxes, FP64 6x6 blocks
        {"name": "rigid_lattice_256", "path": "rigid", "mesh": "lattice", "n": 256, "iterations": 10},
        # an epoch of the learned start's training: minibatches forward, backward, Adam
        {"name": "network_training_32768", "path": "training", "n": 32768, "batch": 4096, "epochs": 1},
        # a substep that starts from the network's prediction: features, inference, smoothing, a few sweeps
        {"name": "learned_cloth_400", "path": "learned", "mesh": "cloth", "n": 400, "iterations": 4},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    path = rng.choice(["vbd", "vbd", "vbd", "tolerance", "xpbd", "xpbd", "implicit", "rigid", "training", "learned"])
    if path == "vbd":
        mesh = rng.choice(["cloth", "cloth", "cube", "batch", "further"])
        n = {"cloth": lambda: _log(rng, 17, 420), "cube": lambda: _log(rng, 5, 48), "batch": lambda: rng.randint(2, 24),
             "further": lambda: _log(rng, 20, 251)}[mesh]()
        return {"path": path, "mesh": mesh, "n": n, "iterations": rng.randint(4, 20), "substeps": rng.randint(1, 2)}
    if path == "tolerance":
        return {"path": path, "mesh": "cloth", "n": _log(rng, 40, 256), "iterations": rng.randint(8, 60), "rel_tol": 1e-4}
    if path == "xpbd":
        mesh = rng.choice(["cloth", "cube"])
        n = _log(rng, 17, 400) if mesh == "cloth" else _log(rng, 4, 32)
        return {"path": path, "mesh": mesh, "n": n, "substeps": rng.randint(2, 20)}
    if path == "implicit":
        return {"path": path, "mesh": "cloth", "n": _log(rng, 24, 200)}
    if path == "rigid":
        return {"path": path, "mesh": "lattice", "n": _log(rng, 4, 256), "iterations": rng.randint(4, 10)}
    if path == "training":
        return {"path": path, "n": _log(rng, 500, 40000), "batch": 64 * _log(rng, 4, 64), "epochs": rng.randint(1, 2)}
    return {"path": path, "mesh": "cloth", "n": _log(rng, 17, 400), "iterations": rng.randint(1, 8)}


# ------------------------------------------------------------------------------------------------
# Inputs
# ------------------------------------------------------------------------------------------------

def _cloth(n, seed, young, bending=1e-4, **kw):
    """A 1 m cloth hung by its top row, its vertices displaced by up to 0.3% of the edge length."""
    return scenes.cloth(n, young=young, poisson=0.3, thickness=1e-3, bending=bending, mass=1e-3 * (32.0 / n) ** 2,
                        pin="top_row", noise=1e-4 * 32.0 / n, seed=seed, **kw)


def _sides(count):
    """Sides of a batch's cloths, 16 to 128, in a fixed mixed order: the same work for every seed."""
    return np.random.default_rng(7).permutation(np.linspace(16, 128, count).round().astype(int)).tolist()


def _scenes(case, seed):
    """The scenes of a particle case, positions as a mesh file gives them: 32-bit."""
    n, mesh = case["n"], case["mesh"]
    if mesh == "cloth":
        made = [_cloth(n, seed, 1e5 if case["path"] == "tolerance" else 1e4)]
    elif mesh == "further":
        # slightly stretched, as a hung cloth is, so that the membrane carries tension
        made = [_cloth(n, seed, 1e4, membrane="membrane_bw", bending_kind="bending_bw", edge_springs="spring_continuum",
                       edge_k=1.0, stretch=1.02)]
    elif mesh == "cube":
        made = [scenes.cube(n)]
        rng = np.random.default_rng(seed)
        made[0].x = made[0].x + (rng.random(made[0].x.shape) - 0.5) * (0.02 / n)
    else:
        rng = np.random.default_rng(seed)
        made = [_cloth(s, seed * 1000 + k, 10.0 ** rng.uniform(3, 4), 10.0 ** rng.uniform(-5, -3))
                for k, s in enumerate(_sides(n))]
    for s in made:
        s.x = s.x.astype(np.float32).astype(np.float64)
    return made


def _lattice(case, seed):
    return scenes.rb_lattice(case["n"], seed=seed)


def _network_data(case, seed):
    """Standardised feature rows, and targets that depend on them, of the size that the offsets have (units of h^2 |g|)."""
    rng = np.random.default_rng(seed)
    f = rng.standard_normal((case["n"], native.MLP_FEATURES)).astype(np.float32)
    a = rng.standard_normal((native.MLP_FEATURES, native.MLP_OUTPUTS)) / math.sqrt(native.MLP_FEATURES)
    t = 0.3 * np.tanh(f @ a) + 0.02 * rng.standard_normal((case["n"], native.MLP_OUTPUTS))
    return f, t.astype(np.float32)


def _start_weights(seed):
    """Weights whose predictions are a few percent of h^2 |g|, as a trained network's are on a cloth that moves smoothly."""
    w = native.Mlp(device=0, seed=seed).params()
    w[-(native.MLP_SHAPES[-1][0] * (native.MLP_SHAPES[-1][1] + 1)):] *= 0.02
    return w


def prepare(case, seed):
    path = case["path"]
    if path == "training":
        f, t = _network_data(case, seed)
        net = native.Mlp(device=0, seed=seed)
        return {"case": case, "net": net, "weights": net.params(), "f": f, "t": t}
    if path == "rigid":
        s = _lattice(case, seed)
        return {"case": case, "ctx": native.RigidContext([s])}
    made = _scenes(case, seed)
    if path == "xpbd":
        ctx = native.XpbdContext([s.xpbd_object() for s in made], parallel_gauss_seidel=True)
        ctx.save_state()
    elif path == "implicit":
        ctx = native.ImplicitContext([s.vbd_object() for s in made], "baraff_witkin")
    else:
        ctx = native.VbdContext([s.vbd_object() for s in made])
        ctx.autotune(trials=4)
        ctx.set_launch(use_graph=1 if path == "vbd" else 0)
        if path == "learned":
            ctx.step(DT, 1, LEARNED_FIRST, G)  # the substep whose offsets the features hold
        ctx.save_state()
    state = {"case": case, "ctx": ctx, "objects": len(made), "start": made[0].x, "still": np.zeros_like(made[0].x)}
    if path == "learned":
        state["net"] = native.Mlp(device=0, seed=seed)
        state["net"].set_params(_start_weights(seed))
    return state


def run(state):
    case = state["case"]
    path = case["path"]
    if path == "training":
        net = state["net"]
        net.set_params(state["weights"])
        loss = net.train(state["f"], state["t"], epochs=case["epochs"], batch=case["batch"], lr=LEARNING_RATE, seed=1,
                         standardize=False)
        return {"loss": loss, "weights": net.params()}
    ctx = state["ctx"]
    if path == "rigid":  # each pass is the next frame
        ctx.step(DT, 1, case["iterations"], G)
        return ctx.state()
    if path == "implicit":
        ctx.set_state(0, state["start"], state["still"])
        ctx.step(DT, 1, G)
        return ctx.state()
    ctx.restore_state()
    if path == "xpbd":
        ctx.step(DT, case["substeps"], G)
        return ctx.state()
    if path == "tolerance":
        ctx.begin_substep(DT, G)
        _, rho = ctx.iterate_to_tolerance(case["rel_tol"], case["iterations"], 4)
        ctx.end_substep()
        return {"rho": rho, "state": ctx.state()}
    if path == "learned":
        ctx.begin_substep(DT, G)
        ctx.warm_start(state["net"], gate=False, smoothing=SMOOTHING)
        ctx.iterate(case["iterations"])
        ctx.end_substep()
        return ctx.state()
    ctx.step(DT, case["substeps"], case["iterations"], G)
    return [ctx.state(o) for o in range(state["objects"])]


# ------------------------------------------------------------------------------------------------
# Work and tolerances
# ------------------------------------------------------------------------------------------------

def _counts(mesh, n):
    """Particles and elements by kind of one object."""
    if mesh == "cube":
        return {"particles": (n + 1) ** 3, "tets": 6 * n ** 3}
    c = {"particles": n * n, "triangles": 2 * (n - 1) ** 2, "hinges": 3 * (n - 1) ** 2 - 2 * (n - 1)}
    if mesh == "further":
        c["springs"] = 3 * (n - 1) ** 2 + 2 * (n - 1)
    return c


# bytes of an element's record in 32 bits (vertex indices and coefficients), read once a sweep or projection
_VBD_BYTES = {"triangles": 40, "hinges": 24, "tets": 64, "springs": 16}
_XPBD_BYTES = {"triangles": 52, "hinges": 24, "tets": 68, "springs": 16}
# operations of one element: gradients and diagonal blocks of all its vertices; one projection
_VBD_FLOPS = {"triangles": 450, "hinges": 900, "tets": 800, "springs": 100}
_XPBD_FLOPS = {"triangles": 200, "hinges": 220, "tets": 300, "springs": 40}


def work(case):
    path, n = case["path"], case["n"]
    weights = sum(o * i for o, i in native.MLP_SHAPES)
    if path == "training":
        steps = case["epochs"] * -(-n // case["batch"])
        return {"bytes": case["epochs"] * n * 4.0 * 27 + steps * 24.0 * native.MLP_NUM_PARAMS,
                "flops": case["epochs"] * 6.0 * n * weights}
    if path == "rigid":
        pairs = 2 * n * (n - 1)
        # a body's pose and step state (96 + 240 bytes) and a joint's points and stiffness (64 + 8), a sweep; the state out
        return {"bytes": case["iterations"] * (336.0 * n * n + 72.0 * pairs) + 96.0 * n * n,
                "flops": case["iterations"] * (600.0 * n * n + 2 * 700.0 * pairs)}
    sides = [n] if case["mesh"] != "batch" else _sides(n)
    total = {"bytes": 0.0, "flops": 0.0}
    for s in sides:
        c = _counts(case["mesh"], s)
        p = c.pop("particles")
        if path == "implicit":
            # assembly (every element's Hessian once into 3x3 blocks) and conjugate gradients at their cap of 300
            blocks = p + c["triangles"] * 3 // 2 + c["hinges"]
            total["bytes"] += 300 * (76.0 * blocks + 6 * 24.0 * p) + 72.0 * blocks + 96.0 * p
            total["flops"] += 300 * (2 * 18.0 * blocks + 30.0 * p)
            continue
        if path == "xpbd":
            per = sum(_XPBD_BYTES[k] * v for k, v in c.items()) + 48.0 * p
            flops = sum(_XPBD_FLOPS[k] * v for k, v in c.items())
            passes = case["substeps"]
        else:
            if path == "learned":  # the feature rows' inputs and the network
                total["bytes"] += 100.0 * p
                total["flops"] += 2.0 * weights * p
            per = sum(_VBD_BYTES[k] * v for k, v in c.items()) + 40.0 * p
            flops = sum(_VBD_FLOPS[k] * v for k, v in c.items()) + 80.0 * p
            # a solve to 1e-4 takes about 16 sweeps
            passes = min(case["iterations"], 16 if path == "tolerance" else 1000) * case.get("substeps", 1)
        total["bytes"] += passes * per + 96.0 * p  # the state out in 64 bits, x and v in
        total["flops"] += passes * flops
    return total


def tolerance(case):
    """About four times the largest error against `exact` seen over these ranges. Velocities are differences of 32-bit
    positions over h, so more substeps lose more of them; the network's operands are bfloat16; the residual ratio is a
    small difference of large forces; the implicit and rigid solvers are 64-bit throughout."""
    return {"vbd": {"rel": 2e-4}, "tolerance": {"rel": 3e-2}, "xpbd": {"rel": 8e-3}, "implicit": {"rel": 1e-9},
            "rigid": {"rel": 1e-9}, "training": {"rel": 6e-3}, "learned": {"rel": 1e-4}}[case["path"]]


# ------------------------------------------------------------------------------------------------
# The same in 64 bits
# ------------------------------------------------------------------------------------------------

F8 = torch.float64


def _device():
    return "cuda" if torch.cuda.is_available() else "cpu"


def _t(a, dtype=F8):
    return torch.as_tensor(np.ascontiguousarray(a), dtype=dtype, device=_device())


def _F(xs, dm):
    """Deformation gradient [x1 - x0, ...] Dm^-1; dm: the flattened inverse."""
    k = xs.shape[0] - 1
    return (xs[1:] - xs[0]).T @ dm.reshape(k, k)


def _hinge_xy(xs):
    e0, e3, e4 = xs[1] - xs[0], xs[2] - xs[1], xs[3] - xs[1]
    n1, n2 = torch.linalg.cross(e0, e3), -torch.linalg.cross(e0, e4)
    return torch.dot(torch.linalg.cross(n1, n2), e0), torch.dot(n1, n2), e0


def _det3(f):
    return torch.dot(f[:, 0], torch.linalg.cross(f[:, 1], f[:, 2]))


def _c_spring(xs, p):
    return ((xs[0] - xs[1]).norm() / p[0] - 1.0)[None]


def _c_stvk(xs, p):
    f = _F(xs, p[:4])
    return torch.stack([0.5 * (f[:, 0] @ f[:, 0] - 1), 0.5 * (f[:, 1] @ f[:, 1] - 1), f[:, 0] @ f[:, 1]])


def _c_membrane_bw(xs, p):
    f = _F(xs, p[:4])
    return torch.stack([f[:, 0].norm() - 1, f[:, 1].norm() - 1, f[:, 0] @ f[:, 1]])


def _c_bending(xs, p):
    y, x, e0 = _hinge_xy(xs)
    return torch.atan2(y / e0.norm(), x)[None] - p[:1]


def _c_bending_bw(xs, p):  # p[1]: 1 / |e0| at the positions of the evaluation, a constant to the derivative
    y, x, _ = _hinge_xy(xs)
    return torch.atan2(y * p[1], x)[None] - p[:1]


def _c_snh(xs, p):
    f = _F(xs, p[:9])
    return torch.stack([_det3(f) - p[9], f.norm()])


_CONSTRAINT = {"spring_continuum": _c_spring, "stvk": _c_stvk, "membrane_bw": _c_membrane_bw, "bending": _c_bending,
               "bending_bw": _c_bending_bw, "snh": _c_snh}


def _e_anchor(xs, p, k):
    d = xs[0] - p
    return 0.5 * k[0, 0] * torch.dot(d, d)


def _e_snh(xs, p, k):
    f = _F(xs, p[:9])
    return 0.5 * k[0, 0] * (_det3(f) - p[9]) ** 2 + 0.5 * k[1, 1] * ((f * f).sum() - 3.0)


def _energy(kind):
    if kind in ("anchor", "snh"):
        return {"anchor": _e_anchor, "snh": _e_snh}[kind]
    c = _CONSTRAINT[kind]

    def e(xs, p, k):
        v = c(xs, p)
        return 0.5 * torch.dot(v, k @ v)
    return e


class _Elements:
    """The elements of one energy: stencils, parameters, stiffness matrices."""

    def __init__(self, kind, stencils, raw, x0):
        self.kind, self.ids = kind, np.asarray(stencils, dtype=np.int64)
        self.st = _t(self.ids, torch.int64)
        raw, m = _t(raw), len(self.ids)
        r = _t(x0)[self.st]
        if kind == "anchor":
            self.p, self.k = raw[:, :3], raw[:, 3].reshape(m, 1, 1)
        elif kind == "spring_continuum":
            self.p, self.k = raw[:, :1], (raw[:, 0] * raw[:, 1]).reshape(m, 1, 1)
        elif kind in ("stvk", "membrane_bw"):
            dm = (r[:, 1:, :2] - r[:, :1, :2]).transpose(1, 2).contiguous()
            area = 0.5 * (dm[:, 0, 0] * dm[:, 1, 1] - dm[:, 0, 1] * dm[:, 1, 0])
            self.p = torch.linalg.inv(dm).reshape(m, 4)
            if kind == "stvk":
                y, nu = raw[:, 0], raw[:, 1]
                c, z = y / (1 - nu * nu), torch.zeros_like(y)
                k = torch.stack([c, c * nu, z, c * nu, c, z, z, z, c * (1 - nu) / 2], 1).reshape(m, 3, 3)
            else:
                k = torch.diag_embed(raw)
            self.k = k * area[:, None, None]
        elif kind in ("bending", "bending_bw"):
            e0, e3, e4 = r[:, 1] - r[:, 0], r[:, 2] - r[:, 1], r[:, 3] - r[:, 1]
            a1, a2 = torch.linalg.cross(e0, e3), torch.linalg.cross(e0, e4)
            y = (torch.linalg.cross(a1, -a2) * e0).sum(1) / e0.norm(dim=1)
            self.p = torch.stack([torch.atan2(y, -(a1 * a2).sum(1)), 1.0 / e0.norm(dim=1)], 1)
            f = 2 * 3 * (e0 * e0).sum(1) / (0.5 * (a1.norm(dim=1) + a2.norm(dim=1))) if kind == "bending" else 1.0
            self.k = (raw[:, 1] * f).reshape(m, 1, 1)
        else:
            dm = (r[:, 1:] - r[:, :1]).transpose(1, 2).contiguous()
            mu = raw[:, 0] / (2 * (1 + raw[:, 1]))
            lam = mu / (1 - 2 * raw[:, 1])
            vol = torch.linalg.det(dm) / 6
            self.p = torch.cat([torch.linalg.inv(dm).reshape(m, 9), (1 + mu / lam)[:, None]], 1)
            self.k = torch.diag_embed(torch.stack([lam, mu], 1)) * vol[:, None, None]

    def params(self, x, rows=None):
        p = self.p if rows is None else self.p[rows]
        if self.kind == "bending_bw":
            st = self.st if rows is None else self.st[rows]
            p = torch.stack([p[:, 0], 1.0 / (x[st[:, 1]] - x[st[:, 0]]).norm(dim=1)], 1)
        return p


def _elements(scene):
    return [_Elements(kind, st, raw, scene.x0) for kind, st, raw in scene.energies]


def _vertex_colors(els, n):
    pairs = []
    for e in els:
        s = e.ids.shape[1]
        pairs += [e.ids[:, [a, b]] for a in range(s) for b in range(a)]
    if not pairs:
        return np.zeros(n, np.int64)
    pairs = np.sort(np.concatenate(pairs), axis=1)
    pairs = np.unique(pairs[:, 1] * np.int64(n) + pairs[:, 0])
    hi, lo = (pairs // n), (pairs % n).tolist()
    ptr = np.searchsorted(hi, np.arange(n + 1)).tolist()
    col = [0] * n
    for v in range(n):
        used = 0
        for k in range(ptr[v], ptr[v + 1]):
            used |= 1 << col[lo[k]]
        c = ~used & (used + 1)
        col[v] = c.bit_length() - 1
    return np.array(col)


def _stencil_colors(ids):
    n = int(ids.max()) + 1 if len(ids) else 0
    used, out = [0] * n, []
    for st in ids.tolist():
        m = 0
        for v in st:
            m |= used[v]
        b = ~m & (m + 1)
        for v in st:
            used[v] |= b
        out.append(b.bit_length() - 1)
    return np.array(out, dtype=np.int64)


def _block_fn(kind):
    """Gradient and diagonal block of the energy in one stencil vertex, over a batch of elements."""
    e = _energy(kind)

    def at(d, xs, hot, p, k):
        return e(xs + hot[:, None] * d, p, k)
    g = torch.func.grad(at)

    def both(d, xs, hot, p, k):
        return g(d, xs, hot, p, k), torch.func.jacfwd(g)(d, xs, hot, p, k)
    return torch.func.vmap(both, in_dims=(None, 0, 0, 0, 0))


class _Vbd:
    def __init__(self, scene):
        self.els, self.n = _elements(scene), scene.n
        self.m = _t(scene.m)
        col = _vertex_colors(self.els, self.n)
        self.groups = []
        for c in range(int(col.max()) + 1):
            parts = []
            for e in self.els:
                rows, slots = np.nonzero(col[e.ids] == c)
                if len(rows):
                    rows, slots = _t(rows, torch.int64), _t(slots, torch.int64)
                    parts.append((e, rows, torch.nn.functional.one_hot(slots, e.st.shape[1]).to(F8), e.st[rows, slots]))
            self.groups.append((_t(np.flatnonzero(col == c), torch.int64), parts))
        self.fns = {e.kind: _block_fn(e.kind) for e in self.els}

    def sweep(self, x, xt, h):
        zero = torch.zeros(3, dtype=F8, device=x.device)
        for verts, parts in self.groups:
            w = self.m / (h * h)
            f = -w[:, None] * (x - xt)
            H = w[:, None, None] * torch.eye(3, dtype=F8, device=x.device)
            for e, rows, hot, owner in parts:
                g, b = self.fns[e.kind](zero, x[e.st[rows]], hot, e.params(x, rows), e.k[rows])
                f.index_add_(0, owner, -g)
                H = H.index_add(0, owner, b)
            f, H = f[verts], H[verts]
            ok = torch.linalg.det(H) > 1e-10
            x[verts[ok]] += torch.linalg.solve(H[ok], f[ok])

    def residual(self, x, xt, h):
        y = x.clone().requires_grad_()
        for e in self.els:
            torch.func.vmap(_energy(e.kind))(y[e.st], e.params(x), e.k).sum().backward()
        return float((-y.grad - (self.m / (h * h))[:, None] * (x - xt)).norm())


def _vbd_exact(scene, case):
    s, out = _Vbd(scene), {}
    h = DT / case.get("substeps", 1)
    x, v, g = _t(scene.x), torch.zeros(scene.n, 3, dtype=F8, device=_device()), _t(np.array(G))
    for _ in range(case.get("substeps", 1)):
        old = x.clone()
        v = v + h * g
        x = x + h * v
        xt = x.clone()
        if case["path"] == "tolerance":
            r0, done, rho = s.residual(x, xt, h), 0, 1.0
            while rho > case["rel_tol"] and done < case["iterations"]:
                for _ in range(min(4, case["iterations"] - done)):
                    s.sweep(x, xt, h)
                    done += 1
                rho = s.residual(x, xt, h) / r0
            out["rho"] = rho
        else:
            for _ in range(case["iterations"]):
                s.sweep(x, xt, h)
        v = (x - old) / h
    out["state"] = (x.cpu().numpy(), v.cpu().numpy())
    return out


def _xpbd_exact(scene, case):
    els, n = _elements(scene), scene.n
    h = DT / case["substeps"]
    w = _t(np.where(scene.m == 0, 0.0, 1.0 / np.where(scene.m == 0, 1.0, scene.m)))
    plan = []
    for e in els:
        col = _stencil_colors(e.ids)
        for c in range(int(col.max()) + 1):
            rows = _t(np.flatnonzero(col == c), torch.int64)
            plan.append((e, e.st[rows], e.p[rows], torch.linalg.inv(e.k[rows]) / (h * h)))
    jac = {e.kind: torch.func.vmap(torch.func.jacrev(_CONSTRAINT[e.kind])) for e in els if e.kind != "anchor"}
    val = {e.kind: torch.func.vmap(_CONSTRAINT[e.kind]) for e in els if e.kind != "anchor"}
    x, v, g = _t(scene.x), torch.zeros(n, 3, dtype=F8, device=_device()), _t(np.array(G))
    for _ in range(case["substeps"]):
        old = x.clone()
        v = v + h * g
        x = x + h * v
        for e, st, p, a in plan:
            if e.kind == "anchor":
                d = x[st[:, 0]] - p
                c = d.norm(dim=1, keepdim=True)
                nrm = torch.where(c > 0, d / c.clamp_min(1e-300), torch.zeros_like(d))
                ww = w[st]
                x[st[:, 0]] = x[st[:, 0]] - ww * nrm * c / (ww * (c > 0) + a[:, 0] + 1e-10)
                continue
            xs = x[st]
            C = val[e.kind](xs, p)
            J = jac[e.kind](xs, p).reshape(len(st), C.shape[1], -1)
            ww = w[st].repeat_interleave(3, dim=1)
            A = (J * ww[:, None, :]) @ J.transpose(1, 2).contiguous() + a
            A = A + 1e-10 * torch.eye(C.shape[1], dtype=F8, device=x.device)
            dl = -torch.linalg.solve(A, C[:, :, None])
            x[st.reshape(-1)] = (xs + (ww * (J * dl).sum(1)).reshape(xs.shape)).reshape(-1, 3)
        v = (x - old) / h
    return x.cpu().numpy(), v.cpu().numpy()


def _implicit_exact(scene):
    els, n, h = _elements(scene), scene.n, DT
    x, g, m = _t(scene.x), _t(np.array(G)), _t(scene.m)
    f, hess, diag = m[:, None] * g, [], m[:, None].repeat(1, 3)
    for e in els:
        fn = _energy(e.kind)
        p, xs = e.params(x), x[e.st]
        gr = torch.func.vmap(torch.func.grad(fn))(xs, p, e.k)
        H = torch.func.vmap(torch.func.jacfwd(torch.func.grad(fn)))(xs, p, e.k)
        q = 3 * e.st.shape[1]
        H = H.reshape(len(e.st), q, q)
        f = f.index_add(0, e.st.reshape(-1), -gr.reshape(-1, 3))
        diag = diag.index_add(0, e.st.reshape(-1), h * h * torch.diagonal(H, dim1=1, dim2=2).reshape(-1, 3))
        hess.append((e.st, H))

    def product(y):
        out = m[:, None] * y
        for st, H in hess:
            out.index_add_(0, st.reshape(-1), (h * h * (H @ y[st].reshape(len(st), -1, 1))).reshape(-1, 3))
        return out
    b = h * f  # at rest: no velocity term
    sol, r = torch.zeros_like(b), b.clone()
    limit = max(1e-10 * float((b * b).sum()), 2.3e-308)
    inv = torch.where(diag != 0, 1.0 / diag, torch.ones_like(diag))
    p = inv * r
    rz, it = float((r * p).sum()), 0
    while it < 300 and float((r * r).sum()) >= limit:
        q = product(p)
        a = rz / float((p * q).sum())
        sol, r = sol + a * p, r - a * q
        z = inv * r
        old, rz = rz, float((r * z).sum())
        p, it = z + (rz / old) * p, it + 1
    return (x + h * sol).cpu().numpy(), sol.cpu().numpy()


def _cross_matrix(v):
    z = torch.zeros_like(v[..., 0])
    return torch.stack([z, -v[..., 2], v[..., 1], v[..., 2], z, -v[..., 0], -v[..., 1], v[..., 0], z], -1).reshape(*v.shape, 3)


def _rotation(t):
    a = t.norm(dim=-1)[..., None, None]
    k = _cross_matrix(t / t.norm(dim=-1, keepdim=True).clamp_min(1e-300))
    return torch.eye(3, dtype=F8, device=t.device) + torch.sin(a) * k + (1 - torch.cos(a)) * (k @ k)


def _axis_angle(R):
    """Rotations away from a half turn, as the lattice's are."""
    q = torch.sqrt((R.diagonal(dim1=-2, dim2=-1).sum(-1) + 1).clamp_min(1e-300))
    v = 0.5 / q[..., None] * torch.stack([R[..., 2, 1] - R[..., 1, 2], R[..., 0, 2] - R[..., 2, 0], R[..., 1, 0] - R[..., 0, 1]], -1)
    n = v.norm(dim=-1)
    return v * (2 * torch.atan2(n, 0.5 * q) / n.clamp_min(1e-300))[..., None]


def _rb_points(d, com, R, loc):
    r = (R @ loc[..., None])[..., 0]
    return com + d[:, :3] + r + torch.linalg.cross(d[:, 3:], r)


def _rb_anchor(d, com, R, p):
    q = _rb_points(d, com, R, p[None, :3])[0] - p[3:6]
    return 0.5 * p[6] * torch.dot(q, q)


def _rb_spring(d, com, R, p):
    q = _rb_points(d, com, R, p[:6].reshape(2, 3))
    return 0.5 * p[7] * ((q[0] - q[1]).norm() - p[6]) ** 2


def _rb_alignment(d, com, R, p):
    T = (torch.eye(3, dtype=F8, device=d.device) + _cross_matrix(d[:, 3:])) @ R
    c = torch.linalg.cross(T[0].T, T[1].T)
    return 0.5 * p[0] * (c * c).sum() ** 2


def _rigid_exact(scene, case):
    h, nb = DT, scene.nb
    x, R, I0 = _t(scene.x), _rotation(_t(scene.theta)), _t(scene.inertia)
    old_x, old_R, m = x.clone(), R.clone(), _t(scene.m)
    x = x + h * h * _t(np.array(G))  # at rest: no gyroscopic term, no rotation
    xt, eye = x.clone(), torch.eye(3, dtype=F8, device=x.device)

    class E:
        def __init__(self, st):
            self.ids = np.asarray(st, dtype=np.int64)
    col = _vertex_colors([E(st) for _, st, _ in scene.energies], nb)
    fns = {}
    for kind, fn in (("rb_anchor", _rb_anchor), ("rb_spring", _rb_spring), ("rb_alignment", _rb_alignment)):
        def at(d, hot, com, R_, p, fn=fn):
            return fn(hot[:, None] * d, com, R_, p)

        def both(d, hot, com, R_, p, at=at):
            return torch.func.grad(at)(d, hot, com, R_, p), torch.func.jacfwd(torch.func.grad(at))(d, hot, com, R_, p)
        fns[kind] = torch.func.vmap(both, in_dims=(None, 0, 0, 0, 0))
    zero = torch.zeros(6, dtype=F8, device=x.device)
    for _ in range(case["iterations"]):
        for c in range(int(col.max()) + 1):
            I = R @ I0 @ R.transpose(1, 2).contiguous()
            dw = _axis_angle(R @ old_R.transpose(1, 2).contiguous()) / h
            f = torch.cat([-(m / (h * h))[:, None] * (x - xt), -(I @ dw[..., None])[..., 0] / h], 1)
            H = torch.zeros(nb, 6, 6, dtype=F8, device=x.device)
            H[:, :3, :3] = (m / (h * h))[:, None, None] * eye
            H[:, 3:, 3:] = I / (h * h)
            for kind, st, p in scene.energies:
                rows, slots = np.nonzero(col[st] == c)
                if not len(rows):
                    continue
                s = _t(st[rows], torch.int64)
                hot = torch.nn.functional.one_hot(_t(slots, torch.int64), s.shape[1]).to(F8)
                g, b = fns[kind](zero, hot, x[s], R[s], _t(p[rows]))
                owner = s[torch.arange(len(s), device=s.device), _t(slots, torch.int64)]
                f.index_add_(0, owner, -g)
                H.index_add_(0, owner, b)
            v = _t(np.flatnonzero(col == c), torch.int64)
            d = torch.linalg.solve(H[v], f[v])
            x[v] += d[:, :3]
            R[v] = _rotation(d[:, 3:]) @ R[v]
    omega = _axis_angle(R @ old_R.transpose(1, 2).contiguous()) / h
    return tuple(a.cpu().numpy() for a in (x, _axis_angle(R), (x - old_x) / h, omega))


def _network(p, y):
    k = 0
    for i, (o, n) in enumerate(native.MLP_SHAPES):
        y = y @ p[k:k + o * n].reshape(o, n).T + p[k + o * n:k + o * n + o]
        k += o * n + o
        if i < len(native.MLP_SHAPES) - 1:
            y = torch.nn.functional.silu(y)
    return y


def _shuffles(n, epochs):
    """The rows of each epoch: Fisher-Yates from the last row down, draws of splitmix64 with seed 1."""
    u = scenes.SplitMix64(1).uniforms(epochs * (n - 1))
    for e in range(epochs):
        p = list(range(n))
        for q, i in zip(u[e * (n - 1):(e + 1) * (n - 1)].tolist(), range(n - 1, 0, -1)):
            j = int(q * (i + 1))
            p[i], p[j] = p[j], p[i]
        yield p


def _training_exact(case, seed):
    f, t = _network_data(case, seed)
    f, t, n, batch = _t(f), _t(t), case["n"], case["batch"]
    p = _t(native.Mlp(device=0, seed=seed).params())
    m, v, step, losses = torch.zeros_like(p), torch.zeros_like(p), 0, []
    last = case["epochs"] * -(-n // batch) - 1
    for order in _shuffles(n, case["epochs"]):
        order, total = _t(np.array(order), torch.int64), 0.0
        for b in range(0, n, batch):
            rows = order[b:b + batch]
            w = p.clone().requires_grad_()
            loss = ((_network(w, f[rows]) - t[rows]) ** 2).sum()
            (loss / len(rows)).backward()
            total += float(loss)
            lr = LEARNING_RATE * (0.05 + 0.475 * (1 + math.cos(math.pi * step / last if last else 0.0)))
            step += 1
            m = 0.9 * m + 0.1 * w.grad
            v = 0.999 * v + 0.001 * w.grad ** 2
            p = p - lr * (m / (1 - 0.9 ** step)) / ((v / (1 - 0.999 ** step)).sqrt() + 1e-8)
        losses.append(total / n)
    return {"loss": np.array(losses), "weights": p.cpu().numpy()}


def _learned_exact(scene, case, seed):
    s, n, h = _Vbd(scene), scene.n, DT
    g = _t(np.array(G))
    x = _t(scene.x)
    v = (h * g).expand(n, 3)
    xt = x + h * v
    y = xt.clone()
    for _ in range(LEARNED_FIRST):
        s.sweep(y, xt, h)
    c, v, x = y - xt, (y - x) / h, y
    # one ring: the pairs of vertices that share a triangle
    tri = next(e.ids for e in s.els if e.kind == "stvk")
    pairs = np.concatenate([tri[:, [a, b]] for a in range(3) for b in range(3) if a != b])
    pairs = _t(np.unique(pairs, axis=0), torch.int64)
    i, j = pairs[:, 0], pairs[:, 1]
    deg = torch.zeros(n, dtype=F8, device=x.device).index_add(0, i, torch.ones(len(i), dtype=F8, device=x.device))[:, None]

    def mean(a):
        return torch.zeros(n, a.shape[1], dtype=F8, device=x.device).index_add(0, i, a) / deg

    def most(a, how="amax"):
        out = torch.zeros(n, a.shape[1], dtype=F8, device=x.device)
        return out.scatter_reduce(0, i[:, None].expand_as(a), a, how, include_self=False)
    sc, u = h * h * float(g.norm()), h * float(g.norm())
    xt = x + h * (v + h * g)
    x0 = _t(scene.x0)
    strain = ((xt[j] - xt[i]).norm(dim=1) / (x0[j] - x0[i]).norm(dim=1) - 1.0)[:, None]
    held = np.zeros((n, 1))
    stiff = {kind: raw for kind, _, raw in scene.energies}
    held[next(st for kind, st, _ in scene.energies if kind == "anchor")[:, 0]] = 1.0
    one = torch.ones(n, 1, dtype=F8, device=x.device)
    f = torch.cat([c / sc, v / u, mean(c[j]) / sc, most((c[j] - c[i]).abs()) / sc, mean(v[j]) / u,
                   most((v[j] - v[i]).abs()) / u, math.log10(stiff["stvk"][0, 0]) * one,
                   math.log10(stiff["bending"][0, 1]) * one, _t(held), mean(strain), most(strain), most(strain, "amin")], 1)
    y = _network(_t(_start_weights(seed)), f)
    for _ in range(SMOOTHING):
        y = (y + mean(y[j]) * deg) / (1 + deg)
    old, x = x, xt + sc * y
    for _ in range(case["iterations"]):
        s.sweep(x, xt, h)
    return x.cpu().numpy(), ((x - old) / h).cpu().numpy()


def exact(case, seed):
    path = case["path"]
    if path == "training":
        return _training_exact(case, seed)
    if path == "rigid":
        return _rigid_exact(_lattice(case, seed), case)
    made = _scenes(case, seed)
    if path == "xpbd":
        return _xpbd_exact(made[0], case)
    if path == "implicit":
        return _implicit_exact(made[0])
    if path == "tolerance":
        return _vbd_exact(made[0], case)
    if path == "learned":
        return _learned_exact(made[0], case, seed)
    return [_vbd_exact(s, case)["state"] for s in made]
