"""Performance cases of the nbody library: one pass each through the public
entry points (include/utcnb.h, by way of the utc_amd binding).

Every case is a plain dict; ``kind`` says which entry points it goes through:

  field    utcnb_accel_noalloc on device arrays: the field of one set of
           positions, the smallest call there is
  step     utcnb_set_state / utcnb_step / utcnb_get_state on device arrays: a
           program hands a state over, advances it and takes it back
  slice    utcnb_step_slice: one GPU's slice of the bodies against all sources
           (the multi-GPU task's step)
  share    utcnb_share_pairs / utcnb_share_finish: one GPU's share by wave
           blocks, each unordered pair once
  ref      utcnb_integrate_f32/_f64: the reference's arithmetic, at kernel level
  adjoint  utcnb_set_state / utcnb_adjoint: gradients of a trajectory loss
  batch    utcnb_batch_set_state / utcnb_batch_run: many uneven systems, forward
           alone or with the adjoint

The mixed and plain FP32 paths evaluate their pair terms in FP32; a program
that takes their field or gradients keeps them in FP32, as the cases do, and
hands its state over in the type the case names (``io``).

FLOPs are counted as the reference counts them: 20 per ordered pair of a force
sum (benchapps/nbody/seq/bodysystem.h:75-92), and 40 per ordered pair of a
vector-Jacobian product.
"""
import ctypes as C
import math

import numpy as np
import torch

import utc_amd as U

PRECISIONS = {"mixed": U.PREC_MIXED, "fp32": U.PREC_FP32, "fp64": U.PREC_FP64}


def listed():
    return [
        # one field evaluation of a small set of bodies: the call's own latency
        {"name": "field_1500", "kind": "field", "precision": "mixed", "n": 1500, "masses": "equal", "shape": "cube",
         "newton": False, "eps": 0.01},
        # the golden run's length (100 steps) at its size, one body short of
        # a round number of tiles: step latency
        {"name": "step_mixed_1000_x100", "kind": "step", "precision": "mixed", "n": 1000, "steps": 100,
         "masses": "equal", "shape": "cube", "newton": False, "eps": 0.01, "dt": 1e-3, "kick": "physical",
         "damping": 1.0, "io": "f32"},
        # the reference's default size order on the plain FP32 path, its own kick
        {"name": "step_fp32_4096_x10", "kind": "step", "precision": "fp32", "n": 4096, "steps": 10,
         "masses": "equal", "shape": "cube", "newton": False, "eps": 0.01, "dt": 1e-3, "kick": "reference",
         "damping": 0.995, "io": "f32"},
        # a ragged mid-size system with unequal masses
        {"name": "step_mixed_6001_logm", "kind": "step", "precision": "mixed", "n": 6001, "steps": 10,
         "masses": "log", "shape": "cube", "newton": False, "eps": 0.01, "dt": 1e-3, "kick": "physical",
         "damping": 1.0, "io": "f32"},
        # the gradient workload's size, forward, with the handle's default flags
        {"name": "step_mixed_16384_newton", "kind": "step", "precision": "mixed", "n": 16384, "steps": 10,
         "masses": "log", "shape": "cube", "newton": True, "eps": 0.01, "dt": 1e-3, "kick": "physical",
         "damping": 1.0, "io": "f32"},
        # the plain FP32 benchmark system
        {"name": "step_fp32_65536", "kind": "step", "precision": "fp32", "n": 65536, "steps": 2,
         "masses": "equal", "shape": "plummer", "newton": False, "eps": 0.005, "dt": 5e-4, "kick": "physical",
         "damping": 1.0, "io": "f32"},
        # the headline system
        {"name": "step_mixed_262144", "kind": "step", "precision": "mixed", "n": 262144, "steps": 1,
         "masses": "equal", "shape": "plummer", "newton": False, "eps": 0.002, "dt": 2.5e-4, "kick": "physical",
         "damping": 1.0, "io": "f64"},
        # one of eight GPUs' slice of the headline system, one body more than a
        # power of two in all
        {"name": "slice_0of8_262145", "kind": "slice", "precision": "mixed", "n": 262145, "shares": 8, "share": 0,
         "masses": "equal", "shape": "plummer", "newton": False, "eps": 0.002, "dt": 2.5e-4, "kick": "physical",
         "damping": 1.0, "io": "f64"},
        # one of eight GPUs' share by wave blocks
        {"name": "share_3of8_131072", "kind": "share", "precision": "mixed", "n": 131072, "shares": 8, "share": 3,
         "masses": "equal", "shape": "plummer", "newton": False, "eps": 0.002, "dt": 2.5e-4, "kick": "physical",
         "damping": 1.0, "io": "f64"},
        # the drop-in launch of the reference's kernel
        {"name": "ref_f32_16384", "kind": "ref", "io": "f32", "n": 16384, "steps": 2, "masses": "equal",
         "shape": "cube", "eps": 0.01, "dt": 1e-3, "damping": 0.995},
        # the gradient workload
        {"name": "adjoint_16384", "kind": "adjoint", "precision": "mixed", "n": 16384, "steps": 50, "ckpt": 10,
         "masses": "log", "shape": "cube", "newton": False, "eps": 0.01, "dt": 1e-3, "kick": "physical",
         "damping": 1.0},
        # many uneven systems with gradients, one captured run
        {"name": "batch_adjoint_96", "kind": "batch", "systems": 96, "smallest": 256, "largest": 8192, "steps": 20,
         "ckpt": 10, "adjoint": True, "masses": "equal", "shape": "plummer", "eps": 0.01, "dt": 1e-3,
         "damping": 1.0},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["field", "step", "step", "step", "step", "slice", "share", "ref", "adjoint", "batch", "fp64"])
    masses = rng.choice(["equal", "equal", "log"])
    eps = rng.choice([0.002, 0.005, 0.01])
    dt = {0.002: 2.5e-4, 0.005: 5e-4, 0.01: 1e-3}[eps]
    common = {"masses": masses, "newton": rng.random() < 0.25, "eps": eps}
    move = {"dt": dt, "kick": rng.choice(["physical", "physical", "reference"]),
            "damping": rng.choice([1.0, 1.0, 0.995])}
    if kind == "field":
        return {"kind": "field", "precision": rng.choice(["mixed", "fp32"]), "n": _log_int(rng, 64, 32000),
                "shape": rng.choice(["cube", "plummer"]), **common}
    if kind == "step":
        n = _log_int(rng, 256, 262144)
        most = max(1, min(100, int(1.5e10 / (float(n) * n)) + 1))
        steps = _log_int(rng, 1, most)
        precision = rng.choice(["mixed", "mixed", "fp32"])
        io = "f64" if precision == "mixed" and steps == 1 and n >= 32768 else "f32"
        return {"kind": "step", "precision": precision, "n": n, "steps": steps, "io": io,
                "shape": "plummer" if io == "f64" else rng.choice(["cube", "plummer"]), **common, **move}
    if kind == "slice":
        n = _log_int(rng, 32768, 262144)
        shares = rng.choice([2, 3, 4, 7, 8]) if n < 131072 else rng.choice([4, 7, 8])
        return {"kind": "slice", "precision": "mixed", "n": n, "shares": shares, "share": rng.randrange(shares),
                "io": "f64", "shape": "plummer", **common, **move}
    if kind == "share":
        shares = rng.choice([2, 4, 5, 8])
        return {"kind": "share", "precision": "mixed", "shares": shares, "share": rng.randrange(shares),
                "n": 1024 * shares * _log_int(rng, 32768 / (1024 * shares), 262144 / (1024 * shares)),
                "io": "f64", "shape": "plummer", **common, **move}
    if kind == "ref":
        io = rng.choice(["f32", "f32", "f64"])
        return {"kind": "ref", "io": io, "n": _log_int(rng, 512, 50000 if io == "f32" else 30000),
                "steps": rng.choice([1, 2, 3]), "masses": masses, "shape": rng.choice(["cube", "plummer"]),
                "eps": eps, "dt": dt, "damping": move["damping"]}
    if kind == "adjoint":
        n = _log_int(rng, 1024, 16384)
        return {"kind": "adjoint", "precision": "mixed", "n": n, "steps": rng.randrange(5, 41),
                "ckpt": rng.choice([1, 5, 10]), "shape": rng.choice(["cube", "plummer"]), **common, **move}
    if kind == "batch":
        return {"kind": "batch", "systems": _log_int(rng, 8, 90), "smallest": 256,
                "largest": rng.choice([2048, 4096, 8192]), "steps": rng.choice([5, 10, 20]),
                "ckpt": rng.choice([5, 10]), "adjoint": rng.random() < 0.5, "masses": masses, "shape": "plummer",
                "eps": 0.01, "dt": 1e-3, "damping": move["damping"]}
    return {"kind": "step", "precision": "fp64", "n": _log_int(rng, 1024, 32768), "steps": 1, "io": "f64",
            "shape": rng.choice(["cube", "plummer"]), **common, **move}


# ---- inputs ------------------------------------------------------------------------
def _isotropic(g, n):
    v = g.standard_normal((n, 3))
    return v / np.maximum(np.linalg.norm(v, axis=1, keepdims=True), 1e-300)


def _bodies(shape, masses, n, seed):
    """pos [n,4] = (x,y,z,m), vel [n,4] = (vx,vy,vz,1), FP64 on the host."""
    g = np.random.default_rng(seed)
    pos, vel = np.empty((n, 4)), np.empty((n, 4))
    if shape == "cube":
        pos[:, :3] = g.uniform(-1.0, 1.0, (n, 3))
        vel[:, :3] = g.normal(0.0, 0.01, (n, 3))
    else:  # Plummer sphere, a = 1, total mass 1, the outer 0.1% of the mass cut
        r = 1.0 / np.sqrt(g.uniform(1e-6, 0.999, n) ** (-2.0 / 3.0) - 1.0)
        q = np.empty(0)
        while len(q) < n:
            x, y = g.random(4 * n + 64), 0.1 * g.random(4 * n + 64)
            q = np.concatenate([q, x[y < x * x * (1.0 - x * x) ** 3.5]])
        pos[:, :3] = r[:, None] * _isotropic(g, n)
        vel[:, :3] = (q[:n] * math.sqrt(2.0) * (1.0 + r * r) ** -0.25)[:, None] * _isotropic(g, n)
        pos[:, :3] -= pos[:, :3].mean(axis=0)
        vel[:, :3] -= vel[:, :3].mean(axis=0)
    m = np.full(n, 1.0) if masses == "equal" else np.exp(g.uniform(math.log(0.5), math.log(2.0), n))
    pos[:, 3] = m / n
    vel[:, 3] = 1.0
    return pos, vel


def _bodies_io(case, seed):
    pos, vel = _bodies(case["shape"], case["masses"], case["n"], seed)
    t = np.float32 if case.get("io", "f32") == "f32" else np.float64
    return pos.astype(t), vel.astype(t)


def _targets(n, seed):
    return np.random.default_rng([seed, 1]).normal(0.0, 0.5, (n, 3))


def _batch_sizes(case):
    """Log-uniform sizes, one from each of `systems` equal parts, in mixed order."""
    g = np.random.default_rng(case["systems"])
    u = (g.permutation(case["systems"]) + g.random(case["systems"])) / case["systems"]
    return [int(round(x)) for x in case["smallest"] * (case["largest"] / case["smallest"]) ** u]


def _batch_bodies(case, seed):
    sizes = _batch_sizes(case)
    both = [_bodies(case["shape"], case["masses"], n, [seed, 3, k]) for k, n in enumerate(sizes)]
    return sizes, np.concatenate([b[0] for b in both]), np.concatenate([b[1] for b in both])


def _slice(case):
    """(start, count) of a share's bodies: the first n % shares shares take one more."""
    per, extra = divmod(case["n"], case["shares"])
    return case["share"] * per + min(case["share"], extra), per + (case["share"] < extra)


def _handle(case):
    return U.System(case["n"], PRECISIONS[case["precision"]], case["eps"] ** 2, case["dt"], case["damping"],
                    kick=U.KICK_REFERENCE if case["kick"] == "reference" else U.KICK_PHYSICAL,
                    flags=0 if case["newton"] else U.FLAG_NO_NEWTON)


def _p(t):
    return C.c_void_p(t.data_ptr())


def prepare(case, seed):
    kind = case["kind"]
    s = {"case": case}
    if kind == "batch":
        sizes, s["pos"], s["vel"] = _batch_bodies(case, seed)
        s["target"] = _targets(len(s["pos"]), seed) if case["adjoint"] else None
        s["batch"] = U.Batch(sizes, case["eps"] ** 2, case["dt"], case["damping"])
        # the first run tunes the kernels and captures the graph that a program replays
        s["batch"].set_state(s["pos"], s["vel"])
        s["batch"].run(case["steps"], 0, case["ckpt"], s["target"])
        return s
    pos, vel = _bodies_io(case, seed)
    if kind == "adjoint":
        s["pos"], s["vel"] = pos.astype(np.float64), vel.astype(np.float64)
        s["target"] = _targets(case["n"], seed)
        s["system"] = _handle(case)
        return s
    s["pos"], s["vel"] = torch.from_numpy(pos).cuda(), torch.from_numpy(vel).cuda()
    s["new_pos"], s["new_vel"] = torch.empty_like(s["pos"]), torch.empty_like(s["vel"])
    if kind == "field":
        s["acc"] = torch.empty((case["n"], 3), dtype=torch.float64, device="cuda")
    elif kind == "ref":
        s["old_pos"] = torch.empty_like(s["pos"])
    else:
        s["system"] = _handle(case)
    if kind == "share":
        # what the other GPUs' shares deliver: the reactions summed over all shares
        h, total = s["system"], None
        s["react"] = torch.empty((case["n"], 3), dtype=torch.float64, device="cuda")
        U.check(U.lib().utcnb_set_state(h.h, _p(s["pos"]), _p(s["vel"]), U.F64, U.DEVICE), "set_state")
        for k in range(case["shares"]):
            h.share_pairs(case["shares"], k, s["react"].data_ptr())
            h.sync()
            total = s["react"].clone() if total is None else total + s["react"]
        start, count = h.share_range(case["shares"], case["share"])
        s["react_sum"] = total[start:start + count].contiguous()
        torch.cuda.synchronize()
    return s


def run(state):
    case = state["case"]
    kind = case["kind"]
    L = U.lib()
    if kind == "field":
        U.check(L.utcnb_accel_noalloc(_p(state["pos"]), case["n"], case["eps"] ** 2, PRECISIONS[case["precision"]], 0,
                                      0 if case["newton"] else U.FLAG_NO_NEWTON, _p(state["acc"]), None), "field")
        return state["acc"].to(torch.float32)
    if kind == "ref":
        f32 = case["io"] == "f32"
        fn, r = (L.utcnb_integrate_f32, np.float32) if f32 else (L.utcnb_integrate_f64, np.float64)
        state["new_vel"].copy_(state["vel"])
        src, bufs = state["pos"], (state["new_pos"], state["old_pos"])
        for k in range(case["steps"]):
            dst = bufs[k % 2]
            U.check(fn(_p(src), _p(dst), _p(state["new_vel"]), case["n"], r(case["dt"]), r(case["eps"]) ** 2,
                       r(case["damping"]), 0, None), "integrate")
            src = dst
        return src, state["new_vel"]
    if kind == "adjoint":
        state["system"].set_state(state["pos"], state["vel"])
        loss, dx, dv, dm = state["system"].adjoint(case["steps"], case["ckpt"], state["target"])
        return [np.float32(loss), dx.astype(np.float32), dv.astype(np.float32), dm.astype(np.float32)]
    if kind == "batch":
        b = state["batch"]
        b.set_state(state["pos"], state["vel"])
        r = b.run(case["steps"], 0, case["ckpt"], state["target"])
        outs = r[1:] if case["adjoint"] else b.get_state()
        return [x.astype(np.float32) for x in outs]
    h = state["system"]
    io = U.F32 if case["io"] == "f32" else U.F64
    U.check(L.utcnb_set_state(h.h, _p(state["pos"]), _p(state["vel"]), io, U.DEVICE), "set_state")
    if kind == "step":
        h.step(case["steps"])
    elif kind == "slice":
        h.step_slice(*_slice(case))
    else:
        h.share_pairs(case["shares"], case["share"], state["react"].data_ptr())
        h.share_finish(case["shares"], case["share"], state["react_sum"].data_ptr())
    U.check(L.utcnb_get_state(h.h, _p(state["new_pos"]), _p(state["new_vel"]), io, U.DEVICE), "get_state")
    if kind == "share":
        return state["new_pos"], state["new_vel"], state["react"].to(torch.float32)
    return state["new_pos"], state["new_vel"]


def work(case):
    kind = case["kind"]
    if kind == "batch":
        sizes = _batch_sizes(case)
        n, n2 = float(sum(sizes)), float(sum(k * k for k in sizes))
        out = 56 + 24 if case["adjoint"] else 64
        return {"bytes": n * (64 + out), "flops": case["steps"] * n2 * (60 if case["adjoint"] else 20)}
    n = float(case["n"])
    word = 4 if case.get("io", "f32") == "f32" else 8
    if kind == "field":
        return {"bytes": n * (16 + 24), "flops": 20 * n * n}
    if kind == "adjoint":
        return {"bytes": n * (64 + 24 + 56), "flops": 60 * n * n * case["steps"]}
    if kind == "slice":
        count = _slice(case)[1]
        return {"bytes": n * 64 + count * 64, "flops": 20 * n * count}
    if kind == "share":
        return {"bytes": n * 64 + n * 24 + n / case["shares"] * (64 + 24), "flops": 20 * n * n / case["shares"]}
    return {"bytes": n * 16 * word, "flops": 20 * n * n * case["steps"]}


# ---- the same in 64 bits, plain torch -----------------------------------------------
def _rows(n):
    return max(1, (1 << 27) // n)


def _pairs64(x, i, j, eps2):
    """d^2 + eps2 of rows i:j against all, FP64."""
    d2 = None
    for c in range(3):
        t = x[None, :, c] - x[i:j, c, None]
        d2 = t.square_().add_(eps2) if d2 is None else d2.add_(t.square_())
    return d2


def _field64(x, m, eps2, start=0, count=None):
    """sum_j m_j r_ij (|r_ij|^2 + eps2)^-3/2 of rows [start, start + count)."""
    n = len(x)
    end = n if count is None else start + count
    one = torch.cat([x, torch.ones_like(x[:, :1])], 1) * m[:, None]
    out = torch.empty((end - start, 3), dtype=torch.float64, device=x.device)
    for i in range(start, end, _rows(n)):
        j = min(end, i + _rows(n))
        y = _pairs64(x, i, j, eps2).rsqrt_()
        s = y.square().mul_(y) @ one
        out[i - start:j - start] = s[:, :3] - x[i:j] * s[:, 3:]
    return out


def _vjp64(x, m, a, eps2):
    """(xbar, mbar) that the field passes on for the field's adjoint a."""
    xb, mb = torch.empty_like(x), torch.empty_like(m)
    own = (a * x).sum(1)
    for i in range(0, len(x), _rows(len(x))):
        j = min(len(x), i + _rows(len(x)))
        y = _pairs64(x, i, j, eps2).rsqrt_()
        y2 = y.square()
        y3 = y.mul_(y2)
        arj = own[None, :] - x[i:j] @ a.T
        ari = a[i:j] @ x.T - own[i:j, None]
        mb[i:j] = -(y3 * arj).sum(1)
        q = (m[i:j, None] * arj).sub_(m[None, :] * ari).mul_(y2).mul_(y3).mul_(3.0)
        xb[i:j] = m[i:j, None] * (y3 @ a) - a[i:j] * (y3 @ m)[:, None]
        xb[i:j] -= q @ x - x[i:j] * q.sum(1, keepdim=True)
    return xb, mb


def _kick_drift64(x, v, acc, w, dt, damping):
    v = (v + acc * w[:, None] * dt) * damping if w is not None else (v + acc * dt) * damping
    return x + v * dt, v


def _forward64(pos, vel, case, steps, eps2, dt, damping, keep=None):
    x, m, v = pos[:, :3].clone(), pos[:, 3].clone(), vel[:, :3].clone()
    w = m if case.get("kick", "physical") == "reference" else None
    for _ in range(steps):
        if keep is not None:
            keep.append(x)
        x, v = _kick_drift64(x, v, _field64(x, m, eps2), w, dt, damping)
    return x, m, v


def _adjoint64(pos, vel, target, case):
    eps2, dt, damping = case["eps"] ** 2, case["dt"], case["damping"]
    refkick = case.get("kick", "physical") == "reference"
    kept = []
    x, m, v = _forward64(pos, vel, case, case["steps"], eps2, dt, damping, kept)
    d = x - target
    loss = d.square().sum() / len(x)
    xb, vb, mb = 2.0 * d / len(x), torch.zeros_like(x), torch.zeros_like(m)
    for x in reversed(kept):
        vb = (vb + dt * xb) * damping
        a = vb * dt
        if refkick:
            mb = mb + (a * _field64(x, m, eps2)).sum(1)
            a = a * m[:, None]
        px, pm = _vjp64(x, m, a, eps2)
        xb, mb = xb + px, mb + pm
    return loss, xb, vb, mb


def _whole(x, m, v, vel):
    return torch.cat([x, m[:, None]], 1), torch.cat([v, vel[:, 3:]], 1)


def _up(a):
    return torch.from_numpy(np.ascontiguousarray(a, dtype=np.float64)).cuda()


def exact(case, seed):
    kind = case["kind"]
    if kind == "batch":
        sizes, pos, vel = _batch_bodies(case, seed)
        target = _targets(len(pos), seed)
        outs, at = [], 0
        for n in sizes:
            p, v, t = (_up(a[at:at + n]) for a in (pos, vel, target))
            at += n
            if case["adjoint"]:
                loss, dx, dv, dm = _adjoint64(p, v, t, case)
                outs.append((loss.reshape(1), dx, dv, dm))
            else:
                outs.append(_whole(*_forward64(p, v, case, case["steps"], case["eps"] ** 2, case["dt"],
                                               case["damping"]), v))
        return [torch.cat(x) for x in zip(*outs)]
    pos, vel = _bodies_io(case, seed)
    p, v = _up(pos), _up(vel)
    if kind == "adjoint":
        return list(_adjoint64(p, v, _up(_targets(case["n"], seed)), case))
    if kind == "field":
        return _field64(p[:, :3], p[:, 3], case["eps"] ** 2)
    if kind in ("slice", "share"):
        if kind == "slice":
            start, count = _slice(case)
        else:
            count = case["n"] // case["shares"]
            start = count * case["share"]
        rows = slice(start, start + count)
        w = p[rows, 3] if case["kick"] == "reference" else None
        acc = _field64(p[:, :3], p[:, 3], case["eps"] ** 2, start, count)
        p, v = p.clone(), v.clone()
        p[rows, :3], v[rows, :3] = _kick_drift64(p[rows, :3], v[rows, :3], acc, w, case["dt"], case["damping"])
        return (p, v) if kind == "slice" else (p, v, None)
    if kind == "ref":
        r = np.float32 if case["io"] == "f32" else np.float64
        eps2, dt, damping = float(r(case["eps"]) ** 2), float(r(case["dt"])), float(r(case["damping"]))
        return _whole(*_forward64(p, v, {"kick": "reference"}, case["steps"], eps2, dt, damping), v)
    return _whole(*_forward64(p, v, case, case["steps"], case["eps"] ** 2, case["dt"], case["damping"]), v)
