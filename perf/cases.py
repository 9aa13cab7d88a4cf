"""The batched rigid-body workloads this framework is timed on.

Each case is one call (or the short sequence of calls that a control, simulation or
trajectory-optimisation program makes together) through ``pinocchio_amd.Engine`` or
``pinocchio_amd.MixedBatch``, with the robots of ``pinocchio_amd.models`` and a generated
tree that has no kernels of its own (what a user's robot is).  A case is

  op      rnea | aba | step | mass | derivatives | kinematics | contact | dynamics | mixed
  robot   a sample model, or "tree" (with n: revolute joints, tree: the tree's seed)
  batch   configurations per call
  dtype   f32 | f64
  layout  col (one configuration per row of memory, the default of Engine and the
          reference's Eigen layout) | batch (batch index fastest)

``exact`` evaluates the same quantities with plain torch in 64 bits: spatial quantities
swept over the joints for the whole batch, M as the sum of J_i^T I_i J_i, dense elimination
for the solves, and automatic differentiation of inverse dynamics for the derivatives.
"""
import math

import torch

import pinocchio_amd as pa
from pinocchio_amd import models

# instances per robot in a mixed batch, as shares of the whole
MIX = (("arm7", 0.40), ("quadruped18", 0.40), ("humanoid36", 0.15), ("random60", 0.05))


def listed():
    return [
        # one forward-dynamics evaluation inside a control loop: launches and latency only
        {"name": "aba_quadruped_1", "op": "aba", "robot": "quadruped18", "batch": 1, "dtype": "f64", "layout": "col"},
        # inverse dynamics of an industrial arm for a sampled controller, double precision
        {"name": "rnea_arm_4096_f64", "op": "rnea", "robot": "manipulator6", "batch": 4096, "dtype": "f64",
         "layout": "col"},
        # whole-body inverse dynamics for a reinforcement-learning batch kept as (B, n) tensors
        {"name": "rnea_humanoid_50021", "op": "rnea", "robot": "humanoid36", "batch": 50021, "dtype": "f32",
         "layout": "col"},
        # the benchmark step: forward dynamics, mass matrix and its FP64 tree factor
        {"name": "step_humanoid_65536", "op": "step", "robot": "humanoid36", "batch": 65536, "dtype": "f32",
         "layout": "batch"},
        # linearised dynamics of every sample of a large sampled planner
        {"name": "derivatives_humanoid_16384", "op": "derivatives", "robot": "humanoid36", "batch": 16384,
         "dtype": "f32", "layout": "batch"},
        # linearised dynamics at every knot of a few trajectories (shooting solver, FP64, Eigen matrices)
        {"name": "derivatives_quadruped_2000_f64", "op": "derivatives", "robot": "quadruped18", "batch": 2000,
         "dtype": "f64", "layout": "col"},
        # mass matrix and its inverse for operational-space control, one matrix per row of memory
        {"name": "mass_humanoid_10007", "op": "mass", "robot": "humanoid36", "batch": 10007, "dtype": "f32",
         "layout": "col"},
        # placements, velocities, accelerations and Jacobians of every joint
        {"name": "kinematics_humanoid_30011", "op": "kinematics", "robot": "humanoid36", "batch": 30011,
         "dtype": "f32", "layout": "col"},
        # forward dynamics with both feet held on the ground
        {"name": "contact_humanoid_16384", "op": "contact", "robot": "humanoid36", "batch": 16384, "dtype": "f32",
         "layout": "batch"},
        # a user's own robot, which has no prebuilt kernels: simulation and its mass matrix
        {"name": "dynamics_tree_16384", "op": "dynamics", "robot": "tree", "n": 27, "tree": 41, "batch": 16384,
         "dtype": "f32", "layout": "col"},
        # the same kind of robot in a trajectory optimiser
        {"name": "derivatives_tree_3001", "op": "derivatives", "robot": "tree", "n": 23, "tree": 42, "batch": 3001,
         "dtype": "f32", "layout": "col"},
        # a fleet of different robots stepped together
        {"name": "mixed_100000", "op": "mixed", "robot": "mix", "batch": 100000, "dtype": "f32", "layout": "batch"},
    ]


def draw(rng):
    def size(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    op = rng.choice(["rnea", "aba", "step", "mass", "derivatives", "kinematics", "contact", "dynamics", "derivatives",
                     "mixed"])
    c = {"op": op, "dtype": "f32", "layout": rng.choice(["col", "batch"])}
    if op in ("rnea", "aba"):
        c.update(robot=rng.choice(["manipulator6", "arm7", "quadruped18", "humanoid36", "random60"]),
                 batch=size(1, 65536), dtype=rng.choice(["f32", "f64"]))
    elif op == "step":
        c.update(robot=rng.choice(["arm7", "quadruped18", "humanoid36"]), batch=size(1000, 65536))
    elif op == "mass":
        c.update(robot=rng.choice(["manipulator6", "quadruped18", "humanoid36"]), batch=size(64, 30000))
    elif op == "kinematics":
        c.update(robot=rng.choice(["arm7", "quadruped18", "humanoid36"]), batch=size(64, 50000))
    elif op == "contact":
        c.update(robot=rng.choice(["quadruped18", "humanoid36"]), batch=size(256, 16384))
    elif op == "mixed":
        c.update(robot="mix", batch=size(2000, 100000), layout="batch")
    elif op == "dynamics":
        c.update(robot="tree", n=rng.randint(8, 32), tree=rng.randrange(1000), batch=size(64, 16384))
    elif rng.random() < 0.3:
        c.update(robot="tree", n=rng.randint(8, 28), tree=rng.randrange(1000), batch=size(64, 4096))
    else:
        c.update(robot=rng.choice(["manipulator6", "arm7", "quadruped18", "humanoid36"]), batch=size(64, 16384),
                 dtype=rng.choice(["f32", "f32", "f64"]))
    return c


# ---------------------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------------------
def _desc(case):
    if case["robot"] == "tree":
        return models.random_tree(case["n"], models.MODEL_SEED_BASE + 1000 + case["tree"], free_flyer=True, compact=True)
    return models.SAMPLE_MODELS[case["robot"]]()


def _inputs(desc, batch, dtype, gen):
    """(batch, rows) tensors q, v, a, tau: angles uniform, base within a metre of the origin
    in any orientation, velocities, accelerations and torques normal."""
    dev = gen.device
    uniform = lambda *s: torch.rand(*s, generator=gen, device=dev, dtype=torch.float64)  # noqa: E731
    q = (2 * uniform(batch, desc.nq) - 1) * math.pi
    for j, i in enumerate(desc.idx_q):
        if desc.jtype[j] == models.JT_FREEFLYER:
            x = torch.randn(batch, 4, generator=gen, device=dev, dtype=torch.float64)
            q[:, i:i + 3] /= math.pi
            q[:, i + 3:i + 7] = x / x.norm(dim=1, keepdim=True)
    v, a, tau = (torch.randn(batch, desc.nv, generator=gen, device=dev, dtype=torch.float64) for _ in range(3))
    return tuple(x.to(dtype) for x in (q, v, a, tau))


def _case_inputs(case, seed):
    dev = torch.device("cuda" if torch.cuda.is_available() else "cpu")
    gen = torch.Generator(device=dev)
    gen.manual_seed(seed * 1000003 + 17)
    dtype = torch.float64 if case["dtype"] == "f64" else torch.float32
    if case["op"] == "mixed":
        counts = [max(1, int(case["batch"] * share)) for _, share in MIX]
        descs = [models.SAMPLE_MODELS[name]() for name, _ in MIX]
        return [(d, _inputs(d, n, dtype, gen)) for d, n in zip(descs, counts)]
    d = _desc(case)
    return d, _inputs(d, case["batch"], dtype, gen)


def _feet(desc):
    """Last joint of the first two limbs (humanoid: 6-D contacts) or of all four (quadruped: points)."""
    tips = [j for j in range(1, desc.njoints) if j not in set(int(p) for p in desc.parents[1:])]
    return tips[:2] if desc.name == "humanoid36" else tips[:4]


_FOOT = (1.0, 0.0, 0.0, 0.0, 1.0, 0.0, 0.0, 0.0, 1.0, 0.02, -0.01, -0.08)  # sole in the last joint's frame


def _contacts(desc):
    kind = pa.CONTACT_6D if desc.name == "humanoid36" else pa.CONTACT_3D
    return [pa.RigidConstraintModel(kind, j, _FOOT) for j in _feet(desc)]


def prepare(case, seed):
    batch_fastest = case["layout"] == "batch"
    lay = (lambda x: x.t().contiguous()) if batch_fastest else (lambda x: x.contiguous())
    ctx = pa.Context(0)
    s = {"op": case["op"], "ctx": ctx}
    if case["op"] == "mixed":
        groups = [(pa.Model(ctx, d), *(lay(x) for x in xs)) for d, xs in _case_inputs(case, seed)]
        s["mix"] = pa.MixedBatch(ctx, groups)
        return s
    d, xs = _case_inputs(case, seed)
    s["q"], s["v"], s["a"], s["tau"] = (lay(x) for x in xs)
    s["eng"] = pa.Engine(pa.Model(ctx, d), case["layout"])
    if case["op"] == "contact":
        s["contacts"] = _contacts(d)
    return s


def run(s):
    op = s["op"]
    if op == "mixed":
        return s["mix"].run()
    e, q, v, a, tau = s["eng"], s["q"], s["v"], s["a"], s["tau"]
    if op == "rnea":
        return e.rnea(q, v, a)
    if op == "aba":
        return e.aba(q, v, tau)
    if op == "step":  # queued on the engine's stream; the last call waits
        ddq = e.aba(q, v, tau, async_=True)
        M = e.crba(q, async_=True)
        U, D = e.cholesky_decompose(M)
        return ddq, M, U, D
    if op == "mass":
        return e.crba(q), e.compute_minverse(q)
    if op == "derivatives":
        return e.aba_derivatives(q, v, tau)
    if op == "kinematics":
        return (*e.forward_kinematics(q, v, a), e.joint_jacobians(q))
    if op == "contact":
        return e.constraint_dynamics(q, v, tau, s["contacts"])
    return e.rnea(q, v, a), e.aba(q, v, tau), e.crba(q)  # dynamics


# ---------------------------------------------------------------------------------------
# what one pass cannot do without
# ---------------------------------------------------------------------------------------
def _work(case, d, batch):
    """Bytes of inputs and outputs; multiply-adds of the tree recursions (counted for the
    reference's sweeps, per joint) as two operations each."""
    nq, nv, nj = d.nq, d.nv, d.njoints - 1
    parent = {}  # dof -> next dof towards the root
    for j in range(1, d.njoints):
        iv, p = int(d.idx_v[j]), int(d.parents[j])
        parent[iv] = int(d.idx_v[p] + d.nvs[p] - 1) if p else -1
        for k in range(1, int(d.nvs[j])):
            parent[iv + k] = iv + k - 1
    nnz = 0
    for c in range(nv):
        x = parent[c]
        while x >= 0:
            nnz, x = nnz + 1, parent[x]
    S = 8 if case["dtype"] == "f64" else 4
    rnea, aba, crba, chol = 330 * nj, 860 * nj, 260 * nj + 22 * nnz, 12 * nnz
    op = case["op"]
    if op in ("rnea", "aba"):
        b, f = S * (nq + 3 * nv), rnea if op == "rnea" else aba
    elif op == "step":
        b, f = S * (nq + 3 * nv + nv * nv) + 8 * (nnz + nv), aba + crba + chol
    elif op == "mass":
        b, f = S * (nq + 2 * nv * nv), crba + chol + 4 * nv * nnz
    elif op == "derivatives":
        b, f = S * (nq + 3 * nv + 3 * nv * nv), aba + 70 * nnz + 1500 * nj + chol + 12 * nv * nnz
    elif op == "kinematics":
        b, f = S * (nq + 2 * nv + 24 * nj + 6 * nv), 250 * nj
    elif op == "contact":
        nc = 12
        b, f = S * (nq + 3 * nv + nc), rnea + crba + chol + 4 * (nc + 1) * nnz + 2 * nc * nc * nv + nc ** 3
    elif op == "mixed":
        b, f = S * (nq + 5 * nv), rnea + aba
    else:
        b, f = S * (nq + 5 * nv + nv * nv), rnea + aba + crba
    return batch * b, batch * f


def work(case):
    if case["op"] == "mixed":
        parts = [_work(case, models.SAMPLE_MODELS[n](), max(1, int(case["batch"] * share))) for n, share in MIX]
    else:
        parts = [_work(case, _desc(case), case["batch"])]
    return {"bytes": sum(p[0] for p in parts), "flops": sum(p[1] for p in parts)}


def tolerance(case):
    # about four times what the 64-bit evaluation below is away from the kernels; the solves
    # lose the conditioning of M (and of J M^-1 J^T)
    if case["dtype"] == "f64":
        return {"rel": 1e-12, "max": 1e-10}
    if case["op"] in ("rnea", "kinematics"):
        return {"rel": 1e-6, "max": 1e-4}
    if case["op"] in ("step", "dynamics", "mixed", "aba"):
        return {"rel": 8e-6, "max": 2e-3}
    return {"rel": 6e-5, "max": 8e-3}


# ---------------------------------------------------------------------------------------
# the same quantities in 64 bits with plain torch
# ---------------------------------------------------------------------------------------
def _cross(a, b):
    return torch.linalg.cross(a, b, dim=-1)


def _mv(R, x):
    return (R * x.unsqueeze(-2)).sum(-1)


def _mtv(R, x):
    return (R * x.unsqueeze(-1)).sum(-2)


def _mm(a, b):
    return (a.unsqueeze(-1) * b.unsqueeze(-3)).sum(-2)


def _quat(q):
    x, y, z, w = q.unbind(-1)
    return torch.stack([1 - 2 * (y * y + z * z), 2 * (x * y - z * w), 2 * (x * z + y * w),
                        2 * (x * y + z * w), 1 - 2 * (x * x + z * z), 2 * (y * z - x * w),
                        2 * (x * z - y * w), 2 * (y * z + x * w), 1 - 2 * (x * x + y * y)], -1).reshape(-1, 3, 3)


def _skew(w):
    x, y, z = w.unbind(-1)
    o = torch.zeros_like(x)
    return torch.stack([o, -z, y, z, o, -x, -y, x, o], -1).reshape(*w.shape[:-1], 3, 3)


class _Tree:
    """Joint frames of a batch: R (B, 3, 3) and p (B, 3) of each joint in its parent; with
    `step` (B, nv) a first-order step of the configuration along its tangent."""

    def __init__(self, d, q, step=None):
        self.d, self.n, dev = d, q.shape[0], q.device
        c = lambda x: torch.tensor(x, dtype=torch.float64, device=dev)  # noqa: E731
        self.R, self.p, self.body = [None], [None], [None]
        eye = torch.eye(3, dtype=torch.float64, device=dev)
        for j in range(1, d.njoints):
            Rp, pp = c(d.placement[j, :9].reshape(3, 3)), c(d.placement[j, 9:])
            iq, iv = int(d.idx_q[j]), int(d.idx_v[j])
            if d.jtype[j] == models.JT_FREEFLYER:
                Rq, pq = _quat(q[:, iq + 3:iq + 7]), q[:, iq:iq + 3]
                if step is not None:
                    pq = pq + _mv(Rq, step[:, iv:iv + 3])
                    Rq = _mm(Rq, eye + _skew(step[:, iv + 3:iv + 6]))
                R, p = _mm(Rp.expand(self.n, 3, 3), Rq), _mv(Rp, pq) + pp
            else:
                t = q[:, iq] if step is None else q[:, iq] + step[:, iv]
                K = _skew(eye[int(d.jtype[j]) - models.JT_RX])
                s, k = t.sin()[:, None, None], (1 - t.cos())[:, None, None]
                R = _mm(Rp.expand(self.n, 3, 3), eye + s * K + k * (K @ K))
                p = pp.expand(self.n, 3)
            self.R.append(R)
            self.p.append(p)
            m, com, I = d.inertia[j, 0], c(d.inertia[j, 1:4]), d.inertia[j, 4:]
            I3 = c([[I[0], I[1], I[3]], [I[1], I[2], I[4]], [I[3], I[4], I[5]]])
            C = _skew(com)
            self.body.append((float(m), com, I3 - float(m) * (C @ C)))  # about the joint frame's origin

    def down(self, j, m):  # a motion of the parent frame, in joint j's
        lin, ang = m
        return _mtv(self.R[j], lin + _cross(ang, self.p[j])), _mtv(self.R[j], ang)

    def force(self, j, m):  # inertia of body j times a motion
        lin, ang = m
        mass, com, I = self.body[j]
        com = com.expand_as(lin)
        return mass * (lin + _cross(ang, com)), mass * _cross(com, lin) + _mv(I, ang)

    def of_dofs(self, j, x):  # S_j x_j
        iv = int(self.d.idx_v[j])
        if self.d.jtype[j] == models.JT_FREEFLYER:
            return x[:, iv:iv + 3], x[:, iv + 3:iv + 6]
        ax = int(self.d.jtype[j]) - models.JT_RX
        ang = torch.zeros(self.n, 3, dtype=x.dtype, device=x.device)
        ang = torch.cat([ang[:, :ax], x[:, iv:iv + 1], ang[:, ax + 1:]], 1)
        return torch.zeros_like(ang), ang

    def motions(self, v, a, gravity):
        d, V, A = self.d, [None], [None]
        g = torch.tensor(d.gravity, dtype=torch.float64, device=v.device) * (-1.0 if gravity else 0.0)
        zero = torch.zeros(self.n, 3, dtype=torch.float64, device=v.device)
        V[0], A[0] = (zero, zero), (zero + g[:3], zero + g[3:])
        for j in range(1, d.njoints):
            p = int(d.parents[j])
            vJ, aJ = self.of_dofs(j, v), self.of_dofs(j, a)
            vp, ap = self.down(j, V[p]), self.down(j, A[p])
            vl, va = vp[0] + vJ[0], vp[1] + vJ[1]
            V.append((vl, va))
            A.append((ap[0] + aJ[0] + _cross(va, vJ[0]) + _cross(vl, vJ[1]), ap[1] + aJ[1] + _cross(va, vJ[1])))
        return V, A

    def rnea(self, v, a):
        d = self.d
        V, A = self.motions(v, a, True)
        F = [None] * d.njoints
        for j in range(1, d.njoints):
            h, f = self.force(j, V[j]), self.force(j, A[j])
            vl, va = V[j]
            F[j] = (f[0] + _cross(va, h[0]), f[1] + _cross(va, h[1]) + _cross(vl, h[0]))
        tau = [None] * d.njoints
        for j in range(d.njoints - 1, 0, -1):
            l, n = F[j]
            if d.jtype[j] == models.JT_FREEFLYER:
                tau[j] = torch.cat([l, n], 1)
            else:
                ax = int(d.jtype[j]) - models.JT_RX
                tau[j] = n[:, ax:ax + 1]
            p = int(d.parents[j])
            if p:
                up = _mv(self.R[j], l)
                F[p] = (F[p][0] + up, F[p][1] + _mv(self.R[j], n) + _cross(self.p[j], up))
        arm = torch.tensor(d.armature, dtype=torch.float64, device=v.device)
        return torch.cat(tau[1:], 1) + arm * a

    def world(self):
        R, p = [None], [None]
        for j in range(1, self.d.njoints):
            k = int(self.d.parents[j])
            R.append(_mm(R[k], self.R[j]) if k else self.R[j])
            p.append(p[k] + _mv(R[k], self.p[j]) if k else self.p[j])
        return R, p

    def local_jacobians(self):  # (B, 6, nv) of each joint in its own frame
        d, dev = self.d, self.R[1].device
        J = [None]
        for j in range(1, d.njoints):
            p = int(d.parents[j])
            Jj = torch.zeros(self.n, 6, d.nv, dtype=torch.float64, device=dev)
            if p:
                lin, ang = J[p][:, :3], J[p][:, 3:]
                Rt = self.R[j].transpose(1, 2).contiguous()
                Jj[:, :3] = torch.bmm(Rt, lin - torch.bmm(_skew(self.p[j]), ang))
                Jj[:, 3:] = torch.bmm(Rt, ang)
            iv = int(d.idx_v[j])
            if d.jtype[j] == models.JT_FREEFLYER:
                for k in range(6):
                    Jj[:, k, iv + k] += 1
            else:
                Jj[:, 3 + int(d.jtype[j]) - models.JT_RX, iv] += 1
            J.append(Jj)
        return J

    def mass(self):
        d, dev = self.d, self.R[1].device
        eye = torch.eye(3, dtype=torch.float64, device=dev)
        M = torch.diag(torch.tensor(d.armature, dtype=torch.float64, device=dev)).repeat(self.n, 1, 1)
        for j, J in enumerate(self.local_jacobians()):
            if j:
                m, com, I = self.body[j]
                C = _skew(com)
                Y = torch.zeros(6, 6, dtype=torch.float64, device=dev)
                Y[:3, :3], Y[:3, 3:], Y[3:, :3], Y[3:, 3:] = m * eye, -m * C, m * C, I
                M += torch.bmm(J.transpose(1, 2).contiguous(), torch.matmul(Y, J))
        return M


def _udut(M):
    """M = U D U^T by dense elimination from the last column: unit upper U and D."""
    A, n = M.clone(), M.shape[1]
    U, D = torch.zeros_like(M), torch.empty_like(M[:, 0])
    for j in range(n - 1, -1, -1):
        D[:, j] = A[:, j, j]
        U[:, :j, j] = A[:, :j, j] / D[:, j:j + 1]
        U[:, j, j] = 1
        A[:, :j, :j] -= U[:, :j, j, None] * A[:, None, :j, j]
    return U, D


def _solve(UD, X):
    U, D = UD
    X, n = X.clone(), D.shape[1]
    for j in range(n - 1, 0, -1):
        X[:, :j] -= U[:, :j, j, None] * X[:, j:j + 1]
    X /= D[:, :, None]
    for j in range(n - 1):
        X[:, j + 1:] -= U[:, j, j + 1:, None] * X[:, j:j + 1]
    return X


def _pattern(d):
    """Strictly upper entries of the packed factor: column by column, ancestors from the root down."""
    rows, cols, above = [], [], {}
    for j in range(1, d.njoints):
        up = above.get(int(d.parents[j]), [])
        for k in range(int(d.nvs[j])):
            c = int(d.idx_v[j]) + k
            rows += up
            cols += [c] * len(up)
            up = up + [c]
        above[j] = up
    return rows, cols


def _aba(d, T, v, tau):
    UD = _udut(T.mass())
    return _solve(UD, (tau - T.rnea(v, torch.zeros_like(v)))[:, :, None])[:, :, 0], UD


def _derivatives(d, q, v, tau):
    ddq, UD = _aba(d, _Tree(d, q), v, tau)
    with torch.enable_grad():
        step = torch.zeros_like(v).requires_grad_()
        vel = v.clone().requires_grad_()
        t = _Tree(d, q, step).rnea(vel, ddq)
        rows = [torch.autograd.grad(t[:, k].sum(), (step, vel), retain_graph=True) for k in range(d.nv)]
    dq, dv = (torch.stack([r[k] for r in rows], 1) for k in (0, 1))
    eye = torch.eye(d.nv, dtype=torch.float64, device=q.device).repeat(q.shape[0], 1, 1)
    return -_solve(UD, dq), -_solve(UD, dv), _solve(UD, eye), ddq


def _contact(d, q, v, tau):
    """q'' and multipliers under J q'' + drift = 0, drift the frames' acceleration at q'' = 0:
    spatial for a 6-D contact, that of the material point for a point contact."""
    T = _Tree(d, q)
    V, A = T.motions(v, torch.zeros_like(v), False)
    J, rows, drift = T.local_jacobians(), [], []
    p = torch.tensor(_FOOT[9:], dtype=torch.float64, device=q.device)
    for j in _feet(d):
        lin = J[j][:, :3] - torch.matmul(_skew(p), J[j][:, 3:])
        pe = p.expand(q.shape[0], 3)
        vl, al = V[j][0] + _cross(V[j][1], pe), A[j][0] + _cross(A[j][1], pe)
        if d.name == "humanoid36":
            rows.append(torch.cat([lin, J[j][:, 3:]], 1))
            drift.append(torch.cat([al, A[j][1]], 1))
        else:
            rows.append(lin)
            drift.append(al + _cross(V[j][1], vl))
    J, drift = torch.cat(rows, 1), torch.cat(drift, 1)
    free, UD = _aba(d, T, v, tau)
    Y = _solve(UD, J.transpose(1, 2).contiguous())
    lam = _solve(_udut(torch.bmm(J, Y)), -(torch.bmm(J, free[:, :, None]) + drift[:, :, None]))
    return free + torch.bmm(Y, lam)[:, :, 0], lam[:, :, 0]


def _exact_of(case, d, xs):
    q, v, a, tau = (x.double() for x in xs)
    op, T = case["op"], _Tree(d, q)
    if op == "rnea":
        return [T.rnea(v, a)]
    if op == "aba":
        return [_aba(d, T, v, tau)[0]]
    if op == "mixed":
        return [T.rnea(v, a), _aba(d, T, v, tau)[0]]
    if op == "dynamics":
        return [T.rnea(v, a), _aba(d, T, v, tau)[0], T.mass()]
    if op == "step":
        ddq, (U, D) = _aba(d, T, v, tau)
        rows, cols = _pattern(d)
        return [ddq, T.mass(), U[:, rows, cols], D]
    if op == "mass":
        M = T.mass()
        return [M, _solve(_udut(M), torch.eye(d.nv, dtype=torch.float64, device=q.device).repeat(len(q), 1, 1))]
    if op == "derivatives":
        return list(_derivatives(d, q, v, tau))
    if op == "contact":
        return list(_contact(d, q, v, tau))
    R, p = T.world()
    V, A = T.motions(v, a, False)
    oM, J = [], []
    for j in range(1, d.njoints):
        oM.append(torch.cat([R[j].reshape(-1, 9), p[j]], 1))
        zero = torch.zeros_like(p[j])
        if d.jtype[j] == models.JT_FREEFLYER:
            J += [torch.cat([R[j][:, :, k], zero], 1) for k in range(3)]
        for k in (0, 1, 2) if d.jtype[j] == models.JT_FREEFLYER else (int(d.jtype[j]) - models.JT_RX,):
            w = R[j][:, :, k]
            J.append(torch.cat([_cross(p[j], w), w], 1))
    return [torch.cat(oM, 1), torch.cat([torch.cat(x, 1) for x in V[1:]], 1),
            torch.cat([torch.cat(x, 1) for x in A[1:]], 1), torch.cat(J, 1)]


def exact(case, seed):
    def lay(x):
        if case["layout"] == "col":  # matrices column by column
            return x.transpose(1, 2).contiguous() if x.dim() == 3 else x
        return x.permute(2, 1, 0).reshape(-1, x.shape[0]) if x.dim() == 3 else x.t().contiguous()

    if case["op"] == "mixed":
        return [[lay(x) for x in _exact_of(case, d, xs)] for d, xs in _case_inputs(case, seed)]
    d, xs = _case_inputs(case, seed)
    out = [lay(x) for x in _exact_of(case, d, xs)]
    return out[0] if case["op"] in ("rnea", "aba") else out
