"""Tree-parallel kernels and vector stores of row outputs against the FP64 oracle at the sizes where their tiles of eight
configurations, levels and rounds can go wrong, on every route of the dispatch (prebuilt
and run-time topologies, both layouts and precisions, padded leading dimensions).

Bars (per configuration, infinity norm, relative): FP32 sums over a tree of at most 40
joints as the other kernels' tests (M 1e-5; products with M^-1 4e-4, its conditioning);
FP64 1e-12 and 1e-9.
"""
import ctypes

import numpy as np
import pytest

import oracle
import pinocchio_amd as pa
from helpers import f32_round, inputs, rel_err_cols, rel_err_mats
from pinocchio_amd import models as M

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")

TREES = [M.manipulator6, M.quadruped18, M.humanoid36, M.free_body, M.pendulum,
         lambda: M.random_tree(27, 41), lambda: M.random_tree(20, 7, free_flyer=False),
         lambda: M.serial_chain(30, 3)]
BATCHES = [1, 7, 8, 9, 200]


@pytest.fixture(scope="module")
def ctx():
    return pa.Context(0)


def _inputs(d, B, dt):
    x = inputs(d, B)
    return f32_round(*x) if dt == torch.float32 else x


def _dev(x, layout, dt):
    return torch.tensor(np.ascontiguousarray(x.T if layout == "col" else x), dtype=dt, device="cuda")


@pytest.mark.parametrize("tree", range(len(TREES)))
@pytest.mark.parametrize("dt,bar,bar_inv", [(torch.float32, 1e-5, 4e-4), (torch.float64, 1e-12, 1e-9)])
def test_crba_and_minverse(ctx, tree, dt, bar, bar_inv):
    d = TREES[tree]()
    for runtime in (False, True):
        m = pa.Model(ctx, d, runtime_topology=runtime)
        for B in BATCHES:
            q = _inputs(d, B, dt)[0]
            ref = oracle.crba(d, q)
            inv = np.linalg.inv(ref)
            up = np.triu(ref)
            if d.jtype[1] == M.JT_FREEFLYER:  # upper-only keeps a joint's own block full
                up[:, :6, :6] = ref[:, :6, :6]
            for layout in ("col", "batch"):
                e = pa.Engine(m, layout)
                x = _dev(q, layout, dt)
                num = lambda t: e.mats_to_numpy(t, layout, d.nv)  # noqa: E731
                assert rel_err_mats(num(e.crba(x)), ref).max() < bar, (d.name, B, layout)
                assert rel_err_mats(num(e.crba(x, upper_only=True)), up).max() < bar, (d.name, B, layout)
                assert rel_err_mats(num(e.compute_minverse(x)), inv).max() < bar_inv, (d.name, B, layout)


@pytest.mark.parametrize("tree", range(len(TREES)))
@pytest.mark.parametrize("dt,bar_rnea,bar_aba", [(torch.float32, 1e-5, 1e-4), (torch.float64, 1e-12, 1e-10)])
def test_rnea_and_aba(ctx, tree, dt, bar_rnea, bar_aba):
    d = TREES[tree]()
    m = pa.Model(ctx, d, runtime_topology=True)
    for B in BATCHES:
        q, v, a, tau = _inputs(d, B, dt)
        refs = oracle.rnea(d, q, v, a), oracle.aba(d, q, v, tau)
        for layout in ("col", "batch"):
            e = pa.Engine(m, layout)
            Q, V, A, T = (_dev(x, layout, dt) for x in (q, v, a, tau))
            for out, ref, bar in ((e.rnea(Q, V, A), refs[0], bar_rnea), (e.aba(Q, V, T), refs[1], bar_aba)):
                x = out.double().cpu().numpy()
                assert rel_err_cols(x.T if layout == "col" else x, ref).max() < bar, (d.name, B, layout)
        e = pa.Engine(m, "col")  # inputs that are zero for every configuration
        g = e.generalized_gravity(_dev(q, "col", dt)).double().cpu().numpy().T
        assert rel_err_cols(g, oracle.rnea(d, q, 0 * v, 0 * a)).max() < 2 * bar_rnea, (d.name, B)


@pytest.mark.parametrize("pad", [1, 3, 4])
def test_crba_padded_leading_dimension(ctx, pad):
    """Rows that are not 16-byte aligned, and gaps that stay as the caller had them."""
    d = M.humanoid36()
    m = pa.Model(ctx, d)
    B, nv = 83, d.nv
    q = f32_round(inputs(d, B)[0])[0]
    ref = oracle.crba(d, q)
    for layout, shape in (("col", (B, nv * nv + pad)), ("batch", (nv * nv, B + pad))):
        x = _dev(q, layout, torch.float32)
        out = torch.full(shape, 7.0, dtype=torch.float32, device="cuda")
        flags = pa.RBD_LAYOUT_BATCH if layout == "batch" else 0
        ld = out.stride(0)
        pa._check(pa.lib().rbd_crba(ctx.handle, m.handle, pa._i64(B), pa.RBD_F32, pa._ptr(x), pa._i64(x.stride(0)),
                                    pa._ptr(out), pa._i64(ld), ctypes.c_uint32(flags)))
        o = out.double().cpu().numpy()
        if layout == "col":
            got, gap = o[:, :nv * nv].reshape(B, nv, nv).transpose(0, 2, 1), o[:, nv * nv:]
        else:
            got, gap = o[:, :B].reshape(nv, nv, B).transpose(2, 1, 0), o[:, B:]
        assert rel_err_mats(got, ref).max() < 1e-5
        assert (gap == 7.0).all()


@pytest.mark.parametrize("tree", range(len(TREES)))
@pytest.mark.parametrize("dt,bar", [(torch.float32, 4e-4), (torch.float64, 1e-9)])
def test_aba_derivatives(ctx, tree, dt, bar):
    d = TREES[tree]()
    for B in BATCHES:
        q, v, _, tau = _inputs(d, B, dt)
        ref = oracle.aba_derivatives(d, q, v, tau)
        ddq = oracle.aba(d, q, v, tau)
        for runtime in (False, True):
            m = pa.Model(ctx, d, runtime_topology=runtime)
            for layout in ("col", "batch"):
                e = pa.Engine(m, layout)
                out = e.aba_derivatives(*(_dev(x, layout, dt) for x in (q, v, tau)))
                err = [rel_err_mats(e.mats_to_numpy(o, layout, d.nv), r).max() for o, r in zip(out[:3], ref[:3])]
                a = out[3].double().cpu().numpy()
                err.append(rel_err_cols(a.T if layout == "col" else a, ddq).max())
                assert max(err) < bar, (d.name, B, layout, runtime, err)


def test_aba_derivatives_in_chunks(ctx):
    """A batch beyond one chunk of the packed workspace: bit-identical to its parts."""
    d = M.humanoid36()
    e = pa.Engine(pa.Model(ctx, d), "col")
    B = 10_603
    x = [_dev(y, "col", torch.float64) for y in (lambda t: (t[0], t[1], t[3]))(inputs(d, B))]
    whole = e.aba_derivatives(*x)
    for lo, hi in ((0, 300), (B - 331, B)):
        part = e.aba_derivatives(*(y[lo:hi].contiguous() for y in x))
        for a, b in zip(whole, part):
            assert torch.equal(a[lo:hi], b)


def test_aba_derivatives_captured_after_a_smaller_workspace(ctx):
    """A capture whose workspace an eager call of the other route reserved (it holds all packed tiles)."""
    d = M.quadruped18()
    c = pa.Context(0)
    e = pa.Engine(pa.Model(c, d), "batch")
    big = [_dev(y, "batch", torch.float32) for y in (lambda t: (t[0], t[1], t[3]))(inputs(d, 20_000))]
    small = [y[:, :3000].contiguous() for y in big]
    e.aba_derivatives(*big)  # reserves for 20,000 configurations of the other route
    out = [torch.empty((d.nv * d.nv, 3000), device="cuda") for _ in range(3)]
    ddq = torch.empty((d.nv, 3000), device="cuda")
    with c.capture() as cap:
        e.aba_derivatives(*small, out=out, ddq_out=ddq, async_=True)
    ref = e.aba_derivatives(*small)
    for _ in range(3):
        for o in (*out, ddq):
            o.zero_()
        torch.cuda.synchronize()
        cap.graph.launch()
        for a, b in zip((*out, ddq), ref):
            assert ((a - b).abs().max() <= 2e-4 * b.abs().max()).item()


def test_aba_derivatives_captured_in_the_chunks_that_fit(ctx):
    """A capture for which only the other route's smaller workspace was reserved: the packed tiles go in
    the chunks that it holds, bit-identical to the eager call (the other route's sums differ)."""
    d = M.quadruped18()
    c = pa.Context(0)
    m = pa.Model(c, d)
    x = [_dev(y, "batch", torch.float32) for y in (lambda t: (t[0], t[1], t[3]))(inputs(d, 20_000))]
    pa.Engine(m, "batch").aba_derivatives(*x)  # reserves (99 + 36) scalars per configuration
    e, B = pa.Engine(m, "col"), 9000           # wants 18 + 549, of which 4,616 configurations fit
    rows = [y[:, :B].t().contiguous() for y in x]
    out = [torch.empty((B, d.nv, d.nv), device="cuda") for _ in range(3)]
    ddq = torch.empty((B, d.nv), device="cuda")
    with c.capture() as cap:
        e.aba_derivatives(*rows, out=out, ddq_out=ddq, async_=True)
    ref = pa.Engine(pa.Model(ctx, d), "col").aba_derivatives(*rows)
    for _ in range(3):
        for o in (*out, ddq):
            o.zero_()
        torch.cuda.synchronize()
        cap.graph.launch()
        assert all(torch.equal(a, b) for a, b in zip((*out, ddq), ref))
    cap.graph.close()


def test_aba_derivatives_capture_refused_without_a_workspace():
    """Without kernels of its own a tree has no other path that would allocate nothing: a capture whose
    workspace holds not even one tile is refused as any other, and the context stays usable."""
    d = M.random_tree(20, 7)
    c = pa.Context(0)
    e = pa.Engine(pa.Model(c, d), "batch")
    x = [_dev(y, "batch", torch.float32) for y in (lambda t: (t[0], t[1], t[3]))(inputs(d, 16))]
    one = [y[:, :1].contiguous() for y in x]
    e.aba_derivatives(*one)
    out = [torch.empty((d.nv * d.nv, 16), device="cuda") for _ in range(3)]
    with pytest.raises(ValueError, match="workspace"):
        with c.capture():
            e.aba_derivatives(*x, out=out, async_=True)
    e.aba_derivatives(*x, out=out)


@pytest.mark.parametrize("dt,bar", [(torch.float32, 2e-6), (torch.float64, 1e-13)])
@pytest.mark.parametrize("pad", [0, 1, 2, 4])
def test_kinematics_rows(ctx, dt, bar, pad):
    """Row outputs whose runs are and are not aligned to the vector stores, with gaps that stay
    as the caller had them; against the oracle (FP32: rounding of at most 30 composed
    placements in one coordinate of the largest)."""
    for d, runtime in ((M.arm7(), False), (M.humanoid36(), False), (M.humanoid36(), True), (M.random_tree(12, 5), False)):
        m = pa.Model(ctx, d, runtime_topology=runtime)
        nj, nv, B = d.njoints - 1, d.nv, 131
        q, v, a, _ = _inputs(d, B, dt)
        Q, V, A = (_dev(x, "col", dt) for x in (q, v, a))
        rows = {"M": 12 * nj, "v": 6 * nj, "a": 6 * nj, "J": 6 * nv}
        out = {k: torch.full((B, n + pad), 7.0, dtype=dt, device="cuda") for k, n in rows.items()}
        code = pa.RBD_F32 if dt == torch.float32 else pa.RBD_F64
        p, i = pa._ptr, pa._i64
        pa._check(pa.lib().rbd_forward_kinematics(
            ctx.handle, m.handle, i(B), code, p(Q), i(d.nq), p(V), i(nv), p(A), i(nv), p(out["M"]),
            i(out["M"].stride(0)), p(out["v"]), p(out["a"]), i(out["v"].stride(0)), ctypes.c_uint32(0)))
        pa._check(pa.lib().rbd_joint_jacobians(ctx.handle, m.handle, i(B), code, p(Q), i(d.nq), p(out["J"]),
                                               i(out["J"].stride(0)), ctypes.c_uint32(0)))
        oM, ov, oa = oracle.forward_kinematics(d, q, v, a)
        ref = {"M": oM[:, 1:].reshape(B, -1) if oM.shape[1] == nj + 1 else oM.reshape(B, -1),
               "v": ov[:, 1:].reshape(B, -1) if ov.shape[1] == nj + 1 else ov.reshape(B, -1),
               "a": oa[:, 1:].reshape(B, -1) if oa.shape[1] == nj + 1 else oa.reshape(B, -1),
               "J": oracle.joint_jacobians(d, q).transpose(0, 2, 1).reshape(B, -1)}
        for k, n in rows.items():
            x = out[k].double().cpu().numpy()
            assert rel_err_cols(x[:, :n].T, ref[k].T).max() < bar, (d.name, k, pad)
            assert (x[:, n:] == 7.0).all()


@pytest.mark.parametrize("dt,bar", [(torch.float32, 2e-6), (torch.float64, 1e-13)])
def test_kinematics_rows_staged(ctx, dt, bar):
    """The batch sizes whose row outputs go through LDS, with a last tile of one
    configuration and gaps between the rows; against the batch-fastest outputs (the same sums
    per configuration: the bar of the test above)."""
    for d, B in ((M.arm7(), 32769), (M.random60(), 32769), (M.humanoid36(), 32769), (M.quadruped18(), 8193)):
        m = pa.Model(ctx, d)
        q, v, a = (_dev(x, "col", dt) for x in _inputs(d, B, dt)[:3])
        eb = pa.Engine(m, "batch")
        ref = [*eb.forward_kinematics(*(x.t().contiguous() for x in (q, v, a))), eb.joint_jacobians(q.t().contiguous())]
        code = pa.RBD_F32 if dt == torch.float32 else pa.RBD_F64
        p, i = pa._ptr, pa._i64
        out = [torch.full((B, r.numel() // B + pad), 7.0, dtype=dt, device="cuda") for r, pad in zip(ref, (4, 2, 2, 6))]
        ld = [i(x.stride(0)) for x in out]
        pa._check(pa.lib().rbd_forward_kinematics(
            ctx.handle, m.handle, i(B), code, p(q), i(d.nq), p(v), i(d.nv), p(a), i(d.nv), p(out[0]), ld[0],
            p(out[1]), p(out[2]), ld[1], ctypes.c_uint32(0)))
        pa._check(pa.lib().rbd_joint_jacobians(ctx.handle, m.handle, i(B), code, p(q), i(d.nq), p(out[3]), ld[3],
                                               ctypes.c_uint32(0)))
        for x, r in zip(out, ref):
            r = r.reshape(-1, B).t()
            n = r.shape[1]
            assert ((x[:, :n] - r).abs().amax(1) <= bar * r.abs().amax(1)).all(), d.name
            assert (x[:, n:] == 7.0).all()

