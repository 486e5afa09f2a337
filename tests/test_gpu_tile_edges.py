"""Bit equality with the oracle at the sizes where the marching kernels can go
wrong: one column more or less than a tile, level counts around the chunk
lengths the dispatch picks, every vertical boundary code."""
import numpy as np
import pytest
import torch

from fdd3260_amd import Advection, MultiDomain, _lib, cases
from oracle.oracle import Oracle

from helpers import case2d, case3d
from test_gpu_adjoint import _case as adjoint_case, _check_dot, _dirs, _interior_only, _mask, _tlm

pytestmark = pytest.mark.gpu


def _dev(cuda, *arrs):
    return [torch.from_numpy(np.ascontiguousarray(a)).to(cuda) for a in arrs]


@pytest.mark.parametrize("dims", [(31, 7, 8), (32, 8, 9), (33, 9, 17), (65, 17, 35), (6, 6, 8), (64, 0, 9), (65, 0, 33)])
@pytest.mark.parametrize("bc", ["nnf", "ope", "per"])
@pytest.mark.parametrize("ntime,lavisc", [(0, True), (1, True), (1, False)])
def test_momentum_tile_edges(cuda, dims, bc, ntime, lavisc):
    print(f"case momentum {dims} {bc} ntime={ntime} lavisc={lavisc}", flush=True)
    bcl = ("per", "per", "per", "per", bc, bc)
    mx, my, nz = dims
    g, u, v, w, _ = case3d(mx, my, nz, bcl=bcl) if my else case2d(mx, nz, bcl=bcl)
    rng = np.random.default_rng(9)
    mom = [a * (1.0 + 0.1 * rng.standard_normal(a.shape)) for a in (u, v, w)]
    ref = Oracle(g, lavisc=lavisc).qnadv_uvw(ntime, *mom, u, v, w)
    with Advection(g, lavisc=lavisc) as a:
        d = _dev(cuda, *mom, u, v, w)
        outs = [torch.full(g.shape, 7.0, dtype=torch.float64, device=cuda) for _ in range(3)]
        a.qnadv_uvw(ntime, d[:3], d[3:], outs)
        a.stream_sync()
        for c in (0, 1, 2) if my else (0, 2):
            assert np.array_equal(outs[c].cpu().numpy(), ref[c]), f"component {c}"


@pytest.mark.parametrize("scheme", ["weno", "weno5", "muscl", "ppm"])
@pytest.mark.parametrize("dims", [(139, 117, 75), (6, 6, 8), (33, 9, 8), (15, 17, 33), (300, 0, 41), (1500, 0, 301)])
def test_scalar_chunk_lengths(cuda, scheme, dims):
    """Grids for which the dispatch takes one level per item, a few (with a
    shorter last chunk) and several; the other tests' grids take one."""
    print(f"case chunks {scheme} {dims}", flush=True)
    mx, my, nz = dims
    g, u, v, w, q = case3d(mx, my, nz) if my else case2d(mx, nz)
    ref = np.zeros(g.shape)
    Oracle(g, scal_adv=scheme, muscllimiter="VL").scalar_tendency(1.0, u, v, w, q, ref)
    with Advection(g, scal_adv=scheme, muscllimiter="VL") as a:
        du, dv, dw, dq, dx = _dev(cuda, u, v, w, q, np.zeros(g.shape))
        a.scalar_tendency(1.0, du, dv, dw, [dq], [dx])
        a.stream_sync()
        assert np.array_equal(dx.cpu().numpy(), ref)


@pytest.mark.parametrize("what", ["heun", "ssprk3", "euler", "positive", "batch", "adjoint"])
@pytest.mark.parametrize("two_d", [False, True])
def test_scratch_contents_do_not_matter(cuda, what, two_d):
    """A context whose scratch arrays hold NaN from an earlier call gives the
    same bits as a fresh one: every value a stage reads was written by this
    call."""
    print(f"case scratch {what} 2d={two_d}", flush=True)
    g, u, v, w, q = case2d(40, 20) if two_d else case3d(37, 21, 18)
    wind = _dev(cuda, u, v, w)
    integ = {"heun": 2, "euler": 1}.get(what, 3)

    def call(a, field):
        if what == "batch":
            f = [field.float(), field.clone()]
            a.batch_advance(3, 2, 0.5, *[x.float() for x in wind], f)
        elif what == "adjoint":
            qbar, bars = field.clone(), [torch.zeros_like(x) for x in wind]
            a.adjoint_advance(3, 3, 0.5, *wind, field, qbar, *bars, checkpoint=2)
            f = [qbar] + bars
        else:
            f = [field.clone()]
            a.advance(integ, 2, 0.5, *wind, f, positive=what == "positive")
        a.stream_sync()
        return [x.cpu().numpy() for x in f]

    (field,) = _dev(cuda, q)
    torch.cuda.synchronize()
    with Advection(g) as a, Advection(g) as b:
        a.set_stream(0)
        b.set_stream(0)
        call(a, torch.full_like(field, float("nan")))
        for x, y in zip(call(a, field), call(b, field)):
            assert np.isfinite(x).all() and np.array_equal(x, y)


@pytest.mark.parametrize("dirs", [1, 2, 4, 5, 7])
@pytest.mark.parametrize("bc", ["nnf", "ope", "per"])
@pytest.mark.parametrize("side", ["per", "ope"])
def test_ppm_directions_and_boundaries(cuda, dirs, bc, side):
    """Every direction subset, vertical boundary code and side code (the
    non-periodic sides take another flux at the last interior cell), flux and
    advective form, on a grid of several tiles and chunks."""
    print(f"case ppm dirs={dirs} {bc} {side}", flush=True)
    g, u, v, w, q = case3d(47, 19, 75, bcl=(side,) * 4 + (bc, bc))
    for adv in (False, True):
        ref = np.full(g.shape, 0.25)
        Oracle(g, scal_adv="ppm").scalar_tendency(2.0, u, v, w, q, ref, adv, dirs)
        with Advection(g, scal_adv="ppm") as a:
            du, dv, dw, dq, dx = _dev(cuda, u, v, w, q, np.full(g.shape, 0.25))
            a.scalar_tendency(2.0, du, dv, dw, [dq], [dx], [adv], dirs=dirs)
            a.stream_sync()
            assert np.array_equal(dx.cpu().numpy(), ref)


@pytest.mark.parametrize("scheme,lim", [("weno", "MC"), ("ppm", "MC"), ("muscl", "minmod"), ("muscl", "MC"),
                                        ("muscl", "VL"), ("muscl", "Fromm")])
@pytest.mark.parametrize("data", ["tiny", "huge", "zeros", "constant", "steps"])
def test_scalar_extreme_values(cuda, scheme, lim, data):
    """Values at the ends of the exponent range, exact zeros, constants and
    jumps: the quotients without operand scaling and the limiter gates."""
    print(f"case extreme {scheme} {lim} {data}", flush=True)
    g, u, v, w, q = case3d(35, 18, 20, zero_frac=0.5 if data == "zeros" else 0.0)
    q = {"tiny": q * 1e-295, "huge": q * 1e150, "zeros": q, "constant": np.full_like(q, 3.25),
         "steps": np.where(q > 1e-4, 1.0, -2.0)}[data]
    ref = np.zeros(g.shape)
    Oracle(g, scal_adv=scheme, muscllimiter=lim).scalar_tendency(1.0, u, v, w, q, ref)
    with Advection(g, scal_adv=scheme, muscllimiter=lim) as a:
        du, dv, dw, dq, dx = _dev(cuda, u, v, w, q, np.zeros(g.shape))
        a.scalar_tendency(1.0, du, dv, dw, [dq], [dx])
        a.stream_sync()
        got = dx.cpu().numpy()
    # 'weno' forms the upwind side only: where the other side overflows to NaN
    # in the reference's sum, its value is not the reference's NaN
    fin = np.isfinite(ref) if scheme == "weno" else np.ones(g.shape, bool)
    assert fin.any() and np.array_equal(got[fin], ref[fin])


@pytest.mark.parametrize("scheme,lim", [("ppm", "MC"), ("muscl", "minmod"), ("muscl", "VL")])
@pytest.mark.parametrize("value", [float("nan"), float("inf"), -float("inf")])
def test_scalar_non_finite_values(cuda, scheme, lim, value):
    """A few non-finite cells: what they reach is what they reach in the
    reference's formulas, which look at both sides of a face."""
    print(f"case non-finite {scheme} {lim} {value}", flush=True)
    g, u, v, w, q = case3d(35, 18, 20)
    for k, j, i in ((0, 8, 9), (7, 12, 20), (19, 6, 30), (10, 15, 33)):
        q[k, j, i] = value
    ref = np.zeros(g.shape)
    with np.errstate(all="ignore"):
        Oracle(g, scal_adv=scheme, muscllimiter=lim).scalar_tendency(1.0, u, v, w, q, ref)
    with Advection(g, scal_adv=scheme, muscllimiter=lim) as a:
        du, dv, dw, dq, dx = _dev(cuda, u, v, w, q, np.zeros(g.shape))
        a.scalar_tendency(1.0, du, dv, dw, [dq], [dx])
        a.stream_sync()
        got = dx.cpu().numpy()
    assert not np.isfinite(got).all()
    assert np.array_equal(got, ref, equal_nan=True)


def _batch(cuda, mx, my, nz, nspec):
    """Batch of momenta, two FP64 scalars and FP32 species on FP32-representable inputs."""
    g, u, v, w, _ = case3d(mx, my, nz) if my else case2d(mx, nz)
    u, v, w = (a.astype(np.float32) for a in (u, v, w))
    rng = np.random.default_rng(17)
    mom = [a * (1.0 + 0.1 * rng.standard_normal(a.shape)).astype(np.float32) for a in (u, v, w)]
    f64 = [1.0 + rng.random(g.shape) for _ in range(2)]
    f32 = [np.exp(rng.standard_normal(g.shape)).astype(np.float32) for _ in range(nspec)]
    return g, _dev(cuda, u, v, w), _dev(cuda, *mom), _dev(cuda, *f64, *f32)


@pytest.mark.parametrize("scheme", ["weno", "weno5", "muscl"])
@pytest.mark.parametrize("dims", [(6, 6, 8), (33, 9, 17), (44, 37, 24), (130, 100, 40), (65, 0, 33)])
def test_batch_field_split(cuda, scheme, dims):
    """A batch whose fields are spread over work items, in whole or short chunks,
    has the bits of each field advected alone and of chunks of a set length."""
    print(f"case batch_field_split {scheme} {dims}", flush=True)
    g, vel, _, fields = _batch(cuda, *dims, nspec=15)
    with Advection(g, scal_adv=scheme, muscllimiter="MC") as a:
        def run(which, kchunk):
            a.set_tuning(kchunk=kchunk)
            outs = [torch.zeros_like(f) for f in which]
            a.batch_tendency(*vel, which, outs)
            a.stream_sync()
            return outs
        base = run(fields, 0)
        for kchunk in (5, 8):
            for n, o in enumerate(run(fields, kchunk)):
                assert torch.equal(o, base[n]), f"kchunk {kchunk} field {n}"
        for n in (0, 1, 2, 9, 16):
            assert torch.equal(run([fields[n]], 0)[0], base[n]), f"field {n} alone"


@pytest.mark.parametrize("dims", [(33, 9, 17), (100, 90, 40), (139, 117, 33), (200, 190, 41)])
def test_batch_momentum_chunk_lengths(cuda, dims):
    """The FP32 momenta against the FP64 operator, whose bits are the oracle's,
    where the dispatch takes one, two and more levels per work item.  Bound:
    2e-6 of the field maximum, as for the other batched momenta."""
    print(f"case batch_momentum_chunks {dims}", flush=True)
    g, vel, mom, fields = _batch(cuda, *dims, nspec=1)
    with Advection(g, scal_adv="weno") as a:
        ref = [torch.zeros(g.shape, dtype=torch.float64, device=cuda) for _ in range(3)]
        mom64, vel64 = [m.double() for m in mom], [x.double() for x in vel]  # alive until the sync
        a.qnadv_uvw(0, mom64, vel64, ref)
        ins = mom + fields
        outs = [torch.zeros_like(f) for f in ins]
        a.batch_tendency(*vel, ins, outs, momentum=True)
        a.stream_sync()
        I = g.interior()
        for c in range(3):
            want, got = -ref[c][I], outs[c].double()[I]
            assert float((got - want).abs().max() / want.abs().max()) <= 2e-6, f"component {c}"


@pytest.mark.parametrize("dims", [(6, 6, 8), (7, 45, 9), (251, 9, 8), (60, 0, 9)])
@pytest.mark.parametrize("sides", [("per", "per", "per", "per"), ("per", "per", "nnf", "ope"),
                                   ("ope", "nnf", "per", "per")])
def test_fill_of_many_fields(cuda, dims, sides):
    """Ghosts of a list of fields, more than one launch takes and one of them
    listed twice, next to the oracle's of each field."""
    print(f"case fill_many {dims} {sides}", flush=True)
    mx, my, nz = dims
    bcl = sides + ("nnf", "nnf")
    g = (case3d(mx, my, nz, bcl=bcl) if my else case2d(mx, nz, bcl=bcl))[0]
    rng = np.random.default_rng(3)
    xs = [rng.standard_normal(g.shape) for _ in range(11)]
    with Advection(g) as a:
        d = _dev(cuda, *xs)
        a.fill_halo(d[:4] + [d[2]] + d[4:])
        a.stream_sync()
    ora = Oracle(g)
    for n, x in enumerate(xs):
        ora.fill_scalar(x)
        assert np.array_equal(d[n].cpu().numpy(), x), f"field {n}"


@pytest.mark.parametrize("dims", [(6, 6, 8), (64, 9, 33), (130, 65, 40), (60, 0, 33)])
def test_advection_1d_of_many_fields(cuda, dims):
    """Lists longer than a launch takes, one tendency listed twice (both
    fields add to it in order) and one field that is its own tendency."""
    print(f"case advection_1d_many {dims}", flush=True)
    mx, my, nz = dims
    g = (case3d(mx, my, nz) if my else case2d(mx, nz))[0]
    rng = np.random.default_rng(8)
    w0 = rng.standard_normal(g.nz)
    qs = [rng.standard_normal(g.shape) for _ in range(11)]
    ts = [rng.standard_normal(g.shape) for _ in range(11)]
    dens = 1.0 + rng.random(g.shape)
    qi, ti = list(range(11)) + [3], list(range(11)) + [4]
    with Advection(g) as a:
        dq, dt, dd = _dev(cuda, *qs), _dev(cuda, *ts), _dev(cuda, dens)[0]
        a.advection_1d(w0, [dq[n] for n in qi] + [dq[0]], [dt[n] for n in ti] + [dq[0]], dens=dd)
        a.stream_sync()
    ora = Oracle(g)
    for n, m in zip(qi, ti):
        ora.advection_1d(w0, qs[n], ts[m], dref3=dens)
    own = qs[0].copy()
    ora.advection_1d(w0, qs[0], own, dref3=dens)
    for n in range(11):
        assert np.array_equal(dt[n].cpu().numpy(), ts[n]), f"tendency {n}"
    assert np.array_equal(dq[0].cpu().numpy(), own)


@pytest.mark.parametrize("dims", [(6, 6, 8), (17, 15, 65), (256, 9, 8), (300, 130, 9), (6, 0, 8), (600, 0, 130)])
def test_totalav_sizes(cuda, dims):
    """Mean and budget next to sums in extended precision; n additions of
    positive values are within n units of round-off, relatively."""
    print(f"case totalav {dims}", flush=True)
    mx, my, nz = dims
    g = (case3d(mx, my, nz) if my else case2d(mx, nz))[0]
    x = np.random.default_rng(5).random(g.shape)
    with Advection(g) as a:
        mean, budget = a.totalav(_dev(cuda, x)[0])
    inner = x[g.interior()].astype(np.longdouble)
    tol = inner.size * 2.0 ** -53
    assert abs(mean - float(inner.mean())) <= tol * mean
    want = float((inner.reshape(nz, -1).sum(axis=1) * np.asarray(g.dzw, dtype=np.longdouble)).sum())
    assert abs(budget - want) <= tol * want


@pytest.mark.parametrize("scheme", ["weno", "weno5", "muscl", "ppm", "quick"])
@pytest.mark.parametrize("dims", [(6, 6, 8), (45, 33, 20), (70, 0, 33)])
@pytest.mark.parametrize("overlap", [False, True])
def test_scalar_list_is_its_fields(cuda, scheme, dims, overlap):
    """A list of fields, longer than a launch takes, of both forms, has the bits
    of one call per field; so has one with a tendency that two fields add to
    and one that is a later field's input."""
    print(f"case scalar_list {scheme} {dims} overlap={overlap}", flush=True)
    mx, my, nz = dims
    g, u, v, w, _ = case3d(mx, my, nz) if my else case2d(mx, nz)
    rng = np.random.default_rng(6)
    n = 11
    arrays = [1.0 + rng.random(g.shape) for _ in range(2 * n)]
    form = [k % 2 for k in range(n)]
    with Advection(g, scal_adv=scheme, muscllimiter="MC") as a:
        vel = _dev(cuda, u, v, w)

        def run(split):
            d = _dev(cuda, *arrays)
            q, xs = d[:n], d[n:]
            if overlap:
                xs[5] = xs[2]
                xs[6] = q[7]
            if split:
                for f in range(n):
                    a.scalar_tendency(0.5, *vel, [q[f]], [xs[f]], adv=[form[f]])
            else:
                a.scalar_tendency(0.5, *vel, q, xs, adv=form)
            a.stream_sync()
            return d
        for k, (x, y) in enumerate(zip(run(False), run(True))):
            assert torch.equal(x, y), f"array {k}"


@pytest.mark.parametrize("scheme", ["weno", "weno5"])
@pytest.mark.parametrize("dims", [(6, 6, 8), (63, 7, 9), (64, 8, 33), (65, 9, 17), (17, 16, 10), (130, 33, 12),
                                  (64, 0, 9), (65, 0, 20)])
def test_adjoint_tile_edges(cuda, scheme, dims):
    """<lam, L' d> = <L'^T lam, d> with the oracle's tangent one cell around the
    tiles of both instances, to the 1e-13 of the other dot products; a second
    call writes the same qbar and adds to the velocity adjoints again."""
    print(f"case adjoint_edges {scheme} {dims}", flush=True)
    mx, my, nz = dims
    g, u, v, w, q = adjoint_case(my > 0, "gaussian", maxx=mx, maxy=my, nz=nz)
    rng = np.random.default_rng(72)
    dq, du, dv, dw = _dirs(g, rng, np.abs(q).mean())
    lam = _interior_only(g, rng.standard_normal(g.shape))
    _, tl = _tlm(Oracle(g, scal_adv=scheme), scheme)(q, dq, u, v, w, du, dv, dw)
    with Advection(g, scal_adv=scheme) as a:
        U, V, W, Q, L = _dev(cuda, u, v, w, q, lam)
        bars = [torch.zeros_like(Q) for _ in range(4)]
        a.adjoint_tendency(U, V, W, Q, L, *bars)
        a.stream_sync()
        once = [x.cpu().numpy() for x in bars]
        a.adjoint_tendency(U, V, W, Q, L, *bars)
        a.stream_sync()
        twice = [x.cpu().numpy() for x in bars]
    I = g.interior()
    assert np.all(once[0][~_mask(g)] == 0.0), "ghost entries of qbar were written"
    _check_dot([lam[I] * tl[I]], [d * x for d, x in zip((dq, du, dv, dw), once)])
    assert np.array_equal(once[0], twice[0])
    for n, (x, y) in enumerate(zip(once[1:], twice[1:])):
        scale = max(float(np.abs(x).max()), 1e-300)
        assert float(np.abs(y - 2.0 * x).max()) <= 4 * 2.0 ** -52 * scale, f"velocity {n}"


@pytest.mark.parametrize("counts", [(1, 7), (16, 3, 5), (1,), (18, 0, 2, 11, 4, 9)])
@pytest.mark.parametrize("dims", [(20, 16, 12), (190, 180, 30)])
def test_multi_field_split(cuda, counts, dims):
    """Field counts that the split over work items divides and does not, on
    subdomains too small to fill the chip and large enough, have the bits of
    a batch of each subdomain."""
    print(f"case multi_field_split {counts} {dims}", flush=True)
    advs, vels, fields, refs = [], [], [], []
    for d, nf in enumerate(counts):
        g, u, v, w, _ = case3d(*dims, seed=5 + d)
        rng = np.random.default_rng(40 + d)
        q = [cases.fill_periodic(g, np.exp(rng.standard_normal(g.shape))).astype(np.float32) for _ in range(nf)]
        vels.append(tuple(_dev(cuda, *(a.astype(np.float32) for a in (u, v, w)))))
        fields.append(_dev(cuda, *q))
        refs.append(_dev(cuda, *q))
        advs.append(Advection(g, scal_adv=("weno", "muscl", "weno5")[d % 3], muscllimiter="MC"))
    torch.cuda.synchronize()
    with MultiDomain(advs, vels, fields) as m:
        m.advance(_lib.INT_SSPRK3, 2, [0.5] * len(counts))
    for a, vel, fl, ref in zip(advs, vels, fields, refs):
        if ref:
            a.batch_advance(_lib.INT_SSPRK3, 2, 0.5, *vel, ref)
            a.stream_sync()
        for n, (x, y) in enumerate(zip(fl, ref)):
            assert torch.equal(x, y), f"field {n}"
        a.close()
