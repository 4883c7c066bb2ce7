"""Kernels and dispatch branches at the sizes where they can go wrong: tile
and launch edges, remainders, the smallest and largest of their range."""
import ctypes

import numpy as np
import pytest
import torch

from aquagpusph_amd import _lib

pytestmark = pytest.mark.gpu


def _stream():
    return ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)


def _dp(t):
    return ctypes.c_void_p(t.data_ptr())


def _dev(a):
    return torch.from_numpy(np.ascontiguousarray(a)).cuda()


@pytest.mark.parametrize("cells,cap", [(7, 7), (1000, 60_000_000),
                                       (524_288, 524_289),
                                       (1_100_003, 1_500_000)])
def test_ihoc_table_of_wide_grids(cuda, cells, cap):
    """The head-of-chain table of grids below, at and beyond one pass of the
    bounded launch (2048 x 256 cells), under a wider capacity: every cell in
    use is written, nothing past them."""
    rng = np.random.default_rng(cells)
    n = 5000
    ic = np.sort(rng.integers(0, cells, n)).astype(np.int32)
    ic[-1] = cells - 1
    want = np.full(cells, n, np.int32)
    first = np.r_[True, ic[1:] != ic[:-1]]
    want[ic[first]] = np.flatnonzero(first)
    ihoc = torch.full((cap,), -7, dtype=torch.int32, device="cuda")
    nc = _dev(np.array([cells, 1, 1, cells], np.int32))
    icd, st = _dev(ic), _dev(np.zeros(1, np.int32))
    _lib.call("aq_linklist_ihoc", _dp(icd), _dp(ihoc), n, _dp(nc), cap,
              _dp(st), _stream())
    got = ihoc.cpu().numpy()
    np.testing.assert_array_equal(got[:cells], want)
    assert (got[cells:] == -7).all()


# one workgroup's sizes, the tile sizes and their remainders, the line of the
# separate scan, and one to four passes (three write through the inverse)
@pytest.mark.parametrize("bits", [4, 16, 20, 32])
@pytest.mark.parametrize("n", [1, 63, 1024, 1025, 2049, 4097, 8192, 8193,
                               65536, 65537, 131072, 131073, 2_097_152,
                               2_097_153])
def test_radix_sort_edges(cuda, n, bits):
    """Keys, permutation and its inverse (with and without it asked for)
    against a stable sort of the digits in use, whole passes of 8 bits."""
    L = _lib.lib()
    rng = np.random.default_rng(n + bits)
    keys = rng.integers(0, 1 << 32, n, dtype=np.uint32)
    keys[n // 3: 2 * n // 3] &= np.uint32(0xFF00FF0F)
    mask = np.uint32((1 << (8 * ((bits + 7) // 8))) - 1)
    want = np.argsort(keys & mask, kind="stable").astype(np.uint32)
    size = int(L.aq_radix_sort_workspace(ctypes.c_uint32(n)))
    for with_inv in (True, False):
        kd = _dev(keys.view(np.int32))
        pd, iv = (torch.full((n + 1,), -7, dtype=torch.int32, device="cuda")
                  for _ in range(2))
        ws = torch.full((size + 64,), 123, dtype=torch.uint8, device="cuda")
        _lib.call("aq_radix_sort", _dp(kd), _dp(pd),
                  _dp(iv) if with_inv else None, n, bits, _dp(ws), _stream())
        np.testing.assert_array_equal(pd[:n].cpu().numpy(), want)
        np.testing.assert_array_equal(kd.cpu().numpy().view(np.uint32),
                                      keys[want])
        if with_inv:
            inv = np.empty(n, np.int32)
            inv[want] = np.arange(n)
            np.testing.assert_array_equal(iv[:n].cpu().numpy(), inv)
        assert int(pd[n]) == -7 and int(iv[n]) == -7
        assert bool((ws[size:] == 123).all())


@pytest.mark.parametrize("n,most", [(65536, 65537), (65000, 65600),
                                    (2_097_152, 2_097_153),
                                    (2_097_000, 2_100_000)])
def test_radix_sort_in_a_larger_sorts_workspace(cuda, n, most):
    """A sort of n keys in the workspace of a sort of `most`, across the
    lines where the tiles double: nothing behind the workspace is written."""
    f = _lib.lib().aq_radix_sort_workspace
    # allocated so that even a sort that overran it would stay in bounds
    size, room = f(most), max(f(most), f(n)) + 64
    keys = np.random.default_rng(n).integers(0, 1 << 20, n, dtype=np.uint32)
    want = np.argsort(keys, kind="stable").astype(np.uint32)
    kd = _dev(keys.view(np.int32))
    pd, iv = (torch.empty(n, dtype=torch.int32, device="cuda")
              for _ in range(2))
    ws = torch.full((room,), 123, dtype=torch.uint8, device="cuda")
    _lib.call("aq_radix_sort", _dp(kd), _dp(pd), _dp(iv), n, 20, _dp(ws),
              _stream())
    np.testing.assert_array_equal(pd.cpu().numpy(), want)
    assert bool((ws[size:] == 123).all())


def _run(tmp_path, case, presets, tag, steps=3):
    from aquagpusph_amd import casefiles
    from aquagpusph_amd.sim import Simulation
    d = tmp_path / tag
    sim = Simulation(casefiles.write_case(case, str(d), presets=presets,
                                          load=False), case["dims"])
    casefiles.upload(sim, case)
    sim.step(steps, graph=True)
    out = {k: sim.get(k) for k in ("id", "r", "u", "rho", "p", "dudt",
                                   "drhodt", "grad_p", "lap_u", "div_u",
                                   "lap_p", "shepard")}
    sim.close()
    return out


def _stir(case, seed):
    """Displaced fluid particles and a velocity field (a flow out of its
    lattice order, so that cells hold uneven numbers of particles)."""
    rng = np.random.default_rng(seed)
    fl, D = case["imove"] == 1, case["dims"]
    n = int(fl.sum())
    case["r"][fl, :D] += 0.3 * case["params"]["dr"] * rng.uniform(
        -1, 1, (n, D))
    case["u"][fl, :D] = rng.normal(0, 0.3, (n, D))
    return case


def _spray(case, seed, factor):
    """The fluid scattered over `factor` times its extent along each axis, in
    a wider domain box: cells of one or a few particles."""
    rng = np.random.default_rng(seed)
    fl, D = case["imove"] == 1, case["dims"]
    x = case["r"][fl, :D]
    lo, ext = x.min(0), x.max(0) - x.min(0)
    case["r"][fl, :D] = lo + ext * (
        0.5 + factor * (rng.random(x.shape) - 0.5))
    P = case["params"]
    P["domain_min"] = [a - factor * e for a, e in zip(P["domain_min"], ext)]
    P["domain_max"] = [a + factor * e for a, e in zip(P["domain_max"], ext)]
    P["dt_min"] = 1e-9
    case["u"][fl, :D] = rng.normal(0, 0.3, x.shape)
    return case


# aq_walk_lanes: the walks and the lanes per particle of their launches
FLUID, KAHAN, ELEMENTS, LES = range(4)


def _lanes(kernel, case, periodic=0):
    return _lib.lib().aq_walk_lanes(kernel, case["dims"], case["N"], periodic)


# sizes on both sides of the lines between 16 and 4 lanes per particle
@pytest.mark.parametrize("dims,dr,kind", [
    (2, 0.06, "wall"), (2, 0.011, "wall"), (2, 0.0028, "wall"),
    (2, 0.011, "kahan"), (2, 0.0031, "kahan"), (3, 0.05, "wall"),
    (3, 0.031, "wall"), (3, 0.0187, "wall"), (3, 0.031, "kahan"),
    (3, 0.0187, "kahan"), (2, 1 / 41, "box"), (2, 1 / 160, "box"),
    (3, 1 / 17, "box"), (3, 1 / 33, "box"), (2, 0.011, "morris"),
    (3, 0.031, "morris"), (2, 0.011, "spray"), (2, 0.0028, "spray"),
    (3, 0.031, "spray"), (3, 0.0187, "spray"), (3, 0.0187, "cloud")])
def test_lanes_per_particle_are_bit_identical(cuda, tmp_path, monkeypatch,
                                              dims, dr, kind):
    """The fused walk with 4 or 16 lanes per particle against the one-lane
    walk (asked for by an explicit grid), bit for bit: every sum takes the
    same terms in the same order."""
    from aquagpusph_amd import casefiles, cases
    pres = casefiles.PBI_PRESETS
    if kind == "box":
        case = cases.periodic_box(dims, int(round(1 / dr)), seed=3)
        pres = casefiles.PPER_PRESETS
    else:
        case = cases.dam_break(dims, dr)
        if kind == "kahan":
            pres = pres + ("resources/Presets/precision.xml",)
    assert _lanes(KAHAN if kind == "kahan" else FLUID, case,
                  kind == "box") > 1
    if kind in ("spray", "cloud"):
        case = _spray(case, 7, 5.0 if kind == "spray" else 2.0)
    else:
        case = _stir(case, 7)
    extra = ""
    if kind == "morris":
        from aquagpusph_amd import casefiles as cf
        orig = cf.write_case
        extra = ('    <Definitions><Define name="__LAP_FORMULATION__" '
                 'value="2" evaluate="false"/></Definitions>')
        monkeypatch.setattr(
            cf, "write_case",
            lambda *a, **k: orig(*a, **dict(k, extra_xml=extra)))
    got = _run(tmp_path, case, pres, "lanes")
    monkeypatch.setenv("AQ_WALK_BLOCKS", "300")
    want = _run(tmp_path, case, pres, "one")
    for k in want:
        np.testing.assert_array_equal(got[k], want[k], err_msg=k)


# just above the lines to one lane per particle
@pytest.mark.parametrize("dr,kahan", [(0.0083, False), (0.01, True)])
def test_one_lane_walk_matches_oracle(cuda, tmp_path, dr, kahan):
    """The fused walk with one lane per particle, as launched by default, and
    the element kernels over its near list against the oracle's float32
    walk, bit for bit: 3D dam breaks of 252,576 and, with compensated sums,
    153,600 particles."""
    from aquagpusph_amd import casefiles, cases
    from aquagpusph_amd.sim import Simulation
    from oracle import pipeline as op
    case = _stir(cases.dam_break(3, dr), 13)
    assert _lanes(KAHAN if kahan else FLUID, case) == 1
    pres = casefiles.PBI_PRESETS
    if kahan:
        pres = pres + ("resources/Presets/precision.xml",)
    sim = Simulation(casefiles.write_case(case, str(tmp_path), load=False,
                                          presets=pres), 3)
    casefiles.upload(sim, case)
    o = op.OracleSim(case, precision=kahan)
    for _ in range(2):
        o.step()
    sim.step(2)
    for k in ("id", "r", "u", "rho", "p", "dudt", "drhodt", "shepard",
              "grad_p", "lap_u", "div_u", "lap_p"):
        np.testing.assert_array_equal(
            sim.get(k).ravel().view(o.f[k].dtype), o.f[k].ravel(), err_msg=k)
    sim.close()


# 16, 4 and one lane per particle in a periodic box, one with relaxed math
@pytest.mark.parametrize("dims,n,relaxed", [
    (2, 60, False), (2, 150, False), (3, 17, False), (3, 30, False),
    (3, 64, False), (2, 60, True), (3, 30, True)])
def test_fluid_pairs_at_the_edge_of_the_support(cuda, tmp_path, dims, n,
                                                relaxed):
    """Neighbours of zero density up to 2e-5 beyond the support radius (the
    walk's distance test accepts some of them): they add nothing, so the
    sums of the particle they are out of reach of stay finite."""
    from aquagpusph_amd import casefiles, cases
    from aquagpusph_amd.sim import Simulation
    case = cases.periodic_box(dims, n, seed=2)
    # a row of particles i, 11 apart, and their neighbours j, 4 spacings on
    x, dr, h = case["r"], case["params"]["dr"], case["params"]["h"]
    x[:, :dims] = x[:, :dims].astype(np.float32)
    key = np.lexsort(np.round(x[:, :dims] / dr, 2).T)
    row = key[:n] if dims == 2 else key[n * (n // 2):][:n]
    i = row[np.arange(2, n - 6, 11)]
    j = row[np.arange(2, n - 6, 11) + 4]
    assert np.allclose(x[j, 0] - x[i, 0], 4 * dr, rtol=1e-4)
    assert np.allclose(2 * h, 4 * dr, rtol=1e-6)
    x[j] = x[i]
    x[j, 0] += 2 * h * (1 + np.linspace(2e-6, 2e-5, len(i)))
    case["rho"][j] = 0
    case["u"][:] = 0  # the predictor leaves the positions
    kw = {}
    if relaxed:
        kw["extra_xml"] = ('<Settings><Device platform="0" device="0" '
                           'compile_flags="-cl-fast-relaxed-math" />'
                           '</Settings>')
    sim = Simulation(casefiles.write_case(
        case, str(tmp_path), load=False, presets=casefiles.PPER_PRESETS,
        **kw), dims)
    casefiles.upload(sim, case)
    sim.step(1)
    ids = sim.get("id")
    mine = np.isin(ids, i)
    for k in ("grad_p", "lap_u", "div_u", "lap_p", "shepard"):
        assert np.isfinite(sim.get(k).reshape(len(ids), -1)[mine]).all(), k
    sim.close()


# element kernels: 16 lanes per owner below 100 k (2D) / 600 k (3D)
# particles, 4 above (one for BI Interactions above 1 M in 3D, the last case);
# wall edges and corners hold more than one group
@pytest.mark.parametrize("dims,dr,hfac,lanes", [
    (2, 0.06, 2.0, 16), (2, 0.011, 2.0, 16), (2, 0.00135, 2.0, 4),
    (3, 0.05, 2.0, 16), (3, 0.031, 3.3, 16), (3, 0.0061, 2.0, 16),
    (3, 0.0059, 2.0, 4), (3, 0.005, 2.0, 4)])
def test_element_groups_match_one_lane_walks(cuda, tmp_path, monkeypatch,
                                             dims, dr, hfac, lanes):
    """The boundary-integral element kernels with 4 or 16 lanes per owner
    over the owner, wet and near lists against one lane per owner over every
    cell (AQ_BI_WALK=cells), bit for bit."""
    from aquagpusph_amd import casefiles, cases
    case = _stir(cases.dam_break(dims, dr, hfac=hfac), 11)
    assert _lanes(ELEMENTS, case) == lanes
    got = _run(tmp_path, case, casefiles.PBI_PRESETS, "groups", 2)
    monkeypatch.setenv("AQ_BI_WALK", "cells")
    want = _run(tmp_path, case, casefiles.PBI_PRESETS, "cells", 2)
    for k in want:
        np.testing.assert_array_equal(got[k], want[k], err_msg=k)


@pytest.mark.parametrize("dims,n,lanes", [(2, 23, 16), (2, 150, 4),
                                          (3, 17, 16), (3, 30, 4),
                                          (3, 63, 1)])
def test_les_groups_match_oracle(cuda, tmp_path, dims, n, lanes):
    """The LES gradient and viscous term (periodic box, Smagorinsky) with 16
    and with 4 lanes per particle (2D above 16 k, 3D above 24 k particles)
    and with one (3D above 250 k: 63^3 = 250,047) against the oracle's
    float32 walk, bit for bit."""
    from aquagpusph_amd import casefiles, cases
    from aquagpusph_amd.sim import Simulation
    from oracle import pipeline as op
    case = _stir(cases.periodic_box(dims, n), 5)
    assert _lanes(LES, case, 1) == lanes
    sim = Simulation(casefiles.write_case(
        case, str(tmp_path), load=False, presets=casefiles.PPER_PRESETS +
        ("resources/Presets/cfd/LES-smagorinsky.xml",)), dims)
    casefiles.upload(sim, case)
    o = op.OracleSim(case, bi=False, domain=False, les={"Cs": 0.15},
                     periodic=case["params"]["periodic"])
    steps = 2 if n < 60 or dims == 2 else 1
    for _ in range(steps):
        o.step()
    sim.step(steps)
    for k in ("grad_u", "nu_t", "dudt", "u", "r"):
        np.testing.assert_array_equal(sim.get(k).ravel(), o.f[k].ravel(),
                                      err_msg=k)
    sim.close()


@pytest.mark.parametrize("dims,dr,lanes,spray", [
    (2, 0.011, 16, 0), (3, 0.0187, 4, 0), (3, 0.0083, 1, 0), (3, 0.031, 16, 4),
    (3, 0.0187, 4, 2), (3, 0.0187, 4, 5)])
def test_les_walls_match_oracle(cuda, tmp_path, dims, dr, lanes, spray):
    """The LES kernels of a dam break with its walls (no periodic images), as
    a flow and as a spray, against the oracle's float32 walk, bit for bit."""
    from aquagpusph_amd import casefiles, cases
    from aquagpusph_amd.sim import Simulation
    from oracle import pipeline as op
    case = cases.dam_break(dims, dr)
    case = _spray(case, 5, spray) if spray else _stir(case, 5)
    assert _lanes(LES, case) == lanes
    sim = Simulation(casefiles.write_case(
        case, str(tmp_path), load=False, presets=casefiles.PBI_PRESETS +
        ("resources/Presets/cfd/LES-smagorinsky.xml",)), dims)
    casefiles.upload(sim, case)
    o = op.OracleSim(case, les={"Cs": 0.15})
    o.step()
    sim.step(1)
    for k in ("grad_u", "nu_t", "dudt", "u", "r"):
        np.testing.assert_array_equal(sim.get(k).ravel(), o.f[k].ravel(),
                                      err_msg=k)
    sim.close()


@pytest.mark.parametrize("dims,n", [(2, 23), (2, 150), (3, 17), (3, 30),
                                    (3, 63)])
def test_les_gradient_of_an_empty_particle(cuda, tmp_path, dims, n):
    """A particle of zero density is no neighbour of itself: its own velocity
    gradient stays finite (16, 4 and one lane per particle)."""
    from aquagpusph_amd import casefiles, cases
    from aquagpusph_amd.sim import Simulation
    case = _stir(cases.periodic_box(dims, n), 5)
    empty = np.array([case["N"] // 2])
    case["rho"][empty] = 0
    sim = Simulation(casefiles.write_case(
        case, str(tmp_path), load=False, presets=casefiles.PPER_PRESETS +
        ("resources/Presets/cfd/LES-smagorinsky.xml",)), dims)
    casefiles.upload(sim, case)
    sim.step(1)
    g, ids = sim.get("grad_u").reshape(case["N"], -1), sim.get("id")
    sim.close()
    mine = np.isin(ids, empty)
    assert mine.sum() == empty.size
    assert np.isfinite(g[mine]).all()


def _abi_linklist(dims, r, h):
    """Device link-list (icell, ihoc, n_cells) of the positions r, and the
    permutation that sorts them."""
    n, vs = r.shape
    extent = (r.max(0) - r.min(0))[:dims]
    cap = int(np.prod(np.floor(extent / (2 * h)) + 8))
    d = {k: _dev(v) for k, v in dict(
        lo=np.zeros(vs, np.float32), hi=np.zeros(vs, np.float32),
        sup=np.float32([2]), h=np.float32([h]), nc=np.zeros(4, np.int32),
        ic=np.zeros(n, np.int32), pu=np.zeros(n, np.int32),
        ps=np.zeros(n, np.int32), hoc=np.zeros(cap, np.int32),
        st=np.zeros(1, np.int32), r=r).items()}
    ws = torch.empty(int(_lib.lib().aq_linklist_workspace(
        ctypes.c_uint32(n))), dtype=torch.uint8, device="cuda")
    _lib.call("aq_linklist", dims, _dp(d["r"]), n, _dp(d["lo"]),
              _dp(d["hi"]), _dp(d["sup"]), _dp(d["h"]), _dp(d["nc"]),
              _dp(d["ic"]), _dp(d["pu"]), _dp(d["ps"]), _dp(d["hoc"]), cap,
              _dp(d["st"]), _dp(ws), _stream())
    assert int(d["st"].item()) == 0
    return d, d["pu"].cpu().numpy()


def _check_abi_pair_kernels(rng, dims, lap, h, r, u, rho, m, p, im):
    """aq_shepard (both variants), aq_interactions and aq_lapp against the
    oracle's float32 walk, bit for bit, accumulating onto given values."""
    from oracle import pipeline as op
    f32 = lambda a: np.ascontiguousarray(a, np.float32)  # noqa: E731
    n, vs = r.shape
    d, perm = _abi_linklist(dims, r, h)
    r, u, rho, m, p, im = (np.ascontiguousarray(a[perm])
                           for a in (r, u, rho, m, p, im))
    H = op.definition(h)
    CONW = op.definition(1.0 / float(h) ** dims)
    CONF = op.definition(1.0 / float(h) ** (dims + 2))
    D = _lib.Defs(H, CONW, CONF, float(dims), lap)
    g = {k: _dev(v) for k, v in dict(r=r, u=u, rho=rho, m=m, p=p,
                                     im=im).items()}
    ll = (n, _dp(d["ic"]), _dp(d["hoc"]), _dp(d["nc"]), D)
    hic, hhoc, hnc = (d[k].cpu().numpy() for k in ("ic", "hoc", "nc"))
    oll = tuple(op._p(a) for a in (hic, hhoc, hnc))
    fn = lambda k: getattr(op.lib(), "orc_%s_f32_%dd" % (k, dims))  # noqa
    cf, cu = ctypes.c_float, ctypes.c_uint
    for cfd in (0, 1):
        want = f32(rng.normal(0, 1, n))
        got = _dev(want)
        _lib.call("aq_shepard", dims, _dp(g["im"]), _dp(g["r"]),
                  _dp(g["rho"]), _dp(g["m"]), _dp(got), *ll, cfd, _stream())
        fn("shepard")(op._p(im), op._p(r), op._p(rho), op._p(m),
                      op._p(want), cu(n), *oll, cf(H), cf(CONW),
                      ctypes.c_int(cfd))
        np.testing.assert_array_equal(got.cpu().numpy(), want)
    w = [f32(rng.normal(0, 1, (n, vs))), f32(rng.normal(0, 1, (n, vs))),
         f32(rng.normal(0, 1, n)), f32(rng.normal(0, 1, n))]
    t = [_dev(a) for a in w]
    _lib.call("aq_interactions", dims, _dp(g["im"]), _dp(g["r"]),
              _dp(g["u"]), _dp(g["rho"]), _dp(g["m"]), _dp(g["p"]),
              *(_dp(a) for a in t[:3]), *ll, _stream())
    _lib.call("aq_lapp", dims, _dp(g["im"]), _dp(g["r"]), _dp(g["rho"]),
              _dp(g["m"]), _dp(g["p"]), _dp(t[3]), *ll, _stream())
    fn("interactions")(op._p(im), op._p(r), op._p(u), op._p(rho), op._p(m),
                       op._p(p), *(op._p(a) for a in w[:3]), cu(n), *oll,
                       cf(H), cf(CONF), ctypes.c_int(lap))
    fn("lapp")(op._p(im), op._p(r), op._p(rho), op._p(m), op._p(p),
               op._p(w[3]), cu(n), *oll, cf(H), cf(CONF))
    for a, b in zip(t, w):
        np.testing.assert_array_equal(a.cpu().numpy(), b)


# single particles, cells of more than 64, around the lines of the launch by
# groups alone (16384) and between 16 and 4 lanes per particle (50000), and
# about one particle per cell beyond them (the per-particle form)
@pytest.mark.parametrize("dims,n,cell,lap", [
    (2, 1, 3, 1), (2, 65, 3, 2), (2, 16384, 4, 1), (2, 16385, 4, 2),
    (2, 30011, 12, 1), (3, 1, 3, 1), (3, 63, 2, 1), (3, 5000, 6, 2),
    (3, 16384, 4, 1), (3, 20011, 4, 1), (2, 50000, 4, 2), (2, 50001, 5, 1),
    (3, 50001, 4, 2), (2, 16385, 1, 1), (2, 60001, 1, 2), (3, 50001, 1, 1),
    (3, 110003, 1, 2)])
def test_abi_pair_kernels_match_oracle(cuda, dims, n, cell, lap):
    """The pair kernels of the C ABI on disordered particles of every kind,
    about cell^dims of them per cell."""
    rng = np.random.default_rng(n + dims)
    vs = 2 if dims == 2 else 4
    side = max(1.0, (n / cell ** dims) ** (1 / dims))  # in cells
    h = np.float32(0.05)
    r = np.zeros((n, vs), np.float32)
    r[:, :dims] = rng.uniform(0, side * 2 * h, (n, dims))
    u = np.zeros_like(r)
    u[:, :dims] = rng.normal(0, 1, (n, dims))
    f32 = lambda a: np.ascontiguousarray(a, np.float32)  # noqa: E731
    rho = f32(1000 + rng.normal(0, 5, n))
    m = f32(rng.uniform(0.5, 1.5, n))
    p = f32(rng.normal(0, 100, n))
    im = rng.choice(np.array([1, 1, 1, 1, 1, 0, -3, 2, 3, -256], np.int32), n)
    _check_abi_pair_kernels(rng, dims, lap, h, r, u, rho, m, p, im)


@pytest.mark.parametrize("dims,sites,lap", [(2, 60, 1), (2, 2100, 2),
                                            (3, 60, 2), (3, 2100, 1)])
def test_abi_pairs_at_the_edge_of_the_support(cuda, dims, sites, lap):
    """Pairs within 4e-5 of the support radius (the walk's distance test
    accepts some of those beyond it) whose neighbour has an infinite, NaN or
    zero field, and particles that meet themselves with such a field: a pair
    out of reach, or a particle with itself, adds nothing.  Each site is a
    bunch of 24 particles and a broken one a support radius away; 60 sites
    run with 16 lanes per particle, 2100 with 4."""
    rng = np.random.default_rng(sites + dims)
    vs = 2 if dims == 2 else 4
    h = np.float32(0.05)
    k, B = np.arange(sites), 25
    n = sites * B
    r = np.zeros((sites, B, vs))
    r[:, :, 0] = (0.61 * (k % 20))[:, None]
    r[:, :, 1] = (0.61 * (k // 20))[:, None]
    r[:, :-1, 1] += 1e-3 * h * rng.uniform(-1, 1, (sites, B - 1))
    r[:, -1, 0] += 2 * h * (1 + 4e-5 * rng.uniform(-1, 1, sites))
    r = np.ascontiguousarray(r.reshape(n, vs), np.float32)
    u = np.zeros_like(r)
    u[:, :dims] = rng.normal(0, 1, (n, dims))
    f32 = lambda a: np.ascontiguousarray(a, np.float32)  # noqa: E731
    rho, m, p = (f32(1000 + rng.normal(0, 5, n)),
                 f32(rng.uniform(0.5, 1.5, n)), f32(rng.normal(0, 100, n)))
    last = np.arange(sites) * B + B - 1
    for kind, (a, v) in enumerate([(p, np.inf), (p, np.nan), (rho, 0),
                                   (m, np.inf), (u, np.nan)]):
        a[last[kind::5]] = v
    _check_abi_pair_kernels(rng, dims, lap, h, r, u, rho, m, p,
                            np.ones(n, np.int32))
