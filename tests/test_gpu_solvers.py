"""The interpolation solvers' device-resident control flow.

soint (ps_solver + ps_cgstep), soint2dc(prec=1) (ps_solver_prec) and sint
(ps_conjgrad) keep every scalar on the device, so the iterations are queued
without host round trips; one iteration is captured into a HIP graph and
replayed (SH_SOLVER_GRAPH=0 launches the kernels directly).  Checked here:
 * graph replays and direct launches give identical bits, on repeated calls
   (the graph is captured anew per call and replayed niter times, with the
   host's own work and synchronisations in between);
 * long solves on small problems, which stop early on the reference's
   tolerance tests, equal the FP32 oracle bit for bit (a missed or late
   stop would move the model);
 * the LDS-tiled i2 <-> i3 permutation of sint3d equals the plain one."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def canon(a):
    a = np.asarray(a, np.float32).ravel(order="F")
    return np.where(a == 0, np.float32(0), a).view(np.uint32)


def same(a, b, what=""):
    assert np.array_equal(canon(a), canon(b)), what


def F(a):
    return np.asarray(a, np.float32).ravel(order="F")


@pytest.fixture(scope="module")
def ps():
    import pyseistr_amd
    return pyseistr_amd


def _case3(shape, seed):
    rng = np.random.default_rng(seed)
    d = rng.standard_normal(shape).astype(np.float32)
    m = (rng.random(shape[1:]) > 0.6).astype(np.float32)[None] * np.ones(shape, np.float32)
    p = (0.6 * rng.standard_normal(shape)).astype(np.float32)
    q = (0.6 * rng.standard_normal(shape)).astype(np.float32)
    return (d * m).astype(np.float32), m, p, q


def _calls(ps, d, m, p, q):
    d2, m2, p2 = d[:, :, 0], m[:, :, 0], p[:, :, 0]
    return {
        "soint3d": lambda: ps.soint3dc(d, m, p, q, order=2, niter=12, report=True),
        "soint3d drift": lambda: ps.soint3dc(d, m, 3 * p, 3 * q, order=1, niter=7, drift=1, report=True),
        "soint2d": lambda: ps.soint2dc(d2, m2, p2, order=2, niter=12, report=True),
        "soint2d prec": lambda: ps.soint2dc(d2, m2, p2, order=2, niter=6, prec=1, report=True),
        "sint3d": lambda: ps.sint3dc(d, m, p, q, niter=9, eps=0.01, ns1=2, ns2=2, order1=2, order2=2, report=True),
        "sint2d": lambda: ps.sint2dc(d2, m2, p2, niter=9, eps=0.01, ns=3, order=2, report=True),
    }


def test_graph_replays_equal_direct_launches(ps, monkeypatch):
    d, m, p, q = _case3((48, 20, 16), 5)
    calls = _calls(ps, d, m, p, q)
    graph = {k: f() for k, f in calls.items()}
    again = {k: f() for k, f in calls.items()}
    monkeypatch.setenv("SH_SOLVER_GRAPH", "0")
    direct = {k: f() for k, f in calls.items()}
    monkeypatch.delenv("SH_SOLVER_GRAPH")
    for k in calls:
        print(k, "iterations", graph[k][1], flush=True)
        same(graph[k][0], direct[k][0], k)
        same(again[k][0], direct[k][0], k + " (second call)")
        assert graph[k][1] == direct[k][1] == again[k][1], k


@pytest.mark.parametrize("graph", ["1", "0"])
def test_long_solves_stop_like_the_oracle(ps, monkeypatch, graph):
    from oracle import oracle as O
    monkeypatch.setenv("SH_SOLVER_GRAPH", graph)
    rng = np.random.default_rng(17)
    n1, n2 = 24, 10
    d = rng.standard_normal((n1, n2)).astype(np.float32)
    m = (rng.random((n1, n2)) > 0.5).astype(np.float32)
    d = d * m
    p = (0.4 * rng.standard_normal((n1, n2))).astype(np.float32)
    s = (n1, n2)
    got, it = ps.sint2dc(d, m, p, niter=400, eps=0.01, ns=2, order=2, report=True)
    same(got, O.sint2d(F(d), F(m), F(p), s, niter=400, eps=0.01, ns=2, order=2), "sint2d")
    print("sint2d stopped after", it, flush=True)
    got, it2 = ps.soint2dc(d, m, p, order=2, niter=400, report=True)
    same(got, O.soint2d(F(d), F(m), F(p), s, order=2, niter=400), "soint2d")
    print("soint2d stopped after", it2, flush=True)
    got, it3 = ps.soint2dc(d, m, p, order=2, niter=300, prec=1, report=True)
    same(got, O.soint2d(F(d), F(m), F(p), s, order=2, niter=300, prec=1), "soint2d prec")
    print("soint2d prec stopped after", it3, flush=True)
    assert it < 400 or it2 < 400 or it3 < 300, "no solve stopped early; the test no longer covers the stop"


def test_tiled_permutation_equals_plain(ps, monkeypatch):
    d, m, p, q = _case3((40, 37, 45), 8)
    a = ps.sint3dc(d, m, p, q, niter=4, eps=0.01, ns1=2, ns2=1, order1=2, order2=2)
    monkeypatch.setenv("SH_PERMUTE_PLAIN", "1")
    b = ps.sint3dc(d, m, p, q, niter=4, eps=0.01, ns1=2, ns2=1, order1=2, order2=2)
    monkeypatch.delenv("SH_PERMUTE_PLAIN")
    same(a, b)


def test_spray2_prefetch_distances_identical(ps, monkeypatch):
    """The 2-D chain kernels' load rings at 8 and 16 samples ahead, and their
    buffer-resource and pointer accessors (SH_SPRAY2_BUF=0), give the same
    bits (spray, adjoint spray, somean2d and sint3d's shaping CG)."""
    d, m, p, q = _case3((60, 23, 9), 11)
    d2, p2 = d[:, :, 0], p[:, :, 0]
    rng = np.random.default_rng(3)
    u = rng.standard_normal(60 * 23 * 7).astype(np.float32)

    from pyseistr_amd import filters

    def calls():
        return [filters.pwspray2d(d2, p2, 3, 2, 0.01),
                filters.pwspray2d_adjoint(u, p2, 3, 2, 0.01, (60, 23)),
                ps.somean2dc(d, p, 4, 2, 0.01),
                ps.sint3dc(d, m, p, q, niter=5, eps=0.01, ns1=3, ns2=2, order1=2, order2=2)]

    out = {}
    for pf in ("8", "16"):
        monkeypatch.setenv("SH_SPRAY2_PF", pf)
        out[pf] = calls()
    monkeypatch.delenv("SH_SPRAY2_PF")
    monkeypatch.setenv("SH_SPRAY2_BUF", "0")
    out["ptr"] = calls()
    monkeypatch.delenv("SH_SPRAY2_BUF")
    for k, (a, b, c) in enumerate(zip(out["8"], out["16"], out["ptr"])):
        same(a, b, f"call {k}")
        same(a, c, f"call {k}, pointers")


@pytest.mark.parametrize("n1,n2,n3,ns,order", [(8, 1, 1, 2, 1), (9, 2, 3, 3, 2), (17, 5, 1, 6, 4), (31, 33, 2, 2, 3),
                                                (300, 17, 1, 4, 2), (515, 40, 1, 3, 2), (1030, 9, 1, 2, 3),
                                                (2100, 6, 1, 2, 2), (4000, 5, 1, 1, 1), (33, 70, 33, 2, 2)])
def test_chain_blocks_equal_single_threads(ps, monkeypatch, n1, n2, n3, ns, order):
    """The spray chains by blocks of threads and one thread each
    (SH_SPRAY2_PF selects the latter) give the same bits: one trace, fewer
    traces than radii, pieces and blocks that do not divide, traces too long
    for the blocks, and enough chains for the long pieces."""
    from pyseistr_amd import filters
    rng = np.random.default_rng(n1 + n2)
    d = rng.standard_normal((n1, n2, n3)).astype(np.float32)
    p = rng.uniform(-2, 2, (n1, n2, n3)).astype(np.float32)
    u = rng.standard_normal(n1 * n2 * (2 * ns + 1)).astype(np.float32)

    def calls():
        return [filters.pwspray2d(d[:, :, 0], p[:, :, 0], ns, order, 0.01),
                filters.pwspray2d_adjoint(u, p[:, :, 0], ns, order, 0.01, (n1, n2)),
                ps.somean2dc(d, p, ns, order, 0.01), ps.somean2dc(d, p, ns, order, 0.01, adj=1)]

    a = calls()
    monkeypatch.setenv("SH_SPRAY2_PF", "8")
    for k, (x, y) in enumerate(zip(a, calls())):
        same(x, y, f"call {k}")


@pytest.mark.parametrize("n1,n2,order", [(48, 1, 1), (49, 3, 1), (32, 40, 3), (35, 17, 4), (33, 70, 2), (65, 8, 2),
                                         (515, 9, 2), (97, 1100, 2)])
def test_chain_blocks_take_nothing_past_the_factors(ps, monkeypatch, n1, n2, order):
    """The block chains read whole groups of factor rows, past a trace's last
    one where its length is no multiple: with NaN all over the workspace
    before every call, the same bits as one thread per chain."""
    from pyseistr_amd import filters
    rng = np.random.default_rng(n1)
    d = rng.standard_normal((n1, n2)).astype(np.float32)
    p = rng.uniform(-2, 2, (n1, n2)).astype(np.float32)
    u = rng.standard_normal(n1 * n2 * 5).astype(np.float32)
    big = np.ones((600, 96), np.float32)

    def dirty():
        monkeypatch.setenv("SH_SPRAY2_PF", "8")  # writes every plane of the factors' buffer
        filters.pwspray2d(big, np.nan * big, 1, 4, 0.01)
        ps.somean2dc(big, np.nan * big, 1, 4, 0.01)
        monkeypatch.delenv("SH_SPRAY2_PF")

    calls = [lambda: filters.pwspray2d(d, p, 2, order, 0.01),
             lambda: filters.pwspray2d_adjoint(u, p, 2, order, 0.01, (n1, n2)),
             lambda: ps.somean2dc(d, p, 2, order, 0.01), lambda: ps.somean2dc(d, p, 2, order, 0.01, adj=1)]
    for k, f in enumerate(calls):
        dirty()
        a = f()
        monkeypatch.setenv("SH_SPRAY2_PF", "8")
        b = f()
        monkeypatch.delenv("SH_SPRAY2_PF")
        assert np.isfinite(a).all()
        same(a, b, f"call {k}")


@pytest.mark.parametrize("n1,n2,order", [(15000, 600, 2), (15150, 513, 1), (14600, 1024, 3), (14400, 600, 4), (15000, 3, 2),
                                         (15352, 2, 1), (16000, 2, 1), (130, 1100, 2), (300, 1100, 1)])
def test_chain_block_limits(ps, monkeypatch, n1, n2, order):
    """The longest traces that blocks of chains hold, with one spray and with
    two at once (the forward smoothing), and past them, where each chain has
    a thread; more than 2048 chains with several pieces a trace: the same
    bits as one thread per chain."""
    from pyseistr_amd import filters
    rng = np.random.default_rng(n1)
    d = rng.standard_normal((n1, n2)).astype(np.float32)
    p = rng.uniform(-2, 2, (n1, n2)).astype(np.float32)
    calls = [lambda: filters.pwspray2d(d, p, 1, order, 0.01), lambda: ps.somean2dc(d, p, 1, order, 0.01),
             lambda: ps.somean2dc(d, p, 1, order, 0.01, adj=1)]
    a = [f() for f in calls]
    monkeypatch.setenv("SH_SPRAY2_PF", "8")
    for k, f in enumerate(calls):
        same(a[k], f(), f"call {k}")


def test_spray3_level_paths_identical(ps, monkeypatch):
    """The 3-D spray levels give the same bits through buffer resources (the
    default) and through pointers (SH_SPRAY_BUF=0), at every prefetch
    distance (SH_SPRAY_PF) and with two-source slots grouped per thread
    (SH_SPRAY_GROUP): pwspray3d, somean3dc and somf3dc, PWD orders 1-3."""
    d, _, p, q = _case3((52, 17, 14), 31)

    def calls():
        return [ps.pwspray3d(d, p, q, 2, 3, 2, 0.01), ps.pwspray3d(d, p, q, 1, 2, 1, 0.05),
                ps.pwspray3d(d, p, q, 2, 1, 3, 0.01), ps.somean3dc(d, p, q, 3, 2, 0.01, 2),
                ps.somf3dc(d, p, q, 4, 4, 0.01, 2)]

    ref = calls()
    for env in ({"SH_SPRAY_BUF": "0"}, {"SH_SPRAY_PF": "4"}, {"SH_SPRAY_PF": "8"},
                {"SH_SPRAY_PF": "2", "SH_SPRAY_BUF": "0"}, {"SH_SPRAY_PF": "0"}, {"SH_SPRAY_GROUP": "2"}):
        for k, v in env.items():
            monkeypatch.setenv(k, v)
        for k, (a, b) in enumerate(zip(calls(), ref)):
            same(a, b, f"{env} call {k}")
        for k in env:
            monkeypatch.delenv(k)


def test_pwd_virtual_blocks_identical(ps, monkeypatch):
    """soint's operator kernels give the same bits with 1, 2 or 4 groups of
    samples per block (the partial-sum partition is unchanged), with and
    without drift, in 3-D and 2-D."""
    d, m, p, q = _case3((45, 19, 13), 21)
    d2, m2, p2 = d[:, :, 0], m[:, :, 0], p[:, :, 0]

    def calls():
        return [ps.soint3dc(d, m, p, q, order=2, niter=9, report=True),
                ps.soint3dc(d, m, 3 * p, 3 * q, order=1, niter=6, drift=1, report=True),
                ps.soint2dc(d2, m2, p2, order=3, niter=9, report=True)]

    out = {}
    for v in ("1", "2", "4"):
        monkeypatch.setenv("SH_PWD_V", v)
        out[v] = calls()
    monkeypatch.delenv("SH_PWD_V")
    for v in ("2", "4"):
        for k, ((a, ia), (b, ib)) in enumerate(zip(out["1"], out[v])):
            same(a, b, f"V={v} call {k}")
            assert ia == ib


@pytest.mark.parametrize("shape,order,njs", [((8, 2, 2), 1, (1, 1)), ((13, 5, 1), 3, (1, 1)), ((252, 3, 4), 2, (1, 3)),
                                             ((301, 19, 1), 2, (2, 1)), ((257, 7, 9), 6, (5, 1)),
                                             ((140, 5, 6), 2, (16, 16)), ((140, 5, 6), 2, (17, 1)),
                                             ((31, 150, 140), 2, (1, 2)), ((2100, 130, 7), 3, (1, 1))])
def test_pwd_ranges_equal_single_samples(ps, monkeypatch, shape, order, njs):
    """soint's operators over ranges of samples (one sum a block, the
    adjoint's products handed over in LDS) and one sum per 256 samples
    (SH_PWD_V): traces as long as a range's inner part and off it by some,
    stencils that reach over a trace's ends and to the rule's edge, more
    ranges than blocks.  Float operations agree; the order of the double sums
    may round a scalar to another float: a few 2^-24 an iteration."""
    d, m, p, q = _case3(shape, 41)
    if shape[2] == 1:
        d, m, p = d[:, :, 0], m[:, :, 0], p[:, :, 0]

    def call():
        if shape[2] == 1:
            return ps.soint2dc(d, m, p, order=order, njs=list(njs), niter=5, report=True)
        return ps.soint3dc(d, m, p, q, order=order, njs=list(njs), niter=5, report=True)

    new, it = call()
    monkeypatch.setenv("SH_PWD_V", "1")
    old, it0 = call()
    assert it == it0
    assert np.abs(new - old).max() <= 5 * 8 * 2.0**-24 * max(np.abs(old).max(), 1.0)


@pytest.mark.parametrize("shape,r,order", [((40, 9, 8), (1, 1), 1), ((33, 16, 16), (2, 3), 2), ((64, 17, 15), (3, 0), 2),
                                           ((24, 64, 33), (4, 4), 2), ((9, 3, 2), (4, 4), 1), ((30, 50, 41), (2, 2), 3)])
def test_levels_in_one_launch_equal_two(ps, monkeypatch, shape, r, order):
    """A spray level's one- and two-source nodes in one launch and in one
    each (SH_SPRAY_PF selects the latter): the same bits, from volumes
    smaller than the radius to a few blocks of traces."""
    d, _, p, q = _case3(shape, 5)
    kw = dict(order=order, eps=0.01, verb=0)
    new = [ps.somf3dc(d, p, q, r[0], r[1], **kw), ps.somean3dc(d, p, q, r[0], r[1], **kw)]
    monkeypatch.setenv("SH_SPRAY_PF", "6")
    old = [ps.somf3dc(d, p, q, r[0], r[1], **kw), ps.somean3dc(d, p, q, r[0], r[1], **kw)]
    for a, b in zip(new, old):
        same(a, b, str(shape))


@pytest.mark.parametrize("shape,rect", [((64, 32, 5), (5, 5, 5)), ((65, 33, 4), (2, 9, 3)), ((63, 31, 6), (9, 2, 2)),
                                        ((129, 7, 8), (5, 12, 2)), ((9, 40, 7), (13, 3, 4)), ((3, 2, 2), (4, 5, 2)),
                                        ((200, 95, 3), (20, 27, 2)), ((70, 40, 500), (3, 3, 3)), ((130, 70, 3), (40, 2, 2))])
def test_pair_of_axes_equals_single_axes(ps, monkeypatch, shape, rect):
    """The 3-D dip with axes 1 and 2 smoothed in one pass and one axis a pass
    (SH_SMOOTH_WAVE): planes of a tile, a sample more or less, smaller than
    the radii, radii to the largest that fits a tile, more tiles than blocks.
    The same operations in the same order: the same bits."""
    d = np.random.default_rng(sum(shape)).standard_normal(shape).astype(np.float32)
    mask = (np.random.default_rng(1).random(shape) > 0.1).astype(np.float32)
    for m in (None, mask):
        kw = dict(niter=2, liter=4, order=1, rect=list(rect), verb=0)
        if m is not None:
            kw["mask"] = m
        new = ps.dip3dc(d, **kw)
        monkeypatch.setenv("SH_SMOOTH_WAVE", "1")
        old = ps.dip3dc(d, **kw)
        monkeypatch.delenv("SH_SMOOTH_WAVE")
        for a, b in zip(new, old):
            same(a, b, str(shape))


@pytest.mark.parametrize("shape,rect,order,masked", [((8, 2), (3, 2), 1, False), ((31, 15), (1, 1), 2, False),
                                                     ((33, 17), (10, 20), 2, True), ((64, 32), (5, 1), 3, False),
                                                     ((130, 70), (1, 9), 2, True), ((515, 257), (10, 20), 2, False),
                                                     ((1030, 260), (20, 20), 1, False), ((1500, 600), (4, 4), 2, False)])
def test_resident_section_equals_launches(ps, monkeypatch, shape, rect, order, masked):
    """The dip of a 2-D section in one resident launch and as a sequence of
    launches (SH_SMOOTH_WAVE selects it): the float operations are the same,
    only double sums are added in another order, so the decisions agree and
    the dips differ by no more than a rounding of a step length moves them.
    Tile edges, radii past the section, one tile, every tile shape, and a
    section with too many tiles, which takes the launches either way."""
    rng = np.random.default_rng(shape[0])
    d = rng.standard_normal(shape).astype(np.float32)
    init = rng.uniform(-0.5, 0.5, shape).astype(np.float32)
    mask = (rng.random(shape) > 0.02).astype(np.float32) if masked else None
    kw = dict(niter=3, liter=12, order=order, rect=[rect[0], rect[1], 1], mask=mask, init=init, report=True)
    a, ra = ps.dip2dc(d, **kw)
    monkeypatch.setenv("SH_SMOOTH_WAVE", "1")
    b, rb = ps.dip2dc(d, **kw)
    assert ra["cg_iters"] == rb["cg_iters"] and ra["ls_step"] == rb["ls_step"]
    assert np.abs(a - b).max() <= 1e-6 * max(1.0, np.abs(b).max())


def test_resident_sections_from_threads(ps):
    """Sections estimated at once from several threads and streams, and into
    the data's own buffer, equal the ones estimated alone."""
    import threading

    import torch
    from pyseistr_amd import dip
    rng = np.random.default_rng(5)
    shapes = [(512, 512, 1), (300, 90, 1), (512, 512, 1), (128, 64, 1)]
    data = [torch.from_numpy(rng.standard_normal(a * b).astype(np.float32)).cuda() for a, b, _ in shapes]
    alone = [dip.dip_device(x, s, niter=2, rect=(6, 6, 1)).cpu().numpy() for x, s in zip(data, shapes)]
    got = [None] * len(shapes)

    def work(k):
        with torch.cuda.stream(torch.cuda.Stream()):
            for _ in range(3):
                got[k] = dip.dip_device(data[k], shapes[k], niter=2, rect=(6, 6, 1)).cpu().numpy()

    torch.cuda.synchronize()
    th = [threading.Thread(target=work, args=(k,)) for k in range(len(shapes))]
    [t.start() for t in th]
    [t.join() for t in th]
    for k, (x, y) in enumerate(zip(got, alone)):
        assert np.array_equal(x, y), k
    buf = data[1].clone()
    dip.dip_device(buf, shapes[1], niter=2, rect=(6, 6, 1), out=buf)
    assert np.array_equal(buf.cpu().numpy(), alone[1])


def test_section_whose_blocks_do_not_meet_is_an_error(ps, monkeypatch):
    """With no polls allowed (SH_DIP2_POLLS=0) every block of a section gives
    up at its first barrier: NaN dips, and an error from the call where it
    waits (drop-in, report, host pointers), else from the next sh_sync or
    estimate, once.  The estimates after it are as before."""
    import ctypes

    import torch
    from pyseistr_amd import _lib, dip
    shape = (130, 70, 1)
    d = np.random.default_rng(9).standard_normal(shape[:2]).astype(np.float32)
    x = _lib.to_device(d)
    kw = dict(niter=2, liter=6, rect=(6, 6, 1))
    good = dip.dip_device(x, shape, **kw).cpu().numpy()
    lib, ctx = _lib.load(), _lib.context()
    flat, out = F(d), np.empty(good.size, np.float32)
    args = [ctx, flat.ctypes.data_as(ctypes.c_void_p), None, None, *shape, 2, 6, 2, 0.01, 6, 6, 1,
            out.ctypes.data_as(ctypes.c_void_p), None]
    monkeypatch.setenv("SH_DIP2_POLLS", "0")
    with pytest.raises(_lib.SeistrError, match="did not meet"):
        ps.dip2dc(d, niter=2, liter=6, rect=[6, 6, 1])
    with pytest.raises(_lib.SeistrError, match="did not meet"):
        ps.dip2dc(d, niter=2, liter=6, rect=[6, 6, 1], report=True)
    assert lib.sh_ctx_set_flags(ctx, _lib.FLAG_HOST_PTRS) == 0
    rc = lib.sh_dip(*args)
    assert lib.sh_ctx_set_flags(ctx, 0) == 0
    assert rc == -4 and np.isnan(out).all()
    assert torch.isnan(dip.dip_device(x, shape, **kw)).all()
    assert lib.sh_sync(ctx) == -4 and lib.sh_sync(ctx) == 0
    dip.dip_device(x, shape, **kw)
    torch.cuda.synchronize()
    monkeypatch.delenv("SH_DIP2_POLLS")
    with pytest.raises(_lib.SeistrError, match="did not meet"):
        dip.dip_device(x, shape, **kw)
    assert np.array_equal(dip.dip_device(x, shape, **kw).cpu().numpy(), good)
    assert lib.sh_sync(ctx) == 0
