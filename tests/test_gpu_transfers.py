"""Region transfers through the C ABI vs the oracle: bit-exact."""
import numpy as np
import pytest

import oracle
from helpers import okeys
from test_oracle_transfers import setup

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    import bigdft_hip
    assert torch.cuda.is_available(), "GPU tests need a HIP device"
    c = bigdft_hip.Context(0)
    yield c
    c.close()


def dev(a):
    return torch.from_numpy(np.ascontiguousarray(a)).cuda()


def test_transfers_batch_bit_exact(ctx):
    cases = [setup(s) for s in (1, 2, 3)]
    glob = cases[0][0]
    ng = cases[0][2]
    g = ctx.region(glob)
    locs = [ctx.region(c[1]) for c in cases]
    ns = np.array([c[4] for c in cases], dtype=np.int32)
    rng = np.random.default_rng(7)
    gpsi = rng.standard_normal((3, glob.ncoef))
    lnc = [c[1].ncoef for c in cases]
    loff = np.concatenate([[0], np.cumsum(lnc)[:-1]])
    lpsi = torch.full((sum(lnc),), np.nan, dtype=torch.float64, device="cuda")
    ctx.psi_to_locreg(g, locs, ns, dev(gpsi), lpsi)
    got = lpsi.cpu().numpy()
    for i, (gl, lo, _, nl, nsi) in enumerate(cases):
        exp = oracle.psi_to_locreg2(nl, ng, nsi, okeys(lo), okeys(gl), gpsi[i])
        assert np.array_equal(got[loff[i]:loff[i] + lnc[i]], exp)
    # local -> global onto a global array holding other values
    lsrc = rng.standard_normal(sum(lnc))
    base = rng.standard_normal((3, glob.ncoef))
    gout = dev(base)
    ctx.locreg_to_psi(g, locs, ns, dev(lsrc), gout)
    got = gout.cpu().numpy()
    for i, (gl, lo, _, nl, nsi) in enumerate(cases):
        exp, n = oracle.lpsi_to_global2(nl, ng, nsi, okeys(lo), okeys(gl),
                                        lsrc[loff[i]:loff[i] + lnc[i]], base[i])
        assert n == lo.nvctr_c + lo.nvctr_f
        assert np.array_equal(got[i], exp)
    for l in locs:
        l.close()
    g.close()


def test_locreg_to_psi_rejects_points_outside(ctx):
    import bigdft_hip
    from bigdft_hip.descriptors import region_from_grids
    glob, loc, ng, nl, ns = setup(4)
    full = np.ones(tuple(x + 1 for x in nl), dtype=bool)
    loc2 = region_from_grids("F", nl, loc.hgrid, full, np.zeros_like(full))
    g, l = ctx.region(glob), ctx.region(loc2)
    gpsi = torch.zeros(glob.ncoef, dtype=torch.float64, device="cuda")
    lp = dev(np.ones(loc2.ncoef))
    with pytest.raises(bigdft_hip.BigDFTError, match="DESC"):
        ctx.locreg_to_psi(g, [l], np.array(ns, dtype=np.int32), lp, gpsi)
    # the other direction fills the missing points with zeros
    out = torch.full((loc2.ncoef,), np.nan, dtype=torch.float64, device="cuda")
    ctx.psi_to_locreg(g, [l], np.array(ns, dtype=np.int32),
                      dev(np.arange(glob.ncoef, dtype=np.float64)), out)
    assert not torch.isnan(out).any()
    l.close()
    g.close()


def test_transfers_sphere_batch_round_trip(ctx):
    """48 compressed spheres of a 64^3 free global box (tiles of several
    thousand coefficients, coarse and fine parts of many sizes): local
    orbitals equal the oracle's psi_to_locreg2, and writing them back into
    a zero global orbital restores exactly the points each sphere holds"""
    from bigdft_hip import workloads
    from bigdft_hip.descriptors import dense_region
    sb = workloads.sphere_batch(48, 5, n_glob=63, device="cuda")
    regs = sb["regions"]
    ng = (63, 63, 63)
    glob = dense_region("F", ng, (0.4,) * 3)
    g = ctx.region(glob)
    cache = {}
    lrs = [cache.setdefault(id(r), ctx.region(r)) for r in regs]
    ns = np.array(sb["nl"], dtype=np.int32).reshape(-1, 3)
    rng = np.random.default_rng(8)
    gh = rng.standard_normal((len(regs), glob.ncoef))
    goff = np.arange(len(regs), dtype=np.int64) * glob.ncoef
    loff = sb["psi_off"]
    lp = torch.full_like(sb["psi"], np.nan)
    ctx.psi_to_locreg(g, lrs, ns, dev(gh.ravel()), lp, goff=goff, loff=loff)
    lh = lp.cpu().numpy()
    gk = okeys(glob)
    for i in rng.choice(len(regs), 5, replace=False):
        r = regs[i]
        exp = oracle.psi_to_locreg2(r.n, ng, sb["nl"][i], okeys(r), gk, gh[i])
        assert np.array_equal(lh[loff[i]:loff[i] + r.ncoef], exp)
    back = torch.zeros(len(regs) * glob.ncoef, dtype=torch.float64, device="cuda")
    ctx.locreg_to_psi(g, lrs, ns, lp, back, loff=loff, goff=goff)
    bh = back.cpu().numpy().reshape(len(regs), -1)
    for i in range(len(regs)):
        nz = bh[i] != 0.0
        assert np.array_equal(bh[i][nz], gh[i][nz])
        assert nz.sum() == regs[i].ncoef
    # the same batch again (descriptors reused) on other values
    lp2 = torch.full_like(sb["psi"], np.nan)
    ctx.psi_to_locreg(g, lrs, ns, dev(2.0 * gh.ravel()), lp2, goff=goff, loff=loff)
    assert np.array_equal(lp2.cpu().numpy(), 2.0 * lh)
    for l in cache.values():
        l.close()
    g.close()


@pytest.mark.parametrize("nl", [(0, 0, 0), (1, 0, 2), (2, 6, 0), (0, 7, 8), (8, 1, 6), (15, 16, 3),
                                (16, 14, 17)], ids=lambda v: "x".join(map(str, v)))
def test_transfers_box_extents(ctx, nl):
    """local grids of one point, powers of two and their neighbours along x
    and y (the split of a grid index), a tile's remainder in the coarse and
    the fine part, a local box without fine points: bit-exact"""
    from bigdft_hip.descriptors import dense_region, region_from_grids
    h = (0.4, 0.4, 0.4)
    ng = (19, 18, 20)
    glob = dense_region("F", ng, h)
    rng = np.random.default_rng(sum(nl) + 3)
    cm = rng.random(tuple(x + 1 for x in nl)) < 0.7
    cm[0, 0, 0] = True
    locs = [dense_region("F", nl, h), region_from_grids("F", nl, h, cm, np.zeros_like(cm)),
            region_from_grids("F", nl, h, cm, cm & (rng.random(cm.shape) < 0.5))]
    ns = [[int(rng.integers(0, ng[d] - nl[d] + 1)) for d in range(3)] for _ in locs]
    g, lrs = ctx.region(glob), [ctx.region(r) for r in locs]
    gpsi = rng.standard_normal((3, glob.ncoef))
    lnc = [r.ncoef for r in locs]
    lp = torch.full((sum(lnc),), np.nan, dtype=torch.float64, device="cuda")
    ctx.psi_to_locreg(g, lrs, np.array(ns, dtype=np.int32), dev(gpsi), lp)
    base = rng.standard_normal((3, glob.ncoef))
    back = dev(base)
    ctx.locreg_to_psi(g, lrs, np.array(ns, dtype=np.int32), lp, back)
    got = np.split(lp.cpu().numpy(), np.cumsum(lnc)[:-1])
    for i, r in enumerate(locs):
        exp = oracle.psi_to_locreg2(nl, ng, ns[i], okeys(r), okeys(glob), gpsi[i])
        assert np.array_equal(got[i], exp)
        full, n = oracle.lpsi_to_global2(nl, ng, ns[i], okeys(r), okeys(glob), exp, base[i])
        assert n == r.nvctr_c + r.nvctr_f
        assert np.array_equal(back[i].cpu().numpy(), full)
    for lr in lrs:
        lr.close()
    g.close()


def test_missing_points_are_counted_on_every_call(ctx):
    """the count of points without a counterpart is that of the one call:
    failing, good and failing calls in turn, on one batch and on another"""
    import bigdft_hip
    from bigdft_hip.descriptors import dense_region, region_from_grids
    h = (0.4, 0.4, 0.4)
    full = np.ones((9, 8, 7), dtype=bool)
    holes = full.copy()
    holes[2:4, 3, 1:6] = False
    glob = region_from_grids("F", (8, 7, 6), h, holes, np.zeros_like(full))
    g = ctx.region(glob)
    small, big = dense_region("F", (1, 1, 1), h), dense_region("F", (8, 7, 6), h)
    for loc, ns, missing in [(big, (0, 0, 0), (9 * 8 * 7 * 2) - glob.nvctr_c),
                             (small, (2, 3, 1), 12), (big, (0, 0, 0), 9 * 8 * 7 * 2 - glob.nvctr_c)]:
        lr = ctx.region(loc)
        lp = dev(np.ones(loc.ncoef))
        out = torch.zeros(glob.ncoef, dtype=torch.float64, device="cuda")
        for _ in range(2):
            with pytest.raises(bigdft_hip.BigDFTError, match=f"{missing} local points"):
                ctx.locreg_to_psi(g, [lr], np.array(ns, dtype=np.int32), lp, out)
            # to the local region the missing points are zeros, not an error
            ctx.psi_to_locreg(g, [lr], np.array(ns, dtype=np.int32), out, lp)
            lp.fill_(1.0)
        lr.close()
    ok = region_from_grids("F", (8, 7, 6), h, holes, np.zeros_like(full))
    lr = ctx.region(ok)
    out = torch.zeros(glob.ncoef, dtype=torch.float64, device="cuda")
    ctx.locreg_to_psi(g, [lr], np.zeros(3, dtype=np.int32), dev(np.ones(ok.ncoef)), out)
    assert torch.equal(out, torch.ones_like(out))
    lr.close()
    g.close()


def test_alternating_sets_of_regions(ctx):
    """calls that alternate between sets of regions (new descriptors each time,
    of more and of fewer regions), gathers before the context's first scatter,
    and a set with missing points among them: bit-exact, every count its own"""
    import bigdft_hip
    from bigdft_hip.descriptors import region_from_grids
    h = (0.4, 0.4, 0.4)
    ng = (12, 11, 10)
    cm = np.ones(tuple(x + 1 for x in ng), dtype=bool)
    cm[10:, 9:, 8:] = False
    glob = region_from_grids("F", ng, h, cm, np.zeros_like(cm))
    own = bigdft_hip.Context(0)
    g = own.region(glob)
    # regions of coarse points only, as the global one
    full = {n: np.ones(tuple(x + 1 for x in n), dtype=bool) for n in ((3, 2, 4), (6, 5, 3))}
    small, big = (region_from_grids("F", n, h, m, np.zeros_like(m)) for n, m in full.items())
    hl = {id(r): own.region(r) for r in (small, big)}
    # 24 regions of one kind, 5 of both, 1 that reaches into the hole
    sets = [([small] * 24, [(i % 5, i % 4, i % 3) for i in range(24)], 0),
            ([big, small, big, small, small], [(0, 1, 2), (5, 4, 2), (3, 3, 3), (1, 0, 0), (6, 6, 3)], 0),
            ([big], [(6, 6, 7)], 27)]
    rng = np.random.default_rng(17)
    psi = rng.standard_normal(glob.ncoef)
    want = []
    for regs, ns, miss in sets:
        want.append(np.concatenate([oracle.psi_to_locreg2(r.n, ng, list(o), okeys(r), okeys(glob), psi)
                                    for r, o in zip(regs, ns)]))
    d_psi = dev(psi)
    goff = {k: np.zeros(len(s[0]), dtype=np.int64) for k, s in enumerate(sets)}
    for scatter in (False, True, True):
        for _ in range(2):
            for k, (regs, ns, miss) in enumerate(sets):
                lrs = [hl[id(r)] for r in regs]
                o = np.array(ns, dtype=np.int32)
                lp = torch.full((want[k].size,), np.nan, dtype=torch.float64, device="cuda")
                own.psi_to_locreg(g, lrs, o, d_psi, lp, goff=goff[k])
                assert np.array_equal(lp.cpu().numpy(), want[k])
                if not scatter:
                    continue
                back = d_psi.clone()
                if miss:
                    with pytest.raises(bigdft_hip.BigDFTError, match=f"^.*{miss} local points"):
                        own.locreg_to_psi(g, lrs, o, lp, back, goff=goff[k])
                else:
                    own.locreg_to_psi(g, lrs, o, lp, back, goff=goff[k])
                assert torch.equal(back, d_psi)
    for l in hl.values():
        l.close()
    g.close()
    own.close()
