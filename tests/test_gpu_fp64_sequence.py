"""The FP64 plane-fused sequence (bdft_fp64.hip) against the oracle at the
edges of its launch rules: extents where an in-plane work-group changes its
shape (8, 12 or 16 waves, one or more per CU), where the planes stop fitting
and x and y go as tiles of 64 lines, where those lines stop fitting, z lines where the z kernels change their
chunks per wave or stop fitting, and coarse planes that leave a partly empty
last run of 16 columns.

FP64 sums of at most 2 x 31 (G, G^T) and 58 (kinetic) products per axis, in
another order than the oracle's: 1e-12 per element (guarded relative) and in
the energies, the bar of every FP64 parity test.
"""
import numpy as np
import pytest

import oracle
from helpers import dense_region, okeys, random_pot, random_psi, region_from_grids, rel_err

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

TOL = 1e-12


@pytest.fixture(scope="module")
def ctx():
    import bigdft_hip
    assert torch.cuda.is_available(), "GPU tests need a HIP device"
    c = bigdft_hip.Context(0)
    yield c
    c.close()


def dev(a):
    return torch.from_numpy(np.ascontiguousarray(a)).cuda()


def lr_dims(reg):
    """real-space grid points per axis"""
    extra = 0 if reg.geocode == "P" else 29
    return tuple(2 * (x + 1) + extra for x in reg.n)


# n (coarse points - 1) per axis
SIZES = [("P", n) for n in [
    (0, 0, 0), (15, 0, 4), (4, 3, 1), (7, 15, 2), (16, 16, 1),   # column runs, 4 waves
    (22, 22, 1), (31, 31, 0), (38, 41, 1),                       # 8 waves
    (48, 48, 1), (49, 49, 1), (54, 55, 0),                       # half a CU's LDS, 12 waves
    (63, 63, 0), (69, 69, 0), (70, 70, 0), (84, 40, 0),          # 16 waves, beyond
    (1, 2, 31), (2, 1, 32), (1, 2, 47), (2, 1, 48), (1, 2, 63), (2, 1, 64),
    (1, 0, 158), (0, 1, 159), (71, 70, 3), (127, 128, 0), (156, 90, 0), (90, 156, 0),
    (157, 90, 0), (90, 157, 0)]] + [("F", n) for n in [
    (0, 0, 0), (4, 3, 1), (15, 16, 1), (20, 21, 0), (25, 26, 1),
    (35, 35, 0), (36, 36, 0), (40, 30, 1), (55, 55, 0), (56, 57, 0),
    (1, 2, 31), (2, 1, 32), (1, 2, 48), (2, 1, 64), (1, 0, 144), (0, 1, 146),
    (57, 63, 2), (141, 60, 0), (60, 141, 0), (142, 60, 0), (60, 142, 0)]]


@pytest.mark.parametrize("geo,n", SIZES, ids=[f"{g}{n[0]}x{n[1]}x{n[2]}" for g, n in SIZES])
@pytest.mark.parametrize("keys", ["dense", "sparse"])
def test_launch_edges_match_the_oracle(ctx, geo, n, keys):
    reg = dense_region(geo, n, (0.45, 0.4, 0.5))
    if keys == "sparse":   # half the coarse points, a quarter of them fine
        rng = np.random.default_rng(sum(n) + 5)
        lg = rng.random(tuple(x + 1 for x in n)) < 0.5
        lg[0, 0, 0] = True
        fine = lg & (rng.random(lg.shape) < 0.5)
        fine[0, 0, 0] = True
        reg = region_from_grids(geo, n, (0.45, 0.4, 0.5), lg, fine)
    print(f"case {geo} n={n} {keys} nvctr=({reg.nvctr_c},{reg.nvctr_f})", flush=True)
    norb = 2
    psi, h0 = random_psi(reg, norb, 31), random_psi(reg, norb, 32)
    pot = random_pot(reg, 33)
    lr = ctx.region(reg)
    d_h = dev(h0)
    ek = torch.zeros(norb, dtype=torch.float64, device="cuda")
    ep = torch.zeros_like(ek)
    ctx.locham(lr, dev(pot), dev(psi), d_h, ek, ep)
    ctx.sync()
    lr.close()
    ho, eo, po = oracle.locham(geo, reg.n, reg.nfl, reg.nfu, reg.hgrid, okeys(reg), pot, psi, h0)
    # element by element against the sums' own scale: an isolated point's
    # value may cancel to far below the terms it is made of
    h = d_h.cpu().numpy()
    assert np.abs(h - ho).max() < TOL * np.abs(ho - h0).max()
    if keys == "dense":
        assert rel_err(h - h0, ho - h0) < TOL
    assert rel_err(ek.cpu().numpy(), eo) < TOL
    assert rel_err(ep.cpu().numpy(), po) < TOL


def test_large_and_small_boxes_of_one_batch(ctx):
    """boxes beyond LDS planes and small ones in one batch (all on x and y
    lines): a potential box smaller than the grid and offset from it, and a
    confining term, each against the oracle; the batch through the fixed
    device array gives the same bits"""
    import bigdft_hip
    regs = [dense_region("P", (71, 72, 2), (0.45, 0.4, 0.5)),
            dense_region("F", (5, 4, 3), (0.45, 0.4, 0.5)),
            dense_region("P", (40, 90, 3), (0.45, 0.4, 0.5))]
    psi = [random_psi(r, 1, 61 + i)[0] for i, r in enumerate(regs)]
    dims = [lr_dims(r) for r in regs]
    assert [r.n_isf for r in regs] == [int(np.prod(d)) for d in dims]
    # potential boxes: four points less on x and y, offset by one and two
    pots = [random_pot(r, 71 + i).reshape(d[::-1]) for i, (r, d) in enumerate(zip(regs, dims))]
    sub = [np.ascontiguousarray(p[:, 2:-2, 1:-3]) for p in pots]
    full = [np.zeros_like(p) for p in pots]
    for a, b in zip(full, sub):
        a[:, 2:-2, 1:-3] = b
    lrs = [ctx.region(r) for r in regs]

    def run(ps, conf=None, fixed=False, **kw):
        off = np.cumsum([0] + [p.size for p in ps[:-1]])
        po = np.cumsum([0] + [p.size for p in psi[:-1]])
        x = dev(np.concatenate(psi))
        h = torch.zeros_like(x)
        ek = torch.zeros(3, dtype=torch.float64, device="cuda")
        ep = torch.zeros_like(ek)
        fn = ctx.locham_batch_fixed if fixed else ctx.locham_batch
        if conf is not None:
            kw["conf"] = conf
        fn(lrs, dev(np.concatenate([p.ravel() for p in ps])), x, h, ek, ep, pot_off=off,
           psi_off=po, **kw)
        ctx.sync()
        return np.split(h.cpu().numpy(), po[1:]), ek.cpu().numpy(), ep.cpu().numpy()

    kw = dict(potdim=np.array([s.shape[::-1] for s in sub], dtype=np.int32).ravel(),
              ishift=np.array([(1, 2, 0)] * 3, dtype=np.int32).ravel())
    confs = [dict(args=(4, 1e-4, (0.2,) * 3, (3.0, 4.0, 1.0), (-1, -15, 2)[i:i + 1] * 3))
             for i in range(3)]
    gconf = np.concatenate([bigdft_hip.confpot(*c["args"]) for c in confs])
    got = [run(sub, **kw), run(pots, conf=gconf)]
    for g, ps, cf in ((got[0], full, None), (got[1], pots, confs)):
        for i, r in enumerate(regs):
            print(f"box {i} conf={cf is not None}", flush=True)
            h, ek, ep = oracle.locham(r.geocode, r.n, r.nfl, r.nfu, r.hgrid, okeys(r),
                                      ps[i].ravel(), psi[i][None],
                                      conf=oracle.confpot(*cf[i]["args"]) if cf else None)
            assert np.abs(g[0][i] - h[0]).max() < TOL * np.abs(h).max()
            assert rel_err(g[1][i:i + 1], ek) < TOL
            assert rel_err(g[2][i:i + 1], ep) < TOL
    fx = run(sub, fixed=True, **kw)
    for a, b in zip(fx[0], got[0][0]):
        assert np.array_equal(a, b)
    assert np.array_equal(fx[1], got[0][1]) and np.array_equal(fx[2], got[0][2])
    for lr in lrs:
        lr.close()


# (geo, n, spins): one work-group shape each, groups of one spin that are
# full, partly full, single or (all orbitals spin down) missing
DENSITY = [("P", (0, 0, 0), [0]), ("P", (4, 3, 5), [1, 0, 1]), ("P", (22, 21, 2), [1, 1]),
           ("P", (38, 41, 0), [0, 1, 0, 0, 1]), ("P", (48, 48, 1), [0, 0]),
           ("P", (49, 50, 0), [1, 0]), ("P", (63, 63, 0), [0, 1]),
           ("F", (4, 3, 1), [0, 1]), ("F", (20, 21, 0), [1]), ("F", (35, 35, 0), [0, 1]),
           ("F", (40, 30, 1), [0]), ("P", (1, 2, 2), [k % 2 for k in range(2000)])]


@pytest.mark.parametrize("geo,n,spin", DENSITY,
                         ids=[f"{g}{n[0]}x{n[1]}x{n[2]}-{len(s)}" for g, n, s in DENSITY])
def test_density_launch_edges_match_the_oracle(ctx, geo, n, spin):
    """rho += hfac psir^2 within 1e-12 of max rho: every point sums squares
    of sums of 3 x 31 products"""
    reg = dense_region(geo, n, (0.45, 0.4, 0.5))
    norb = len(spin)
    print(f"case {geo} n={n} norb={norb}", flush=True)
    psi = random_psi(reg, norb, 41)
    hfac = np.random.default_rng(42).uniform(0.1, 2.0, norb)
    rho0 = np.random.default_rng(43).uniform(0.0, 1.0, (2, reg.n_isf))
    lr = ctx.region(reg)
    rho = dev(rho0)
    ctx.density(lr, dev(psi), hfac, rho, spin=spin, nspin=2)
    lr.close()
    want = oracle.density(geo, reg.n, reg.nfl, reg.nfu, okeys(reg), psi, hfac, spin, 2)
    got = rho.cpu().numpy() - rho0
    assert np.abs(got - want.reshape(2, -1)).max() < TOL * max(np.abs(want).max(), 1.0)


@pytest.mark.parametrize("geo,n", [("P", (4, 3, 5)), ("P", (22, 22, 32)), ("P", (48, 48, 1)),
                                   ("P", (49, 49, 2)), ("P", (63, 63, 0)), ("P", (70, 69, 0)),
                                   ("F", (15, 16, 48)), ("F", (35, 36, 1)), ("F", (49, 50, 1)),
                                   ("F", (2, 1, 144)), ("F", (2, 1, 147))],
                         ids=lambda v: v if isinstance(v, str) else "x".join(map(str, v)))
@pytest.mark.parametrize("keys", ["dense", "sparse"])
def test_precond_launch_edges_match_the_oracle(ctx, geo, n, keys):
    """three steps, every update in another kernel than the oracle's: 1e-10
    of max|x|, the bar of the preconditioner's parity tests"""
    reg = dense_region(geo, n, (0.45, 0.4, 0.5))
    if keys == "sparse":
        rng = np.random.default_rng(sum(n) + 7)
        lg = rng.random(tuple(x + 1 for x in n)) < 0.6
        lg[0, 0, 0] = True
        reg = region_from_grids(geo, n, (0.45, 0.4, 0.5), lg, lg & (rng.random(lg.shape) < 0.5))
    print(f"case {geo} n={n} {keys}", flush=True)
    b, x0 = random_psi(reg, 2, 51), 0.05 * random_psi(reg, 2, 52)
    cpr = [0.3, 0.9]
    lr = ctx.region(reg)
    x = dev(x0.ravel())
    ctx.precond_cg([lr, lr], cpr, 3, x, dev(b.ravel()))
    got = x.cpu().numpy().reshape(2, -1)
    lr.close()
    for i in range(2):
        want = oracle.precond_cg(geo, reg.n, reg.hgrid, cpr[i], 3, okeys(reg), x0[i], b[i])
        assert np.abs(got[i] - want).max() < 1e-10 * np.abs(want).max()


@pytest.mark.parametrize("geo,n,norb", [("P", (0, 0, 0), 1), ("P", (15, 15, 15), 1),
                                        ("P", (22, 20, 21), 6), ("P", (31, 31, 3), 5),
                                        ("P", (32, 31, 9), 2), ("P", (40, 44, 2), 2),
                                        ("P", (54, 53, 1), 1), ("P", (55, 54, 1), 1),
                                        ("P", (3, 3, 0), 5461), ("P", (3, 3, 0), 5462),
                                        ("F", (3, 2, 47), 2), ("F", (9, 8, 7), 11)],
                         ids=lambda v: v if isinstance(v, str) else str(v).replace(", ", "x"))
def test_small_batches_share_the_first_launch(ctx, geo, n, norb):
    """small batches run G_z and the x-y kinetic in one launch of 256, 512 or
    768 threads, up to 16384 work-groups (5461 of the three of a 4x4x1 box);
    with stage timing on every kernel has its own: the same sums in the same
    order, so the same bits"""
    reg = dense_region(geo, n, (0.45, 0.4, 0.5))
    print(f"case {geo} n={n} norb={norb}", flush=True)
    psi, pot, lr = dev(random_psi(reg, norb, 81)), dev(random_pot(reg, 82)), ctx.region(reg)

    def run():
        h = torch.zeros_like(psi)
        ek = torch.zeros(norb, dtype=torch.float64, device="cuda")
        ep = torch.zeros_like(ek)
        ctx.locham(lr, pot, psi, h, ek, ep)
        ctx.sync()
        return h, ek, ep
    one = run()
    ctx.profile(True)
    try:
        each = run()
    finally:
        ctx.profile_read()
        ctx.profile(False)
    lr.close()
    for a, b in zip(one, each):
        assert torch.equal(a, b)


@pytest.mark.parametrize("copies", [1, 2, 5])
def test_uneven_batches_in_one_and_in_several_launches(ctx, copies):
    """boxes of every launch shape in one batch: few planes (one launch per
    pass), more than 512 (potential pass by shape), against the oracle, and
    cut into chunks the same bits"""
    ns = [(4, 3, 5), (20, 17, 9), (27, 30, 12), (36, 35, 20), (49, 51, 7)]
    regs = [dense_region("F", n, (0.4, 0.4, 0.4)) for n in ns]
    psi = [random_psi(r, 1, 91 + i)[0] for i, r in enumerate(regs)]
    pots = [random_pot(r, 95 + i) for i, r in enumerate(regs)]
    lrs = [ctx.region(r) for r in regs] * copies
    po = np.cumsum([0] + [p.size for p in pots])
    so = np.cumsum([0] + [p.size for p in psi * copies])
    x, pot = dev(np.concatenate(psi * copies)), dev(np.concatenate(pots))

    def run():
        h = torch.zeros_like(x)
        ek = torch.zeros(len(lrs), dtype=torch.float64, device="cuda")
        ep = torch.zeros_like(ek)
        ctx.locham_batch(lrs, pot, x, h, ek, ep, pot_off=np.tile(po[:-1], copies), psi_off=so[:-1])
        ctx.sync()
        return h.cpu().numpy(), ek.cpu().numpy(), ep.cpu().numpy()
    got = run()
    ctx.set_option("chunk_mb", 8)
    try:
        cut = run()
    finally:
        ctx.set_option("chunk_mb", 0)
    for a, b in zip(got, cut):
        assert np.array_equal(a, b)
    h = np.split(got[0], so[1:-1])
    for i, r in enumerate(regs):
        print(f"box {i} of {copies}", flush=True)
        ho, eo, vo = oracle.locham("F", r.n, r.nfl, r.nfu, r.hgrid, okeys(r), pots[i],
                                   psi[i][None])
        for k in range(i, len(lrs), len(regs)):
            assert np.abs(h[k] - ho[0]).max() < TOL * np.abs(ho).max()
            assert rel_err(got[1][k:k + 1], eo) < TOL
            assert rel_err(got[2][k:k + 1], vo) < TOL
    for lr in lrs[:len(regs)]:
        lr.close()


@pytest.mark.parametrize("how", ["chunks", "fixed"])
def test_parts_of_a_batch_sum_ekin_as_the_whole(ctx, how):
    """z lines of 40, 60 and 75 points in one batch: the back pass's launch
    shape decides which chunks of a line one wave sums, so a part that holds
    only shorter lines than the batch's longest has to run the whole batch's
    shape.  The same bits as in one piece, for cuts into parts of one length,
    of two, and of all"""
    # 1.2, 1.8 and 2.3 MB of grids a box: chunks of 4 MiB, or 128 MiB of the fixed array
    times = 1 if how == "chunks" else 30
    regs = {k: dense_region("P", (12, 8, k - 1), (0.45, 0.4, 0.5)) for k in (40, 60, 75)}
    lr = {k: ctx.region(r) for k, r in regs.items()}
    psi = {k: random_psi(r, 1, 101 + k)[0] for k, r in regs.items()}
    pot = {k: random_pot(r, 103 + k) for k, r in regs.items()}
    for lens in ([40] * 7 + [60] * 3, [60, 40, 40, 40, 40, 40, 40], [75, 40, 40, 60, 60, 60, 40]):
        print(f"case {how} {lens}", flush=True)
        lens = [k for k in lens for _ in range(times)]
        so = np.cumsum([0] + [psi[k].size for k in lens])[:-1]
        po = np.cumsum([0] + [pot[k].size for k in lens])[:-1]
        x, v = dev(np.concatenate([psi[k] for k in lens])), dev(np.concatenate([pot[k] for k in lens]))

        def run(fn):
            h = torch.zeros_like(x)
            ek = torch.zeros(len(lens), dtype=torch.float64, device="cuda")
            ep = torch.zeros_like(ek)
            fn([lr[k] for k in lens], v, x, h, ek, ep, pot_off=po, psi_off=so)
            ctx.sync()
            return h, ek, ep
        whole = run(ctx.locham_batch)
        if how == "chunks":
            ctx.set_option("chunk_mb", 4)
            try:
                cut = run(ctx.locham_batch)
            finally:
                ctx.set_option("chunk_mb", 0)
        else:
            cut = run(ctx.locham_batch_fixed)
        for a, b in zip(whole, cut):
            assert torch.equal(a, b)
    for l in lr.values():
        l.close()


# z lines beyond the 64-line tiles (159 periodic, 145 free points), in tiles of
# 32: the first lengths, a partly empty last tile of eight columns, lines whose
# last pair of chunks is half empty, the longest lines of the library
LONG = [("P", n) for n in [(1, 0, 159), (4, 3, 160), (2, 2, 163), (6, 5, 199), (3, 4, 255)]] + \
       [("F", n) for n in [(0, 1, 145), (4, 3, 146), (5, 2, 180), (3, 4, 255)]]
LONG_IDS = [f"{g}{n[0]}x{n[1]}x{n[2]}" for g, n in LONG]


@pytest.mark.parametrize("geo,n", LONG, ids=LONG_IDS)
@pytest.mark.parametrize("keys", ["dense", "sparse"])
def test_long_z_lines_match_the_oracle(ctx, geo, n, keys):
    test_launch_edges_match_the_oracle(ctx, geo, n, keys)
    if keys == "dense":
        test_density_launch_edges_match_the_oracle(ctx, geo, n, [0, 1, 1])
    test_precond_launch_edges_match_the_oracle(ctx, geo, n, keys)


def test_long_z_lines_keep_the_plane_kernels(ctx):
    """a batch with z lines of 20, 60, 200 and 256 points: boxes in z-line tiles of
    both widths, no line pass runs; against the oracle, and the same bits in
    chunks and in the fixed device array.  Then the preconditioner on it."""
    ns = [("P", (23, 23, 199)), ("F", (7, 5, 19)), ("F", (4, 5, 255)), ("P", (5, 3, 59)),
          ("F", (9, 7, 150))]
    regs = [dense_region(g, n, (0.45, 0.4, 0.5)) for g, n in ns]
    psi = [random_psi(r, 1, 121 + i)[0] for i, r in enumerate(regs)]
    pots = [random_pot(r, 131 + i) for i, r in enumerate(regs)]
    lrs = [ctx.region(r) for r in regs]
    po = np.cumsum([0] + [p.size for p in pots])
    so = np.cumsum([0] + [p.size for p in psi])
    x, pot = dev(np.concatenate(psi)), dev(np.concatenate(pots))

    def run(fn):
        h = torch.zeros_like(x)
        ek = torch.zeros(len(lrs), dtype=torch.float64, device="cuda")
        ep = torch.zeros_like(ek)
        fn(lrs, pot, x, h, ek, ep, pot_off=po[:-1], psi_off=so[:-1])
        ctx.sync()
        return h.cpu().numpy(), ek.cpu().numpy(), ep.cpu().numpy()
    got = run(ctx.locham_batch)
    ctx.set_option("chunk_mb", 4)
    try:
        cut = run(ctx.locham_batch)
    finally:
        ctx.set_option("chunk_mb", 0)
    for other in (cut, run(ctx.locham_batch_fixed)):
        for a, b in zip(got, other):
            assert np.array_equal(a, b)
    ctx.profile(True)
    try:
        run(ctx.locham_batch)
        stages = ctx.profile_read()[0]
    finally:
        ctx.profile(False)
    busy = sorted(stages, key=stages.get)[-4:]
    assert set(busy) == {"z_grow", "xy_kin", "xy_pot", "z_back"}, stages
    h = np.split(got[0], so[1:-1])
    cpr, b = [0.3, 0.5, 0.7, 0.9, 1.1], [random_psi(r, 1, 141 + i)[0] for i, r in enumerate(regs)]
    x0 = 0.05 * x
    ctx.precond_cg(lrs, cpr, 3, x0, dev(np.concatenate(b)), psi_off=so[:-1])
    x0 = np.split(x0.cpu().numpy(), so[1:-1])
    for i, r in enumerate(regs):
        print(f"box {i}", flush=True)
        ho, eo, vo = oracle.locham(r.geocode, r.n, r.nfl, r.nfu, r.hgrid, okeys(r), pots[i],
                                   psi[i][None])
        assert np.abs(h[i] - ho[0]).max() < TOL * np.abs(ho).max()
        assert rel_err(got[1][i:i + 1], eo) < TOL
        assert rel_err(got[2][i:i + 1], vo) < TOL
        want = oracle.precond_cg(r.geocode, r.n, r.hgrid, cpr[i], 3, okeys(r), 0.05 * psi[i], b[i])
        assert np.abs(x0[i] - want).max() < 1e-10 * np.abs(want).max()
    for lr in lrs:
        lr.close()


@pytest.mark.parametrize("geo", ["P", "F"])
@pytest.mark.parametrize("n3", [1, 2, 7, 8, 9, 15, 16, 17])
def test_flat_batches_match_the_oracle(ctx, geo, n3):
    """more than 512 z-line tiles of short lines: the back pass runs two or four
    waves per work-group (up to 8 or 16 points), in the chunks of a cut batch
    (one box of 27 tiles or so each) eight; the same bits"""
    reg = dense_region(geo, (19, 20, n3 - 1), (0.45, 0.4, 0.5))
    norb = 20
    print(f"case {geo} n3={n3}", flush=True)
    psi, h0, pot = random_psi(reg, norb, 151), random_psi(reg, norb, 152), random_pot(reg, 153)
    lr = ctx.region(reg)
    d_pot, d_psi = dev(pot), dev(psi)

    def run():
        h = dev(h0)
        ek = torch.zeros(norb, dtype=torch.float64, device="cuda")
        ep = torch.zeros_like(ek)
        ctx.locham(lr, d_pot, d_psi, h, ek, ep)
        ctx.sync()
        return h.cpu().numpy(), ek.cpu().numpy(), ep.cpu().numpy()
    got = run()
    ctx.set_option("chunk_mb", 1)
    try:
        cut = run()
    finally:
        ctx.set_option("chunk_mb", 0)
    for a, b in zip(got, cut):
        assert np.array_equal(a, b)
    ho, eo, po = oracle.locham(geo, reg.n, reg.nfl, reg.nfu, reg.hgrid, okeys(reg), pot, psi, h0)
    assert np.abs(got[0] - ho).max() < TOL * np.abs(ho - h0).max()
    assert rel_err(got[1], eo) < TOL
    assert rel_err(got[2], po) < TOL
    lr.close()


# group sizes of every kind: all orbitals in one group, several trips of groups,
# a last group partly full in both spins, one orbital of a spin, one spin empty
GROUPS = [("F", (43, 43, 0), [0] * 40 + [1]), ("F", (39, 39, 1), [1] * 33),
          ("F", (53, 53, 53), [0, 1]), ("P", (49, 49, 5), [k % 2 for k in range(25)]),
          ("P", (3, 3, 3), [int(k % 3 == 0) for k in range(257)]),
          ("P", (11, 9, 149), [k % 2 for k in range(9)])]


@pytest.mark.parametrize("geo,n,spin", GROUPS,
                         ids=[f"{g}{n[0]}x{n[1]}x{n[2]}-{len(s)}" for g, n, s in GROUPS])
def test_density_groups_match_the_oracle(ctx, geo, n, spin):
    test_density_launch_edges_match_the_oracle(ctx, geo, n, spin)


@pytest.mark.parametrize("n", [(42, 40, 0), (57, 59, 0), (57, 60, 1), (66, 60, 2)],
                         ids=lambda n: "x".join(map(str, n)))
def test_flat_free_batches_on_line_passes_match_the_oracle(ctx, n):
    """flat free boxes with large planes: z first up to 512 planes, then the line
    passes, of the whole batch also where it is cut into parts of fewer planes"""
    reg = dense_region("F", n, (0.45, 0.4, 0.5))
    psi, pot, lr = random_psi(reg, 20, 161), random_pot(reg, 162), ctx.region(reg)
    for norb in (14, 20):   # 434 to 490 planes; 620 to 700
        print(f"case {n} norb={norb}", flush=True)
        x, v = dev(psi[:norb]), dev(pot)

        def run():
            h = torch.zeros_like(x)
            ek = torch.zeros(norb, dtype=torch.float64, device="cuda")
            ep = torch.zeros_like(ek)
            ctx.locham(lr, v, x, h, ek, ep)
            ctx.sync()
            return h.cpu().numpy(), ek.cpu().numpy(), ep.cpu().numpy()
        got = run()
        ctx.set_option("chunk_mb", 4)
        try:
            cut = run()
        finally:
            ctx.set_option("chunk_mb", 0)
        for a, b in zip(got, cut):
            assert np.array_equal(a, b)
        ho, eo, po = oracle.locham("F", reg.n, reg.nfl, reg.nfu, reg.hgrid, okeys(reg), pot,
                                   psi[:norb], np.zeros_like(psi[:norb]))
        assert np.abs(got[0] - ho).max() < TOL * np.abs(ho).max()
        assert rel_err(got[1], eo) < TOL
        assert rel_err(got[2], po) < TOL
    lr.close()


@pytest.mark.parametrize("geo,n,norb,mb", [("F", (49, 49, 1), 64, 64), ("P", (23, 23, 23), 48, 32),
                                           ("P", (71, 72, 5), 24, 48)],
                         ids=["flat_free", "periodic", "lines"])
def test_chunks_keep_to_their_size(ctx, geo, n, norb, mb):
    """a plan cut into chunks of mb MiB holds at most that much in working grids
    (FP64: K and TZ, 2.9 MB a flat free box, and TX on lines) and not less than
    half of it; with the bits of one chunk"""
    reg = dense_region(geo, n, (0.45, 0.4, 0.5))
    lr = ctx.region(reg)
    psi, pot = dev(random_psi(reg, norb, 171)).ravel(), dev(random_pot(reg, 172))

    def run():
        h = torch.zeros_like(psi)
        ek = torch.zeros(norb, dtype=torch.float64, device="cuda")
        ep = torch.zeros_like(ek)
        torch.cuda.synchronize()
        before = torch.cuda.mem_get_info()[0]
        plan = ctx.plan([lr] * norb, pot, psi, h, ek, ep)
        used = before - torch.cuda.mem_get_info()[0]
        plan.execute()
        ctx.sync()
        plan.close()
        return used, (h, ek, ep)
    run()   # (the first plan also sets up what the runtime keeps)
    whole, one = run()
    ctx.set_option("chunk_mb", mb)
    try:
        used, cut = run()
    finally:
        ctx.set_option("chunk_mb", 0)
    print(f"case {geo} {n}: {whole >> 20} MiB in one chunk, {used >> 20} of {mb}", flush=True)
    assert whole > 1.3 * mb * 2 ** 20
    assert mb * 2 ** 19 < used < (mb + 8) * 2 ** 20   # tables and allocation units beside
    for a, b in zip(one, cut):
        assert torch.equal(a, b)
    lr.close()


@pytest.mark.parametrize("ns", [[(23, 22, 24)], [(9, 8, 20), (27, 30, 24), (38, 41, 27)]],
                         ids=["one_group", "several"])
def test_potential_planes_in_either_order(ctx, ns):
    """more than 512 planes, in one launch and in one per box shape: both tile
    orders give the same bits"""
    regs = [dense_region("P", n, (0.4, 0.4, 0.4)) for n in ns] * 12
    psi = [random_psi(r, 1, 181 + i)[0] for i, r in enumerate(regs[:len(ns)])] * 12
    pots = [random_pot(r, 185 + i) for i, r in enumerate(regs[:len(ns)])]
    lr = [ctx.region(r) for r in regs[:len(ns)]]
    lrs = lr * 12
    po = np.tile(np.cumsum([0] + [p.size for p in pots[:-1]]), 12)
    so = np.cumsum([0] + [p.size for p in psi])[:-1]
    x, v = dev(np.concatenate(psi)), dev(np.concatenate(pots))
    outs = []
    for order in (0, 1):
        print(f"case {ns} order {order}", flush=True)
        ctx.set_option("tile_order", order)
        try:
            h = torch.zeros_like(x)
            ek = torch.zeros(len(lrs), dtype=torch.float64, device="cuda")
            ep = torch.zeros_like(ek)
            ctx.locham_batch(lrs, v, x, h, ek, ep, pot_off=po, psi_off=so)
            ctx.sync()
        finally:
            ctx.set_option("tile_order", 0)
        outs.append((h, ek, ep))
    for a, b in zip(*outs):
        assert torch.equal(a, b)
    for l in lr:
        l.close()
