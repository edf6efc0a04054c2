"""Edges of the kernels that choose their work split by size: tile remainders, the smallest and the
first size past each split, against the oracle or a plain restatement."""
import numpy as np
import pytest

from miluphpc_amd import ics
from conftest import print_case

pytestmark = pytest.mark.gpu


def load_ctx(lib, s, params):
    ctx = lib.Context(len(s["x"]), params)
    ctx.load(**{k: v for k, v in s.items() if k in lib.FIELD_ID})
    return ctx


def mlp_inputs(seed, n):
    rng = np.random.default_rng(seed)
    p = (rng.uniform(-1, 1, 4801) * 0.3).astype(np.float32)
    X = rng.normal(size=(n, 8)).astype(np.float32)
    X[:, 7] = 0.0
    return p, X, rng.normal(size=n).astype(np.float32)


@pytest.mark.parametrize("n", [1, 15, 17, 65, 16384, 16385, 40000])
def test_mlp_gradient_is_the_sum_over_its_samples(gpu_lib, n):
    """The gradient of n samples is the mean of the gradients of its parts: the first and the rest,
    which split over wavefronts, blocks (256 x 64 samples fill one step) and steps differently.
    Every sample's terms are the same BF16 products in both, scaled by a power of two at most
    apart in dy before rounding; the sums are FP32, so parts and whole differ by BF16 roundings of
    dz (2^-9 each, random) and FP32 sums."""
    print_case(f"mlp gradient parts n={n}")
    p, X, T = mlp_inputs(n, n)
    with gpu_lib.Context(64) as ctx:
        ctx.mlp_set_params(p)
        g, loss = ctx.mlp_gradient(X, T)
        g2, loss2 = ctx.mlp_gradient(X, T)
        assert np.array_equal(g, g2) and loss == loss2   # deterministic
        if n > 1:
            k = max(1, n // 3)
            ga, la = ctx.mlp_gradient(X[:k], T[:k])
            gb, lb = ctx.mlp_gradient(X[k:], T[k:])
            both = (k * ga.astype(np.float64) + (n - k) * gb) / n
            assert loss == pytest.approx((k * la + (n - k) * lb) / n, rel=1e-4)
            assert np.linalg.norm(g - both) <= 1e-2 * np.linalg.norm(both)
    assert np.all(g[:512].reshape(64, 8)[:, 7] == 0.0)   # the padding input


@pytest.mark.parametrize("nsamples", [1, 100, 16500])
def test_mlp_train_step_is_adam_on_the_sampled_gradient(gpu_lib, nsamples):
    """One training step equals Adam (its first step) on the gradient of the sampled pairs."""
    print_case(f"mlp train step nsamples={nsamples}")
    s = ics.sedov_lattice(12)
    lr, seed = 1e-3, 5
    flags = gpu_lib.RHS_SPH | gpu_lib.RHS_VARIABLE_SML | gpu_lib.RHS_FEATURES
    with load_ctx(gpu_lib, s, ics.params_sedov()) as ctx:
        n = ctx.n
        ctx.mlp_init(3)
        norm = np.zeros(18, np.float32)
        norm[:7] = [-1.0, 1.0, 0.0, 0.0, 0.0, 0.0, 0.0]
        norm[8:15] = 1.0
        norm[17] = 0.1
        ctx.mlp_set_norm(norm)
        h0 = ctx.download("sml")
        ctx.rhs(flags)
        X, h1 = ctx.mlp_download_features(), ctx.download("sml")
        T = (np.log(h1 / h0) / np.float64(norm[17])).astype(np.float32)
        M = (1 << 64) - 1

        def mix(z):
            z = ((z ^ (z >> 30)) * 0xBF58476D1CE4E5B9) & M
            z = ((z ^ (z >> 27)) * 0x94D049BB133111EB) & M
            return z ^ (z >> 31)

        idx = np.array([mix((seed * 0x9E3779B97F4A7C15 + i) & M) % n for i in range(nsamples)])
        p0 = ctx.mlp_get_params()
        g, loss_g = ctx.mlp_gradient(X[idx], T[idx])
        loss = ctx.mlp_train(nsamples=nsamples, iters=1, lr=lr, seed=seed)
        p1 = ctx.mlp_get_params()
    assert loss == pytest.approx(loss_g, rel=1e-6)
    g = g.astype(np.float64)
    # the first step with the FP32 bias corrections; a dozen FP32 roundings of it, and one of p.
    # Below |g| = 1e-6 the step is not saturated and follows the rounding of g itself
    f32 = np.float32
    bc1, bc2 = float(f32(1) - f32(0.9)), float(f32(1) - f32(0.999))
    step = lr * (float(f32(0.1)) * g / bc1) / (np.sqrt(float(f32(0.001)) * g * g / bc2) + 1e-8)
    sure = (np.abs(g) > 1e-6) | (g == 0.0)
    assert sure.mean() > 0.5
    assert np.abs((p1 - p0.astype(np.float64)) + step)[sure].max() <= 12 * 2.0 ** -24 * lr + 2.0 ** -24 * np.abs(p0).max()


@pytest.mark.parametrize("n", [1000, 1025, 300000])
def test_diagnostics_of_ragged_counts(gpu_lib, n):
    """Global sums of counts around the block split (1024 per block; more than one particle per
    thread above 262,144), every term's exact sum in extended precision to FP64 rounding."""
    print_case(f"diagnostics n={n}")
    rng = np.random.default_rng(n)
    f = {k: rng.normal(size=n) + 0.5 for k in ("x", "y", "z", "vx", "vy", "vz")}
    f.update(mass=rng.uniform(0.5, 1.5, n), e=rng.uniform(0, 1, n))
    with gpu_lib.Context(n) as ctx:
        ctx.load(**f)
        ctx.upload("u", -f["mass"])
        d = ctx.diagnostics()
    L = {k: v.astype(np.longdouble) for k, v in f.items()}
    m = L["mass"]
    # each term takes at most 6 roundings before the compensated sum's one or two
    checks = [("mass", d["mass"], m), ("potential", d["potential"], -m), ("internal", d["internal"], m * L["e"]),
              ("kinetic", d["kinetic"], 0.5 * m * (L["vx"] ** 2 + L["vy"] ** 2 + L["vz"] ** 2))]
    checks += [(f"momentum {a}", d["momentum"][a], m * L[t]) for a, t in enumerate(("vx", "vy", "vz"))]
    for name, got, terms in checks:
        assert abs(got - float(terms.sum())) <= 8 * 2.0 ** -53 * float(np.abs(terms).sum()), name


@pytest.mark.parametrize("quad,precision", [(0, 0), (1, 0), (0, 1), (1, 1)])
@pytest.mark.parametrize("vote", [0, 1])
@pytest.mark.parametrize("n", [70, 2100, 33000])
def test_barnes_hut_shared_groups(gpu_lib, orc, n, vote, quad, precision):
    """Groups shared by several wavefronts (8 below 512 groups without quadrupole, else 4) give the
    oracle walk's interactions and forces, with and without softening, with potential."""
    print_case(f"shared groups n={n} vote={vote} quad={quad} precision={precision}")
    s = ics.plummer(n, seed=n)
    for eps2 in (1e-6, 0.0):
        p = gpu_lib.default_params(theta=0.6, smoothing=eps2, curve=1, quadrupole=quad, bh_accept=vote,
                                   precision=precision)
        with load_ctx(gpu_lib, s, p) as ctx:
            st = ctx.rhs(gpu_lib.RHS_GRAVITY | gpu_lib.RHS_POTENTIAL)
            g = np.stack([ctx.download(k) for k in ("g_ax", "g_ay", "g_az")])
            u = ctx.download("u")
        o = orc.gravity_rhs(s, 0.6, eps2, curve=1, quad=bool(quad), vote=bool(vote), potential=True)
        assert st["n_cell_interactions"] == o["n_cell"] and st["n_part_interactions"] == o["n_part"]
        go = np.stack([o["ax"], o["ay"], o["az"]])
        uo = 0.5 * s["mass"] * o["phi"]
        size = np.sqrt((go ** 2).sum(0))
        err = np.sqrt(((g - go) ** 2).sum(0)) / np.maximum(size, np.sqrt((size ** 2).mean()))
        if precision == 0:
            tol = 1e-12 if not quad else 2e-7   # quadrupoles are stored in FP32
            assert err.max() <= tol
            assert np.abs(u - uo).max() <= tol * np.abs(uo).max()
        else:
            assert np.percentile(err, 99) < 1e-5
            assert np.percentile(np.abs(u / uo - 1.0), 99) < 1e-5


@pytest.mark.parametrize("side", [25, 33])
@pytest.mark.parametrize("curve", [0, 1])
def test_neighbours_of_groups_that_straddle_a_curve_jump(gpu_lib, orc, side, curve):
    """On lattices whose side is no power of two some runs of 64 Lebesgue keys span the domain; the
    walks split them.  Lists, h and counts equal the oracle's, in both list structures."""
    print_case(f"split groups side={side} curve={curve}")
    s = ics.sedov_lattice(side)
    rng = np.random.default_rng(side)
    for k in "xyz":
        s[k] = s[k] + rng.uniform(-0.02, 0.02, side ** 3) / side
    s["sml"] = s["sml"] * rng.uniform(0.95, 1.05, side ** 3)   # some particles change h
    p = ics.params_sedov(curve=curve, sml_max=4.0 * float(s["sml"].max()))
    o = orc.sph_rhs(s, sml_max=p.sml_max)
    for spec in (0, gpu_lib.RHS_SPECULATIVE_NN):
        with load_ctx(gpu_lib, s, p) as ctx:
            ctx.rhs(gpu_lib.RHS_SPH | gpu_lib.RHS_VARIABLE_SML | spec)
            nnl, noi = ctx.neighbour_lists(180)
            h, rho = ctx.download("sml"), ctx.download("rho")
        assert np.array_equal(h, o["sml"])
        assert np.array_equal(noi, o["noi"])
        assert np.max(np.abs(rho / o["rho"] - 1.0)) <= 1e-12
        used = np.arange(180) < noi[:, None]
        assert np.array_equal(np.sort(np.where(used, nnl, -1), 1), np.sort(np.where(used, o["nnl"], -1), 1))


@pytest.mark.parametrize("n", [1, 63, 64, 65, 2047, 8192, 8193, 20000, 98304, 98305])
def test_key_sort_by_rank_edges(gpu_lib, n):
    """The allocation-free key sort at the edges of its forms (one launch to 8,192 keys, tiles of
    2,048 merged to 98,304, radix passes above) on full 64-bit keys with ties, the largest key among
    them, and with the outputs over the inputs: numpy's stable sort."""
    import ctypes as C
    print_case(f"key sort n={n}")
    rng = np.random.default_rng(n)
    key = rng.integers(0, 1 << 64, n, dtype=np.uint64)
    key[rng.random(n) < 0.5] &= np.uint64(7)
    key[rng.random(n) < 0.1] = np.uint64(0xFFFFFFFFFFFFFFFF)
    order = np.argsort(key, kind="stable")
    with gpu_lib.Context(64) as ctx:
        dk, ds, dv = ctx.device_alloc(8 * n), ctx.device_alloc(8 * n), ctx.device_alloc(4 * n)
        for out in (ds, dk):   # separate, then in place
            ctx.device_upload(dk, key)
            st = gpu_lib.LIB.mhpc_sort_keys_noalloc(C.c_void_p(dk), n, C.c_void_p(out), C.c_void_p(dv), None)
            assert st == gpu_lib.OK
            assert np.array_equal(ctx.device_download(out, n, np.uint64), key[order])
            assert np.array_equal(ctx.device_download(dv, n, np.int32), order)
        for p in (dk, ds, dv):
            ctx.device_free(p)


@pytest.mark.parametrize("curve", [0, 1])
def test_partial_radix_sort_falls_back(gpu_lib, orc, curve):
    """Above the rank sort's range a context sorts only the levels its last tree needed, and in full
    when two particles then share them: both orders are the stable sort's."""
    print_case(f"partial radix sort, 47^3, curve {curve}")
    s = ics.sedov_lattice(47)
    with load_ctx(gpu_lib, s, gpu_lib.default_params(curve=curve)) as ctx:
        for step in range(3):
            if step == 2:
                for c in "xyz":
                    s[c][1] = s[c][0]
                ctx.load(x=s["x"], y=s["y"], z=s["z"])
            box = ctx.bbox()
            ctx.keys()
            ctx.sort()
            perm = ctx.download("sorted")
            if step < 2:
                ctx.build_tree()
                ctx.centres_of_mass()
            assert np.array_equal(perm, orc.sort(orc.keys(s["x"], s["y"], s["z"], box, curve)))


@pytest.mark.parametrize("n", [2, 257, 4096, 4097, 262144, 262145])
def test_tree_and_com_at_the_tile_and_launch_splits(gpu_lib, orc, n):
    """Octree and centres of mass bit-exact where the tree's tile (256 or 1024 positions) and the
    bottom-up pass's launches (one to 4,096 particles) change."""
    print_case(f"tree n={n}")
    s = ics.plummer(n, seed=n)
    with load_ctx(gpu_lib, s, gpu_lib.default_params(quadrupole=1)) as ctx:
        box = ctx.bbox()
        ctx.keys()
        ctx.sort()
        ctx.build_tree()
        ctx.centres_of_mass()
        t = ctx.tree()
    o = orc.Tree(s["x"], s["y"], s["z"], box)
    o.com(s["mass"])
    assert len(t["mass"]) == o.ncells
    lev = np.asarray(o.level[n:n + o.ncells])
    assert np.array_equal(np.bincount(t["level"]), np.bincount(lev))
    # the two number cells differently: compare as sets of (level, mass, centre)
    nm, nx, ny, nz = (np.asarray(a)[n:n + o.ncells] for a in (o.nm, o.nx, o.ny, o.nz))
    a = np.array(sorted(zip(t["level"], t["mass"], t["x"], t["y"], t["z"])))
    b = np.array(sorted(zip(lev, nm, nx, ny, nz)))
    assert np.array_equal(a, b)


@pytest.mark.parametrize("curve", [0, 1])
def test_relists_around_boxes_the_direct_search_declines(gpu_lib, orc, curve):
    """A jittered 33^3 lattice (35,937 particles: group walks, an odd last group) where some h are
    several times and a few are hundreds of times the others', so that their search boxes hold more
    particles than the direct search takes: h, iteration counts and neighbour sets of the speculative
    lists equal the plain iteration's and the oracle's."""
    print_case(f"declined boxes, 33^3 curve={curve}")
    s = ics.sedov_lattice(33)
    rng = np.random.default_rng(91)
    n = len(s["x"])
    for a in "xyz":
        s[a] = s[a] + rng.uniform(-0.2, 0.2, n) / 33
    u = rng.uniform(size=n)
    h0 = s["sml"] * rng.uniform(0.9, 1.25, n) * np.where(u < 0.05, 6.0, 1.0)
    h0[rng.choice(n, 12, replace=False)] = 3.0 * (s["x"].max() - s["x"].min())
    base = gpu_lib.RHS_SPH | gpu_lib.RHS_VARIABLE_SML
    out = {}
    for name, flags in (("plain", base), ("spec", base | gpu_lib.RHS_SPECULATIVE_NN)):
        with load_ctx(gpu_lib, {**s, "sml": h0}, gpu_lib.default_params(curve=curve)) as ctx:
            ctx.rhs(flags)
            out[name] = {k: ctx.download(k) for k in ("sml", "h_iters", "noi", "rho")}
            nnl, noi = ctx.neighbour_lists(180)
        out[name]["sets"] = [frozenset(nnl[i, :noi[i]].tolist()) for i in range(n)]
    a, b = out["plain"], out["spec"]
    st, oh, oiters, _ = orc.h_iterate(s["x"], s["y"], s["z"], h0)
    assert np.array_equal(b["h_iters"], oiters) and np.array_equal(b["sml"], oh)
    for k in ("sml", "h_iters", "noi"):
        assert np.array_equal(a[k], b[k]), k
    assert a["sets"] == b["sets"]
    assert np.max(np.abs(a["rho"] - b["rho"])) <= 1e-12 * a["rho"].max()   # order of 180 terms at most


@pytest.mark.parametrize("scale,offset,mixed", [(1.0, 0.0, True), (1.0, 0.0, False), (2.0 ** 60, 0.0, True),
                                                (2.0 ** -60, 0.0, True), (1.0, 2.0 ** 20, True),
                                                (1.0, 0.0, "far"), (1.0, 0.0, "random")])
def test_group_walks_decide_pairs_at_the_radius_exactly(gpu_lib, orc, scale, offset, mixed):
    """Lattice distances are whole, and the radii are whole or one rounding to either side: a pair's
    squared distance equals, just misses or just meets h^2, in both particles' h.  The walks' matrix
    tests cannot tell these apart and must leave them to the FP64 test: neighbour sets and counts are
    the oracle's, at scales whose squares leave FP32, far from the origin, and (`far`) in groups whose
    box is too large against h for the matrix tests."""
    print_case(f"pairs at the radius scale={scale} offset={offset} mixed={mixed}")
    side = 33
    n = side ** 3
    rng = np.random.default_rng(3)
    g = np.stack(np.meshgrid(*[np.arange(side, dtype=np.float64)] * 3, indexing="ij")).reshape(3, n)
    r = np.array([2.0, 3.0, 2.5, 2.0])
    r = np.concatenate([r, np.nextafter(r, 9.0), np.nextafter(r, 0.0)])
    h = rng.choice(r, n) if mixed else np.full(n, np.nextafter(3.0, 9.0))
    if mixed == "far":
        h = np.where(rng.uniform(size=n) < 0.5, 1.0, np.nextafter(1.0, 2.0))
        g = g * np.where(np.arange(3) < 2, 1.0, 40.0)[:, None]
    if mixed == "random":
        g = rng.uniform(0.0, side, (3, n))
        h = rng.uniform(1.5, 2.6, n)
    p = (g + offset) * scale
    h = h * scale
    s = dict(x=p[0], y=p[1], z=p[2], mass=np.full(n, 1.0 / n), sml=h)
    st, onnl, onoi = orc.nn_grid(p[0], p[1], p[2], h, 180)
    assert st == 0
    with load_ctx(gpu_lib, s, gpu_lib.default_params(curve=0)) as ctx:
        ctx.bbox(); ctx.keys(); ctx.sort(); ctx.build_tree()
        ctx.neighbours()
        nnl, noi = ctx.neighbour_lists(180)
    assert np.array_equal(noi, onoi)
    used = np.arange(180) < noi[:, None]
    assert np.array_equal(np.sort(np.where(used, nnl, -1), 1), np.sort(np.where(used, onnl, -1), 1))
    # the counting and the list-writing passes of the h-iteration, from the same h
    oh, oiters = orc.h_iterate(p[0], p[1], p[2], h)[1:3]
    for spec in (0, gpu_lib.RHS_SPECULATIVE_NN):
        with load_ctx(gpu_lib, s, gpu_lib.default_params(curve=0)) as ctx:
            ctx.rhs(gpu_lib.RHS_SPH | gpu_lib.RHS_VARIABLE_SML | spec)
            assert np.array_equal(ctx.download("sml"), oh)
            assert np.array_equal(ctx.download("h_iters"), oiters)


@pytest.mark.parametrize("scale", [2.0 ** 500, 2.0 ** -500, 2.0 ** -520])
def test_group_walks_where_squares_leave_the_normal_numbers(gpu_lib, orc, scale):
    """Radii whose squares come close to the largest FP64 number, or are denormal (exact multiples of
    the lattice's, so the comparison still has one answer): neighbour sets are the oracle's."""
    print_case(f"extreme scales scale={scale}")
    side = 33
    n = side ** 3
    rng = np.random.default_rng(4)
    p = np.stack(np.meshgrid(*[np.arange(side, dtype=np.float64)] * 3, indexing="ij")).reshape(3, n)
    h = rng.choice([2.0, 2.5, 3.0], n)
    st, onnl, onoi = orc.nn_grid(p[0], p[1], p[2], h, 180)   # scaling by a power of two changes nothing
    assert st == 0
    s = dict(x=p[0] * scale, y=p[1] * scale, z=p[2] * scale, mass=np.full(n, 1.0 / n), sml=h * scale)
    with load_ctx(gpu_lib, s, gpu_lib.default_params(curve=0)) as ctx:
        ctx.bbox(); ctx.keys(); ctx.sort(); ctx.build_tree()
        ctx.neighbours()
        nnl, noi = ctx.neighbour_lists(180)
    assert np.array_equal(noi, onoi)
    used = np.arange(180) < noi[:, None]
    assert np.array_equal(np.sort(np.where(used, nnl, -1), 1), np.sort(np.where(used, onnl, -1), 1))


def gas_in_units(side, h, v, rho, cs, seed=17):
    """A jittered lattice of gas with smoothing length h and random velocities of size v, density rho
    and sound speed cs, in whatever units these are."""
    s = ics.sedov_lattice(side)
    rng = np.random.default_rng(seed)
    n = side ** 3
    L = h / float(s["sml"][0])
    for a in "xyz":
        s[a] = L * (s[a] + 0.1 / side * rng.uniform(-1, 1, n))
        s["v" + a] = v * rng.normal(size=n)
    s["sml"] = L * s["sml"]
    s["mass"] = np.full(n, rho * L ** 3 / n)
    s["e"] = cs ** 2 / (5.0 / 3.0 * 2.0 / 3.0) * rng.uniform(0.9, 1.1, n)
    s["p"] = 2.0 / 3.0 * rho * s["e"]
    s["rho"] = np.full(n, rho)
    return s


def compare_fp32_rhs(gpu_lib, orc, s):
    """The FP32 SPH RHS against the FP64 oracle.  A pair term carries about a dozen roundings
    (7e-7) and a sum's terms add up to some 30 times the field's RMS."""
    p = gpu_lib.default_params(precision=gpu_lib.PREC_FP32_KAHAN)
    with load_ctx(gpu_lib, s, p) as ctx:
        ctx.rhs(gpu_lib.RHS_SPH | gpu_lib.RHS_VARIABLE_SML)
        g = {k: ctx.download(k) for k in ("sml", "rho", "ax", "ay", "az", "drhodt", "dedt", "dsmldt")}
    o = orc.sph_rhs(s)
    assert np.array_equal(g["sml"], o["sml"])
    assert np.max(np.abs(g["rho"] / o["rho"] - 1.0)) < 5e-6
    for k in ("ax", "ay", "az", "drhodt", "dedt", "dsmldt"):
        scale = np.maximum(np.abs(o[k]), np.sqrt(np.mean(o[k] ** 2)))
        assert np.all(np.isfinite(g[k])), k
        assert np.max(np.abs(g[k] - o[k]) / scale) < 5e-5, k


@pytest.mark.parametrize("side", [16, 37])   # shared lists; windows
@pytest.mark.parametrize("h,v,rho,cs", [(1e5, 1e4, 3e3, 5e3), (5e4, 3e3, 3e3, 5e3), (1e6, 1e6, 3.0, 5e5),
                                        (1e-5, 1.0, 1e-18, 0.5), (1.0, 1.0, 1.0, 0.5)])
def test_fp32_forces_in_physical_units(gpu_lib, orc, side, h, v, rho, cs):
    """FP32 pair sums where lengths are far from one: rock in SI and cgs units, thin gas at small h."""
    print_case(f"fp32 forces side={side} h={h} v={v} rho={rho}")
    compare_fp32_rhs(gpu_lib, orc, gas_in_units(side, h, v, rho, cs))


@pytest.mark.parametrize("sigma", [2e-2, 3e-4])
@pytest.mark.parametrize("curve", [0, 1])
def test_groups_that_straddle_a_dense_clump(gpu_lib, orc, curve, sigma):
    """Half of 40,000 particles in a small ball, the others spread around it with h hundreds of times
    as large: groups that hold both test the clump in FP64, and split parts whose box holds it go to
    the per-particle searches.  h, iteration counts, counts and neighbour sets are the oracle's."""
    print_case(f"dense clump sigma={sigma} curve={curve}")
    n, k = 40000, 20000
    rng = np.random.default_rng(2)
    p = np.concatenate([sigma * rng.normal(size=(k, 3)) + 0.3, rng.uniform(-1, 1, (n - k, 3))])
    h = np.concatenate([np.full(k, 1.2 * sigma * (64 / (4.19 * k / 15.75)) ** (1 / 3)),
                        np.full(n - k, (64 * 8 / (4.19 * (n - k))) ** (1 / 3))])
    s = dict(x=p[:, 0].copy(), y=p[:, 1].copy(), z=p[:, 2].copy(), mass=np.full(n, 1.0 / n), sml=h)
    st, oh, oiters, _ = orc.h_iterate(s["x"], s["y"], s["z"], h, max_nb=400)
    assert st == 0
    st, onnl, onoi = orc.nn_grid(s["x"], s["y"], s["z"], oh, 400)
    assert st == 0
    used = np.arange(400) < onoi[:, None]
    for spec in (0, gpu_lib.RHS_SPECULATIVE_NN):
        with load_ctx(gpu_lib, s, gpu_lib.default_params(curve=curve, max_nb=400)) as ctx:
            ctx.rhs(gpu_lib.RHS_SPH | gpu_lib.RHS_VARIABLE_SML | spec)
            nnl, noi = ctx.neighbour_lists(400)
            assert np.array_equal(ctx.download("sml"), oh) and np.array_equal(ctx.download("h_iters"), oiters)
        assert np.array_equal(noi, onoi)
        assert np.array_equal(np.sort(np.where(used, nnl, -1), 1), np.sort(np.where(used, onnl, -1), 1))


@pytest.mark.parametrize("side", [20, 33])   # per particle; groups
@pytest.mark.parametrize("curve", [0, 1])
def test_neighbours_beside_particles_that_are_no_numbers(gpu_lib, orc, side, curve):
    """Particles with a NaN coordinate or a NaN h, alone and side by side in a group, have no neighbours
    and are nobody's; every other particle's list, h and iteration count is that of a set without
    them."""
    print_case(f"nan particles side={side} curve={curve}")
    s = ics.sedov_lattice(side)
    n = side ** 3
    rng = np.random.default_rng(side)
    for a in "xyz":
        s[a] = s[a] + rng.uniform(-0.1, 0.1, n) / side
    s["sml"] = s["sml"] * rng.uniform(0.85, 1.15, n)
    bad = np.array([n // 3, n // 2, n // 2 + 1, 2 * n // 3])
    ok = np.setdiff1d(np.arange(n), bad)
    st, oh, oiters, _ = orc.h_iterate(s["x"][ok], s["y"][ok], s["z"][ok], s["sml"][ok])
    assert st == 0
    s["x"][bad[0]] = np.nan
    s["z"][bad[1]] = np.nan
    s["sml"][bad[2]] = np.nan
    s["sml"][bad[3]] = np.nan

    def listed(h):
        st, nnl, noi = orc.nn_grid(s["x"][ok], s["y"][ok], s["z"][ok], h, 180)
        assert st == 0
        return nnl, noi

    p = gpu_lib.default_params(curve=curve)
    with load_ctx(gpu_lib, s, p) as ctx:
        ctx.bbox(); ctx.keys(); ctx.sort(); ctx.build_tree()
        ctx.neighbours()
        nnl, noi = ctx.neighbour_lists(180)
    onnl, onoi = listed(s["sml"][ok])
    assert np.all(noi[bad] == 0)
    assert np.array_equal(noi[ok], onoi)
    used = np.arange(180) < onoi[:, None]
    want = np.sort(np.where(used, ok[onnl.clip(0, len(ok) - 1)], -1), 1)
    assert np.array_equal(np.sort(np.where(used, nnl[ok], -1), 1), want)

    onnl, onoi = listed(oh)
    st, orho = orc.density(*(s[k][ok] for k in ("x", "y", "z", "mass")), oh, onnl, onoi)
    assert st == 0
    for spec in (0, gpu_lib.RHS_SPECULATIVE_NN):
        with load_ctx(gpu_lib, s, p) as ctx:
            with pytest.raises(gpu_lib.MhpcError):   # particles without neighbours or density
                ctx.rhs(gpu_lib.RHS_SPH | gpu_lib.RHS_VARIABLE_SML | spec)
            assert np.array_equal(ctx.download("sml")[ok], oh)
            assert np.array_equal(ctx.download("h_iters")[ok], oiters)
            noi, rho = ctx.download("noi"), ctx.download("rho")
        assert np.array_equal(noi[ok], onoi) and np.all(noi[bad] == 0)
        assert np.max(np.abs(rho[ok] / orho - 1.0)) <= 1e-12


@pytest.mark.parametrize("side", [16, 37])   # shared lists; windows
@pytest.mark.parametrize("precision", [0, 1])
@pytest.mark.parametrize("kernel", [1, 2])
def test_density_of_coincident_particles(gpu_lib, orc, side, precision, kernel):
    """Two particles on either side of the middle of the box, so close that their squared distance is
    zero: each counts with the kernel's value at zero in the other's density."""
    print_case(f"coincident pair side={side} precision={precision} kernel={kernel}")
    s = ics.sedov_lattice(side)
    n = side ** 3
    rng = np.random.default_rng(side)
    for a in "xyz":
        s[a] = s[a] + rng.uniform(-0.1, 0.1, n) / side
    for a in "xyz":
        s[a][0], s[a][-1] = -0.5, 0.5   # the box is [-0.5, 0.5]: its middle is 0
    i, j = n // 2, n // 2 + 1
    d = 1e-170 if precision == 0 else 1e-30
    s["x"][i], s["x"][j] = -d, d
    for a in "yz":
        s[a][j] = s[a][i]
    p = gpu_lib.default_params(precision=precision, smoothing_kernel=kernel)
    with load_ctx(gpu_lib, s, p) as ctx:
        ctx.rhs(gpu_lib.RHS_SPH)
        g = {k: ctx.download(k) for k in ("noi", "rho", "ax", "ay", "az", "dedt")}
    st, nnl, noi = orc.nn_grid(s["x"], s["y"], s["z"], s["sml"], 180)
    assert st == 0 and j in nnl[i, :noi[i]]
    st, rho = orc.density(s["x"], s["y"], s["z"], s["mass"], s["sml"], nnl, noi, kernel=kernel)
    assert np.array_equal(g["noi"], noi)
    assert np.max(np.abs(g["rho"] / rho - 1.0)) < (1e-12 if precision == 0 else 5e-6)
    for k in ("ax", "ay", "az", "dedt"):
        assert np.all(np.isfinite(g[k])), k


def fp32_pair_sums(s, rho, p, cs, nnl, noi):
    """Density and de/dt as FP32 pair terms (cubic spline) with correctly rounded square roots and
    quotients, added in 64 bits."""
    f = np.float32
    fma = lambda a, b, c: (a.astype(np.float64) * b + c).astype(f)   # the product is exact in 64 bits
    i = np.repeat(np.arange(len(noi)), noi)
    j = nnl[np.arange(nnl.shape[1]) < noi[:, None]]
    d = [(s[a][i] - s[a][j]).astype(f) for a in "xyz"]
    v = [(s["v" + a][i] - s["v" + a][j]).astype(f) for a in "xyz"]
    h = (0.5 * (s["sml"][i] + s["sml"][j])).astype(f)
    r2 = fma(d[0], d[0], fma(d[1], d[1], d[2] * d[2]))
    r, ih = np.sqrt(r2), f(1) / h
    q = r * ih
    t, norm = f(1) - q, f(8 / np.pi) * ih * ih * ih
    w = np.where(q <= f(0.5), norm * fma(f(6) * q * q, q - f(1), f(1)), f(2) * norm * t * t * t)
    dw = np.where(q <= f(0.5), f(6) * norm * ih * q * fma(f(3) * np.ones_like(q), q, f(-2)), f(-6) * norm * ih * t * t)
    inside = q <= f(1)
    add = lambda terms: np.bincount(i, np.where(inside, terms, f(0)).astype(np.float64), len(noi))
    m = s["mass"][j].astype(f)
    g = [dw / r * c for c in d]
    vv = fma(v[0], g[0], fma(v[1], g[1], v[2] * g[2]))
    vr = fma(v[0], d[0], fma(v[1], d[1], v[2] * d[2]))
    c = f(0.5) * (cs[i].astype(f) + cs[j].astype(f))
    mu = h * vr / fma(h * h, f(0.01), r2)
    visc = np.where(vr < 0, m * (f(2) * mu - f(1) * c) * mu / (f(0.5) * (rho[i].astype(f) + rho[j].astype(f))), f(0))
    pr = p / (rho * rho)
    press = -m * (pr[i].astype(f) + pr[j].astype(f))
    return s["mass"] * (8 / np.pi) / s["sml"] ** 3 + add(m * w), 0.5 * add((visc - press) * vv)


@pytest.mark.parametrize("side", [31, 37])   # shared lists; windows
def test_fp32_pair_sums_are_as_accurate_as_rounded_roots_and_quotients(gpu_lib, orc, side):
    """The FP32 pair terms come from hardware estimates: their RMS error against 64 bits is within
    one per cent of that with correctly rounded square roots and divisions, on the same particles."""
    print_case(f"fp32 accuracy side={side}")
    s = gas_in_units(side, 1.0, 1.0, 1.0, 0.5, seed=side)
    s["sml"] = s["sml"] * np.random.default_rng(side).uniform(0.95, 1.05, side ** 3)
    with load_ctx(gpu_lib, s, gpu_lib.default_params(precision=gpu_lib.PREC_FP32_KAHAN)) as ctx:
        ctx.rhs(gpu_lib.RHS_SPH)
        g = {k: ctx.download(k) for k in ("rho", "p", "cs", "dedt")}
    st, nnl, noi = orc.nn_grid(s["x"], s["y"], s["z"], s["sml"], 180)
    assert st == 0
    st, rho = orc.density(s["x"], s["y"], s["z"], s["mass"], s["sml"], nnl, noi)
    o = orc.forces(*(s[k] for k in ("x", "y", "z", "vx", "vy", "vz", "mass", "sml")), g["rho"], g["p"], g["cs"], nnl,
                   noi)
    rho32, dedt32 = fp32_pair_sums(s, g["rho"], g["p"], g["cs"], nnl, noi)
    rms = lambda a: np.sqrt(np.mean(a ** 2))
    errs = (rms(g["rho"] - rho), rms(rho32 - rho), rms(g["dedt"] - o["dedt"]), rms(dedt32 - o["dedt"]))
    print("rms errors: density %.4g (rounded %.4g), de/dt %.4g (rounded %.4g)" % errs)
    assert errs[0] <= 1.01 * errs[1] < 1e-6 * rms(rho)
    assert errs[2] <= 1.01 * errs[3] < 1e-5 * rms(o["dedt"])


@pytest.mark.parametrize("eps2", [1e-6, 0.0])
@pytest.mark.parametrize("vote", [0, 1])
def test_barnes_hut_with_strays_beyond_the_square_of_fp64(gpu_lib, orc, vote, eps2):
    """Two particles so far out that their squared distances are infinite act on nothing (1 / sqrt(inf)
    = 0); the others, one per octant around the middle, keep the oracle's forces."""
    print_case(f"far strays vote={vote} eps2={eps2}")
    rng = np.random.default_rng(8)
    corner = np.array([[i & 1, i >> 1 & 1, i >> 2 & 1] for i in range(8)]) * 2.0 - 1.0
    p = np.concatenate([corner * rng.uniform(0.5, 1.5, (8, 3)), [[1e160] * 3, [-1e160] * 3]])
    s = dict(x=p[:, 0].copy(), y=p[:, 1].copy(), z=p[:, 2].copy(), mass=rng.uniform(0.5, 1.5, 10))
    with load_ctx(gpu_lib, s, gpu_lib.default_params(theta=0.5, smoothing=eps2, curve=0, bh_accept=vote,
                                                     precision=gpu_lib.PREC_FP64)) as ctx:
        ctx.rhs(gpu_lib.RHS_GRAVITY)
        g = np.stack([ctx.download(k) for k in ("g_ax", "g_ay", "g_az")])
    d = p[None, :8] - p[:8, None]
    r2 = (d ** 2).sum(2) + eps2
    np.fill_diagonal(r2, 1.0)
    want = (s["mass"][None, :8, None] * d / r2[..., None] ** 1.5).sum(1).T
    assert np.abs(g[:, :8] - want).max() <= 1e-13 * np.abs(want).max()
    assert np.all(g[:, 8:] == 0.0)


@pytest.mark.parametrize("fraction", [0.02, 1.0])
@pytest.mark.parametrize("curve", [0, 1])
def test_relists_of_few_and_of_many_changed_particles(gpu_lib, orc, curve, fraction):
    """41^3 particles of which a few or all change h after pass 0 (32,768 changes part the re-lists per
    particle from those by groups): h, counts and neighbour sets are the oracle's."""
    print_case(f"re-lists fraction={fraction} curve={curve}")
    side = 41
    n = side ** 3
    s = ics.sedov_lattice(side)
    rng = np.random.default_rng(12)
    for a in "xyz":
        s[a] = s[a] + rng.uniform(-0.1, 0.1, n) / side
    s["sml"] = np.where(rng.uniform(size=n) < fraction, 1.15, 1.0) * s["sml"]
    p = gpu_lib.default_params(curve=curve, sml_max=4.0 * float(s["sml"].min()))
    o = orc.sph_rhs(s, sml_max=p.sml_max)
    changed = int((o["h_iters"] > 1).sum())
    assert changed > 32768 if fraction == 1.0 else 0 < changed < 32768
    with load_ctx(gpu_lib, s, p) as ctx:
        ctx.rhs(gpu_lib.RHS_SPH | gpu_lib.RHS_VARIABLE_SML | gpu_lib.RHS_SPECULATIVE_NN)
        nnl, noi = ctx.neighbour_lists(180)
        h = ctx.download("sml")
    assert np.array_equal(h, o["sml"]) and np.array_equal(noi, o["noi"])
    used = np.arange(180) < noi[:, None]
    assert np.array_equal(np.sort(np.where(used, nnl, -1), 1), np.sort(np.where(used, o["nnl"], -1), 1))


@pytest.mark.parametrize("vote", [0, 1])
def test_fp32_potential_rounding(gpu_lib, vote):
    """FP32 potentials against the FP64 ones of the same walk.  Terms of one sign added in chains of 32
    leave a batch 1.3 x 2^-24 off (RMS; chains of 64: 1.9), and some ten chains make up a potential."""
    print_case(f"fp32 potential vote={vote}")
    s = ics.plummer(65536, seed=1)
    u = []
    for precision in (gpu_lib.PREC_FP64, gpu_lib.PREC_FP32_KAHAN):
        p = gpu_lib.default_params(theta=0.6, smoothing=1e-6, curve=1, bh_accept=vote, precision=precision)
        with load_ctx(gpu_lib, s, p) as ctx:
            ctx.rhs(gpu_lib.RHS_GRAVITY | gpu_lib.RHS_POTENTIAL)
            u.append(ctx.download("u"))
    assert np.sqrt(np.mean((u[1] / u[0] - 1.0) ** 2)) < 2.0 ** -25


def test_mlp_gradient_divides_by_the_sample_count(gpu_lib):
    """db3 is the mean of y - t.  For these counts the FP32 rounding of 1/n is 5e-8 to 6e-8: scaled by
    it, every gradient would be off by that; divided, the roundings of the terms average out (a few
    2^-24 / sqrt(1000) and those of the sums, over eight counts)."""
    print_case("mlp gradient scale")
    off = []
    for n in (1020, 1008, 1013, 976, 953, 951, 943, 933):
        p, X, T = mlp_inputs(n, n)
        T -= np.float32(6.0)   # every y - t positive
        with gpu_lib.Context(64) as ctx:
            ctx.mlp_set_params(p)
            g, _ = ctx.mlp_gradient(X, T)
            y = ctx.mlp_forward(X).astype(np.float64).ravel()
        assert np.all(y - T > 0)
        scale = float(np.float32(1) / np.float32(n)) * n - 1.0
        assert abs(scale) > 5e-8
        off.append((g[-1] / np.mean(y - T) - 1.0) * np.sign(scale))
    assert abs(np.mean(off)) < 2.0 ** -25


@pytest.mark.parametrize("side", [20, 33])   # per particle; groups
@pytest.mark.parametrize("curve", [0, 1])
def test_neighbours_with_infinite_h(gpu_lib, orc, side, curve):
    """Particles with an infinite h, a few scattered and a compact block of them: their lists hold every
    particle whose own h reaches them, the others' lists are limited by their own h."""
    print_case(f"infinite h side={side} curve={curve}")
    s = ics.sedov_lattice(side)
    n = side ** 3
    rng = np.random.default_rng(side + 1)
    for a in "xyz":
        s[a] = s[a] + rng.uniform(-0.1, 0.1, n) / side
    r2 = sum((s[a] - 0.1) ** 2 for a in "xyz")
    s["sml"][np.argsort(r2)[:90]] = np.inf
    s["sml"][[5, n // 3, n - 9]] = np.inf
    with load_ctx(gpu_lib, s, gpu_lib.default_params(curve=curve, max_nb=400)) as ctx:
        ctx.bbox(); ctx.keys(); ctx.sort(); ctx.build_tree()
        ctx.neighbours()
        nnl, noi = ctx.neighbour_lists(400)
    st, onnl, onoi = orc.nn_brute(s["x"], s["y"], s["z"], s["sml"], 400)
    assert st == 0
    assert np.array_equal(noi, onoi)
    used = np.arange(400) < noi[:, None]
    assert np.array_equal(np.sort(np.where(used, nnl, -1), 1), np.sort(np.where(used, onnl, -1), 1))
