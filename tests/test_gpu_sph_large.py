"""The SPH parity tests past the sizes up to which every search is per particle (32,768) and density
and forces share a particle's list among lanes (49,152): 33^3 particles take the group walks, 37^3
also the windowed density and force kernels."""
import numpy as np
import pytest

import test_gpu_sph as small
from miluphpc_amd import ics
from conftest import print_case

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def sedov33():
    return small.perturbed_sedov(33)


@pytest.fixture(scope="module")
def sedov37():
    return small.perturbed_sedov(37)


def test_neighbour_sets_groups(gpu_lib, orc, sedov33):
    small.test_neighbour_sets_bitexact(gpu_lib, orc, sedov33)


@pytest.mark.parametrize("cap", [0.0, 1.3])
def test_h_iteration_groups(gpu_lib, orc, sedov33, cap):
    small.test_h_iteration_bitexact(gpu_lib, orc, sedov33, cap)


@pytest.mark.parametrize("drop", [104, 92])   # the last window holds 505 particles, 5
def test_lists_ragged_last_window_groups(gpu_lib, orc, sedov33, drop):
    assert (len(sedov33["x"]) - drop) % 512 in (505, 5)
    small.test_lists_ragged_last_window(gpu_lib, orc, sedov33, drop)


def test_outlier_particles_groups(gpu_lib, orc, sedov33):
    small.test_outlier_particles_match_oracle(gpu_lib, orc, sedov33)


@pytest.mark.parametrize("precision", [0, 1])
def test_speculative_lists_groups(gpu_lib, orc, sedov33, precision):
    small.test_speculative_lists_equal_plain(gpu_lib, orc, sedov33, precision)


def test_neighbour_capacity_groups(gpu_lib, sedov33):
    """The walks' append with its capacity check, in the plain and the speculative form."""
    small.test_neighbour_capacity_error(gpu_lib, sedov33)
    p = gpu_lib.default_params(max_nb=16)
    with small.make_ctx(gpu_lib, sedov33, p) as ctx:
        with pytest.raises(gpu_lib.MhpcError) as e:
            ctx.rhs(gpu_lib.RHS_SPH | gpu_lib.RHS_VARIABLE_SML | gpu_lib.RHS_SPECULATIVE_NN)
        assert e.value.status == gpu_lib.E_CAP_NEIGHBOURS


@pytest.mark.parametrize("curve", [0, 1])
def test_clustered_groups(gpu_lib, orc, curve):
    print_case(f"plummer 40000 clustered h, curve {curve}")
    s = small.clustered(40000)
    h0 = 0.7 * s["sml"]
    st, oh, oiters, _ = orc.h_iterate(s["x"], s["y"], s["z"], h0)
    assert st == 0
    st, onnl, onoi = orc.nn_brute(s["x"], s["y"], s["z"], oh, 180)
    assert st == 0
    for spec in (0, gpu_lib.RHS_SPECULATIVE_NN):
        with small.make_ctx(gpu_lib, {**s, "sml": h0}, gpu_lib.default_params(curve=curve)) as ctx:
            ctx.rhs(gpu_lib.RHS_SPH | gpu_lib.RHS_VARIABLE_SML | spec)
            assert np.array_equal(ctx.download("sml"), oh)
            assert np.array_equal(ctx.download("h_iters"), oiters)
            assert small.sets(*ctx.neighbour_lists()) == small.sets(onnl, onoi)


@pytest.mark.parametrize("cap", [1.02, 1.1])
def test_h_iteration_frozen_tail_groups(gpu_lib, orc, cap):
    """Lattice faces held at sml_max (the tail passes repeat the last count): the plain stage and the
    speculative RHS equal the oracle, which iterates every pass."""
    print_case(f"frozen tail 33^3, sml_max {cap} x h0")
    s = ics.sedov_lattice(33)
    h0 = s["sml"].copy()
    sml_max = cap * h0.max()
    H = [orc.h_iterate(s["x"], s["y"], s["z"], h0, max_counts=u + 1, sml_max=sml_max)[1] for u in range(4)]
    st, oh, oiters, onoi = orc.h_iterate(s["x"], s["y"], s["z"], h0, sml_max=sml_max)
    assert st == 0
    F = 2 if cap < 1.05 else 3   # the first pass whose predecessor changed no h
    assert np.array_equal(H[F], H[F - 1]) and not np.array_equal(H[F - 1], H[F - 2])
    assert (oiters == 7).sum() > 100
    p = gpu_lib.default_params(curve=1, sml_max=sml_max)
    with small.make_ctx(gpu_lib, s, p) as ctx:
        ctx.bbox(); ctx.keys(); ctx.sort(); ctx.build_tree()
        ctx.h_iterate()
        for k, o in (("sml", oh), ("h_iters", oiters), ("noi", onoi)):
            assert np.array_equal(ctx.download(k), o), k
    with small.make_ctx(gpu_lib, s, p) as ctx:
        stats = ctx.rhs(gpu_lib.RHS_SPH | gpu_lib.RHS_VARIABLE_SML | gpu_lib.RHS_SPECULATIVE_NN)
        for k, o in (("sml", oh), ("h_iters", oiters), ("noi", onoi)):
            assert np.array_equal(ctx.download(k), o), k
    assert stats["n_h_counts"] == int(oiters.sum())


@pytest.mark.parametrize("precision", [0, 1])
def test_sph_rhs_windows(gpu_lib, orc, sedov37, precision):
    small.test_sph_rhs_parity(gpu_lib, orc, sedov37, precision)


@pytest.mark.parametrize("kernel", [0, 2, 3, 4])
@pytest.mark.parametrize("precision", [0, 1])
def test_smoothing_kernels_windows(gpu_lib, orc, sedov37, kernel, precision):
    small.test_smoothing_kernels_match_oracle(gpu_lib, orc, sedov37, kernel, precision)


@pytest.mark.parametrize("kernel", [1, 2])
@pytest.mark.parametrize("precision", [0, 1])
def test_features_windows(gpu_lib, orc, sedov37, kernel, precision):
    """|curl v| and |grad rho| (the learned smoothing length's inputs) of the windowed force kernel."""
    print_case(f"learned-h features 37^3, kernel {kernel} precision={precision}")
    s = sedov37
    p = gpu_lib.default_params(curve=1, precision=precision, smoothing_kernel=kernel)
    with small.make_ctx(gpu_lib, s, p) as ctx:
        ctx.rhs(gpu_lib.RHS_SPH | gpu_lib.RHS_VARIABLE_SML | gpu_lib.RHS_FEATURES)
        f = {k: ctx.download(k) for k in ("sml", "rho", "curlv", "gradrho")}
        nnl, noi = ctx.neighbour_lists(180)
    curl, grad = orc.sph_features(*(s[k] for k in ("x", "y", "z", "vx", "vy", "vz", "mass")), f["sml"], f["rho"], nnl,
                                  noi, kernel=kernel)
    for got, o in ((f["curlv"], curl), (f["gradrho"], grad)):
        want = np.linalg.norm(o, axis=1)
        # sums of up to 180 signed terms: their rounding against the largest sum
        assert np.abs(got - want).max() <= (1e-12 if precision == 0 else 1e-5) * want.max()
