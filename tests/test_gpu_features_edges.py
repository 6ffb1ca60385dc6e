"""The feature kernel where its waves, pairs and tables end: site counts around
a wave and a workgroup's chunk, the fewest and the most taxa, one and eight
categories, with and without gaps."""
import numpy as np
import pytest

from phylommand_amd import learn as L

from oracle import learn_oracle as LO

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n_taxa,n_sites,n_cat,gap", [
    (4, 1, 1, 0.0), (4, 63, 8, 0.1), (5, 64, 4, 0.0), (17, 65, 4, 0.05), (31, 257, 8, 0.08), (32, 511, 1, 0.02),
    (32, 513, 4, 0.05), (9, 1024, 2, 0.0), (24, 1100, 8, 0.3),
])
def test_features_match_the_oracle_at_the_edges(n_taxa, n_sites, n_cat, gap):
    """Pair features are sums of n_pairs floats of at most 3 / n_pairs in no
    fixed order: off by at most 3 n_pairs 2^-24; the transition / transversion
    ratio relatively by twice that; the deviation's square by as much."""
    print(f"features taxa={n_taxa} sites={n_sites} cat={n_cat} gap={gap}", flush=True)
    d = L.draw_models(3, n_taxa, np.random.default_rng(n_taxa + n_sites))
    d.gap[:] = gap
    f, masks = L.simulate_features(d, n_sites, n_cat=n_cat, seed=5, want_masks=True)
    tol = max(2e-6, 3 * n_taxa * (n_taxa - 1) / 2 * 2.0 ** -24)
    for k in range(3):
        ref = LO.features_from_states(LO.states_from_masks(masks[k]))
        got = f[k].astype(float)
        assert abs(got[185] ** 2 - ref[185] ** 2) <= 4 * tol
        got[185] = ref[185]
        np.testing.assert_allclose(got, ref, atol=tol, rtol=2 * tol, err_msg=f"alignment {k}")
    # the draws are counted by site: fewer sites are a prefix
    short = L.simulate_features(d, max(1, n_sites - 1), n_cat=n_cat, seed=5, want_masks=True)[1]
    np.testing.assert_array_equal(short, masks[:, :, :max(1, n_sites - 1)])
