"""SPRT preemptive verification (inc/preemption/preemption_sprt.h:206-379) in
the engine's main loop, against the oracle run with the same seed: identical
inlier masks and iteration / LO / graph-cut counts, models within 1e-12.

The device walks each pair's candidate models in the loop's order through
the random pool; the host makes the history updates of accepted models, the
validity checks and the best-model updates.  Cases: homography (the class
default ratio 0.01), fundamental with the API's 1e-5 and a larger ratio,
DEGENSAC on a plane-dominated scene (its homography fit takes the SPRT list
in pool order), essential with the reference's defaults, the adaptive
reordering sampler (whose rand() stream the pool shuffle shares), PROSAC,
and a batch mixing SPRT and full-scoring pairs.
"""
import numpy as np
import pytest

from pygcransac import synthetic

pytestmark = pytest.mark.gpu


def _same(st, so, M, Mo, mask, mo, rc, atol=1e-12):
    assert np.array_equal(mask, mo)
    for key in ("iteration_number", "local_optimization_number", "graph_cut_number"):
        assert st[key] == so[key], key
    if rc > 0:
        np.testing.assert_allclose(M, Mo, rtol=1e-12, atol=atol)


@pytest.mark.parametrize("seed,sampler", [(0, 0), (1, 1), (2, 0)])
def test_homography_sprt_matches_oracle(oracle, seed, sampler):
    import pygcransac
    sc = synthetic.homography_scene(synthetic.scene_seed(15, seed), n=2500, inlier_ratio=[0.3, 0.5, 0.15][seed])
    print("homography sprt seed=%d sampler=%d" % (seed, sampler), flush=True)
    H, mask = pygcransac.findHomography(sc["corr"], 480, 640, 480, 640, None, threshold=3.0, conf=0.99,
                                        spatial_coherence_weight=0.975, max_iters=10000, min_iters=50,
                                        use_sprt=True, sampler=sampler, neighborhood=0, neighborhood_size=8.0,
                                        use_space_partitioning=False, lo_number=50, seed=seed)
    st = pygcransac.last_stats()
    p = oracle.params(3.0, 0.99, 0.975, 10000, 50, sampler, 50, 8.0, seed, use_sprt=True)
    rc, Ho, mo, so = oracle.find_homography(sc["corr"], 480, 640, 480, 640, p)
    # at 15 % inliers the class-default test (epsilon 0.01) rejects the true
    # plane almost always: both runs exhaust the iterations without a model
    assert rc > 0 or seed == 2
    _same(st, so, H, Ho, mask, mo, rc)


@pytest.mark.parametrize("ratio,plane", [(1e-5, 0.0), (0.05, 0.0), (1e-5, 0.9)])
def test_fundamental_sprt_matches_oracle(oracle, ratio, plane):
    import pygcransac
    sc = synthetic.fundamental_scene(synthetic.scene_seed(15, 20 + int(plane * 10)), n=3000, inlier_ratio=0.4,
                                     plane_fraction=plane)
    print("fundamental sprt ratio=%g plane=%g" % (ratio, plane), flush=True)
    F, mask = pygcransac.findFundamentalMatrix(sc["corr"], 480, 640, 480, 640, None, threshold=1.0, conf=0.99,
                                               spatial_coherence_weight=0.0, max_iters=10000, min_iters=50,
                                               use_sprt=True, min_inlier_ratio_for_sprt=ratio, sampler=0,
                                               neighborhood=0, neighborhood_size=8.0, lo_number=50, seed=3)
    st = pygcransac.last_stats()
    p = oracle.params(1.0, 0.99, 0.0, 10000, 50, 0, 50, 8.0, 3, use_sprt=True, min_inlier_ratio_for_sprt=ratio)
    rc, Fo, mo, so = oracle.find_fundamental(sc["corr"], 480, 640, 480, 640, p)
    assert rc > 0
    _same(st, so, F, Fo, mask, mo, rc, atol=1e-14)


def test_essential_reference_defaults_with_sprt_match_oracle(oracle):
    import pygcransac
    sc = synthetic.essential_scene(synthetic.scene_seed(15, 40), n=4000, inlier_ratio=0.25)
    E, mask = pygcransac.findEssentialMatrix(sc["corr"], sc["K1"], sc["K2"], 768, 1024, 768, 1024, None,
                                             threshold=0.75, conf=0.99, spatial_coherence_weight=0.1,
                                             max_iters=10000, min_iters=50, use_sprt=True,
                                             min_inlier_ratio_for_sprt=0.01, sampler=0, neighborhood=1,
                                             neighborhood_size=20.0, lo_number=50, seed=8)
    st = pygcransac.last_stats()
    p = oracle.params(0.75, 0.99, 0.1, 10000, 50, 0, 50, 20.0, 8, neighborhood=1, use_sprt=True,
                      min_inlier_ratio_for_sprt=0.01)
    rc, Eo, mo, so = oracle.find_essential(sc["corr"], sc["K1"], sc["K2"], 768, 1024, 768, 1024, p)
    assert rc > 0
    _same(st, so, E, Eo, mask, mo, rc, atol=1e-14)


def test_adaptive_reordering_sampler_with_sprt_matches_oracle(oracle):
    import pygcransac
    sc = synthetic.homography_scene(synthetic.scene_seed(15, 60), n=2000, inlier_ratio=0.35)
    rng = np.random.default_rng(4)
    pr = np.where(sc["gt"], rng.uniform(0.4, 1.0, 2000), rng.uniform(0.0, 0.7, 2000))
    H, mask = pygcransac.findHomography(sc["corr"], 480, 640, 480, 640, pr, threshold=3.0, conf=0.99,
                                        spatial_coherence_weight=0.975, max_iters=5000, min_iters=50,
                                        use_sprt=True, sampler=4, neighborhood=0, neighborhood_size=8.0,
                                        use_space_partitioning=False, lo_number=50, sampler_variance=0.1, seed=6)
    st = pygcransac.last_stats()
    p = oracle.params(3.0, 0.99, 0.975, 5000, 50, 4, 50, 8.0, 6, probabilities=pr, sampler_variance=0.1,
                      use_sprt=True)
    rc, Ho, mo, so = oracle.find_homography(sc["corr"], 480, 640, 480, 640, p)
    _same(st, so, H, Ho, mask, mo, rc)


def test_batch_mixing_sprt_and_full_scoring(oracle):
    import pygcransac
    probs, refs = [], []
    for i in range(6):
        seed = synthetic.scene_seed(15, 80 + i)
        sprt = i % 2 == 0
        if i % 3 == 1:
            sc = synthetic.fundamental_scene(seed, n=2500, inlier_ratio=0.35)
            pb = dict(kind="fundamental", correspondences=sc["corr"], h1=480, w1=640, h2=480, w2=640,
                      threshold=1.0, spatial_coherence_weight=0.0, min_inlier_ratio_for_sprt=1e-5)
            p = oracle.params(1.0, 0.99, 0.0, 10000, 50, 0, 50, 8.0, 40 + i, use_sprt=sprt,
                              min_inlier_ratio_for_sprt=1e-5)
            refs.append(oracle.find_fundamental(sc["corr"], 480, 640, 480, 640, p))
        else:
            sc = synthetic.homography_scene(seed, n=1800, inlier_ratio=0.4)
            pb = dict(kind="homography", correspondences=sc["corr"], h1=480, w1=640, h2=480, w2=640,
                      threshold=3.0, spatial_coherence_weight=0.975, use_space_partitioning=False)
            p = oracle.params(3.0, 0.99, 0.975, 10000, 50, 0, 50, 8.0, 40 + i, use_sprt=sprt)
            refs.append(oracle.find_homography(sc["corr"], 480, 640, 480, 640, p))
        pb.update(conf=0.99, max_iters=10000, min_iters=50, use_sprt=sprt, sampler=0, neighborhood=0,
                  neighborhood_size=8.0, lo_number=50, seed=40 + i)
        probs.append(pb)
    res = pygcransac.findBatch(probs)
    stats = pygcransac.last_batch_stats()
    for i, ((M, mask), (rc, Mo, mo, so)) in enumerate(zip(res, refs)):
        assert stats[i]["status"] == rc, i
        _same(stats[i], so, M, Mo, mask, mo, rc, atol=1e-14)


# Sizes at the edges of the walk's 64-position words and of the 64 words that
# the lanes hold at once (4,096 points), and far beyond (later words come from
# memory), with and without the space partitioning cells.
@pytest.mark.parametrize("n", [8, 63, 64, 65, 129, 4095, 4096, 4097, 65537])
@pytest.mark.parametrize("sp,sampler", [(False, 0), (True, 1)])
def test_homography_sprt_walk_sizes_match_oracle(oracle, n, sp, sampler):
    import pygcransac
    sc = synthetic.homography_scene(synthetic.scene_seed(15, 300 + n), n=n, inlier_ratio=0.6)
    print("homography sprt walk n=%d sp=%d" % (n, sp), flush=True)
    H, mask = pygcransac.findHomography(sc["corr"], 480, 640, 480, 640, None, threshold=3.0, conf=0.99,
                                        spatial_coherence_weight=0.975, max_iters=1000, min_iters=50,
                                        use_sprt=True, sampler=sampler, neighborhood=0, neighborhood_size=16.0,
                                        use_space_partitioning=sp, lo_number=20, seed=n)
    st = pygcransac.last_stats()
    p = oracle.params(3.0, 0.99, 0.975, 1000, 50, sampler, 20, 16.0, n, use_sprt=True, use_space_partitioning=sp)
    rc, Ho, mo, so = oracle.find_homography(sc["corr"], 480, 640, 480, 640, p)
    _same(st, so, H, Ho, mask, mo, rc, atol=1e-9)


@pytest.mark.parametrize("n", [63, 64, 65, 4097])
def test_fundamental_sprt_walk_sizes_match_oracle(oracle, n):
    import pygcransac
    sc = synthetic.fundamental_scene(synthetic.scene_seed(15, 400 + n), n=n, inlier_ratio=0.6)
    F, mask = pygcransac.findFundamentalMatrix(sc["corr"], 480, 640, 480, 640, None, threshold=1.0, conf=0.99,
                                               spatial_coherence_weight=0.0, max_iters=2000, min_iters=50,
                                               use_sprt=True, sampler=0, neighborhood=0, neighborhood_size=8.0,
                                               lo_number=50, seed=n)
    st = pygcransac.last_stats()
    p = oracle.params(1.0, 0.99, 0.0, 2000, 50, 0, 50, 8.0, n, use_sprt=True, min_inlier_ratio_for_sprt=1e-5)
    rc, Fo, mo, so = oracle.find_fundamental(sc["corr"], 480, 640, 480, 640, p)
    _same(st, so, F, Fo, mask, mo, rc, atol=1e-12)


def test_windows_of_eight_models_match_one_window(monkeypatch):
    """The models of a walk come in windows bounded by the bit rows' memory; the
    test's state (delta, A, the pool position, the last tested model and its
    inlier list) passes from one to the next.  A budget that leaves eight models
    a window, and one that the longest slot list crosses a few times, against
    the default: the same bits, with and without space partitioning, SPRT pairs
    beside a fully scored one."""
    import pygcransac
    probs = []
    for i, (kind, n, eps, sp) in enumerate([("homography", 1500, 0.2, False), ("homography", 2100, 0.25, True),
                                            ("fundamental", 1800, 0.3, False), ("homography", 700, 0.3, True),
                                            ("essential", 1200, 0.3, False), ("homography", 900, 0.4, False)]):
        sc = getattr(synthetic, kind + "_scene")(synthetic.scene_seed(15, 500 + i), n=n, inlier_ratio=eps)
        pb = dict(kind=kind, correspondences=sc["corr"], h1=768, w1=1024, h2=768, w2=1024, threshold=2.0, conf=0.99,
                  spatial_coherence_weight=0.5, max_iters=6000, min_iters=3000, use_sprt=i != 5, sampler=i % 2,
                  neighborhood=0, neighborhood_size=8.0, lo_number=20, seed=60 + i, min_inlier_ratio_for_sprt=0.01)
        if kind == "homography":
            pb["use_space_partitioning"] = sp
        if kind == "essential":
            pb.update(K1=sc["K1"], K2=sc["K2"])
        probs.append(pb)
    runs = []
    for words in (None, "1", "40000"):
        if words is None:
            monkeypatch.delenv("GCR_SPRT_WINDOW_WORDS", raising=False)
        else:
            monkeypatch.setenv("GCR_SPRT_WINDOW_WORDS", words)
        print("sprt window words:", words, flush=True)
        runs.append((pygcransac.findBatch(probs), pygcransac.last_batch_stats()))
    (r0, s0) = runs[0]
    assert sum(int(m.sum()) for _, m in r0) > 500
    for r, s in runs[1:]:
        for i, ((Ma, ma), (Mb, mb)) in enumerate(zip(r0, r)):
            assert np.array_equal(ma, mb), i
            assert (Ma is None) == (Mb is None), i
            if Ma is not None:
                assert np.array_equal(Ma.view(np.uint64), Mb.view(np.uint64)), i
            for key in ("iteration_number", "local_optimization_number", "graph_cut_number", "num_inliers", "score",
                        "models_scored"):
                assert s0[i][key] == s[i][key], (i, key)
