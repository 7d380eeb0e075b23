"""Metropolis rendering with few chains runs one wave per chain; with many, a
wavefront over all of them.  Both follow every chain's trajectory exactly: B
and the accepted mutations of every chain equal the oracle's, whatever the
number of chains, bounces and mutations (a launch holds at most 1024 a chain)."""
import numpy as np
import pytest

from barnacle_amd import configs, scene

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("waves", [0, 1 << 20])
@pytest.mark.parametrize("strategy", ["Gaussian", "Kelemen"])
@pytest.mark.parametrize("chains,size,depth", [(1, 12, 8), (1, 33, 1), (2, 16, 0), (257, 30, 16)])
def test_chains_match_the_oracle(ctx, orc, chains, size, depth, strategy, waves):
    info = configs.caustic_scene(width=size, height=size, spp=1, max_depth=depth, freq=4, n_bootstrap=512,
                                 n_chains=chains, sigma=1.0 / 64.0, large_step=0.3)
    info["integrator"]["mutation-strategy"] = strategy
    sc = scene.load_scene(info)
    p = sc.mlt_params()
    print(f"{chains} chains, {size}x{size}, depth {depth}, {strategy}, waves {waves}", flush=True)
    ds = ctx.scene(sc)
    ctx.set_option("mlt_wave_chains", waves)
    try:
        film, st = ds.render_pssmlt(p)
        boot, acc = ds.pssmlt_last(p)
    finally:
        ctx.set_option("mlt_wave_chains", 20480)
        ds.release()
    ofilm, ost, oboot, oacc = orc.scene(sc).render_pssmlt(p)
    assert np.array_equal(boot.view(np.int32), oboot.view(np.int32)) and st["b"] == ost["b"]
    assert np.array_equal(acc, oacc) and st["accepted"] == ost["accepted"]
    ok = np.isfinite(ofilm).all(axis=1)
    assert np.array_equal(ok, np.isfinite(film).all(axis=1))
    # the same contributions added in another order: at most a few hundred float additions a pixel
    assert np.sqrt(np.sum((film[ok] - ofilm[ok]) ** 2)) <= 1e-5 * np.sqrt(np.sum(ofilm[ok] ** 2))
