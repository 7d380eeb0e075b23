"""The kernel that runs one wave per Metropolis chain where it shares a SIMD among
four waves and where a wave runs several chains one after the other (more chains
than the grid has waves: 1024 with one block of 256 per CU), for each way in
which a scene is traversed.  Chain by chain the accepted mutations equal the
wavefront's and the oracle's."""
import numpy as np
import pytest

from barnacle_amd import configs, native, scene
from test_gpu_flat import cubes

pytestmark = pytest.mark.gpu


def metropolis(n_instances, chains, strategy):
    info = configs.caustic_scene(width=61, height=52, spp=2, max_depth=6, freq=4, n_bootstrap=512, n_chains=chains)
    info["integrator"]["mutation-strategy"] = strategy
    return cubes(n_instances, 39.3, info["integrator"]) if n_instances else scene.load_scene(info)


def render(ctx, ds, waves):
    ctx.set_option("mlt_wave_chains", waves)
    p = ds.sc.mlt_params()
    film, st = ds.render_pssmlt(p)
    return film, st, ds.pssmlt_last(p)[1].copy()


def close(a, b):
    # the same contributions added in another order: at most a few hundred float additions a pixel
    ok = np.isfinite(b).all(axis=1)
    return np.array_equal(ok, np.isfinite(a).all(axis=1)) and \
        np.sqrt(np.sum((a[ok] - b[ok]) ** 2)) <= 1e-5 * np.sqrt(np.sum(b[ok] ** 2))


@pytest.mark.parametrize("records", [1, 0])
@pytest.mark.parametrize("strategy", ["Gaussian", "Kelemen"])
@pytest.mark.parametrize("n_instances,chains", [(0, 1024), (0, 1025), (0, 2500), (40, 1025), (40, 2500)])
def test_chains_of_a_wave(ctx, orc, n_instances, chains, strategy, records):
    print(f"{n_instances} instances, {chains} chains, {strategy}, records {records}", flush=True)
    sc = metropolis(n_instances, chains, strategy)
    ctx.set_option("records", records)
    ctx.set_option("trace_blocks_per_cu", 1)
    try:
        ds = ctx.scene(sc)
        film_f, st_f, acc_f = render(ctx, ds, 0)
        film_w, st_w, acc_w = render(ctx, ds, 1 << 20)
        ds.release()
    finally:
        ctx.set_option("records", 1)
        ctx.set_option("trace_blocks_per_cu", 7)
    assert np.array_equal(acc_w, acc_f) and st_w["accepted"] == st_f["accepted"] and st_w["b"] == st_f["b"]
    assert close(film_w, film_f)
    if records:
        ofilm, ost, _, oacc = orc.scene(sc).render_pssmlt(sc.mlt_params())
        assert np.array_equal(acc_w, oacc) and st_w["b"] == ost["b"]
        assert close(film_w, ofilm)


def test_another_limit(ctx):
    ctx.set_option("mlt_wave_chains", 20480)     # which the next test is not to see


def test_the_session_keeps_the_shipped_limit(ctx):
    """24,000 chains take the same kernels on the session's context, which other
    tests have used, and on a new one."""
    kernels = []
    new = native.Context(0)
    for c in (ctx, new):
        ds = c.scene(metropolis(0, 24000, "Gaussian"))
        c.set_option("timing", 1)
        c.reset_kernel_times()
        try:
            ds.render_pssmlt(ds.sc.mlt_params())
            kernels.append(sorted(c.kernel_times()))
        finally:
            c.set_option("timing", 0)
            ds.release()
    new.close()
    assert kernels[0] == kernels[1]
