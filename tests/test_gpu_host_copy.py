"""Results reach the caller's arrays whole: of a few bytes (less than the copy
kernel's 16-byte words), of several parts whose borders lie inside its pieces,
and larger than its 16 MB buffer."""
import numpy as np
import pytest

from barnacle_amd import configs, scene

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("size", [(1, 1), (3, 1), (1365, 1), (1201, 1193)])
def test_first_hits_arrive_whole(ctx, orc, size):
    w, h = size
    sc = scene.load_scene(configs.config1(width=w, height=h, spp=1, freq=6))
    p = sc.pt_params()
    print(f"first hits {w}x{h}", flush=True)
    ds = ctx.scene(sc)
    ref = orc.scene(sc).first_hit(p)
    for _ in range(2):                                      # the second from a buffer that holds the first
        got = ds.first_hit(p)
        for g, r in zip(got, ref):
            assert np.array_equal(g.view(np.int32), r.view(np.int32))
    ds.release()


def test_batched_films_of_odd_sizes_arrive_whole(ctx):
    sc = scene.load_scene(configs.config1(width=64, height=64, spp=1, freq=6, max_depth=2))
    ds = ctx.scene(sc)
    jobs = []
    for w, h in [(1, 1), (37, 3), (1, 5), (129, 65), (1000, 1001), (31, 17)]:
        p = sc.pt_params()
        p.width, p.height = w, h
        jobs.append((ds, p))
    films, _ = ctx.render_batch(jobs)
    for (_, p), film in zip(jobs, films):
        assert np.array_equal(film.view(np.int32), ds.render_pt(p).view(np.int32))
    ds.release()
