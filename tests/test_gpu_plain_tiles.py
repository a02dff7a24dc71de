"""Depth of the plain path's emission tiles (uw_build_chunks_plain): chunk sets on both sides of the counts
where the rule takes deeper or shallower x-slabs, and where the emission goes from a tile per workgroup to
the list of tiles. A chunk's mesh depends on neither: every chunk of a large launch equals the same chunk
in launches of three, bit for bit."""
import numpy as np
import pytest

from underwaterworld_amd import params as PR

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,counts", [(2, (1100, 2100)), (4, (300, 1100, 1600)), (8, (260, 700, 1100)), (12, (200, 600, 2100)),
                                      (14, (300, 1100)), (20, (260, 1100)), (33, (20, 70)), (40, (20, 70))])
def test_tile_depth_leaves_meshes_alone(n, counts):
    import torch
    from underwaterworld_amd import Perlin, build_chunks_plain
    perlin = Perlin(PR.preset("mixed", octaves=3))
    few = [((7 * i) % 13 - 6, (5 * i) % 11 - 5, i % 3 - 2) for i in range(12)]
    want = []
    for k in range(0, len(few), 3):
        b = build_chunks_plain(perlin, few[k:k + 3], n, collision=True)
        torch.cuda.synchronize()
        info = b.info()
        for i in range(3):
            r = info[i]
            col = b.chunk_collision(i, info) if r["n_inds"] else ()
            want.append(((r["flags"], r["n_verts"], r["n_inds"], r["n_active"]), *b.chunk_mesh(i, info), *col))
    assert sum(len(w[2]) for w in want) > 0
    for count in counts:
        b = build_chunks_plain(perlin, [few[i % 12] for i in range(count)], n, collision=True)
        torch.cuda.synchronize()
        info = b.info()
        for i in list(range(12)) + list(range(count - 12, count)):
            w, r = want[i % 12], info[i]
            assert (r["flags"], r["n_verts"], r["n_inds"], r["n_active"]) == w[0], (count, i)
            got = (*b.chunk_mesh(i, info), *(b.chunk_collision(i, info) if r["n_inds"] else ()))
            assert len(got) == len(w) - 1 and all(np.array_equal(x, y) for x, y in zip(got, w[1:])), (count, i)
        for key in ("flags", "n_verts", "n_inds", "n_active"):  # the chunks in between by their sizes
            assert np.array_equal(info[key], np.resize([info[key][i] for i in range(12)], count))
        assert np.array_equal(info["ind_off"], np.cumsum(info["n_inds"].astype(np.int64)) - info["n_inds"])
