"""An infinite vertex gradient: the field's offset gradient is infinite along every axis on which the two
endpoint densities of the vertex move the same way (their terms have one sign), and NaN where they don't.
The terrace bias has no slope, so z follows the rule of x and y."""
import numpy as np
import pytest

from underwaterworld_amd import params as PR

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("volume", [False, True])
def test_offset_gradient_of_an_infinite_vertex_gradient(volume):
    import torch
    from underwaterworld_amd import Perlin, density_at
    from underwaterworld_amd.adjoint import ChunkMesher, VolumeMesher
    n, chunk = 12, (0, 0, -1)
    p = PR.preset("reference", offset=(0.3, 0.4, 0.1))
    assert p["bias_kind"] == PR.BIAS_TERRACE
    perlin = Perlin(p)
    mesher = VolumeMesher(perlin, n, chunk) if volume else ChunkMesher(perlin, [chunk], n)
    rec = mesher.forward()
    torch.cuda.synchronize()
    nv = int(rec.batch.info()["n_verts"][0])
    tape = rec.tape[:nv].cpu().numpy()
    seen = np.zeros((3, 2), int)
    for v in range(0, nv, max(1, nv // 60)):
        # signs of d rho / d offset at the two endpoints, by central differences of the noise alone (the
        # steps of the terrace have no gradient): the bias is taken out by its own value at each point
        ends = []
        for s in tape[v, :2]:
            i = np.array([s // (n + 1) ** 2, s // (n + 1) % (n + 1), s % (n + 1)], np.float64)
            x = (i * (p["chunk_extent"] / n) + np.array(chunk) * p["chunk_extent"]) * p["frequency"]  # (density_at adds the offset)
            h = 1e-3
            pts = np.array([x + k * h * np.eye(3)[a] for a in range(3) for k in (1, -1)])
            rho = density_at(perlin, pts).cpu().numpy().astype(np.float64)
            z = (pts[:, 2] + p["offset"][2] * p["frequency"]).astype(np.float32)
            adj = (z * np.float32(p["bias"][0])) / np.float32(p["bias"][1])
            noise = rho - (adj - np.fmod(adj, np.float32(p["bias"][2]))).astype(np.float64)
            ends.append((noise[0::2] - noise[1::2]) / (2 * h))
        g = torch.zeros((max(nv, rec.batch.verts.shape[0]), 3), device="cuda")
        g[v] = float("inf")  # (only the axis of the vertex's edge counts)
        got = mesher.backward(g, record=rec).grad_off.cpu().numpy().reshape(-1)[:3]
        for a in range(3):
            lo, hi = sorted(abs(e[a]) for e in ends)
            if lo < 0.05:  # too flat for the differences to tell the sign
                continue
            same = np.sign(ends[0][a]) == np.sign(ends[1][a])
            assert np.isinf(got[a]) if same else np.isnan(got[a]), (v, a, got, ends)
            seen[a, int(same)] += 1
    assert (seen[:, 1] > 5).all(), seen
