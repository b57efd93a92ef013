"""Majorants by a lane per cell and by groups of lanes, around the sizes at which one
takes over from the other, against the CPU oracle."""
import numpy as np
import pytest

from mdwtracker_amd import scenes

pytestmark = pytest.mark.gpu


# entries 4096 and 4104 (tables of up to 32 texels), 16384 and 16400 (up to 128),
# 65536 and 65550 (longer ones), with ranges below, at and above the 16 texels that a
# lane takes alone
@pytest.mark.parametrize("cells,texels", [((16, 16, 16), 12), ((19, 18, 12), 32), ((32, 32, 16), 36),
                                          ((41, 40, 10), 128), ((64, 32, 32), 132), ((46, 57, 25), 132),
                                          ((46, 57, 25), 700)])
@pytest.mark.parametrize("conservative", [False, True])
@pytest.mark.parametrize("mode", [2, 5])
def test_both_kernels_match_the_oracle(cells, texels, conservative, mode):
    from mdwtracker_amd import capi
    from oracle import pyoracle
    rng = np.random.default_rng(texels + cells[0])
    # smooth along x, noise in one corner, a constant slab (one value per range)
    v = np.broadcast_to(np.linspace(0, 60000, 70), (40, 160, 70)).astype(np.uint16)
    v[:20, :80] = rng.integers(0, 65536, (20, 80, 70))
    v[30:] = 777
    tfs = [rng.uniform(0, 1, (texels, 4)).astype(np.float32), rng.uniform(0, 1, (max(texels // 3, 1), 4)).astype(np.float32)]
    channels = 1 if mode == 2 else 2
    out = []
    for r in (capi.MdwtRenderer(0), pyoracle.OracleRenderer()):
        for c in range(channels):
            r.push_channel(v if c == 0 else np.ascontiguousarray(v[:, ::-1]))
        r.init(mode, cells, False)
        r.set_conservative_majorants(conservative)
        for c in range(channels):
            r.set_tf(c, tfs[c], 0.7, ((0.0, 1.0), (0.8, 0.2))[c])
        out.append(r.read_majorants().view(np.uint32))
        r.close()
    print(f"[majorants] {cells} texels {texels} mode {mode} conservative {conservative}", flush=True)
    assert len(np.unique(out[1])) > 3
    np.testing.assert_array_equal(*out)
