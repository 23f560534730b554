"""The kernels that take 64 cells per block (csrc/block_rates.h), against the CPU oracle bit for
bit at the sizes where their dispatch and their last block change."""
import numpy as np
import pytest

from pelelmex_amd import workloads as W

pytestmark = pytest.mark.gpu

KEYS = {"ode.rtol": 1e-10, "ode.atol": 1e-10}


def _bits(name, got, ref):
    assert np.array_equal(got, ref, equal_nan=True), \
        f"{name}: {int(np.sum(got != ref))} of {got.size} entries differ from the oracle's"


BOXES = {"LiDryer": W.h2_air_box, "drm19": W.ch4_air_flame_box, "dodecane_lu": W.dodecane_box, "syn53": W.syn53_chunk}


# 256 CUs: the block kernel from 12288 cells (6144 above 32 components); whole last block, one cell
# in it, all but one
@pytest.mark.parametrize("mech,dims", [("drm19", (12288, 1, 1)), ("drm19", (12289, 1, 1)), ("drm19", (85, 17, 9)),
                                       ("drm19", (12287, 1, 1)), ("LiDryer", (31, 21, 19)), ("dodecane_lu", (89, 23, 3)),
                                       ("syn53", (79, 39, 2))])
def test_reaction_rates_64_cells_per_block(gpu, mech, dims):
    """reactionRateRhoY over ragged and masked boxes, in MKS, T started 25 K off."""
    import torch
    from oracle import pyoracle as po
    from pelelmex_amd.reactor import Reactor
    nx, ny, nz = dims
    nc = nx * ny * nz
    box = BOXES[mech](nx=nx, ny=ny, nz=nz)
    m = po.Mech(mech)
    rY, rH = box["rY"] * 1e3, box["rH"] * 0.1
    T0 = box["T"] + 25.0 * np.sin(np.arange(nc))
    ref, _ = m.rate_rhoY(rY, rH, T0)
    mask = np.ones(nc, dtype=np.int32)
    mask[::7] = -1
    mask[-1] = 1
    ref[:, mask == -1] = 0.0
    r = Reactor.create("ReactorCvode", mech, KEYS)
    r.init(2, 1)
    dev = lambda a, *shape: torch.as_tensor(np.ascontiguousarray(a)).reshape(*shape).to(gpu).contiguous()
    out = torch.full((m.nsp, nz, ny, nx), float("nan"), dtype=torch.float64, device=gpu)
    r.reaction_rate_rhoY(dev(rY, m.nsp, nz, ny, nx), dev(rH, nz, ny, nx), dev(T0, nz, ny, nx),
                         mask=dev(mask, nz, ny, nx), rYdot=out)
    r.close()
    _bits("rYdot", out.cpu().numpy().reshape(m.nsp, nc), ref)
