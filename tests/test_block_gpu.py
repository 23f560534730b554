"""Launches whose kernel depends on the number of cells, at the sizes where it changes: the kernels
that take 64 cells per block (csrc/block_rates.h) against the CPU oracle bit for bit, and the BDF's
variants for small launches against the one of large launches."""
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


# the same sizes without a mask (with one the line is five times as high)
@pytest.mark.parametrize("mech,dims", [("drm19", (12288, 1, 1)), ("drm19", (12289, 1, 1)), ("drm19", (85, 17, 9)),
                                       ("LiDryer", (31, 21, 19)), ("dodecane_lu", (89, 23, 3)), ("syn53", (79, 39, 2)),
                                       ("drm19", (61441, 1, 1)), ("dodecane_lu", (30721, 1, 1))])
def test_reaction_rates_64_cells_per_block_without_mask(gpu, mech, dims):
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
    r = Reactor.create("ReactorCvode", mech, KEYS)
    r.init(2, 1)
    dev = lambda a, *shape: torch.as_tensor(np.ascontiguousarray(a)).reshape(*shape).to(gpu).contiguous()
    args = dev(rY, m.nsp, nz, ny, nx), dev(rH, nz, ny, nx), dev(T0, nz, ny, nx)
    _bits("rYdot", r.reaction_rate_rhoY(*args).cpu().numpy().reshape(m.nsp, nc), ref)
    # nothing covered: the masked kernel on either side of its line
    mask = torch.ones((nz, ny, nx), dtype=torch.int32, device=gpu)
    _bits("rYdot", r.reaction_rate_rhoY(*args, mask=mask).cpu().numpy().reshape(m.nsp, nc), ref)
    r.close()


# more rounds of 64 cells than blocks, so that a block's uncovered cells come from several rounds
@pytest.mark.parametrize("mech,dims", [("drm19", (67, 45, 51)), ("dodecane_lu", (61, 29, 23))])
@pytest.mark.parametrize("pattern", ["all", "last", "sparse", "slab", "half"])
def test_reaction_rates_of_mostly_covered_boxes(gpu, mech, dims, pattern):
    """The uncovered cells' rates are those without a mask, whatever else is covered (zero rates there)."""
    import torch
    from pelelmex_amd.reactor import Reactor
    nx, ny, nz = dims
    nc = nx * ny * nz
    box = BOXES[mech](nx=nx, ny=ny, nz=nz)
    covered = {"all": np.ones(nc, bool), "last": np.arange(nc) < nc - 1, "slab": np.arange(nc) >= nc // 5,
               "sparse": np.random.default_rng(1).random(nc) < 0.97, "half": np.random.default_rng(2).random(nc) < 0.5}[pattern]
    r = Reactor.create("ReactorCvode", mech, KEYS)
    r.init(2, 1)
    dev = lambda a, *s: torch.as_tensor(np.ascontiguousarray(a)).reshape(*s, nz, ny, nx).to(gpu).contiguous()
    rY, rH, T = dev(box["rY"] * 1e3, r.nsp), dev(box["rH"] * 0.1), dev(box["T"])
    mask = dev(np.where(covered, -1, 1).astype(np.int32))
    want = r.reaction_rate_rhoY(rY, rH, T)  # against the oracle above
    want[:, mask == -1] = 0.0
    out = torch.full_like(want, float("nan"))
    r.reaction_rate_rhoY(rY, rH, T, mask=mask, rYdot=out)
    r.close()
    assert torch.equal(out, want)


def test_covered_cells_cost_no_rates(gpu):
    """A covered box takes a fraction of the time (about a quarter; 0.8 with rates formed for every cell)."""
    import time
    import torch
    from pelelmex_amd.reactor import Reactor, box_tensors
    t = box_tensors(W.ch4_air_flame_box(nx=64, ny=64, nz=64), gpu)
    rY, rH, out = t["rY"] * 1e3, t["rH"] * 0.1, torch.empty_like(t["rY"])
    r = Reactor.create("ReactorCvode", "drm19", KEYS)
    r.init(2, 1)
    took = []
    for m in (1, -1):
        mask = torch.full(t["T"].shape, m, dtype=torch.int32, device=gpu)
        ts = []
        for _ in range(20):
            torch.cuda.synchronize()
            t0 = time.perf_counter()
            r.reaction_rate_rhoY(rY, rH, t["T"], mask=mask, rYdot=out)
            ts.append(time.perf_counter() - t0)
        took.append(float(np.median(ts)))
    r.close()
    assert took[1] < 0.6 * took[0]


LARGE = {"LiDryer": (16, 3), "drm19": (32, 4), "dodecane_lu": (64, 2), "syn53": (64, 2)}


@pytest.mark.parametrize("mech,cells,lanes,waves", [
    ("LiDryer", 1, 64, 2), ("LiDryer", 2048, 64, 2), ("LiDryer", 2049, 32, 3), ("LiDryer", 7168, 32, 3),
    ("LiDryer", 7169, 16, 3), ("LiDryer", 28673, 16, 4), ("drm19", 1, 64, 2), ("drm19", 6144, 64, 2),
    ("drm19", 6145, 32, 4), ("dodecane_lu", 6144, 64, 2), ("dodecane_lu", 6145, 64, 3), ("syn53", 6145, 64, 3)])
def test_react_variant_by_size(gpu, mech, cells, lanes, waves):
    """A launch's variant follows its cell count unless a key chooses one; the bits do not."""
    import torch
    from pelelmex_amd.reactor import Reactor, box_tensors
    box = BOXES[mech](nx=cells, ny=1, nz=1)
    out = []
    for keys in (KEYS, dict(KEYS, **{"hipbdf.lanes_per_cell": LARGE[mech][0], "hipbdf.waves_per_simd": LARGE[mech][1]})):
        r = Reactor.create("ReactorCvode", mech, dict(keys, **{"cvode.max_order": 4}))
        r.init(2, 1)
        t = box_tensors(box, gpu)
        nfail, _, _ = r.react(t["rY"], t["rYsrc"], t["T"], t["rH"], t["rHsrc"], t["FC"], t["mask"], box["dt"], 0.0)
        torch.cuda.synchronize()
        out.append([t[k].cpu().numpy() for k in ("rY", "T", "rH", "FC")] + [nfail, r.stats()])
        r.close()
    assert (out[0][5]["lanes_per_cell"], out[0][5]["waves_per_simd"]) == (lanes, waves)
    for k in range(4):
        _bits(("rY", "T", "rH", "FC")[k], out[0][k], out[1][k])
    assert out[0][4] == out[1][4] and all(out[0][5][k] == out[1][5][k] for k in ("nst", "nfe", "nje", "nsetups", "nni"))


# 64 cells per block of setTemperature (32 with 8 lanes per cell): one cell, all but one, one more
@pytest.mark.parametrize("mech,cells", [("drm19", 1), ("drm19", 63), ("drm19", 64), ("drm19", 65), ("LiDryer", 17),
                                        ("dodecane_lu", 1), ("dodecane_lu", 31), ("dodecane_lu", 33), ("syn53", 100)])
def test_set_temperature_rows(gpu, mech, cells):
    import torch
    from oracle import pyoracle as po
    from pelelmex_amd.reactor import Reactor
    box = BOXES[mech](nx=cells, ny=1, nz=1)
    m = po.Mech(mech)
    rY, rH = box["rY"] * 1e3, box["rH"] * 0.1
    rho, T0 = rY.sum(0), box["T"] + 25.0 * np.sin(np.arange(cells))
    r = Reactor.create("ReactorCvode", mech, KEYS)
    r.init(2, 1)
    dev = lambda a, *shape: torch.as_tensor(np.ascontiguousarray(a)).reshape(*shape).to(gpu).contiguous()
    T = dev(T0, 1, 1, cells).clone()
    r.set_temperature(dev(rho, 1, 1, cells), dev(rY, m.nsp, 1, 1, cells), dev(rH, 1, 1, cells), T)
    r.close()
    _bits("T", T.cpu().numpy().reshape(-1), m.set_temperature(rho, rY, rH, T0))


# a block writes its cells' Jacobians together: one cell, a part of a block, whole blocks and one more,
# through the LU area (8, 16 lanes), extra LDS (32) and straight from the group (64)
@pytest.mark.parametrize("mech,lanes", [("LiDryer", 8), ("LiDryer", 16), ("drm19", 16), ("drm19", 32), ("drm19", 64),
                                        ("dodecane_lu", 64)])
@pytest.mark.parametrize("cells", [1, 7, 33])
def test_jacobians_by_block(gpu, mech, lanes, cells):
    import torch
    from oracle import pyoracle as po
    from pelelmex_amd.reactor import Reactor
    box = BOXES[mech](nx=cells, ny=1, nz=1)
    m = po.Mech(mech)
    y = np.vstack([box["rY"], box["T"][None, :]])
    ref = np.zeros((m.nsp + 1, m.nsp + 1, cells))
    for c in range(cells):
        ref[:, :, c] = m.jac(m.cell(box["rH"][c], box["rHsrc"][c], box["rYsrc"][:, c]), 0.0, y[:, c])
    r = Reactor.create("ReactorCvode", mech, dict(KEYS, **{"hipbdf.lanes_per_cell": lanes}))
    r.init(2, 1)
    dev = lambda a: torch.as_tensor(np.ascontiguousarray(a), dtype=torch.float64).to(gpu)
    J = r.jac_batch(dev(y), dev(box["rYsrc"]), dev(box["rHsrc"])).cpu().numpy()
    r.close()
    _bits("jac", J, ref)


@pytest.mark.parametrize("lanes,waves", [(64, 2), (32, 3), (16, 4)])
def test_rule_variants_by_key(gpu, lanes, waves):
    """What the size rules launch can be chosen by key too, with the same bits."""
    import torch
    from pelelmex_amd.reactor import Reactor, box_tensors
    box = W.h2_air_box(nx=67, ny=1, nz=1)
    out = []
    for keys in ({"hipbdf.lanes_per_cell": 8}, {"hipbdf.lanes_per_cell": lanes, "hipbdf.waves_per_simd": waves}):
        r = Reactor.create("ReactorCvode", "LiDryer", dict(KEYS, **keys))
        r.init(2, 1)
        t = box_tensors(box, gpu)
        r.react(t["rY"], t["rYsrc"], t["T"], t["rH"], t["rHsrc"], t["FC"], t["mask"], box["dt"], 0.0)
        torch.cuda.synchronize()
        out.append({k: t[k].cpu().numpy() for k in ("rY", "T", "rH", "FC")})
        st = r.stats()
        t = box_tensors(box, gpu)  # the other kernels of the handle take its lanes as well
        y = torch.cat([t["rY"].reshape(-1, 67), t["T"].reshape(1, 67)]).contiguous()
        src, rHsrc = t["rYsrc"].reshape(-1, 67).contiguous(), t["rHsrc"].reshape(67)
        out[-1]["rhs"] = r.rhs_batch(y, src, t["rH"].reshape(67), rHsrc).cpu().numpy()
        out[-1]["jac"] = r.jac_batch(y, src, rHsrc).cpu().numpy()
        out[-1]["rates"] = r.reaction_rate_rhoY(t["rY"] * 1e3, t["rH"] * 0.1, t["T"]).cpu().numpy()
        r.close()
    assert (st["lanes_per_cell"], st["waves_per_simd"]) == (lanes, waves)
    for k in out[0]:
        _bits(k, out[1][k], out[0][k])


def test_autotune_leaves_small_boxes_to_the_size_rules(gpu):
    """A first box too small to tell variants apart chooses none: the launch is the one without the key."""
    from pelelmex_amd.reactor import Reactor, box_tensors
    box = W.h2_air_box(nx=100, ny=1, nz=1)
    r = Reactor.create("ReactorCvode", "LiDryer", dict(KEYS, **{"hipbdf.autotune": 1}))
    r.init(2, 1)
    t = box_tensors(box, gpu)
    r.react(t["rY"], t["rYsrc"], t["T"], t["rH"], t["rHsrc"], t["FC"], t["mask"], box["dt"], 0.0)
    st = r.stats()
    r.close()
    assert (st["lanes_per_cell"], st["waves_per_simd"]) == (64, 2)


def _alike(mech, cells, at):
    """A box of one cell's state, the one at this place in the order of temperatures."""
    full = BOXES[mech](nx=16, ny=16, nz=16)
    box = W.subsample(full, np.full(cells, np.argsort(full["T"])[int(at * (full["T"].size - 1))]))
    if box.get("mask") is not None:
        box["mask"] = np.ones_like(box["mask"])
    return box


# both sides of what the rule's variant holds at once; cells alike, and a flame whose costs spread widely
@pytest.mark.parametrize("noalloc", [False, True])
@pytest.mark.parametrize("mech,cells,alike,want", [
    ("drm19", 2048, True, (64, 2)), ("drm19", 2049, True, (32, 4)), ("drm19", 6144, True, (32, 4)),
    ("drm19", 4096, False, (64, 2)), ("drm19", 6145, True, (32, 4)), ("LiDryer", 6144, True, (32, 3)),
    ("LiDryer", 6145, True, (16, 3)), ("LiDryer", 7168, False, (32, 3))])
def test_variant_by_costs(gpu, mech, cells, alike, want, noalloc):
    """Where every cell costs the same a launch takes the variant that holds them all at once, from the
    second call on (the first knows no costs); the bits do not depend on it."""
    import torch
    from pelelmex_amd.reactor import Reactor, box_tensors
    box = _alike(mech, cells, 0.05) if alike else BOXES[mech](nx=cells, ny=1, nz=1)
    t = box_tensors(box, gpu)
    old = {k: t[k].clone() for k in ("rY", "T", "rH", "FC")}
    out = []
    r = Reactor.create("ReactorCvode", mech, dict(KEYS, **{"cvode.max_order": 4}))
    r.init(2, 1)
    for call in range(3):
        for k in ("rY", "T", "rH"):
            t[k].copy_(old[k])
        status = torch.full((cells,), 7, dtype=torch.int32, device=gpu)
        assert r.react(t["rY"], t["rYsrc"], t["T"], t["rH"], t["rHsrc"], t["FC"], t["mask"], box["dt"], 0.0,
                       status=status, noalloc=noalloc)[0] == 0
        torch.cuda.synchronize()
        assert int(status.abs().sum()) == 0
        out.append(([t[k].clone() for k in old], r.stats()))
    shape = lambda st: (st["lanes_per_cell"], st["waves_per_simd"])
    rule = {"drm19": (64, 2) if cells <= 6144 else (32, 4), "LiDryer": (32, 3)}[mech]
    assert [shape(st) for _, st in out] == [rule, want, want]
    assert all(st["cells"] == cells and st["nfe"] == out[0][1]["nfe"] for _, st in out)
    for got, _ in out[1:]:
        assert all(torch.equal(a, b) for a, b in zip(got, out[0][0]))
    # and as a batch, captured: the costs of each replay decide
    if not noalloc:
        for k in old:
            t[k].copy_(old[k])
        r.react_batch([dict(t, dt=box["dt"])])
        g = torch.cuda.CUDAGraph()
        with torch.cuda.graph(g):
            r.react_batch([dict(t, dt=box["dt"])], enqueue_only=True)
        for first in (True, False, False):
            for k in old:
                if k != "FC" or first:
                    t[k].copy_(old[k])
            g.replay()
            assert r.collect() == 0 and shape(r.stats()) == (rule if first else want)
            assert all(torch.equal(t[k], v) for k, v in zip(old, out[0][0]))
    r.close()


def _free_after(torch, f):
    """Bytes of device memory that f() takes."""
    torch.cuda.synchronize()
    before = torch.cuda.mem_get_info()[0]
    f()
    torch.cuda.synchronize()
    return before - torch.cuda.mem_get_info()[0]


# doubles of a group's global slot (saved Jacobian, five records per reaction, LU factors above 32
# components) times the groups that the waves of the rules up to this size can hold
@pytest.mark.parametrize("mech,cells,slot,groups", [("dodecane_lu", 6145, 2 * 54 * 54 + 5 * 253, 4 * 3),
                                                    ("LiDryer", 28673, 10 * 10 + 5 * 21, 4 * 4 * 64 // 16)])
def test_slots_of_what_can_be_resident(gpu, mech, cells, slot, groups):
    """A launch reserves slots for the groups that can run at once, not for the cells of a smaller rule."""
    import torch
    from pelelmex_amd.reactor import Reactor, box_tensors
    t = box_tensors(BOXES[mech](nx=cells, ny=1, nz=1, dt=1e-9), gpu)

    def react(r):
        r.react(t["rY"], t["rYsrc"], t["T"], t["rH"], t["rHsrc"], t["FC"], t["mask"], 1e-9, 0.0)

    rs = [Reactor.create("ReactorCvode", mech, KEYS) for _ in range(2)]
    for r in rs:
        r.init(2, 1)
    react(rs[0])  # the kernels' own memory
    cus = torch.cuda.get_device_properties(gpu).multi_processor_count
    taken = _free_after(torch, lambda: react(rs[1]))
    for r in rs:
        r.close()
    assert taken <= 8 * slot * groups * cus + (8 << 20)  # tables and cost order: a few pages of 2 MiB


# the cells that fill the default variant (groups of its waves on 256 CUs), and one past the last line
@pytest.mark.parametrize("mech,small,large", [("dodecane_lu", 4 * 2 * 256, 6145),
                                              ("LiDryer", 4 * 3 * 64 // 16 * 256, 28673)])
def test_larger_launches_find_their_slots(gpu, mech, small, large):
    """After a launch that fills the default variant a larger one allocates no slots, so it can be captured."""
    import torch
    from pelelmex_amd.reactor import Reactor, box_tensors
    dt = 1e-9
    rs = [Reactor.create("ReactorCvode", mech, dict(KEYS, **{"hipbdf.cost_order": 0})) for _ in range(2)]
    tl, ts = (dict(box_tensors(BOXES[mech](nx=n, ny=1, nz=1, dt=dt), gpu), dt=dt) for n in (large, small))
    pristine = {k: tl[k].clone() for k in ("rY", "T", "rH", "FC")}

    def restore():
        for k, v in pristine.items():
            tl[k].copy_(v)

    for r in rs:
        r.init(2, 1)
    for t in (tl, ts):  # the kernels' own memory
        rs[0].react_batch([t])
    ref = {k: tl[k].clone() for k in pristine}
    r = rs[1]
    r.react_batch([ts])
    assert _free_after(torch, lambda: r.react_batch([tl])) <= 4 << 20
    r.close()
    r = Reactor.create("ReactorCvode", mech, dict(KEYS, **{"hipbdf.cost_order": 0}))
    r.init(2, 1)
    r.react_batch([ts])
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        r.react_batch([tl], enqueue_only=True)
    for _ in range(3):
        restore()
        g.replay()
        assert r.collect() == 0
        for k, v in ref.items():
            assert torch.equal(tl[k], v), k
    r.close()
    rs[0].close()
