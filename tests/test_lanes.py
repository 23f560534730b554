"""The react kernel's device code with its lanes emulated on the host (tests/lanes): every memory
access inside the array it belongs to, no value that another lane wrote before the next ordering
point, no read of memory that nobody wrote, no conversion out of range - and the oracle's bits."""
import os
import re
import subprocess

import numpy as np
import pytest

from pelelmex_amd import workloads as W

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(os.path.dirname(HERE), "pelelmex_amd", "csrc")

# what the host compiler does not know, in its terms
EDITS = {
    "bdf_kernel.h": [('asm volatile("" : "+s"(c));', "", 1), ('asm volatile("" : "+v"(v));', "", 1),
                     ("__builtin_amdgcn_wave_barrier();", "", 1),
                     ('asm volatile("" ::: "memory");', "emu::sync();", 1),
                     ('asm("v_max_f64 %0, %1, %2" : "=v"(r) : "v"(a), "v"(b));', "r = a > b ? a : b;", 1),
                     ('asm("v_cvt_i32_f64 %0, %1" : "=v"(r) : "v"(v));',
                      "r = v != v ? 0 : (int)(v < -2147483648.0 ? -2147483648.0 : (v > 2147483647.0 ? 2147483647.0 : v));",
                      1)],
    "react_kernel.h": [('asm volatile("" ::: "memory");', "emu::sync();", 1),
                       ("extern __shared__ __align__(16) unsigned char smem[];", "unsigned char* smem = emu_smem();", None),
                       ("double* setup_views(", "double* device_views(", 1),
                       ("// Views of the mechanism tables",
                        'unsigned char* emu_smem();\nconst unsigned char* emu_blob(int from, int to);\n#include "views.h"\n// Views',
                        1)],
}


@pytest.fixture(scope="module")
def lanes(tmp_path_factory):
    d = tmp_path_factory.mktemp("lanes")
    for name, edits in EDITS.items():
        text = open(os.path.join(CSRC, name)).read()
        for old, new, count in edits:
            assert text.count(old) == count or (count is None and old in text), (name, old)
            text = text.replace(old, new)
        (d / name).write_text(text)
    host = open(os.path.join(CSRC, "reactor.hip")).read()
    parts = [host[host.index(a):host.index(b)] for a, b in
             (("std::vector<unsigned char> pack_blob(", "// Tables of the block kernels"),
              ("// Terms of every Jacobian entry", "// The device tables of a mechanism"))]
    (d / "tables.h").write_text("\n".join(parts))
    exe = d / "lanes"
    subprocess.run(["g++", "-std=c++17", "-O1", "-ffp-contract=off", "-fsanitize=float-cast-overflow",
                    "-fno-sanitize-recover=all", "-w", f"-I{d}", f"-I{HERE}/lanes", f"-I{CSRC}",
                    f"{HERE}/lanes/main.cpp", "-o", str(exe)], check=True)
    return str(exe)


def _run(exe, args, data):
    p = subprocess.run([exe, *[str(a) for a in args]], input=data, capture_output=True, timeout=300)
    assert p.returncode == 0, f"status {p.returncode}: {p.stderr.decode()[-400:]}"
    return np.frombuffer(p.stdout)


BOXES = {"LiDryer": W.h2_air_box, "drm19": W.ch4_air_flame_box, "dodecane_lu": W.dodecane_box}


@pytest.mark.parametrize("mech,G,cells,dt", [("LiDryer", 8, 3, 1e-6), ("LiDryer", 16, 6, 1e-6), ("LiDryer", 32, 3, 1e-6),
                                             ("LiDryer", 64, 3, 1e-6), ("drm19", 16, 2, 1e-6), ("drm19", 32, 2, 1e-6),
                                             ("drm19", 64, 2, 1e-6), ("dodecane_lu", 64, 1, 1e-9)])
def test_react_lanes(lanes, mech, G, cells, dt):
    from oracle import pyoracle as po
    box = BOXES[mech](nx=cells, ny=1, nz=1, dt=dt)
    ref = po.Mech(mech).react(box["rY"], box["rYsrc"], box["T"], box["rH"], box["rHsrc"], None, dt, max_order=4)
    want = np.concatenate([ref["rY"].ravel(), ref["T"], ref["rH"], ref["FC"], [0.0]])
    data = np.int64(cells).tobytes() + np.float64(dt).tobytes() + \
        b"".join(np.ascontiguousarray(box[k]).tobytes() for k in ("rY", "rYsrc", "T", "rH", "rHsrc"))
    for fill, at_end in ((255, 1), (63, 0)):  # NaN and about 4.8e-4 in what nobody wrote
        np.testing.assert_array_equal(_run(lanes, (mech, G, fill, at_end), data), want)


def test_exp_log_over_all_arguments(lanes):
    """Any argument, Troe fits with T*** = 1e-30 give -1e33: defined, and the oracle's bits."""
    from oracle import pyoracle as po
    x = np.array([0.0, -0.0, 1.0, -1.0, 699.999, 700.0, 709.7, 709.8, -708.0, -745.0, -745.2, 1e9, -3e9, 1e33, -1e33,
                  1e300, -1e308, np.inf, -np.inf, np.nan, 5e-324, 1e-310])
    out = _run(lanes, ("exp",), np.int64(x.size).tobytes() + x.tobytes())
    L = po.lib()
    want = [[f(v) for v in x] for f in (L.orc_exp, L.orc_log)]
    np.testing.assert_array_equal(out, np.concatenate(want))
