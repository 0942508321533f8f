"""The sums that carry a low part (Mz, Mzb), CPU only: every device function (float& hi, float& lo, float d) of the
kernels' sources, compiled for the host, keeps hi + lo exactly what it adds up, hi + fl(d + lo), also where the increment is
larger than the value (an inversion's zero crossing, a hard pulse)."""

import re
import subprocess
from pathlib import Path

import numpy as np

SRC = Path(__file__).resolve().parent.parent / "blochparty_amd" / "csrc"
HEAD = "__device__ __forceinline__ void "


def test_low_parts_are_exact(tmp_path):
    found = {}
    for path in sorted([*SRC.glob("*.h"), *SRC.glob("*.hip")]):
        text = path.read_text()
        for m in re.finditer(re.escape(HEAD) + r"(\w+)\(float& hi, float& lo, float d\) \{\n.*?\n\}\n", text, re.S):
            found[f"{m.group(1)}_{len(found)}"] = m.group(0)[len(HEAD) + len(m.group(1)):]
    assert found
    code = ["#include <stddef.h>"]
    for name, rest in found.items():
        code.append(f"static void f_{name}{rest}")
        code.append(f'extern "C" void {name}(float* hi, float* lo, const float* d, size_t n) '
                    f"{{ for (size_t i = 0; i < n; ++i) f_{name}(hi[i], lo[i], d[i]); }}")
    (tmp_path / "low.cpp").write_text("\n".join(code))
    lib = tmp_path / "low.so"
    subprocess.run(["g++", "-O1", "-ffp-contract=off", "-shared", "-fPIC", "-o", str(lib), str(tmp_path / "low.cpp")],
                   check=True)
    import ctypes

    rng = np.random.default_rng(0)
    n = 100_000
    hi0 = (rng.normal(size=n) * 2.0 ** rng.integers(-12, 3, n)).astype(np.float32)
    lo0 = (np.spacing(np.abs(hi0)) * rng.uniform(-0.5, 0.5, n)).astype(np.float32)
    d = (rng.normal(size=n) * 2.0 ** rng.integers(-12, 3, n)).astype(np.float32)
    want = hi0.astype(np.float64) + (d + lo0).astype(np.float64)  # exact in float64
    dll = ctypes.CDLL(str(lib))
    for name in found:
        hi, lo = hi0.copy(), lo0.copy()
        ptr = lambda a: a.ctypes.data_as(ctypes.c_void_p)
        getattr(dll, name)(ptr(hi), ptr(lo), ptr(d), ctypes.c_size_t(n))
        off = np.abs(hi.astype(np.float64) + lo.astype(np.float64) - want)
        assert off.max() == 0.0, (name, int((off > 0).sum()))
