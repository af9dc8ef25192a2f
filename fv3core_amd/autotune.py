"""Offline shape autotuner for the del-n and a2b_ord4 row marches.

A march runs strips of columns in segments of rows, one wave to a segment.
The segments follow from the launch's size by the march's cost
(``csrc/strip.hpp``); the most rows a segment may have (del-n: where a SIMD
holds more than three waves), and the waves per workgroup, are macros in
``csrc/tile_config.hpp``.  A shape only changes how the work is
split, never the arithmetic, so every candidate returns the same bits; the
tuner picks the fastest on the GPU it runs on:

1. ``build``: for each candidate, compile every source that holds the kernel
   with the shape's ``-D`` flags and link them with the other objects of the
   in-tree build into ``_tune/lib_<kernel>_<a>_<b>.so`` (CPU only: hipcc
   cross-compiles for gfx950).
2. ``measure``: run a benchmark workload once per library, each in its own
   process, timing the kernel with the library's HIP-event hooks
   (``bench.py --roofline-kernel <kernel>``), and write the mean launch
   times to ``_tune/results.json``.  Candidates that split the workload's
   launches as another does are left out.  ``--workload ensemble`` (the default)
   times the launches of the 32-member C48 batch in the mixed form;
   ``--workload dyncore`` those of the FP64 acoustic step on six C96 tiles.
3. ``apply``: rewrite the defaults in ``tile_config.hpp`` with the fastest
   shape of each kernel (rebuild the library afterwards).

``python -m fv3core_amd.autotune build``, then on a GPU
``python -m fv3core_amd.autotune measure``, then
``python -m fv3core_amd.autotune apply``.
"""
from __future__ import annotations

import argparse
import ctypes
import json
import pathlib
import re
import subprocess
import sys
from typing import Dict, List, Tuple

from . import _lib
from . import build as _build

HERE = pathlib.Path(__file__).resolve().parent
TUNE_DIR = HERE / "_tune"
CONFIG = _build.CSRC / "tile_config.hpp"
REPO = HERE.parent

# kernel -> (file that reads the macros, timing name, macro names, candidate
# (most rows, waves) pairs)
KERNELS: Dict[str, Tuple[str, str, Tuple[str, str], List[Tuple[int, int]]]] = {
    "delnflux": ("delnflux.hpp", "delnflux_kernel", ("FV3_DN_TJ", "FV3_DN_NY"),
                 [(17, 4), (25, 4), (33, 1), (33, 2), (33, 4), (33, 8), (49, 4)]),
    "a2b": ("a2b.hip", "a2b_interp_kernel", ("FV3_AB_TJ", "FV3_AB_NY"),
            [(11, 4), (19, 4), (33, 1), (33, 2), (33, 4), (49, 4), (97, 4)]),
}


# workload -> its launches of the kernels: (cells a side, tiles, levels, FP32)
_LAUNCHES = {"ensemble": [(48, 192, 79, True), (48, 192, 80, False)],
             "dyncore": [(96, 6, 79, False), (96, 6, 80, False)]}


def sources(kernel: str) -> List[pathlib.Path]:
    """The HIP sources that compile the kernel: the file itself or its includers."""
    name = KERNELS[kernel][0]
    if name.endswith(".hip"):
        return [_build.CSRC / name]
    return [s for s in sorted(_build.CSRC.glob("*.hip")) if f'#include "{name}"' in s.read_text()]


def default_shape(kernel: str) -> Tuple[int, int]:
    text = CONFIG.read_text()
    rows, waves = (int(re.search(rf"#define {m} (\d+)", text).group(1))
                   for m in KERNELS[kernel][2])
    return rows, waves


def plan(kernel: str, shape: Tuple[int, int], workload: str) -> tuple:
    """How the shape splits the workload's launches: their segment rows, and the waves."""
    lib = _lib.lib()
    segments = []
    for n, tiles, levels, fp32 in _LAUNCHES[workload]:
        if kernel == "delnflux":  # interfaces, 58 a strip
            rows = n + 1
            planes = -(-rows // 58) * levels * tiles
            segments.append(lib.fv3_plan_delnflux_rows(rows, ctypes.c_int64(planes), int(fp32),
                                                       shape[0]))
        else:  # the corners off the tile edges
            rows = n - 1
            planes = -(-rows // 58) * levels * tiles
            segments.append(lib.fv3_plan_a2b_rows(rows, ctypes.c_int64(planes), shape[0]))
    return tuple(segments) + (shape[1],)


def distinct_shapes(kernel: str, workload: str) -> List[Tuple[int, int]]:
    """The candidates whose plans differ on the workload, the default before the others."""
    shapes, first = KERNELS[kernel][3], default_shape(kernel)
    kept = {}
    for shape in sorted(shapes, key=lambda s: s != first):
        kept.setdefault(plan(kernel, shape, workload), shape)
    return [s for s in shapes if s in kept.values()]


def variant_lib(kernel: str, shape: Tuple[int, int]) -> pathlib.Path:
    return TUNE_DIR / f"lib_{kernel}_{shape[0]}_{shape[1]}.so"


def build_variants(kernels=None) -> List[pathlib.Path]:
    """Compile one library per candidate shape (needs the in-tree objects)."""
    lib = _build.build(verbose=False)
    objdir = lib.parent / "_build"
    TUNE_DIR.mkdir(exist_ok=True)
    made = []
    for kernel in kernels or KERNELS:
        _, _, macros, shapes = KERNELS[kernel]
        srcs = sources(kernel)
        others = [str(o) for o in sorted(objdir.glob("*.o"))
                  if o.stem not in [s.stem for s in srcs]]
        for shape in shapes:
            defs = [f"-D{macros[0]}={shape[0]}", f"-D{macros[1]}={shape[1]}"]
            objs = []
            for src in srcs:
                obj = TUNE_DIR / f"{src.stem}_{shape[0]}_{shape[1]}.o"
                cmd = [_build.hipcc()] + _build.COMMON_FLAGS + defs + ["-c", str(src),
                                                                     "-o", str(obj)]
                res = subprocess.run(cmd, capture_output=True, text=True)
                if res.returncode != 0:
                    raise RuntimeError(f"hipcc failed for {kernel} {shape}:\n{res.stderr}")
                objs.append(obj)
            out = variant_lib(kernel, shape)
            res = subprocess.run([_build.hipcc(), "-shared", "-fPIC",
                                  f"--offload-arch={_build.OFFLOAD_ARCH}"] + others +
                                 [str(o) for o in objs] + ["-o", str(out)],
                                 capture_output=True, text=True)
            if res.returncode != 0:
                raise RuntimeError(f"link failed for {kernel} {shape}:\n{res.stderr}")
            for obj in objs:
                obj.unlink()
            made.append(out)
    return made


_RUNNER = """
import pathlib, runpy, sys
sys.path.insert(0, {repo!r})
from fv3core_amd import _lib
_lib.LIB_PATH = pathlib.Path({lib!r})
sys.argv = ["bench.py", "--workload", {workload!r}, "--steps", "{steps}", "--warmup", "1",
            "--no-cpu-baseline", "--roofline-kernel", {name!r}] + {extra!r}
runpy.run_path({bench!r}, run_name="__main__")
"""


# bench.py options that leave out what the kernel timing does not need
_WORKLOAD_ARGS = {"ensemble": ["--no-graph", "--no-adjoint"], "dyncore": []}


def measure(kernels=None, steps: int = 3, timeout: int = 300,
            workload: str = "ensemble") -> dict:
    """Mean launch time (us) of each variant's kernel inside the workload."""
    if workload not in _WORKLOAD_ARGS:
        raise ValueError(f"unknown workload {workload}")
    results = {}
    for kernel in kernels or KERNELS:
        name = KERNELS[kernel][1]
        for shape in distinct_shapes(kernel, workload):
            lib = variant_lib(kernel, shape)
            if not lib.exists():
                raise FileNotFoundError(f"{lib} is missing: run the build step first")
            code = _RUNNER.format(repo=str(REPO), lib=str(lib), steps=steps, name=name,
                                  bench=str(REPO / "bench.py"), workload=workload,
                                  extra=_WORKLOAD_ARGS[workload])
            res = subprocess.run([sys.executable, "-c", code], capture_output=True, text=True,
                                 timeout=timeout)
            if res.returncode != 0:
                raise RuntimeError(f"timing run failed for {kernel} {shape}:\n{res.stderr[-2000:]}")
            line = [ln for ln in res.stdout.splitlines() if ln.startswith("{")][-1]
            us = float(json.loads(line)["roofline"]["kernel_avg_us"])
            results.setdefault(kernel, {})[f"{shape[0]}x{shape[1]}"] = us
            print(f"{kernel} rows={shape[0]} waves={shape[1]}: {us:.1f} us", flush=True)
    TUNE_DIR.mkdir(exist_ok=True)
    (TUNE_DIR / "results.json").write_text(json.dumps(results, indent=1))
    return results


def best_shapes(results: dict) -> Dict[str, Tuple[int, int]]:
    best = {}
    for kernel, times in results.items():
        key = min(times, key=times.get)
        a, b = key.split("x")
        best[kernel] = (int(a), int(b))
    return best


def rewrite_config(text: str, best: Dict[str, Tuple[int, int]]) -> str:
    """tile_config.hpp text with the defaults of the tuned kernels replaced."""
    for kernel, shape in best.items():
        macros = KERNELS[kernel][2]
        for macro, value in zip(macros, shape):
            pat = re.compile(rf"(#ifndef {macro}\n#define {macro} )(\d+)")
            if not pat.search(text):
                raise ValueError(f"{macro} has no default in tile_config.hpp")
            text = pat.sub(lambda m: m.group(1) + str(value), text)
    return text


def apply(results_path: pathlib.Path = TUNE_DIR / "results.json") -> Dict[str, Tuple[int, int]]:
    best = best_shapes(json.loads(results_path.read_text()))
    CONFIG.write_text(rewrite_config(CONFIG.read_text(), best))
    return best


def main(argv=None) -> int:
    p = argparse.ArgumentParser(description=__doc__.splitlines()[0])
    p.add_argument("step", choices=["build", "measure", "apply"])
    p.add_argument("--kernel", action="append", choices=sorted(KERNELS))
    p.add_argument("--steps", type=int, default=3)
    p.add_argument("--workload", default="ensemble", choices=sorted(_WORKLOAD_ARGS))
    a = p.parse_args(argv)
    if a.step == "build":
        for lib in build_variants(a.kernel):
            print(lib)
    elif a.step == "measure":
        measure(a.kernel, a.steps, workload=a.workload)
    else:
        for kernel, shape in apply().items():
            print(f"{kernel}: rows={shape[0]} waves={shape[1]}")
    return 0


if __name__ == "__main__":
    raise SystemExit(main())
