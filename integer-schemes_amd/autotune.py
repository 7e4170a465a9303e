"""Autotuner of the fused stage kernels' schedule on the device it runs on.

    python integer-schemes_amd/autotune.py [--n 256] [--steps 6] [--space full|quick]
                                           [--write] [--out tuning.json]

The stage kernels' schedule is a set of compile-time knobs (bssn_params.h, bssn_brick.h,
bssn_stage.h): the brick of output points one wave owns (BSSN_BRICK_X/Y/Z, 64 points: the
4x4x4 cube stages the fewest halo cells, the flatter bricks longer z runs), the LDS box's
x-plane stride (BSSN_BOX_XPLANE_MOD32: dense, or padded to a residue modulo 32 doubles that
spreads the brick's lanes over the banks), the order in which an XCD's workgroups take their
bricks (BSSN_BRICK_TILE_XY: z columns in square tiles of columns, or 0 for rows of columns), how
many fields are staged ahead of the one being evaluated (BSSN_STAGE_DEPTH for the RK/MSRK stage
kernels, BSSN_RHS_DEPTH for the bare RHS), how many algebra phases ahead of its store a field's
write-back operands are loaded
(BSSN_WB_LEAD), and how many waves per SIMD the register allocator targets (BSSN_STAGE_WAVES,
BSSN_RHS_WAVES; two waves force one field in flight). A knob moves loads, LDS addresses and
register allocation, not arithmetic, so every variant computes the same RHS.

All but BSSN_BRICK_TILE_XY are knobs of the wave-private kernels, which run the grids that
bssn_dispatch.h leaves to them: all of at most 1024 bricks, and some thin ones. Bricks shared by
four waves (bssn_group.h) read only the brick order. So a candidate is checked on both kinds of
grid and timed where its knobs reach:
  * small: the 26^3 equal-mass binary, whose interior and padded grid are one round of
    wave-private bricks whatever their shape;
  * bench: the n^3 binary (default 256^3, the benchmark workload), candidates with a knob in
    SHARED_KNOBS only.

For every candidate the tuner
  1. builds a variant library (build.build(out=..., defines=...)) under integer-schemes_amd/_tune/;
  2. in a fresh process with that library (BSSN_HIP_LIB), checks the variant against the installed
     library's RK4 steps and RHS on puncture grids of 26^3 and 48^3 (normwise 1e-12: the knobs may
     only move FMA formation) and times the RK4 step and the bare RHS;
and keeps the defaults unless a passing candidate is faster on a step by more than the timing
noise (0.5 %) without slowing anything that it was timed on by more (choose()). With --write the
result goes to tuning.json next to build.py, whose defines build.build() then compiles by default;
the batched launch shape is tuned at run time on each batch (BlockBatch.autotune,
PatchHierarchy.tune_launch).
"""
from __future__ import annotations

import argparse
import json
import os
import subprocess
import sys
import tempfile
from pathlib import Path

PKG = Path(__file__).resolve().parent
TUNING = PKG / "tuning.json"

SPACES = {
    "quick": [
        {},
        {"BSSN_STAGE_DEPTH": 2},
        {"BSSN_BOX_XPLANE_MOD32": 16},
    ],
    "full": [
        {},
        {"BSSN_STAGE_DEPTH": 2},
        {"BSSN_WB_LEAD": 1},
        {"BSSN_WB_LEAD": 3},
        {"BSSN_STAGE_DEPTH": 2, "BSSN_WB_LEAD": 1},
        {"BSSN_STAGE_DEPTH": 2, "BSSN_WB_LEAD": 3},
        {"BSSN_RHS_DEPTH": 1},
        {"BSSN_STAGE_WAVES": 2},
        {"BSSN_RHS_WAVES": 2},
        {"BSSN_BOX_XPLANE_MOD32": 16},
        {"BSSN_BOX_XPLANE_MOD32": 16, "BSSN_WB_LEAD": 3},
        {"BSSN_BRICK_X": 2, "BSSN_BRICK_Y": 4, "BSSN_BRICK_Z": 8},
        {"BSSN_BRICK_X": 4, "BSSN_BRICK_Y": 2, "BSSN_BRICK_Z": 8},
        {"BSSN_BRICK_X": 2, "BSSN_BRICK_Y": 8, "BSSN_BRICK_Z": 4},
        {"BSSN_BRICK_X": 8, "BSSN_BRICK_Y": 4, "BSSN_BRICK_Z": 2},
        {"BSSN_BRICK_X": 2, "BSSN_BRICK_Y": 2, "BSSN_BRICK_Z": 16},
        {"BSSN_BRICK_TILE_XY": 0},
        {"BSSN_BRICK_TILE_XY": 2},
        {"BSSN_BRICK_TILE_XY": 8},
    ],
}
# the brick shapes alone, and the brick orders alone (with the defaults as the baseline every
# space starts with)
SPACES["bricks"] = [{}] + [d for d in SPACES["full"] if "BSSN_BRICK_X" in d]
SPACES["order"] = [{}] + [d for d in SPACES["full"] if "BSSN_BRICK_TILE_XY" in d]

# knobs that the bricks shared by four waves read too
SHARED_KNOBS = {"BSSN_BRICK_TILE_XY"}
SMALL = 26                     # interior points per axis of the small workload (padded 32)
CHECKS = (SMALL, 48)           # of the checks: wave-private and shared bricks
TIMES = ("step_ms", "rhs_ms", "small_step_ms", "small_rhs_ms")


def timed_on(defines: dict) -> tuple:
    """The workloads a candidate's knobs reach; the defaults are timed on both."""
    both = not defines or SHARED_KNOBS & set(defines)
    return ("small", "bench") if both else ("small",)


# Runs in the candidate's process: compare the steps and RHS of the check grids with the installed
# library's (written by the parent), time the workloads.
_CHILD = r"""
import json, sys
sys.path.insert(0, sys.argv[1])
import numpy as np, torch
from bssn3d_hip import initial_data as idata
from bssn3d_hip.evolve import BSSNEvolution
from bssn3d_hip.rhs import rhs_into
from bssn3d_hip.state import PhysicsParams, scalars
n, steps, ref_path, mode = int(sys.argv[2]), int(sys.argv[3]), sys.argv[4], sys.argv[5]
small, checks, workloads = int(sys.argv[6]), sys.argv[7].split(","), sys.argv[8].split(",")
dev = torch.device("cuda:0")
p = PhysicsParams()

def rhs_of(grid, U, out, dt):
    rhs_into(U, out, scalars(p, grid.dx, grid.dy, grid.dz, dt, 0.0), 4)

found = {}
for N in checks:
    g, U, _ = idata.config_single_puncture(seed=3, N=int(N), device=dev)
    ev = BSSNEvolution(g, p, order=4, ko_sigma=0.1, bc="periodic")
    dt = 0.25 * g.dx
    for k in range(2):
        ev.step_(U, k * dt, dt)
    out = torch.empty_like(U)
    rhs_of(g, U, out, dt)
    found["step" + N], found["rhs" + N] = U.cpu().numpy(), out.cpu().numpy()
if mode == "ref":
    np.savez(ref_path, **found)
    print(json.dumps({"ok": True}))
    sys.exit(0)
err = 0.0
with np.load(ref_path) as ref:
    for key, got in found.items():
        den = np.maximum(np.abs(ref[key]).reshape(24, -1).max(axis=1), 1e-12)
        err = max(err, float((np.abs(got - ref[key]).reshape(24, -1).max(axis=1) / den).max()))
del found, U, out
e0, e1 = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)

def timed(fn, reps, trials):
    best = float("inf")
    for _ in range(trials):
        torch.cuda.synchronize()
        e0.record()
        for k in range(reps):
            fn(k)
        e1.record()
        torch.cuda.synchronize()
        best = min(best, e0.elapsed_time(e1) / reps)
    return best

res, ok = {}, True
for name in workloads:
    N, reps, trials = (n, steps, 1) if name == "bench" else (small, 40 * steps, 5)
    pre = "" if name == "bench" else "small_"
    grid, U, _ = idata.config_binary(seed=0, N=N, device=dev)
    ev = BSSNEvolution(grid, p, order=4, ko_sigma=0.1, bc="periodic")
    # the small grid's steps are short ones: its many repetitions stay at early times
    dt = 0.25 * grid.dx * (1.0 if name == "bench" else 1e-3)
    for k in range(2):
        ev.step_(U, k * dt, dt)
    res[pre + "step_ms"] = timed(lambda k: ev.step_(U, (2 + k) * dt, dt), reps, trials)
    out = torch.empty_like(U)
    rhs_of(grid, U, out, dt)
    res[pre + "rhs_ms"] = timed(lambda k: rhs_of(grid, U, out, dt), reps, trials)
    ok = ok and bool(torch.isfinite(U).all())
    del U, out, ev
print(json.dumps({"ok": ok, "err": err, **res}))
"""


# a candidate must beat the defaults' time of a step by more than this fraction (timing noise)
MARGIN = 0.005


def key_of(defines: dict) -> str:
    return "_".join(f"{k.replace('BSSN_', '').lower()}{v}" for k, v in sorted(defines.items())) \
        or "default"


def run_child(lib: Path | None, n: int, steps: int, ref: Path, mode: str,
              workloads=("small", "bench")) -> dict:
    env = dict(os.environ)
    if lib is not None:
        env["BSSN_HIP_LIB"] = str(lib)
    r = subprocess.run([sys.executable, "-c", _CHILD, str(PKG), str(n), str(steps), str(ref), mode,
                        str(SMALL), ",".join(map(str, CHECKS)), ",".join(workloads)],
                       capture_output=True, text=True, env=env, timeout=900)
    if r.returncode != 0:
        raise RuntimeError(f"candidate run failed:\n{r.stdout[-2000:]}\n{r.stderr[-2000:]}")
    return json.loads(r.stdout.strip().splitlines()[-1])


def tune(space: str = "full", n: int = 256, steps: int = 6, tol: float = 1e-12,
         verbose: bool = True) -> dict:
    import importlib.util
    spec = importlib.util.spec_from_file_location("bssn_build", PKG / "build.py")
    build = importlib.util.module_from_spec(spec)
    spec.loader.exec_module(build)
    cands = SPACES[space]
    work = PKG / "_tune"
    libs = {}
    for d in cands:
        k = key_of(d)
        out = work / k / "libbssn_hip.so"
        if verbose:
            print(f"[autotune] building {k}", flush=True)
        libs[k] = build.build(out=out, defines=[f"{a}={b}" for a, b in d.items()])
    results = {}
    with tempfile.TemporaryDirectory() as td:
        ref = Path(td) / "ref.npz"
        run_child(None, n, steps, ref, "ref")          # the installed library's results
        for d in cands:
            k = key_of(d)
            r = run_child(libs[k], n, steps, ref, "time", timed_on(d))
            r["passed"] = bool(r["ok"] and r["err"] <= tol)
            r["defines"] = d
            results[k] = r
            if verbose:
                times = "  ".join(f"{t[:-3]} {r[t]:8.4f}" for t in TIMES if t in r)
                print(f"[autotune] {k:28s} {times} ms  err {r['err']:.1e}  "
                      f"{'ok' if r['passed'] else 'REJECTED'}", flush=True)
    import torch
    return choose(results, workload=f"bssn_rk4_step_{n}^3_fp64_bl_binary", small=SMALL,
                  device=torch.cuda.get_device_name(0), steps_timed=steps)


def choose(results: dict, margin: float = MARGIN, **info) -> dict:
    """The tuning record for measured candidates: the defaults unless a passing candidate is
    faster on a step by more than ``margin`` (run-to-run noise of the timing) without making
    any step or bare RHS that it was timed on slower by more than ``margin``; among those, the
    largest gain on a step."""
    base = results["default"]

    def relative(r):
        return {t: r[t] / base[t] for t in TIMES if t in r and t in base}

    def gain(k):
        return min(v for t, v in relative(results[k]).items() if t.endswith("step_ms"))

    better = [k for k, r in results.items()
              if r["passed"] and gain(k) <= 1.0 - margin
              and max(relative(r).values()) <= 1.0 + margin]
    best = min(better, key=gain) if better else "default"
    return {"defines": [f"{a}={b}" for a, b in results[best]["defines"].items()],
            "best": best, "margin": margin, **info, "candidates": results}


def merge(old: dict, new: dict) -> dict:
    """One record from two runs on the same device and workload: every candidate of both (the
    newer measurement where both have one, the newer defaults as the baseline), chosen again."""
    if any(old.get(k) != new.get(k) for k in ("workload", "small")):
        raise ValueError("records of different workloads")
    cands = dict(old.get("candidates", {}))
    cands.update(new["candidates"])
    info = {k: new[k] for k in ("workload", "small", "device", "steps_timed") if k in new}
    return choose(cands, margin=new.get("margin", MARGIN), **info)


def main(argv=None) -> int:
    ap = argparse.ArgumentParser(description=__doc__.splitlines()[0])
    ap.add_argument("--space", default="full", choices=sorted(SPACES))
    ap.add_argument("--n", type=int, default=256, help="points per axis of the bench workload")
    ap.add_argument("--steps", type=int, default=6)
    ap.add_argument("--write", action="store_true", help="install the result as tuning.json")
    ap.add_argument("--out", default=None, help="also write the result here")
    ap.add_argument("--merge", default=None,
                    help="a record of earlier candidates (same device and workload) to choose "
                         "among together with this run's")
    a = ap.parse_args(argv)
    res = tune(a.space, a.n, a.steps)
    if a.merge:
        res = merge(json.loads(Path(a.merge).read_text()), res)
    text = json.dumps(res, indent=1)
    print(text)
    if a.out:
        Path(a.out).write_text(text + "\n")
    if a.write:
        TUNING.write_text(text + "\n")
    return 0


if __name__ == "__main__":
    sys.exit(main())
