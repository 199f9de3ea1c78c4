"""Autotuner of the generated kernels' per-class register budget.

Each canonical class is compiled with a register budget (doubles per target
group, codegen/gen_eri.plan_class): a larger budget means fewer groups and
less recomputation, a smaller one fewer spills and more waves.  The best value
differs between classes and is measured, not modelled.  The budget concerns the
per-lane kernels (codegen/gen_eri.py): FP32 and Schwarz factors, and FP64 ERI
batches of the classes in gen_rys.LANE_COST.  The Rys kernels (codegen/gen_rys.py)
that serve FP64 otherwise have no budget, so the other classes are tuned by their
FP32 variant (twice as many values).

  python -m libint_amd.tune build   --dir D [--budgets 128,144,160] [--classes 2222,2122]
        (CPU) one library per budget, holding only the tuned classes (ERI
        kernels), under D/b<budget>/
  python -m libint_amd.tune measure --dir D
        (GPU) times every class's ERI kernel in every library on the same
        seeded quartets (s-d classes: the 60-atom s4p3d2 recipe; f classes:
        the 120-atom s4p3d2f1 recipe), each library in a child process;
        writes D/timings.json
  python -m libint_amd.tune select  --dir D [--out libint_amd/tuned.cfg]
        writes the fastest budget of each measured class as a
        class=budget:0:fp32 entry, merged into the file's other entries; the
        Makefile passes them to the generator (CLASSCFG)
  python -m libint_amd.tune fp32 [--classes ...] [--out libint_amd/tuned.cfg]
        (GPU) times each class's FP64 kernel and its FP32 variant in the
        built library on the quartets a mixed batch would run in FP32
        (K K < 1e-6, S S < 16e-6) and sets the fp32 field (1: the FP32
        variant is at least 5 % faster there, so mixed batches route to it
        by default); rebuild the library afterwards
"""
from __future__ import annotations

import argparse
import json
import os
import subprocess
import sys

HERE = os.path.dirname(os.path.abspath(__file__))
DEFAULT_BUDGETS = (128, 144, 160)
DEFAULT_BUDGET = 160  # the Makefile's BUDGET
MODES = "eri,schwarz,fp32"  # of the libraries that are timed: what the shipped one runs ERI batches on


def heavy_classes():
    sys.path.insert(0, os.path.join(HERE, "codegen"))
    import gen_eri
    return ["".join(map(str, c)) for c in gen_eri.canonical_classes(2) if sum(c) >= 5]


def build(args):
    budgets = [int(b) for b in args.budgets.split(",")]
    classes = args.classes or ",".join(heavy_classes())
    procs = []
    for b in budgets:
        d = os.path.join(os.path.abspath(args.dir), f"b{b}")
        os.makedirs(d, exist_ok=True)
        cmd = ["make", "-s", "-C", HERE, f"GEN={d}/gen", f"OBJ={d}/obj", f"LIB={d}/libl2g.so",
               f"ONLY={classes}", f"MODES={MODES}", f"BUDGET={b}", "CLASSCFG=", "-j2"]
        procs.append((b, subprocess.Popen(cmd, stdout=subprocess.DEVNULL, stderr=subprocess.PIPE)))
    for b, p in procs:
        _, err = p.communicate()
        if p.returncode:
            raise SystemExit(f"budget {b}: build failed\n{err.decode()[-2000:]}")
        print(f"budget {b}: built", flush=True)
    with open(os.path.join(args.dir, "classes.txt"), "w") as f:
        f.write(classes)


def time_library(args):
    """Child process: time the ERI kernel of each class with the library
    named by LIBINT_AMD_LIB; prints one JSON object."""
    import numpy as np

    import libint_amd as la
    from libint_amd import molecule
    classes = args.classes.split(",")
    ctx = la.Context(0)
    bases = {}
    out = {}
    rng = np.random.default_rng(11)
    for name in classes:
        la_, lb_, lc_, ld_ = (int(x) for x in name)
        # s-d classes on the 60-atom recipe, f classes on the 120-atom one
        w = 3 if max(la_, lb_, lc_, ld_) == 3 else 2
        if w not in bases:
            m = molecule.make_molecule(w)
            bases[w] = (m.basis, la.Basis(ctx, m.basis))
        B, b = bases[w]
        bra = [(i, j) for i in range(B.nshell) for j in range(B.nshell)
               if B.l[i] == la_ and B.l[j] == lb_ and (la_ != lb_ or i >= j)]
        ket = [(i, j) for i in range(B.nshell) for j in range(B.nshell)
               if B.l[i] == lc_ and B.l[j] == ld_ and (lc_ != ld_ or i >= j)]
        # significant pairs (Schwarz factor >= 1e-9), quartets with
        # K_ab K_cd >= 1e-12, as the workloads screen them
        bra = np.array(bra, np.int32)
        ket = np.array(ket, np.int32)
        kb, sb = la.precision_bounds(b, bra)
        kk, sk = (kb, sb) if (la_, lb_) == (lc_, ld_) else la.precision_bounds(b, ket)
        bra, kb, sb = bra[kb >= 1e-9], kb[kb >= 1e-9], sb[kb >= 1e-9]
        ket, kk, sk = ket[kk >= 1e-9], kk[kk >= 1e-9], sk[kk >= 1e-9]
        i1 = rng.integers(0, len(bra), 1600000)
        i2 = rng.integers(0, len(ket), 1600000)
        sig = kb[i1] * kk[i2] >= 1e-12
        # the quartets a mixed batch at threshold 1e-6 runs in FP32
        # (K K < 1e-6 and S S < 16e-6): where the FP32 variant is compared
        elig = sig & (kb[i1] * kk[i2] < 1e-6) & (sb[i1] * sk[i2] < la.FP32_HRR_FACTOR * 1e-6)
        qe = np.concatenate([bra[i1[elig][:400000]], ket[i2[elig][:400000]]], 1)
        i1, i2 = i1[sig][:400000], i2[sig][:400000]
        q = np.concatenate([bra[i1], ket[i2]], 1)
        variants = [("", 0.0, q)]
        if args.fp32 and max(la_, lb_, lc_, ld_) <= la.fp32_max_l() and len(qe):
            # the eligible quartets in FP64 and, every one below the bounds, in FP32
            variants += [("/e64", 0.0, qe), ("/fp32", 1e300, qe)]
        for suffix, thr, qq in variants:
            ctx.set_fp32_policy(la.FP32_ALWAYS)
            plan = la.EriPlan(b, qq, fp32_threshold=thr)
            ctx.set_fp32_policy(la.FP32_MEASURED)
            if thr and not all(s["fp32"] for s in plan.stats()):
                raise SystemExit(f"{name}: the FP32 plan is not all FP32")
            d = plan.device_output()
            plan.execute(d)
            ctx.synchronize()
            ms = []
            for _ in range(3):
                plan.execute(d)
                ctx.synchronize()
                ms.append(sum(s["ms"] for s in plan.stats()))
            out[name + suffix] = float(np.median(ms))
            del plan
    bases.clear()
    ctx.close()
    print(json.dumps(out), flush=True)


def measure(args):
    classes = open(os.path.join(args.dir, "classes.txt")).read().strip()
    res = {}
    for sub in sorted(os.listdir(args.dir)):
        lib = os.path.join(os.path.abspath(args.dir), sub, "libl2g.so")
        if not (sub.startswith("b") and os.path.exists(lib)):
            continue
        env = dict(os.environ, LIBINT_AMD_LIB=lib)
        print(f"budget {sub[1:]}: timing {classes}", flush=True)
        r = subprocess.run([sys.executable, "-m", "libint_amd.tune", "_time", "--fp32", "--classes", classes],
                           env=env, cwd=os.path.dirname(HERE), capture_output=True, text=True, timeout=900)
        if r.returncode:
            raise SystemExit(f"budget {sub[1:]}: timing failed ({r.returncode})\n{r.stderr[-2000:]}")
        res[sub[1:]] = json.loads(r.stdout.strip().splitlines()[-1])
        print(f"  {res[sub[1:]]}", flush=True)
    with open(os.path.join(args.dir, "timings.json"), "w") as f:
        json.dump(res, f, indent=1)


def read_cfg(path):
    """class -> [budget, waves, fp32] of a tuned.cfg file."""
    out = {}
    try:
        text = open(path).read().strip()
    except OSError:
        return out
    for item in filter(None, text.split(",")):
        k, v = item.split("=")
        f = [int(x) for x in v.split(":")]
        out[k] = (f + [0] * 3)[:3]
    return out


def write_cfg(path, cfg):
    """Entries that differ from the defaults (budget 160, waves 0, fp32 0)."""
    keep = {c: v for c, v in cfg.items() if list(v) != [DEFAULT_BUDGET, 0, 0]}
    with open(path, "w") as f:
        f.write(",".join(f"{c}={v[0]}:{v[1]}:{v[2]}" for c, v in sorted(keep.items())) + "\n")
    print(f"wrote {path}")


def fp32_pays(t64, t32):
    return 1 if t32 is not None and t32 < 0.95 * t64 else 0


def budget_time(c, r):
    """The time of class c, in a library's timings r, that its budget decides: its FP64 kernel's where that is a per-lane
    kernel, else its FP32 variant's (None: nothing of the class depends on the budget)."""
    sys.path.insert(0, os.path.join(HERE, "codegen"))
    import gen_rys
    return r[c] if gen_rys.lane_cost(*map(int, c)) else r.get(c + "/fp32")


def select(args):
    res = json.load(open(os.path.join(args.dir, "timings.json")))
    classes = sorted({c for r in res.values() for c in r if "/" not in c})
    cfg = read_cfg(args.out)
    for c in classes:
        times = {int(b): budget_time(c, r) for b, r in res.items() if c in r}
        if None in times.values():
            print(f"{c}: no kernel with a budget")
            continue
        best = min((t, b) for b, t in times.items())
        r = res[str(best[1])]
        cfg[c] = [best[1], 0, fp32_pays(r.get(c + "/e64", r[c]), r.get(c + "/fp32"))]
        print(f"{c}: budget {best[1]} ({best[0]:.2f} ms), fp32 {cfg[c][2]}; " +
              ", ".join(f"{b}: {t:.2f}" for b, t in sorted(times.items())))
    write_cfg(args.out, cfg)


def fp32(args):
    """FP64 kernel against FP32 variant of each class, with the built library."""
    sys.path.insert(0, os.path.join(HERE, "codegen"))
    import gen_eri
    classes = args.classes or ",".join("".join(map(str, c)) for c in gen_eri.canonical_classes(2))
    r = subprocess.run([sys.executable, "-m", "libint_amd.tune", "_time", "--fp32", "--classes", classes],
                       cwd=os.path.dirname(HERE), capture_output=True, text=True, timeout=1200)
    if r.returncode:
        raise SystemExit(f"timing failed ({r.returncode})\n{r.stderr[-2000:]}")
    res = json.loads(r.stdout.strip().splitlines()[-1])
    cfg = read_cfg(args.out)
    for c in classes.split(","):
        if c not in res:
            continue
        v = cfg.setdefault(c, [DEFAULT_BUDGET, 0, 0])
        t64, t32 = res.get(c + "/e64"), res.get(c + "/fp32")
        v[2] = fp32_pays(t64, t32) if t64 is not None else 0
        print(f"{c}: all significant quartets fp64 {res[c]:.2f} ms; FP32-eligible quartets fp64 "
              f"{t64 if t64 is None else round(t64, 2)} ms, fp32 {t32 if t32 is None else round(t32, 2)} ms "
              f"-> fp32 {v[2]}", flush=True)
    write_cfg(args.out, cfg)


def main():
    ap = argparse.ArgumentParser(description=__doc__, formatter_class=argparse.RawDescriptionHelpFormatter)
    ap.add_argument("step", choices=["build", "measure", "select", "fp32", "_time"])
    ap.add_argument("--fp32", action="store_true", help="_time: also the FP32 variants")
    ap.add_argument("--dir", default="tune_build")
    ap.add_argument("--budgets", default=",".join(map(str, DEFAULT_BUDGETS)))
    ap.add_argument("--classes", default="")
    ap.add_argument("--out", default=os.path.join(HERE, "tuned.cfg"))
    args = ap.parse_args()
    {"build": build, "measure": measure, "select": select, "fp32": fp32,
     "_time": time_library}[args.step](args)


if __name__ == "__main__":
    main()
