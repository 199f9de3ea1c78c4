"""The register-budget autotuner times and chooses by the kernels that run."""
import argparse
import json
import os

import pytest

from libint_amd import tune
from libint_amd.codegen import gen_eri


def test_timed_libraries_hold_the_kernels_that_are_shipped(tmp_path, monkeypatch):
    cmds = []

    class Make:
        returncode = 0

        def __init__(self, cmd, **kw):
            cmds.append(cmd)

        def communicate(self):
            return b"", b""
    monkeypatch.setattr(tune.subprocess, "Popen", Make)
    tune.build(argparse.Namespace(budgets="128,160", classes="2222,1010", dir=str(tmp_path)))
    modes = {x.split("=")[1] for c in cmds for x in c if x.startswith("MODES=")}
    assert len(cmds) == 2 and len(modes) == 1
    # as the tuner's make call generates them: FP64 (dd|dd) on its Rys kernel only, (ps|ps) on either
    gen_eri.generate(str(tmp_path / "gen"), only={"2222", "1010"}, modes=tuple(modes.pop().split(",")))
    table = (tmp_path / "gen" / "eri_table.cpp").read_text()
    for name in ("l2g_rys_eri_2222", "l2g_rys_eri_1010", "l2g_eri_1010", "l2g_eri32_2222", "l2g_schwarz_2222"):
        assert f"&{name}_launch" in table, name
    assert "&l2g_eri_2222_launch" not in table


@pytest.mark.parametrize("timings, cfg", [
    # (dd|dd): FP64 does not depend on the budget; FP32, which does, is best at 144 and slower than FP64
    ({"128": {"2222": 9.0, "2222/e64": 8.9, "2222/fp32": 15.0}, "144": {"2222": 9.1, "2222/e64": 8.9, "2222/fp32": 13.9}},
     {"2222": [144, 0, 0]}),
    # (ds|dd)... on its per-lane kernel in FP64: by that one; FP32 pays there
    ({"128": {"1022": 4.0, "1022/e64": 3.9, "1022/fp32": 1.0}, "176": {"1022": 3.5, "1022/e64": 3.6, "1022/fp32": 3.0}},
     {"1022": [176, 0, 1]}),
    # neither: the entry stays
    ({"128": {"3333": 1.0}}, {"3333": [192, 0, 0]}),
])
def test_choice_of_budget(tmp_path, timings, cfg):
    (tmp_path / "timings.json").write_text(json.dumps(timings))
    out = os.path.join(tmp_path, "tuned.cfg")
    tune.write_cfg(out, {"3333": [192, 0, 0]} if "3333" in cfg else {})
    tune.select(argparse.Namespace(dir=str(tmp_path), out=out))
    got = tune.read_cfg(out)
    assert {c: got[c] for c in cfg} == cfg
