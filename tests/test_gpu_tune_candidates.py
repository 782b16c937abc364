"""The tuner times every plan that modwt_plan_candidates lists: a tile plan that
agrees with a sliding-window plan in depth, segments and threads is another plan,
and FP32 inverses of three to eight levels have the wide tile."""
import re

import pytest
import torch

from wavecuda_amd import device as D

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,J,dtype", [(1 << 10, 5, torch.float64), (1 << 12, 8, torch.float32),
                                       (1 << 9, 3, torch.float32)])
def test_every_candidate_is_timed(n, J, dtype, monkeypatch, capfd):
    monkeypatch.setenv("WH_TUNE_LOG", "1")
    want = {"fwd": set(D.modwt_plan_candidates(False, n, J, "LA8", dtype)),
            "inv": set(D.modwt_plan_candidates(True, n, J, "LA8", dtype))}
    try:
        D.modwt_tune(n, J, "LA8", dtype)
    finally:
        for inverse in (False, True):
            D.modwt_set_plan(inverse, n, J, "LA8", dtype, None)
    log = capfd.readouterr().err
    timed = {"fwd": set(), "inv": set()}
    for direction, plan in re.findall(r"wh_modwt_tune (\w+) [\d.]+ ms (\{.*)", log):
        timed[direction].add(plan.strip())
    for direction, plans in want.items():
        assert {p.strip() for p in plans} <= timed[direction], direction
