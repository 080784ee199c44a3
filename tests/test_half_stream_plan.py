"""The plan walk of tests/test_stream_plan.py over the stream kernel's two-per-CU configuration
(w2 projection, four blocks per unit on 2 waves, twice as many work-groups as CUs)."""
import subprocess

from tests import test_stream_plan as plan


def test_two_work_groups_per_cu_stay_in_bounds(tmp_path, monkeypatch):
    body = plan.CHECKER
    a, b = body.index("kCfgs[] = {"), body.index("};", body.index("kCfgs[] = {"))
    body = body[:a] + 'kCfgs[] = {\n  {"fp8 moe w2, 2 waves", false, 4, 2, true, 1},\n' + body[b:]
    assert "Grids[] = {80, 256, 304}" in body and "const int Ks[] = {128," in body
    body = body.replace("Grids[] = {80, 256, 304}", "Grids[] = {160, 512, 608}")
    body = body.replace("const int Ks[] = {128,", "const int Ks[] = {640, 768, 1792, 128,")
    monkeypatch.setattr(plan, "CHECKER", body)
    res = subprocess.run([str(plan._build(tmp_path))], capture_output=True, text=True, timeout=300)
    assert res.returncode == 0, res.stdout
    assert int(res.stdout.split()[1]) > 500
