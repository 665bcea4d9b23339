"""The autotuner's choices (no GPU): a knob has several values only where they differ, and a case
with nothing to choose starts no timing run."""
import pytest

from minismac_amd import autotune
from minismac_amd._abi import SMAC_FP32_LHS, SMAC_ORDER_ZEBRA
from minismac_amd.case import config_case


@pytest.mark.parametrize("kw", [dict(impsch=2, iturb=0), dict(impsch=2, ivis=0),
                                dict(impsch=2, iturb=0, precision=SMAC_FP32_LHS), dict(impsch=1),
                                dict(impsch=1, line_order=SMAC_ORDER_ZEBRA)])
def test_nothing_to_choose_is_not_timed(tmp_path, monkeypatch, kw):
    def no_probe(*a, **k):
        raise AssertionError("a timing run of settings that launch the same kernels")

    monkeypatch.setattr(autotune, "_Probe", no_probe)
    case, path = config_case(0, **kw), str(tmp_path / "tune.json")
    opts = autotune.tune(case, path=path)
    assert opts == {name: vals[0] for name, vals in autotune._space(case)}
    assert autotune._load(path)[autotune.key(case)]["options"] == opts


def test_scalar_sweeps_have_rows_to_choose():
    assert len(dict(autotune._space(config_case(0, impsch=2)))["lusgs_rows"]) > 1


def test_settings_of_another_build_are_not_taken(tmp_path, monkeypatch):
    case = config_case(0, impsch=2)
    builds = [tmp_path / "a.so", tmp_path / "b.so"]
    keys = []
    for i, b in enumerate(builds):
        b.write_bytes(b"build %d" % i)
        monkeypatch.setattr(autotune, "LIB_PATH", str(b))
        keys.append(autotune.key(case))
    assert keys[0] != keys[1] and all("119x31" in k for k in keys)
    # an entry of a version whose keys did not name the build
    sa = int(case.params.ivis == 1 and case.params.iturb == 1)
    assert f"{autotune._device_name()}|119x31|impsch2|prec0|sa{sa}" not in keys
