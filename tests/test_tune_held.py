"""The kept tuning table is nobody else's: what a caller does to the one it was
given does not reach later launches, and another file is read again."""

import json
import os

from piquasso_amd import tune

ARCH = "gfx950:sramecc+:xnack-"


def _table(units):
    return {"device": "gfx950", "cus": 256, "workloads": {
        "batched_uneven": {"best": {"total_units": units, "persistent": False}, "log2_terms": 15.2}}}


def test_a_callers_changes_stay_its_own(tmp_path):
    path = str(tmp_path / "t.json")
    open(path, "w").write(json.dumps(_table(5120)))
    before = tune.best_config(4096, 256, ARCH, path=path, log2_terms=15.0)
    mine = tune.load_tuning(path)
    mine["workloads"]["batched_uneven"]["best"]["total_units"] = 1
    mine["workloads"].clear()
    assert tune.best_config(4096, 256, ARCH, path=path, log2_terms=15.0) == before == {
        "total_units": 5120, "persistent": False}
    assert tune.load_tuning(path) == _table(5120)


def test_another_file_of_the_same_size_and_time(tmp_path):
    path, other = tmp_path / "t.json", tmp_path / "u.json"
    path.write_text(json.dumps(_table(5120)))
    other.write_text(json.dumps(_table(5248)))
    at = path.stat()
    os.utime(other, ns=(at.st_atime_ns, at.st_mtime_ns))
    assert tune.load_tuning(str(path)) == _table(5120)
    other.replace(path)
    assert tune.load_tuning(str(path)) == _table(5248)
    path.unlink()
    assert tune.load_tuning(str(path)) == {}
