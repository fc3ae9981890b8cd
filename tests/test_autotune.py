"""Tile tables of the GEMM: installing and dropping rules (host only)."""

import ctypes
import json

import pytest


@pytest.fixture
def rules(monkeypatch, tmp_path):
    from qe_python_amd import _native as nat
    from qe_python_amd import autotune
    from qe_python_amd import device as dv
    monkeypatch.setattr(autotune, "TABLE", tmp_path / "none.json")
    autotune.load_table()
    yield nat, autotune, dv
    monkeypatch.undo()
    nat.load().qepw_gemm_clear_rules()
    autotune.load_table()


def plan(nat, m, n, k):
    out = (ctypes.c_int64 * 4)()
    nat.check(nat.load().qepw_gemm_plan(nat.C128, nat.OP_C, m, n, k, out), "plan")
    return list(out)


def test_the_default_drops_rules_and_cached_sizes(rules):
    """Without a table, load_table() restores the built-in choice: rules set
    before, and the workspace sizes that Python keeps for them, go."""
    nat, autotune, dv = rules
    m, n, k = 200, 61, 3000
    built_in = plan(nat, m, n, k)
    ranges = (ctypes.c_int64 * 6)(m, m, n, n, k, k)
    nat.check(nat.load().qepw_gemm_set_rule(nat.C128, nat.OP_C, ranges, 3, 7), "rule")
    forced = plan(nat, m, n, k)
    assert forced[:2] == [3, 7] != built_in[:2]
    dv._GEMM_WORKSPACE[(nat.C128, nat.OP_C, m, n, k)] = 7 * m * n * 16
    assert autotune.load_table() == 0
    assert plan(nat, m, n, k) == built_in
    assert not dv._GEMM_WORKSPACE


def test_a_table_installs_its_rules(rules, tmp_path):
    nat, autotune, _ = rules
    table = tmp_path / "table.json"
    table.write_text(json.dumps({"rules": [
        {"precision": "fp64", "op": "C", "m": [1, 256], "n": [2, 64], "k": [2049, 1 << 40],
         "variant": 6, "splits": 9, "ms": 1.0, "default_ms": 2.0},
        {"precision": "fp64", "op": "C", "m": [1, 256], "n": [65, 128], "k": [2049, 1 << 40],
         "variant": 6, "splits": 9, "ms": 1.0, "default_ms": 1.01}]}))
    wide = plan(nat, 200, 100, 3000)
    assert autotune.load_table(table) == 1
    assert plan(nat, 200, 61, 3000)[:2] == [6, 9]
    assert plan(nat, 200, 100, 3000) == wide
    assert autotune.load_table(tmp_path / "missing.json") == 0
    assert plan(nat, 200, 61, 3000)[:2] == [6, 9]
