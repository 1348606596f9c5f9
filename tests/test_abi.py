"""The C-ABI library loads and exports every entry point the headers declare;
argument validation answers with status codes before touching the GPU."""
import ctypes
import re
from pathlib import Path

import pytest

ROOT = Path(__file__).resolve().parents[1]


def declared_symbols():
    names = set()
    for h in sorted((ROOT / "include").glob("*.h")):
        text = re.sub(r"/\*.*?\*/", "", h.read_text(), flags=re.S)
        names |= set(re.findall(r"\b(lufqhe_\w+)\s*\(", text))
    return sorted(names)


def test_headers_declare_entry_points():
    names = declared_symbols()
    assert "lufqhe_det_batched" in names
    assert len(names) >= 4


def test_library_exports_declared_symbols(lc):
    lib = lc.load()
    missing = [n for n in declared_symbols() if not hasattr(lib, n)]
    assert not missing, missing


def test_status_strings(lc):
    lib = lc.load()
    assert lib.lufqhe_status_string(0) == b"success"
    assert lib.lufqhe_version() >= 100


@pytest.mark.parametrize("n,ld,stride,batch,policy,arith,want", [
    (0, 1, 1, 1, 0, 0, 1),       # n < 1
    (65, 65, 65 * 65, 1, 0, 0, 1),  # n > 64
    (8, 7, 64, 1, 0, 0, 1),      # ld < n
    (8, 8, -1, 1, 0, 0, 1),      # negative stride
    (8, 8, 64, -1, 0, 0, 1),     # negative batch
    (8, 8, 64, 1, 1, 1, 2),      # ABS pivots with reference arithmetic: unsupported
    (8, 8, 64, 1, 7, 0, 2),      # unknown policy
    (8, 8, 64, 0, 0, 0, 0),      # empty batch: no-op success
])
def test_argument_validation(lc, n, ld, stride, batch, policy, arith, want):
    lib = lc.load()
    st = lib.lufqhe_det_batched(None, batch, n, ld, stride, None, None, None, None, None, None,
                                policy, arith, None)
    assert st == want


def test_null_input_rejected(lc):
    lib = lc.load()
    assert lib.lufqhe_det_batched(None, 4, 8, 8, 64, None, None, None, None, None, None,
                                  0, 0, None) == 1


def test_epilogue_argument_validation(lc):
    lib = lc.load()
    assert lib.lufqhe_det_inplace(None, 0, 8, 8, 64, 1, 0, None, None) == 0   # empty batch
    assert lib.lufqhe_det_inplace(None, 4, 8, 8, 64, 1, 0, None, None) == 1   # null A
    assert lib.lufqhe_det_inplace(None, 4, 0, 8, 64, 1, 0, None, None) == 1   # bad n
    assert lib.lufqhe_det_inplace(None, 4, 8, 8, 64, 1, 9, None, None) == 2   # bad policy
    assert lib.lufqhe_global_reduction(None, 4, 64, None, None, None) == 1     # null output
    assert lib.lufqhe_global_reduction(None, 4, 64, None, 1, None) == 1        # null A, pairs > 0
    assert lib.lufqhe_pair_sum(None, None, 4, None, None, None, None) == 1
    assert lib.lufqhe_det_inplace_workspace_bytes(10) == 200
    assert lib.lufqhe_pair_sum_workspace_bytes() > 0


def test_shape_table_api(lc):
    lib = lc.load()
    for n in range(1, 65):
        c = lib.lufqhe_shape_count(n)
        assert 1 <= c <= 4
        for sh in range(c):
            lanes, cols, waves = lc.shape_info(n, sh)
            assert lanes in (4, 8, 16, 32, 64) and cols in (1, 2, 4) and lanes % cols == 0
            assert waves in (1, 2)
    assert lib.lufqhe_shape_count(0) == 0 and lib.lufqhe_shape_count(65) == 0
    assert lib.lufqhe_set_shape(0, 0, 32, 7) == 1          # shape out of range
    assert lib.lufqhe_set_shape(0, 1, 32, 1) == 4          # reference arithmetic: shape 0 only
    assert lib.lufqhe_set_shape(1, 1, 32, 0) == 2          # ABS + reference arithmetic
    assert lib.lufqhe_get_shape(0, 0, 0) == -1
    old = lc.get_shape("crout_ref", "fused", 32)
    assert lc.set_shape("crout_ref", "fused", 32, 2) and lc.get_shape("crout_ref", "fused", 32) == 2
    assert lc.set_shape("crout_ref", "fused", 32, old)


def test_package_reads_a_shape_table_as_json(lc, tmp_path):
    """apply_shape_table reads any valid JSON table, and refuses a damaged one
    whole instead of applying what comes before the damage."""
    import json
    from importlib import import_module
    entries = json.loads(import_module("lion-codes_amd.lucore").SHAPE_TABLE.read_text())["entries"]
    first = next(e for e in entries if e["shape"] != 0)
    text = json.dumps({"note": {"entries": [1]}, "entries": [first] + entries[:3]},
                      separators=(", ", " :\r "))
    p = tmp_path / "t.json"

    def apply(s):
        p.write_text(s, newline="")
        return lc.apply_shape_table(p)
    assert lc.apply_shape_table(tmp_path / "missing.json") == 0
    assert apply("{}") == 0 and apply('{"entries": []}') == 0
    assert apply(text) == 4
    where = (first["policy"], "fused", first["n"])
    assert lc.get_shape(*where) == first["shape"] and lc.set_default_shape(*where, 0)
    for bad in ("", text[:-20], text + "}"):
        with pytest.raises(json.JSONDecodeError):
            apply(bad)
    assert lc.get_shape(*where) == 0
    with pytest.raises(KeyError):
        apply(json.dumps({"entries": [{k: v for k, v in entries[0].items() if k != "n"}]}))
    lc.apply_shape_table()


def test_selection_of_a_shape_round_trips(lc):
    """get_shape, set_shape(x), set_shape(got) restores which kernel uniform
    batches run, small ones included (256 compute units: 1024 matrices of
    n = 17..32, 256 of n >= 49)."""
    lib = lc.load()
    for policy in ("crout_ref", "abs"):
        for n in range(1, 65):
            def routes(p=policy, n=n):
                return [lc.uniform_shape(p, "fused", n, c, 256) for c in (1, limit, limit + 1)]
            limit = 1024 if n <= 32 else 256
            keep = lc.get_shape(policy, "fused", n)
            small = lc.SHAPE_SMALL_BATCH if 17 <= n <= 32 or n >= 49 else keep
            start = [small, small, keep]
            assert routes() == start, (policy, n)
            for s in range(lc.shape_count(n)):
                assert lc.set_shape(policy, "fused", n, s)
                assert lc.get_shape(policy, "fused", n) == s
                assert routes() == (start if s == keep else [s, s, s]), (policy, n, s)
                assert lc.set_shape(policy, "fused", n, s | lc.SHAPE_PINNED)
                assert routes() == [s, s, s], (policy, n, s)
                got = lc.get_shape(policy, "fused", n)  # a pinned selection round trips too
                assert lc.set_shape(policy, "fused", n, 0) and lc.set_shape(policy, "fused", n, got)
                assert routes() == [s, s, s], (policy, n, s)
                assert lc.set_shape(policy, "fused", n, keep)
                assert routes() == start, (policy, n, s)
            # another default: its own round trip
            s = lc.shape_count(n) - 1
            assert lc.set_default_shape(policy, "fused", n, s)
            assert routes() == [s if small == keep else small] * 2 + [s]
            assert lc.set_default_shape(policy, "fused", n, keep)
            assert routes() == start
    for fn in (lib.lufqhe_set_shape, lib.lufqhe_set_default_shape):
        assert fn(0, 0, 32, -1) == 1 and fn(0, 0, 32, 7) == 1 and fn(0, 0, 32, 0x200) == 1
        assert fn(0, 1, 32, 1) == 4 and fn(1, 1, 32, 0) == 2
    assert lib.lufqhe_set_default_shape(0, 0, 32, 0x100) == 1   # a default is never pinned
    assert lib.lufqhe_uniform_shape(0, 1, 32, 10, 256) == 0     # reference arithmetic: its one shape
    for bad in ((9, 0, 32, 10, 256), (0, 0, 0, 10, 256), (0, 0, 32, 0, 256), (0, 0, 32, 10, -1)):
        assert lib.lufqhe_uniform_shape(*bad) == -1


def test_fqhe_argument_validation(lc):
    lib = lc.load()
    args = (None, None, None, None, None, None, 0, 0, None)
    assert lib.lufqhe_fqhe_det(None, 0, 8, 8, None, *args) == 0     # empty batch
    assert lib.lufqhe_fqhe_det(None, 4, 8, 5, None, *args) == 1     # 0 < z_stride < n
    assert lib.lufqhe_fqhe_det(None, 4, 65, 65, None, *args) == 1   # n > 64
    assert lib.lufqhe_fqhe_det(None, 4, 8, 8, None, *args) == 1     # null positions
    assert lib.lufqhe_fqhe_det(None, 4, 8, 0, None, None, None, None, None, None, None,
                               1, 1, None) == 2                      # ABS + reference arithmetic
    assert lib.lufqhe_fqhe_build(None, 4, 8, 8, None, None, None) == 1
    assert lib.lufqhe_fqhe_build(None, 0, 8, 8, None, None, None) == 0


def test_shape_table_loads_from_c(lc, tmp_path):
    """The C loader applies the committed table exactly as the Python one."""
    import json
    lib = lc.load()
    from importlib import import_module
    core = import_module("lion-codes_amd.lucore")
    entries = json.loads(core.SHAPE_TABLE.read_text())["entries"]
    saved = {(e["policy"], e["n"]): lc.get_shape(e["policy"], "fused", e["n"]) for e in entries}
    try:
        for (pol, n) in saved:
            assert lc.set_shape(pol, "fused", n, 0)
        applied = lib.lufqhe_load_shape_table(str(core.SHAPE_TABLE).encode())
        assert applied == len(entries)
        for e in entries:
            assert lc.get_shape(e["policy"], "fused", e["n"]) == e["shape"]
        # an entry whose geometry no longer matches its index is skipped
        bad = dict(entries[0], lanes=entries[0]["lanes"] * 2 if entries[0]["lanes"] < 64 else 4)
        p = tmp_path / "t.json"
        p.write_text(json.dumps({"entries": [bad]}))
        assert lib.lufqhe_load_shape_table(str(p).encode()) == 0
        # and so is one measured on another kernel of the same geometry, by
        # both readers: no "kernel" means a vector kernel
        kinds = {(n, lc.shape_kernel(n, 0), lc.shape_kernel(n, lc.shape_count(n) - 1))
                 for n in (16, 20, 52)}
        assert kinds == {(16, "vector", "vector"), (20, "vector", "panel"), (52, "panel", "panel")}
        for n, sh in ((16, 0), (20, 0), (20, 3), (52, 0), (52, 1)):
            lanes, cols, waves = lc.shape_info(n, sh)
            e = {"policy": "abs", "n": n, "shape": sh, "lanes": lanes, "lane_cols": cols,
                 "waves": waves}
            for kind in (None, "vector", "panel", "other"):
                p.write_text(json.dumps({"entries": [e if kind is None else dict(e, kernel=kind)]}))
                want = int((kind or "vector") == lc.shape_kernel(n, sh))
                assert lib.lufqhe_load_shape_table(str(p).encode()) == want, (n, sh, kind)
                assert lc.apply_shape_table(p) == want, (n, sh, kind)
        assert lib.lufqhe_shape_kernel(16, 2) == -1 and lib.lufqhe_shape_kernel(65, 0) == -1
        assert lib.lufqhe_load_shape_table(str(tmp_path / "missing.json").encode()) == -1
    finally:
        lc.apply_shape_table()
        for (pol, n), sh in saved.items():
            lc.set_shape(pol, "fused", n, sh)
