"""Saved tables of the column tuner (no GPU)."""
import json


def test_table_without_layouts_leaves_them(tmp_path):
    """A table that names no column layouts (written before there were any) sets its
    budgets and leaves the layouts in use: the 8-column layout at 1024 points, which
    it used to select, is the slower one."""
    from pyfwix_amd import autotune
    before = {(k, m): (autotune.get_layout(k, m, 1024), autotune.get(k, m, 1024)) for k in (0, 1) for m in range(3)}
    p = tmp_path / "t.json"
    try:
        p.write_text(json.dumps({"1024": {"fanout": [4, 4, 4], "fanin": [2, 2, 2]}}))
        autotune.load(str(p))
        for (k, m), (layout, _) in before.items():
            assert autotune.get_layout(k, m, 1024) == layout and autotune.get(k, m, 1024) == (2 if k else 4)
        autotune.save(str(p), sizes=(1024,))
        for k in (0, 1):
            for m in range(3):
                autotune.set_layout(k, m, 1024, 0)
        autotune.load(str(p))
        assert all(autotune.get_layout(k, m, 1024) == layout for (k, m), (layout, _) in before.items())
    finally:
        for (k, m), (layout, wpe) in before.items():
            autotune.set_layout(k, m, 1024, layout)
            autotune.set_budget(k, m, 1024, wpe)
