"""Budgets that select the same kernel are one choice for the tuner."""
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,same", [(1024, {"fanout": [{"2", "4", "6"}, {"split2", "split4", "split6"}],
                                            "fanin": [{"2", "4", "6"}, {"split2", "split4", "split6"}]}),
                                    (384, {"fanout": [], "fanin": [{"2", "4"}]})])
def test_budgets_of_one_kernel_share_a_timing(dev, n, same):
    from pyfwix_amd import autotune
    before = {(k, m): (autotune.get_layout(k, m, n), autotune.get(k, m, n)) for k in (0, 1) for m in range(3)}
    try:
        r = autotune.tune_size(n, planes=4, reps=2)
        for key in ("fanout", "fanin", "scatter_fanout", "scatter_fanin"):
            groups = same["fanout" if "fanout" in key else "fanin"]
            for g in groups:
                assert len({r[key][c] for c in g}) == 1, (key, r[key])
            assert all(t > 0 for t in r[key].values())
    finally:
        for (k, m), (layout, wpe) in before.items():
            autotune.set_layout(k, m, n, layout)
            autotune.set_budget(k, m, n, wpe)
