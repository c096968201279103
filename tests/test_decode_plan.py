"""mxfa_decode_plan on the host: the workspace of a plan holds its partials, never shrinks when the
cache grows or the query moves (a caller may size it once, for the longest cache), and with a window
no plan has more partials than key blocks that the query sees (three are rounded up to 4)."""
import random

import mxfa


def _plan(B, Hkv, group, n, D, window, p_rule=0):
    p = mxfa.make_params(B, Hkv * group, Hkv, 1, (n + 31) // 32 * 32, D, causal=True, q_pos0=n - 1, window=window,
                         p_rule=p_rule)
    return mxfa.decode_plan(p)


def test_workspace_covers_shorter_caches(monkeypatch):
    monkeypatch.delenv("MXFA_DECODE_WAVES", raising=False)
    rng = random.Random(5)
    for _ in range(2000):
        B, Hkv, group = rng.randint(1, 80), rng.choice([1, 2, 4, 8, 16]), rng.choice([1, 2, 7, 8, 16, 32])
        D, n, window = rng.choice([64, 128, 256]), rng.randint(1, 20000), rng.choice([0, 100, 4096])
        parts, ws = _plan(B, Hkv, group, n, D, window)
        _, longer = _plan(B, Hkv, group, n + rng.randint(1, 4000), D, window)
        assert longer >= ws
        assert B * Hkv * group * parts * (D + 2) * 4 <= ws
        visible = min(n, window) if window else n
        assert 1 <= parts <= max(4, (visible + 63) // 64 + 1)


def test_partials_that_share_a_workgroup_stay_spread_at_d256(monkeypatch):
    """At D = 256 (one workgroup per CU) a plan of up to 4 partials keeps them with a window: in fewer the
    visible blocks would sit on fewer CUs.  At D = 128 (two workgroups per CU) and in larger plans the
    window still limits them."""
    monkeypatch.delenv("MXFA_DECODE_WAVES", raising=False)
    for B, parts in ((32, 4), (64, 2)):
        for n in (500, 3000):
            assert _plan(B, 8, 4, n, 256, 0)[0] == parts
            assert _plan(B, 8, 4, n, 256, 100)[0] == parts
    assert _plan(64, 8, 4, 3000, 128, 0)[0] == 4
    assert _plan(64, 8, 4, 3000, 128, 100)[0] == 2
    assert _plan(8, 8, 4, 3000, 256, 0)[0] == 16
    assert _plan(8, 8, 4, 3000, 256, 100)[0] == 2
