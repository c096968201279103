"""The edges of the kernels' dispatch and of their tiles: the sizes at which a launch takes
another path or a tile is partly filled."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")

import mxfa  # noqa: E402
import oracle as O  # noqa: E402
from gpuhelp import DEV, MAX_ABS_TOL, REL_L2_TOL, errors, gen_qkv, np_, oracle_params  # noqa: E402

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("D,softcap,ws", [(64, 0.0, False), (128, 0.0, False), (128, 0.0, None), (128, 30.0, None),
                                          (256, 0.0, None), (256, 30.0, False)])
def test_nan_key_code_reaches_every_row_that_sees_it(D, softcap, ws):
    """The saturating conversion mode of the P codes must not be set while the matrix unit works:
    it would turn the NaN scores of a NaN key code into finite ones."""
    _, dev, _ = gen_qkv(1, 8, 1, 192, 192, D, seed=77)
    k = dev["k"].clone()
    k[0, 0, 100, 3] = 0x7F
    p = mxfa.make_params(1, 8, 1, 192, 192, D, causal=True, softcap=softcap)
    o = mxfa.prefill(p, dev["q"], dev["qs"], k, dev["ks"], dev["v"], dev["vs"], workspace=ws)
    torch.cuda.synchronize()
    nan = torch.isnan(o).all(dim=-1)[0]                    # [head][row]
    assert bool(nan[:, 128:].all()) and bool(torch.isfinite(o[0, :, :100]).all())


@pytest.mark.parametrize("parts", [4, 5, 16, 17, 32, 33, 128, 129, 257, 300])
def test_decode_merge_part_counts(monkeypatch, parts):
    """mxfa_decode_combine at the edges of its part groups: one up to 4 partials, then 4, 16 and 32
    groups, with and without a remainder, and a last batch partly past the end."""
    L = 64 * 300 + 32
    monkeypatch.setenv("MXFA_DECODE_WAVES", str(parts))
    monkeypatch.setenv("MXFA_DECODE_COMBINE", "kernel")
    _, dev, host = gen_qkv(1, 3, 1, 1, L, 128, seed=200 + parts)
    p = mxfa.make_params(1, 3, 1, 1, L, 128, causal=True, q_pos0=L - 5)
    n_parts, _ = mxfa.decode_plan(p)
    assert n_parts == parts
    o = mxfa.decode(p, dev["q"], dev["qs"], dev["k"], dev["ks"], dev["v"], dev["vs"])
    torch.cuda.synchronize()
    want = O.attention(oracle_params(p), host["q"], host["qs"], host["k"], host["ks"], host["v"], host["vs"],
                       block_n=mxfa.DEFAULT_BLOCK_N, n_parts=n_parts)
    rel, mab = errors(np_(o), want)
    print(f"   n_parts {n_parts}: rel-L2 {rel:.3e} max-abs {mab:.3e}", flush=True)
    assert rel <= REL_L2_TOL and mab <= MAX_ABS_TOL
