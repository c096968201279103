"""The edges of the kernels' dispatch and of their tiles: the sizes at which a launch takes
another path or a tile is partly filled."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")

import mxfa  # noqa: E402
import oracle as O  # noqa: E402
from gpuhelp import DEV, MAX_ABS_TOL, REL_L2_TOL, errors, gen_qkv, np_, oracle_params  # noqa: E402
from test_gpu_gemm import run_gemm  # noqa: E402

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


@pytest.mark.parametrize("v_fmt", [mxfa.FMT_E4M3, mxfa.FMT_E3M2, mxfa.FMT_E3M2_BLK])
@pytest.mark.parametrize("D,softcap,p_rule", [(64, 0.0, mxfa.P_R1), (128, 0.0, mxfa.P_R1), (128, 30.0, mxfa.P_R1),
                                              (256, 30.0, mxfa.P_R1), (256, 0.0, mxfa.P_R2)])
@pytest.mark.parametrize("where,pos", [("key", 5), ("key", 1000), ("key", 1997), ("scale", 700), ("query", 3),
                                       ("infinite", 600)])
def test_nan_and_infinite_scores_pass_the_split_merge(D, softcap, p_rule, v_fmt, where, pos):
    """A split call (32 key blocks) with a NaN code in the first, a middle or the last key range, a NaN
    scale, a NaN query code or scores that overflow: the rows of mxfa_prefill (one pass) that are
    NaN are NaN, and only they."""
    n = 2000
    _, dev, _ = gen_qkv(1, 4, 2, 8, 2016, D, seed=78, v_fmt=v_fmt)
    if where == "key":
        dev["k"][0, 1, pos, 3] = 0x7F
    elif where == "scale":
        dev["ks"][0, 1, pos, 0] = 255
    elif where == "query":
        dev["q"][0, 2, pos, 1] = 0x7F
    else:                                                  # 448 x 2^127 per product
        dev["ks"][0, 1, pos] = 254
        dev["k"][0, 1, pos] = 0x7E
    p = mxfa.make_params(1, 4, 2, 8, 2016, D, causal=True, q_pos0=n - 8, softcap=softcap, v_fmt=v_fmt, p_rule=p_rule)
    ops = [dev[x] for x in ("q", "qs", "k", "ks", "v", "vs")]
    split = torch.isnan(mxfa.prefill(p, *ops))
    one = torch.isnan(mxfa.prefill(p, *ops, workspace=False))
    torch.cuda.synchronize()
    assert bool(one.any())
    assert torch.equal(split, one)


@pytest.mark.parametrize("waves,combine", [(1, None), (2, None), (4, None), (4, "kernel"), (24, None), (200, None)])
def test_nan_key_code_reaches_the_decoded_row(monkeypatch, waves, combine):
    """Merged inside the workgroup or by mxfa_decode_combine, a partial with a NaN is not left out."""
    monkeypatch.setenv("MXFA_DECODE_WAVES", str(waves))
    if combine:
        monkeypatch.setenv("MXFA_DECODE_COMBINE", combine)
    L = 64 * 200
    _, dev, _ = gen_qkv(1, 4, 2, 1, L, 128, seed=79)
    dev["k"][0, 1, 5000, 3] = 0x7F
    p = mxfa.make_params(1, 4, 2, 1, L, 128, causal=True, q_pos0=L - 5)
    o = mxfa.decode(p, *(dev[x] for x in ("q", "qs", "k", "ks", "v", "vs")))
    torch.cuda.synchronize()
    assert bool(torch.isnan(o[0, 2:]).all()) and bool(torch.isfinite(o[0, :2]).all())


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


@pytest.mark.parametrize("B,Hq,Hkv,Sq,n,D,kw", [
    (1, 8, 2, 1, 1024, 128, {}),                                        # 16 key blocks: the shortest split range
    (1, 8, 2, 32, 2000, 128, dict(v_fmt=mxfa.FMT_E3M2)),                # a full query tile, last block partly filled
    (2, 14, 2, 31, 1100, 64, dict(v_fmt=mxfa.FMT_E3M2_BLK, p_rule=mxfa.P_R2)),
    (1, 4, 2, 5, 3001, 256, dict(softcap=30.0, window=1500)),           # ranges that start inside the window
    (1, 2, 1, 33, 5200, 256, dict(v_fmt=mxfa.FMT_E3M2, softcap=30.0)),  # two query tiles, 82 key blocks
    (1, 16, 4, 100, 5152, 128, {}),                                     # two tiles: the shortest such call
    (1, 8, 4, 40, 6000, 256, dict(window=1200, v_fmt=mxfa.FMT_E3M2_BLK)),
    (1, 3, 3, 64, 5300, 64, dict(causal=False)),
    (1, 4, 1, 17, 4096, 128, dict(short=2200)),                         # queries far before the end: ranges past them empty
])
def test_split_prefill_matches_single_pass(B, Hq, Hkv, Sq, n, D, kw):
    """mxfa_prefill_ws split over the keys against mxfa_prefill (one pass): the same P codes, so O
    differs by fp32 summation order alone.  Each of the at most 32 partials is rounded once more
    when it is scaled and added: 32 x 2^-24 = 2e-6 of the row."""
    Sk = (n + 31) // 32 * 32
    v_fmt = kw.get("v_fmt", mxfa.FMT_E4M3)
    causal = kw.get("causal", True)
    pos0 = kw.get("short", n - Sq) if causal else 0
    _, dev, host = gen_qkv(B, Hq, Hkv, Sq, Sk, D, seed=300 + n, outlier_p=0.01, v_fmt=v_fmt)
    p = mxfa.make_params(B, Hq, Hkv, Sq, Sk, D, causal=causal, q_pos0=pos0, window=kw.get("window", 0),
                         softcap=kw.get("softcap", 0.0), v_fmt=v_fmt, p_rule=kw.get("p_rule", mxfa.P_R1))
    ops = [dev[x] for x in ("q", "qs", "k", "ks", "v", "vs")]
    out = torch.full((B, Hq, Sq, D), float("nan"), dtype=torch.float32, device=DEV)
    ws = torch.full((mxfa.prefill_plan(p),), 255, dtype=torch.uint8, device=DEV)      # NaN wherever a partial is read unwritten
    mxfa.prefill(p, *ops, out=out, workspace=ws)
    one = mxfa.prefill(p, *ops, workspace=False)
    again = mxfa.prefill(p, *ops, workspace=ws)
    torch.cuda.synchronize()
    assert not torch.equal(out, one), "the call was not split"
    assert torch.equal(out, again)
    rel, _ = errors(np_(out), np_(one))
    print(f"   split against one pass: rel-L2 {rel:.3e}", flush=True)
    assert rel <= 2e-6


@pytest.mark.parametrize("Hq,Hkv,Sq,n,D,v_fmt,ranges", [
    (2, 1, 8, 20000, 64, mxfa.FMT_E4M3, 50),                    # merged by 16 groups
    (4, 1, 5, 131072, 128, mxfa.FMT_E3M2_BLK, 128),             # the most of them
    (2, 1, 8, 160000, 64, mxfa.FMT_E3M2, 141),                  # 32 groups
    (2, 1, 3, 300000, 256, mxfa.FMT_E4M3, 193),
])
def test_split_prefill_of_many_ranges(Hq, Hkv, Sq, n, D, v_fmt, ranges):
    """As above for long caches: sqrt(8 x key blocks) ranges.  Every range is rounded once more in the
    merge (2^-24 of the row), and both passes round their own sums over the blocks, independently
    (the root of their number)."""
    Sk = (n + 31) // 32 * 32
    _, dev, _ = gen_qkv(1, Hq, Hkv, Sq, Sk, D, seed=500 + n // 1000, v_fmt=v_fmt)
    p = mxfa.make_params(1, Hq, Hkv, Sq, Sk, D, causal=True, q_pos0=n - Sq, v_fmt=v_fmt)
    ops = [dev[x] for x in ("q", "qs", "k", "ks", "v", "vs")]
    ws = torch.full((mxfa.prefill_plan(p),), 255, dtype=torch.uint8, device=DEV)
    split, one = mxfa.prefill(p, *ops, workspace=ws), mxfa.prefill(p, *ops, workspace=False)
    torch.cuda.synchronize()
    assert not torch.equal(split, one), "the call was not split"
    rel, _ = errors(np_(split), np_(one))
    print(f"   {ranges} ranges against one pass: rel-L2 {rel:.3e}", flush=True)
    assert rel <= (ranges + (Sk / 64) ** 0.5) * 2.0 ** -24


@pytest.mark.parametrize("B,Hq,Hkv,Sq,n,D,kw", [
    (32, 32, 8, 32, 1000, 64, {}),
    (24, 32, 8, 32, 1500, 128, dict(window=1300)),
    (20, 32, 8, 32, 1000, 256, dict(softcap=30.0, p_rule=mxfa.P_R2)),
])
def test_short_prefill_of_many_rows_is_one_pass(B, Hq, Hkv, Sq, n, D, kw):
    """Where the partials of a split would cost more than the shorter walk saves, mxfa_prefill_ws runs
    the single pass: bit-identical with mxfa_prefill."""
    Sk = (n + 31) // 32 * 32
    _, dev, _ = gen_qkv(B, Hq, Hkv, Sq, Sk, D, seed=400 + n)
    p = mxfa.make_params(B, Hq, Hkv, Sq, Sk, D, causal=True, q_pos0=n - Sq, **kw)
    ops = [dev[x] for x in ("q", "qs", "k", "ks", "v", "vs")]
    ws, one = mxfa.prefill(p, *ops), mxfa.prefill(p, *ops, workspace=False)
    torch.cuda.synchronize()
    assert torch.equal(ws, one)


@pytest.mark.parametrize("M,N,K,a_fmt,b_fmt", [
    # 64 x 64 tiles (256 k per stage)
    (48, 64, 64, 0, 0),              # one half: no whole stage
    (80, 144, 192, 0, 0),            # three halves, rows and columns past the tile
    (128, 8192, 256, 0, 0),          # one stage, 256 tiles; three of the four stages hold nothing
    (1024, 1024, 1344, 0, 0),        # 5 whole stages and a half
    (16, 8208, 512, 0, 0),           # more strips than CUs
    # 128 x 128 tiles
    (144, 6208, 64, 0, 0),           # one half step only
    (160, 6160, 192, 0, 0),          # a step and a half, columns and rows past the tile
    (400, 4112, 576, 0, 0),          # 4 whole steps and a half, ragged
    (1024, 4096, 640, 0, 0),         # 256 tiles
    (1024, 4112, 448, 0, 0),         # a second round of tiles: K % 128 = 64 (256 x 256 tiles below K = 1,024 otherwise)
    (1024, 4112, 896, 0, 0), (1040, 4096, 1024, 0, 0),
    (272, 272, 1088, 0, 1), (256, 144, 64, 1, 0), (48, 400, 320, 1, 1),
])
def test_gemm_small_and_mid_tiles_equal_register_staged(monkeypatch, M, N, K, a_fmt, b_fmt):
    """The 64 x 64 and 128 x 128 tiles run the MFMAs of the 256 x 256 kernels on the same operands in
    the same order: C must match bit for bit, fp32 and bf16."""
    g = torch.Generator(device=DEV)
    g.manual_seed(M + N + K)

    def codes(fmt, shape):
        c = torch.randint(0, 256 if fmt == 0 else 64, shape, generator=g, device=DEV, dtype=torch.int32)
        return torch.where((c & 127) == 127, c - 1, c).to(torch.uint8)

    a, b = codes(a_fmt, (M, K)), codes(b_fmt, (K, N))
    sa, sb = (torch.randint(112, 142, (K // 32, n), generator=g, device=DEV, dtype=torch.int32).to(torch.uint8) for n in (M, N))
    for c_fmt, dt in ((mxfa.C_F32, torch.float32), (mxfa.C_BF16, torch.bfloat16)):
        outs = []
        for mode in (None, "reg"):
            if mode:
                monkeypatch.setenv("MXFA_GEMM", mode)
            else:
                monkeypatch.delenv("MXFA_GEMM", raising=False)
            c = torch.full((M, N), float("nan"), dtype=dt, device=DEV)
            mxfa.gemm(a, sa, b, sb, a_fmt, b_fmt, out=c, c_fmt=c_fmt)
            outs.append(c)
        torch.cuda.synchronize()
        assert bool(torch.isfinite(outs[0]).all())
        assert torch.equal(outs[0], outs[1])


@pytest.mark.parametrize("M,N,K,strips", [
    (16, 48, 8256, True), (32, 8192, 1088, True),                # M <= 32: up to 256 strips of 32 columns
    (32, 8208, 1088, False),
    (48, 80, 8256, True), (64, 4096, 14336, True),               # M <= 64: K above 8,192; 129 steps of 64 k, half a strip
    (64, 8192, 8256, True), (64, 8208, 8256, False),
    (64, 96, 8192, False),
    (64, 96, 32768, True), (64, 96, 32832, False),               # the scales fill the strip kernel's LDS exactly; past it
    (80, 96, 8256, False),
])
def test_gemm_strip_kernel_dispatch(monkeypatch, M, N, K, strips):
    """The k-split strip kernel on its side of each line of the dispatch and the tiles (C bit-identical with
    the 256 x 256 kernels) on the other.  Against the 256 x 256 kernels the strips add the same
    products in another order: as in test_gemm_skinny_matches_oracle_and_tiled_kernel, whose
    bound is 2^-12 of the terms' absolute sum; with terms of random sign that sum is about the
    root of K times the result, 2^-12 sqrt(K) of it at most."""
    monkeypatch.delenv("MXFA_GEMM", raising=False)
    g = torch.Generator(device=DEV)
    g.manual_seed(M + N + K)
    a, b = (torch.randint(0, 256, shape, generator=g, device=DEV, dtype=torch.int32) for shape in ((M, K), (K, N)))
    a, b = (torch.where((c & 127) == 127, c - 1, c).to(torch.uint8) for c in (a, b))
    sa, sb = (torch.randint(112, 142, (K // 32, n), generator=g, device=DEV, dtype=torch.int32).to(torch.uint8) for n in (M, N))
    c, again = mxfa.gemm(a, sa, b, sb), mxfa.gemm(a, sa, b, sb)
    c16 = torch.empty((M, N), dtype=torch.bfloat16, device=DEV)
    mxfa.gemm(a, sa, b, sb, out=c16, c_fmt=mxfa.C_BF16)
    monkeypatch.setenv("MXFA_GEMM", "big")
    big = mxfa.gemm(a, sa, b, sb)
    torch.cuda.synchronize()
    assert torch.equal(c, again) and torch.equal(c16, c.to(torch.bfloat16))
    assert torch.equal(c, big) != strips
    rel, _ = errors(np_(c), np_(big))
    assert rel <= 2.0 ** -12 * K ** 0.5


@pytest.mark.parametrize("M,N,K", [(48, 80, 8256), (64, 208, 14336), (64, 48, 9216)])
def test_gemm_two_tile_strip_kernel_matches_oracle(M, N, K):
    """33 to 64 rows on the strip kernel, within the oracle's bound of every mxfa_gemm."""
    run_gemm(M, N, K, seed=M + N + K)


@pytest.mark.parametrize("rows,cols", [(1, 32), (31, 32), (33, 64), (131071, 32), (131072, 32), (131073, 32), (1025, 4128),
                                       (4096, 4064), (4096, 4096), (4097, 4128)])
@pytest.mark.parametrize("fmt", [mxfa.FMT_E4M3, mxfa.FMT_E3M2])
def test_quantize_rows_block_counts(rows, cols, fmt):
    """Workgroups of 32 blocks, or of 128 (four per thread) from 131,072 blocks (E3M2) or 524,288
    (E4M3) on: around both workgroup sizes and the change between them."""
    x = torch.randn(rows, cols, generator=torch.Generator().manual_seed(rows + cols))
    codes, scales = mxfa.quantize_rows(x.to(DEV), fmt)
    want, want_sc = O.quantize_rows(x.numpy(), fmt)
    np.testing.assert_array_equal(np_(codes), want)
    np.testing.assert_array_equal(np_(scales), want_sc)


@pytest.mark.parametrize("mats,rows,cols", [(1, 32, 4), (3, 32, 36), (1, 96, 128), (2, 64, 132), (5, 32, 260)])
@pytest.mark.parametrize("fmt", [mxfa.FMT_E4M3, mxfa.FMT_E3M2, mxfa.FMT_E3M2_BLK])
def test_quantize_cols_column_counts(mats, rows, cols, fmt):
    """Waves of 128 columns, four to a workgroup: a few columns, a whole wave, a few past it, and
    workgroups whose last waves have nothing."""
    x = torch.randn(mats, rows, cols, generator=torch.Generator().manual_seed(mats + rows + cols))
    codes, scales = mxfa.quantize_cols(x.to(DEV), fmt)
    want, want_sc = O.quantize_cols(x.numpy(), O.FMT_E4M3 if fmt == mxfa.FMT_E4M3 else O.FMT_E3M2)
    if fmt == mxfa.FMT_E3M2_BLK:
        want = mxfa.e3m2_to_blk(want)
    np.testing.assert_array_equal(np_(codes), want)
    np.testing.assert_array_equal(np_(scales), want_sc)
