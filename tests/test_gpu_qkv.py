"""GPU parity of the QKV projection with the append in its epilogue
(gkv_qkv_append).

Two contracts:
- qkv_out: x . W^T + bias against the oracle's orc_linear (run.cpp matmul +
  bias add, itself bit-exact with the reference's own code). bf16 products are
  exact and the sums are fp32 on the matrix cores, so the bound is in units of
  the sum of |products|: |gpu - ref| <= 2e-5 * sum_j |x_j w_ij| + 1e-6.
- the cache: every byte of the paged K and V (NaN-poisoned slots that must
  stay untouched included) equals what gkv_kv_append stores for the same
  qkv_out rows, and the stored K/V equal the oracle's orc_kv_append of those
  rows (bit-exact).
"""
import numpy as np
import pytest

from kvcase import INT8_POISON, from_pool

pytestmark = pytest.mark.gpu

D = 64
NAN16 = np.uint16(0x7FC1)


def bf16_round(a):
    u = np.ascontiguousarray(a, dtype=np.float32).view(np.uint32).astype(np.uint64)
    u = ((u + 0x7FFF + ((u >> 16) & 1)) & 0xFFFF0000).astype(np.uint32)
    return u.view(np.float32)


class QkvCase:
    """rows of x (bf16 values), W, bias; a paged cache with a permuted table.
    Decode mode (prompts=None): row b is sequence b at position lens[b]-1.
    Prompt mode: rows are every position of each prompt (row_pos, row_seq)."""

    def __init__(self, seed, Hq, Hkv, hidden, lens=None, prompts=None, window=0, v_int8=False,
                 kv_fp8=False):
        rng = np.random.default_rng(seed)
        self.Hq, self.Hkv, self.hidden, self.window, self.v_int8 = Hq, Hkv, hidden, window, v_int8
        self.kv_fp8 = kv_fp8
        self.N = (Hq + 2 * Hkv) * D
        if prompts is None:
            self.lens = np.asarray(lens, np.int32)
            self.row_seq = np.arange(len(lens), dtype=np.int32)
            self.row_pos = self.lens - 1
            self.decode = True
        else:
            self.lens = np.asarray(prompts, np.int32)
            self.row_seq = np.concatenate([np.full(L, b, np.int32)
                                           for b, L in enumerate(prompts)]).astype(np.int32)
            self.row_pos = np.concatenate([np.arange(L, dtype=np.int32) for L in prompts])
            self.decode = False
        self.B = len(self.lens)
        self.M = len(self.row_pos)
        self.x = bf16_round(rng.standard_normal((self.M, hidden)))
        self.w = bf16_round(rng.standard_normal((self.N, hidden)) * 0.05)
        self.bias = (rng.standard_normal(self.N) * 0.1).astype(np.float32)
        # table: per sequence, blocks for all positions (full) or a ring of W slots
        if window:
            self.n_tbl = window // 16
        else:
            self.n_tbl = int((self.lens.max() + 15) // 16)
        self.NB = self.B * self.n_tbl + 3
        self.table = rng.permutation(self.NB)[:self.B * self.n_tbl].astype(np.int32).reshape(
            self.B, self.n_tbl)


def run(case, gkv, torch, dev, cache=True):
    t = lambda a: torch.from_numpy(np.ascontiguousarray(a)).to(dev)
    x = t(case.x).to(torch.bfloat16)
    w = t(case.w).to(torch.bfloat16)
    cos, sin = gkv.rope_table(int(case.lens.max()) + 1)
    cos_d, sin_d = t(cos), t(sin)
    lens = t(case.lens)
    table = t(case.table)

    def new_cache():
        if case.kv_fp8:  # e4m3 codes poisoned with the NaN code, scales with NaN
            k = t(np.full((case.NB, case.Hkv, 16 * D), 0x7F, np.uint8))
            v = t(np.full((case.NB, case.Hkv, 16 * D), 0x7F, np.uint8))
            vs = t(np.full((case.NB, case.Hkv, 32), np.nan, np.float32))
            return k, v, vs, gkv.cache_view(k, v, table, case.Hkv, ring=case.window, v_scale=vs,
                                            v_format=gkv.KV_FP8)
        k = t(np.full((case.NB, case.Hkv, 16, D), NAN16, np.uint16).view(np.int16))
        vs = None
        if case.v_int8:
            v = t(np.full((case.NB, case.Hkv, 16 * D), INT8_POISON, np.int8))
            vs = t(np.full((case.NB, case.Hkv, 16), np.nan, np.float32))
        else:
            v = t(np.full((case.NB, case.Hkv, D, 16), NAN16, np.uint16).view(np.int16))
        view = gkv.cache_view(k, v, table, case.Hkv, ring=case.window, v_scale=vs)
        return k, v, vs, view

    qkv_out = torch.full((case.M, case.N), float("nan"), dtype=torch.float32, device=dev)
    err = torch.zeros(1, dtype=torch.int32, device=dev)
    k1, v1, vs1, view1 = new_cache()
    row_pos = None if case.decode else t(case.row_pos)
    row_seq = None if case.decode else t(case.row_seq)
    gkv.qkv_append(x, w, t(case.bias), case.Hq, cos_d, sin_d, view1 if cache else None,
                   row_pos=row_pos, row_seq=row_seq, seq_lens=lens, qkv_out=qkv_out,
                   dev_err=err, n_kv_heads=case.Hkv)
    # the same rows through the plain append
    k2, v2, vs2, view2 = new_cache()
    if cache:
        gkv.kv_append(qkv_out, case.Hq, cos_d, sin_d, t(case.row_pos), view2,
                      row_seq=t(case.row_seq), seq_lens=lens)
    torch.cuda.synchronize()
    res = dict(err=int(err.item()), qkv=qkv_out.cpu().numpy(),
               k1=k1.cpu().numpy(), v1=v1.cpu().numpy(), k2=k2.cpu().numpy(),
               v2=v2.cpu().numpy(), cos=cos, sin=sin)
    if case.v_int8 or case.kv_fp8:
        res["vs1"], res["vs2"] = vs1.cpu().numpy(), vs2.cpu().numpy()
    return res


def check_projection(case, res, oracle, rows=None):
    """rows: the rows checked (default: all)."""
    rows = np.arange(case.M) if rows is None else np.asarray(rows)
    ref = oracle.linear(case.x[rows], case.w, case.bias)
    scale = np.abs(case.x[rows]).astype(np.float64) @ np.abs(case.w).astype(np.float64).T
    err = np.abs(res["qkv"][rows].astype(np.float64) - ref)
    bad = err > 2e-5 * scale + 1e-6
    assert not bad.any(), f"{int(bad.sum())} projections out of bound, max err {err.max()}"


def check_cache_fp8(case, res, oracle):
    """e4m3 K/V: every byte and scale equal to gkv_kv_append's, and the codes
    and scales of each stored row equal to the oracle's quantizer on the
    oracle's rotated key and on the value."""
    from kvcase import k_fp8_offsets, v_int8_offsets
    for a, b in (("k1", "k2"), ("v1", "v2")):
        assert np.array_equal(res[a], res[b]), f"{a} differs from gkv_kv_append's"
    assert np.array_equal(res["vs1"].view(np.uint32), res["vs2"].view(np.uint32)), "scales differ"
    _, k_rot, _, _ = oracle.kv_append(res["qkv"], case.Hq, case.Hkv, res["cos"], res["sin"],
                                      case.row_pos)
    v_rows = res["qkv"][:, (case.Hq + case.Hkv) * D:].reshape(case.M, case.Hkv, D)
    kc, ks = oracle.quantize_fp8(np.asarray(k_rot, np.float32).reshape(case.M, case.Hkv, D))
    vc, vsc = oracle.quantize_fp8(v_rows)
    n_checked = 0
    for r in range(case.M):
        b, p = int(case.row_seq[r]), int(case.row_pos[r])
        if case.window and p + case.window < case.lens[b]:
            continue
        slot = p % case.window if case.window else p
        phys, off = case.table[b, slot // 16], slot % 16
        assert np.array_equal(res["k1"][phys][:, k_fp8_offsets(off)], kc[r]), f"K of row {r}"
        assert np.array_equal(res["v1"][phys][:, v_int8_offsets(off)], vc[r]), f"V of row {r}"
        assert np.array_equal(res["vs1"][phys, :, off].view(np.uint32), ks[r].view(np.uint32))
        assert np.array_equal(res["vs1"][phys, :, 16 + off].view(np.uint32),
                              vsc[r].view(np.uint32))
        n_checked += 1
    assert n_checked > 0


def check_cache(case, res, oracle):
    if case.kv_fp8:
        return check_cache_fp8(case, res, oracle)
    assert np.array_equal(res["k1"], res["k2"]), "K cache bytes differ from gkv_kv_append's"
    assert np.array_equal(res["v1"], res["v2"]), "V cache bytes differ from gkv_kv_append's"
    if case.v_int8:
        assert np.array_equal(res["vs1"].view(np.uint32), res["vs2"].view(np.uint32)), \
            "V scales differ"
    # the stored K/V against the oracle's append of the same qkv rows (rows
    # whose ring slot a later row takes are skipped)
    _, _, kb, vb = oracle.kv_append(res["qkv"], case.Hq, case.Hkv, res["cos"], res["sin"],
                                    case.row_pos)
    kl = from_pool(res["k1"].view(np.uint16), "k")
    vl = None if case.v_int8 else from_pool(res["v1"].view(np.uint16), "v")
    n_checked = 0
    for r in range(case.M):
        b, p = int(case.row_seq[r]), int(case.row_pos[r])
        if case.window and p + case.window < case.lens[b]:
            continue
        slot = p % case.window if case.window else p
        phys, off = case.table[b, slot // 16], slot % 16
        assert np.array_equal(kl[phys, :, off, :], kb[r]), f"K of row {r}"
        if vl is not None:
            assert np.array_equal(vl[phys, :, :, off], vb[r]), f"V of row {r}"
        n_checked += 1
    assert n_checked > 0


def test_decode_config2_shape(oracle, gkv, cuda):
    import torch
    rng = np.random.default_rng(2)
    lens = rng.integers(128, 2049, 512)
    case = QkvCase(3, 64, 8, 2880, lens=lens)
    res = run(case, gkv, torch, cuda)
    assert res["err"] == 0
    check_projection(case, res, oracle)
    check_cache(case, res, oracle)


def test_decode_window_ring(oracle, gkv, cuda):
    import torch
    rng = np.random.default_rng(5)
    lens = rng.integers(1, 4097, 96)
    case = QkvCase(6, 64, 8, 576, lens=lens, window=128)
    res = run(case, gkv, torch, cuda)
    assert res["err"] == 0
    check_projection(case, res, oracle)
    check_cache(case, res, oracle)


@pytest.mark.parametrize("window", [0, 128])
def test_prompt_rows(oracle, gkv, cuda, window):
    import torch
    case = QkvCase(11 + window, 8, 2, 256, prompts=[300, 17, 129, 1, 64], window=window)
    res = run(case, gkv, torch, cuda)
    assert res["err"] == 0
    check_projection(case, res, oracle)
    check_cache(case, res, oracle)


def test_int8_v(oracle, gkv, cuda):
    import torch
    rng = np.random.default_rng(8)
    case = QkvCase(9, 16, 4, 512, lens=rng.integers(1, 300, 100), v_int8=True)
    res = run(case, gkv, torch, cuda)
    assert res["err"] == 0
    check_projection(case, res, oracle)
    check_cache(case, res, oracle)


def test_fp8_kv(oracle, gkv, cuda):
    """The e4m3 K/V cache from the projection's epilogue: decode rows on a full
    layer and prompt rows (the 128 x 128 tiles) on a ring."""
    import torch
    rng = np.random.default_rng(31)
    for case in (QkvCase(32, 16, 4, 512, lens=rng.integers(1, 300, 100), kv_fp8=True),
                 QkvCase(33, 64, 8, 2880, prompts=[900, 700, 500], window=128, kv_fp8=True)):
        res = run(case, gkv, torch, cuda)
        assert res["err"] == 0
        check_cache(case, res, oracle)


@pytest.mark.parametrize("hidden", [64, 128, 192])
def test_short_hidden(oracle, gkv, cuda, hidden):
    """Fewer than three K chunks: the row placement finishes after the loop."""
    import torch
    rng = np.random.default_rng(hidden)
    case = QkvCase(hidden, 8, 2, hidden, lens=rng.integers(1, 100, 70))
    res = run(case, gkv, torch, cuda)
    assert res["err"] == 0
    check_projection(case, res, oracle)
    check_cache(case, res, oracle)


def test_odd_head_count_and_ragged_rows(oracle, gkv, cuda):
    """7 heads (the last column block half used) and 77 rows (a partial row block)."""
    import torch
    rng = np.random.default_rng(12)
    case = QkvCase(13, 5, 1, 320, lens=rng.integers(1, 80, 77))
    res = run(case, gkv, torch, cuda)
    assert res["err"] == 0
    check_projection(case, res, oracle)
    check_cache(case, res, oracle)


def test_many_rows_large_tiles(oracle, gkv, cuda):
    """2,000+ rows take the 128 x 128 tiles: prompt rows with a ragged last
    row block and a ring window."""
    import torch
    case = QkvCase(16, 8, 2, 256, prompts=[700, 513, 900, 1], window=128)
    assert case.M >= 2048
    res = run(case, gkv, torch, cuda)
    assert res["err"] == 0
    check_projection(case, res, oracle)
    check_cache(case, res, oracle)


@pytest.mark.parametrize("v_int8", [False, True])
def test_gpt_oss_shape_large_tiles(oracle, gkv, cuda, v_int8):
    """A prompt batch of the gpt-oss shape (Hq 64, Hkv 8, hidden 2880, N 5120)
    past 2,048 rows: the 128 x 128 tiles with their 40 column blocks spread
    over the XCDs, a ragged last row block, bf16 and int8 V. Every cache byte
    is checked; the projection on 300 sampled rows and every row of the last
    row block."""
    import torch
    case = QkvCase(17 + int(v_int8), 64, 8, 2880, prompts=[800, 640, 512, 130], v_int8=v_int8)
    assert case.M >= 2048 and case.M % 128 != 0
    res = run(case, gkv, torch, cuda)
    assert res["err"] == 0
    rng = np.random.default_rng(3)
    rows = np.unique(np.concatenate([rng.choice(case.M, 300, replace=False),
                                     np.arange(case.M // 128 * 128, case.M)]))
    check_projection(case, res, oracle, rows)
    check_cache(case, res, oracle)


def test_projection_only(oracle, gkv, cuda):
    import torch
    case = QkvCase(14, 64, 8, 2880, lens=np.full(33, 5))
    res = run(case, gkv, torch, cuda, cache=False)
    check_projection(case, res, oracle)
    assert np.array_equal(res["k1"], res["k2"]) and np.array_equal(res["v1"], res["v2"])


def test_bad_block_id_flagged(gkv, cuda):
    """A table entry outside the pool: the row is not stored, the error word
    gets GKV_DEVERR_BLOCK_ID, nothing faults."""
    import torch
    case = QkvCase(15, 8, 2, 128, lens=np.array([20, 40, 3]))
    case.table[1, 2] = case.NB + 100  # row 1 sits at position 39: block 2
    res = run(case, gkv, torch, cuda)
    assert res["err"] & 1
    poison = np.full_like(res["k1"], np.int16(np.uint16(0x7FC1).view(np.int16)))
    assert np.array_equal(res["k1"], res["k2"])
    assert not np.array_equal(res["k1"], poison)


@pytest.mark.parametrize("rows", [1, 17, 32, 33, 96, 97, 192, 193, 512, 513, 768, 769, 1985])
def test_launch_shapes(oracle, gkv, cuda, rows):
    """Rows at the edges of the launch shapes of 5120 columns (16-row tiles up
    to 32 rows, 32-row ones up to 192, 64 x 64 up to 512, 128 x 64 up to 768,
    then 128 x 128 and 256 x 256), the last row block full or ragged; hidden
    576 leaves the 256-wide steps of the few-row shape a partial last one."""
    import torch
    rng = np.random.default_rng(rows)
    case = QkvCase(rows, 64, 8, 576, lens=rng.integers(1, 40, rows), v_int8=rows % 3 == 1,
                   kv_fp8=rows % 3 == 2)
    res = run(case, gkv, torch, cuda)
    assert res["err"] == 0
    check_projection(case, res, oracle, np.unique([0, rows // 2, rows - 1] +
                                                  list(range(rows // 64 * 64, rows))))
    check_cache(case, res, oracle)


@pytest.mark.parametrize("rows, heads", [(384, (64, 8)), (385, (64, 8)), (448, (64, 8)),
                                         (449, (64, 8)), (800, (32, 4)), (927, (32, 4))])
def test_launch_shapes_of_two_tiles_per_cu(oracle, gkv, cuda, rows, heads):
    """Rows around 512 and 576 tiles of 64 x 64 (two per CU, and a third on few of
    them), where the row tiles change from 64 to 128 and back, on 80 and 40
    column blocks."""
    import torch
    rng = np.random.default_rng(rows)
    case = QkvCase(rows, heads[0], heads[1], 128, lens=rng.integers(1, 40, rows))
    res = run(case, gkv, torch, cuda)
    assert res["err"] == 0
    check_projection(case, res, oracle, np.unique([0, rows // 2] +
                                                  list(range(rows // 128 * 128, rows))))
    check_cache(case, res, oracle)


@pytest.mark.parametrize("rows, heads", [(1535, (64, 8)), (1537, (64, 8)), (9087, (32, 4)),
                                         (9089, (32, 4))])
def test_launch_shapes_of_many_rows(oracle, gkv, cuda, rows, heads):
    """Rows around the changes from 128 x 128 to 256 x 256 tiles: past 480 of the small
    ones (the next row block makes 520), and past 1420 against two rounds of the
    large ones; the last row block one row short, and of one row."""
    import torch
    rng = np.random.default_rng(rows)
    case = QkvCase(rows, heads[0], heads[1], 64, prompts=[500] * (rows // 500) + [rows % 500])
    assert case.M == rows
    res = run(case, gkv, torch, cuda)
    assert res["err"] == 0
    check_projection(case, res, oracle, np.unique(list(rng.integers(0, rows, 20)) +
                                                  list(range(rows // 256 * 256, rows, 5))))
    check_cache(case, res, oracle)


@pytest.mark.parametrize("fmt", [0, 1, 2])
def test_prompt_rows_large_tiles(oracle, gkv, cuda, fmt):
    """Prompts whose packed rows start at every offset within a 4-token group
    (values stored four tokens at a time, the others alone) in 256 x 256 tiles."""
    import torch
    rng = np.random.default_rng(5 + fmt)
    prompts = [1, 2, 5] + list(rng.integers(3, 70, 54))
    case = QkvCase(fmt, 64, 8, 320, prompts=prompts, v_int8=fmt == 1, kv_fp8=fmt == 2)
    assert case.M > 1792
    res = run(case, gkv, torch, cuda)
    assert res["err"] == 0
    check_projection(case, res, oracle, [0, 777, case.M - 1])
    check_cache(case, res, oracle)


def test_rows_four_gigabytes_apart(gkv, cuda):
    """A row stride whose byte offsets within a tile pass 32 bits: the same
    rows as with the tight stride."""
    import torch
    g = torch.Generator(device="cuda")
    g.manual_seed(3)
    x = torch.empty(2, 128, dtype=torch.bfloat16, device="cuda").normal_(generator=g)
    w = torch.empty(3 * D, 128, dtype=torch.bfloat16, device="cuda").normal_(generator=g)
    far = torch.empty((1 << 31) + 128, dtype=torch.bfloat16, device="cuda")
    far = far.as_strided((2, 128), (1 << 31, 1))
    far.copy_(x)
    out = [torch.empty(2, 3 * D, device="cuda") for _ in range(2)]
    for xi, o in zip((x, far), out):
        gkv.qkv_append(xi, w, None, 1, None, None, None, qkv_out=o, n_kv_heads=1)
    torch.cuda.synchronize()
    ref = (x.double() @ w.double().t()).cpu().numpy()
    scale = (x.double().abs() @ w.double().abs().t()).cpu().numpy()
    for o in out:
        assert (np.abs(o.cpu().numpy() - ref) <= 2e-5 * scale + 1e-6).all()


@pytest.mark.parametrize("rows", [5, 40, 150, 500, 700, 1000, 1700])
def test_rows_bias_and_tables_at_any_float(gkv, cuda, rows):
    """The fp32 rows, the bias and the angle tables one float off a 16-byte boundary
    and with an odd row stride, in every launch shape of 5120 columns: the same
    rows and cache bytes as aligned ones, and nothing written beside them."""
    import torch
    rng = np.random.default_rng(rows)
    case = QkvCase(rows, 64, 8, 64, lens=rng.integers(1, 40, rows))
    t = lambda a: torch.from_numpy(np.ascontiguousarray(a)).to(cuda)  # noqa: E731
    cos, sin = gkv.rope_table(int(case.lens.max()) + 1)
    x, w = t(case.x).to(torch.bfloat16), t(case.w).to(torch.bfloat16)
    lens, table = t(case.lens), t(case.table)

    def off_by_one(a):
        buf = torch.zeros(a.size + 1, device=cuda)
        buf[1:] = t(a.reshape(-1))
        return buf[1:]

    got = []
    for shifted in (False, True):
        put = off_by_one if shifted else t
        buf = torch.full((rows * (case.N + 3) + 1,), float("nan"), device=cuda)
        out = buf[int(shifted):].as_strided((rows, case.N), (case.N + 3 * shifted, 1))
        k = torch.zeros(case.NB, case.Hkv, 16 * D, dtype=torch.int16, device=cuda)
        v = torch.zeros_like(k)
        gkv.qkv_append(x, w, put(case.bias), case.Hq, put(cos), put(sin),
                       gkv.cache_view(k, v, table, case.Hkv), seq_lens=lens, qkv_out=out)
        torch.cuda.synchronize()
        assert int(torch.isnan(buf).sum()) == buf.numel() - rows * case.N
        got.append([z.cpu().numpy() for z in (out.contiguous(), k, v)])
    for a, b in zip(*got):
        assert np.array_equal(a.view(np.int32 if a.dtype == np.float32 else a.dtype),
                              b.view(np.int32 if b.dtype == np.float32 else b.dtype))
