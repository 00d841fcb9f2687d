"""Rows over the whole vocabulary (top-k off or above 1024): the k_full path.

Every row is compared with the CPU oracle (tests/gpu_helpers.compare_rows):
token, top-k set, kept set and probabilities bit for bit, row flags. The
kept sets are large, so the set outputs are sized to V.
"""
import numpy as np
import pytest

from gpu_helpers import compare_rows, run_gpu

pytestmark = pytest.mark.gpu


def _wl(wl, V, rows, params, seed=3, sigma=2.0, dtype="f32", hist_len=0, mask=None):
    x = wl._rows_normal(seed, rows, V, sigma)
    hist = hl = None
    if hist_len:
        hist = (wl.splitmix64(seed * 7 + 1, rows * hist_len) % np.uint64(V)).astype(np.int32).reshape(rows, hist_len)
        hl = np.full(rows, hist_len, np.int64)
    logits = x if dtype == "f32" else wl.to_bf16_bits(x)
    return wl.Workload("full", dtype, logits, [dict(p) for p in params], wl.uniform53(seed + 9, rows),
                       hist, hl, mask)


def test_config3_spike_and_flat_rows(sampler, wl):
    """BASELINE config 3 at its size, B = 256: 128 rows N(0, 1) with 16 spike
    ids at +15 (exact ties, a nucleus of the 16), 128 near-flat rows N(0, 0.1)
    (a nucleus of about 1e5 ids), top-p 0.9 over the full vocabulary. Every
    row is compared with the oracle: token, kept set and probabilities."""
    w = wl.config(3, seed=5)
    assert w.rows == 256
    g = run_gpu(sampler, w, set_cap=w.vocab)
    assert compare_rows(w, g) == 256


@pytest.mark.parametrize("knobs", [
    dict(temperature=1.0),                                   # identity(): plain draw over V
    dict(temperature=0.8, top_p=0.95),
    dict(temperature=1.3, min_p=0.05),
    dict(temperature=0.7, top_p=0.9, min_p=0.02),
    dict(temperature=0.9, top_k=1500, top_p=0.97),            # k above the top-k path's limit
    dict(temperature=0.9, top_k=3000),
])
def test_full_vocab_knobs(sampler, wl, knobs):
    V, rows = 20011, 6
    p = wl.identity_params(**knobs)
    w = _wl(wl, V, rows, [p] * rows)
    g = run_gpu(sampler, w, set_cap=V)
    assert compare_rows(w, g) == rows


def test_full_vocab_with_penalties_and_bf16(sampler, wl):
    V, rows = 30000, 4
    p = wl.identity_params(temperature=0.8, top_p=0.9, rep_penalty=1.15, repeat_last_n=256,
                           frequency_penalty=0.4, presence_penalty=0.2)
    for dtype in ("f32", "bf16"):
        w = _wl(wl, V, rows, [p] * rows, dtype=dtype, hist_len=300)
        g = run_gpu(sampler, w, set_cap=V)
        assert compare_rows(w, g) == rows


@pytest.mark.parametrize("dtype", ["f32", "bf16"])
@pytest.mark.parametrize("V,hist,knobs", [
    (151936, 600, dict(temperature=0.8, top_p=0.95, min_p=0.05, rep_penalty=1.1, repeat_last_n=600)),
    (2047, 64, dict(temperature=1.1, rep_penalty=0.7, repeat_last_n=40, frequency_penalty=-0.3)),   # raising, one block
    (2049, 1, dict(temperature=0.9, top_p=0.8, presence_penalty=0.5, repeat_last_n=8)),             # one id past a block
    (6145, 2500, dict(temperature=0.7, min_p=0.02, rep_penalty=1.3, repeat_last_n=100, dry_multiplier=0.8,
                      dry_last_n=2500, frequency_penalty=0.2)),                                     # three windows of ids
    (511, 300, dict(temperature=1.0, top_p=0.99, dry_multiplier=0.5, dry_last_n=300, rep_penalty=1.2,
                    repeat_last_n=300)),
])
def test_full_vocab_penalised_rows_over_many_blocks(sampler, wl, V, hist, knobs, dtype):
    """Whole-vocabulary rows with penalties and logit bias, whose transform
    counts the history window by window: ids at the windows' and blocks'
    edges and outside the vocabulary, bans and boosts, a masked row, one row
    of the batch without penalties."""
    rows = 4
    plist = [wl.identity_params(**knobs) for _ in range(rows)]
    plist[2] = wl.identity_params(temperature=0.8, top_p=0.9)
    w = _wl(wl, V, rows, plist, seed=V + hist, sigma=3.0, dtype=dtype, hist_len=hist)
    edges = np.array([0, 511, 512, 2047, 2048, V - 1, V, -1, 0, 511], np.int64)
    k = min(hist, edges.size)
    w.hist[1, -k:] = edges[:k]
    w.hist[3] = np.where(np.arange(hist) % 3 == 0, int(np.argmax(w.logits_f32()[3])), w.hist[3])
    w.mask = np.full((rows, (V + 31) // 32), 0xFFFFFFFF, np.uint32)
    w.mask[1, ::5] = 0x00FF00FF
    bias = [{0: 2.0, V - 1: -np.inf, min(512, V - 2): 5.0}, None, None, {int(np.argmax(w.logits_f32()[3])): -4.0}]
    for wb in ((False, True) if dtype == "f32" else (False,)):
        g = run_gpu(sampler, w, bias=bias, writeback=wb, set_cap=V)
        assert compare_rows(w, g, bias=bias, writeback=wb) == rows


def test_full_vocab_penalised_row_of_many_steps(hs, wl):
    """V above a million: windows of two 512-id steps, counted one at a time."""
    V, rows = (1 << 20) + 700, 2
    p = wl.identity_params(temperature=0.8, top_p=0.9, rep_penalty=1.2, repeat_last_n=500, frequency_penalty=0.3)
    w = _wl(wl, V, rows, [p] * rows, seed=5, sigma=3.0, hist_len=500)
    w.hist[0, :6] = [0, 511, 512, 1023, 1024, V - 1]
    s = hs.Sampler(0, max_rows=rows, max_vocab=V)
    assert compare_rows(w, run_gpu(s, w, set_cap=V)) == rows
    s.close()


@pytest.mark.parametrize("V,dtype,align", [(8, "f32", 4), (15, "bf16", 8), (515, "f32", 4), (2053, "bf16", 8),
                                           (4099, "f32", None), (151936, "bf16", None)])
def test_top_p_rows_read_from_the_logits(sampler, wl, V, dtype, align):
    """Batches whose rows all have a top-p or min-p and no penalties: no
    transformed copy of an aligned row is kept, its values are taken from the
    logits -- at ragged ends, with a mask and NaN logits beside them, ties that
    top-p splits, and the write-back (align None: a misaligned or whole row)."""
    rows = 4
    plist = [wl.identity_params(temperature=t, **k) for t, k in
             [(0.8, dict(top_p=0.9)), (1.3, dict(min_p=0.1)), (1.0, dict(top_p=0.5, min_p=0.01)), (0.7, dict(top_p=0.99))]]
    w = _wl(wl, V, rows, plist, seed=V, sigma=2.0, dtype=dtype)
    x = w.logits_f32().copy()
    x[2] = np.float32(0.5)                     # one value: every cut splits a tie
    w.logits = x if dtype == "f32" else wl.to_bf16_bits(x)
    w.mask = np.full((rows, (V + 31) // 32), 0xFFFFFFFF, np.uint32)
    w.mask[3, ::2] = 0x0FF0F0F1
    for wb in ((False, True) if dtype == "f32" else (False,)):
        g = run_gpu(sampler, w, writeback=wb, set_cap=V, row_align=align)
        assert compare_rows(w, g, writeback=wb) == rows


@pytest.mark.parametrize("rows,dtype", [(252, "f32"), (253, "f32"), (253, "bf16")])
def test_whole_row_passes_on_either_side_of_16384_windows(sampler, wl, rows, dtype):
    """65 windows a row: up to 252 rows the first pass takes the batch's windows
    in turn, from 253 rows on each row's in blocks of its own (the last block
    one window)."""
    V = 33000
    knobs = [dict(), dict(top_p=0.9), dict(min_p=0.02)]
    plist = [wl.identity_params(temperature=0.9, **knobs[r % 3]) for r in range(rows)]
    w = _wl(wl, V, rows, plist, seed=rows, dtype=dtype)
    g = run_gpu(sampler, w, set_cap=V)
    assert compare_rows(w, g, rows=[0, 1, 2, 62, 63, 64, 130, rows - 3, rows - 2, rows - 1]) == 10


def test_full_vocab_mixed_with_topk_and_greedy_rows(sampler, wl):
    V, rows = 12000, 6
    plist = [wl.identity_params(temperature=1.0, top_p=0.9),
             wl.identity_params(temperature=0.7, top_k=40),
             wl.identity_params(temperature=0.0),
             wl.identity_params(temperature=1.2),
             wl.identity_params(temperature=0.9, top_k=2048, min_p=0.01),
             wl.identity_params(temperature=0.6, top_k=8, top_p=0.8)]
    w = _wl(wl, V, rows, plist, seed=8)
    g = run_gpu(sampler, w, set_cap=V)
    assert compare_rows(w, g) == rows


@pytest.mark.parametrize("pen", [True, False])
def test_full_vocab_writeback(sampler, wl, pen):
    V, rows = 9000, 3
    if pen:
        p = wl.identity_params(temperature=0.75, top_p=0.8, rep_penalty=1.2, repeat_last_n=64)
    else:   # a plain transform: the many-block passes ahead of k_full
        p = wl.identity_params(temperature=0.75, top_p=0.8)
    w = _wl(wl, V, rows, [p] * rows, hist_len=64)
    g = run_gpu(sampler, w, writeback=True, set_cap=V)
    assert compare_rows(w, g, writeback=True) == rows


def test_full_vocab_all_masked_row_draws_uniformly(sampler, wl):
    V, rows = 4096, 2
    mask = np.zeros((rows, V // 32), np.uint32)
    mask[1, 5] = 1 << 3          # row 1: one allowed id
    p = wl.identity_params(temperature=1.0, top_p=0.9)
    w = _wl(wl, V, rows, [p] * rows, mask=mask)
    g = run_gpu(sampler, w, set_cap=V)
    assert compare_rows(w, g) == rows
    assert int(g["row_flags"][0]) & 16          # nothing finite: uniform over V


@pytest.mark.parametrize("rows,dtype", [(1, "f32"), (3, "f32"), (2, "bf16")])
def test_cli_identity_rows_at_full_vocab(hs, sampler, wl, rows, dtype):
    """The CLI's call (SamplerParams::identity() + temperature,
    apps/ultima-cli/main.cpp:661-674) at V = 151936: its whole-row passes run
    over many blocks (k_fs_*) ahead of k_full; in the bf16 case with a masked
    row."""
    import torch
    V = 151936
    p = wl.identity_params(temperature=0.8)
    mask = None
    if dtype == "bf16":
        mask = np.full((rows, V // 32), 0xFFFFFFFF, np.uint32)
        mask[1, ::3] = 0x0F0F0F0F
    w = _wl(wl, V, rows, [p] * rows, seed=31 + rows, dtype=dtype, mask=mask)
    from gpu_helpers import to_device
    x, u, h, m = to_device(w)
    k = sampler.query_kernels(x, w.params, u, mask=m)
    assert k & hs.KERNELS_FULL
    g = run_gpu(sampler, w, set_cap=V)
    assert compare_rows(w, g) == rows


def test_cli_row_with_nan_logits_is_flagged(hs, sampler, wl):
    """NaN logits in a whole-vocabulary row count as -inf and flag the row
    (the reference's softmax would turn every probability into NaN): the
    token is one of the finite ids, drawn as if the NaN ids were masked."""
    V = 151936
    p = wl.identity_params(temperature=0.8)
    w = _wl(wl, V, 1, [p], seed=41)
    w.logits[0, 5::1000] = np.nan
    g = run_gpu(sampler, w, set_cap=V)
    assert int(g["row_flags"][0]) & hs.ROW_NAN
    assert not np.isnan(w.logits[0, int(g["token"][0])])
    masked = w.logits.copy()
    masked[0, 5::1000] = -np.inf
    wm = _wl(wl, V, 1, [p], seed=41)
    wm.logits[:] = masked
    gm = run_gpu(sampler, wm, set_cap=V)
    assert int(g["token"][0]) == int(gm["token"][0])
    assert int(g["kept_count"][0]) == int(gm["kept_count"][0]) == V - 152


@pytest.mark.parametrize("V", [32000, 151936, 262144])
def test_plain_transform_rows_exact_sums(hs, sampler, wl, V):
    """Rows that take the whole-row passes over many blocks (plain transform:
    temperature and mask only) with sums that leave their binade in different
    places: flat rows (the sum doubles window after window), wide rows (a few
    ids carry it), a constant row (the sum lands on powers of two exactly at
    window ends), rows with long masked-out ranges (empty windows) and a row
    of one allowed id per 4096. The kept probabilities are e * fl(1/S) for
    every id, so they pin the exact index-order sum S bit for bit."""
    rows = 6
    sig = [0.3, 2.0, 8.0, 0.0, 1.0, 3.0]
    x = wl._rows_normal(77, rows, V, sig)
    x[3] = 0.5                                  # constant row
    temps = [1.0, 0.8, 1.7, 1.0, 0.6, 1.1]
    params = [wl.identity_params(temperature=t) for t in temps]
    mask = np.full((rows, (V + 31) // 32), 0xFFFFFFFF, np.uint32)
    lo, hi = V // 10 // 32, V // 2 // 32
    mask[4, lo:hi] = 0                          # a long masked-out range
    mask[5, :] = 0
    mask[5, ::128] = 1                          # one id per 4096
    w = wl.Workload("full", "f32", x, params, wl.uniform53(78, rows), None, None, mask)
    g = run_gpu(sampler, w, set_cap=V)
    assert compare_rows(w, g) == rows


@pytest.mark.parametrize("sigma,top_p,temp", [(3.0, 1.0, 0.8), (3.0, 0.95, 0.8), (0.5, 1.0, 1.0), (0.5, 0.9, 1.0),
                                               (1.5, 0.999, 1.0), (6.0, 0.6, 1.0)])
def test_min_p_at_a_numerators_edge(sampler, wl, sigma, top_p, temp):
    """min_p set to one id's exp(x - max), a float above and a float below
    (the ids the numerators alone do not decide), to 1 and above, to values
    that remove nothing or all but a few ids, alone and after top-p, with
    kept sets of one wave's list and of many thousands; two ids share the
    largest logit. Rows with and without penalties."""
    V = 20011
    row = wl._rows_normal(int(sigma * 10), 1, V, sigma)[0]
    row[7] = row[19000] = np.float32(row.max() + 0.25)
    x = (row * np.float32(1.0 / np.float32(temp))) if temp != 1.0 else row
    e = np.exp((x - x.max()).astype(np.float32).astype(np.float64)).astype(np.float32)
    order = np.sort(e)[::-1]
    edges = []
    for k in (3, 300, 3000):
        v = order[k]
        edges += [v, np.nextafter(v, np.float32(2)), np.nextafter(v, np.float32(0))]
    edges += [np.float32(1), np.float32(1.0000001), np.float32(2), np.float32(1e-25), np.float32(1e-12), np.float32(0.05)]
    for pen in (False, True):
        kw = dict(rep_penalty=1.3, repeat_last_n=32) if pen else {}
        plist = [wl.identity_params(temperature=temp, top_p=top_p, min_p=float(v), **kw) for v in edges]
        w = _wl(wl, V, len(edges), plist, seed=3, hist_len=32 if pen else 0)
        w.logits[:] = row
        g = run_gpu(sampler, w, writeback=pen, set_cap=V)
        assert compare_rows(w, g, writeback=pen) == len(edges)


@pytest.mark.parametrize("sigma,top_p,temp", [(3.0, 1.0, 0.8), (0.5, 0.9, 1.0), (1.5, 0.999, 1.0)])
def test_min_p_at_a_numerators_edge_of_aligned_rows(sampler, wl, sigma, top_p, temp):
    """min_p at one id's exp(x - max) and a float to either side, in aligned
    rows (no transformed copy): with no top-p the threshold times fl(1/S)
    decides, after it the numerators, or the sum of what it left."""
    V = 20012
    row = wl._rows_normal(int(sigma * 10), 1, V, sigma)[0]
    x = row * np.float32(1.0 / np.float32(temp))
    e = np.sort(np.exp((x - x.max()).astype(np.float32).astype(np.float64)).astype(np.float32))[::-1]
    edges = [np.float32(v) for k in (3, 700, 4000) for v in (e[k], np.nextafter(e[k], np.float32(2)), np.nextafter(e[k], np.float32(0)))]
    edges += [np.float32(v) for v in (1.0, 1.0000001, 2.0, 1e-25, 1e-45, 0.05)]
    plist = [wl.identity_params(temperature=temp, top_p=top_p, min_p=float(v)) for v in edges]
    w = _wl(wl, V, len(edges), plist, seed=3)
    w.logits[:] = row
    for wb in (False, True):
        g = run_gpu(sampler, w, writeback=wb, set_cap=V)
        assert compare_rows(w, g, writeback=wb) == len(edges)


def _as(wl, w, dtype):
    if dtype == "bf16":
        w.logits, w.dtype = wl.to_bf16_bits(w.logits), dtype
    return w


def _without_sets(sampler, w, g, align=None):
    """Token, row flags and kept count of the run that asks for no sets."""
    import torch
    from gpu_helpers import to_device
    x, u, h, m = to_device(w)
    if align:
        xp = torch.zeros((w.rows, (w.vocab + align - 1) // align * align), dtype=x.dtype, device=x.device)
        xp[:, :w.vocab] = x
        x = xp[:, :w.vocab]
    out = {"kept_count": torch.empty(w.rows, dtype=torch.int32, device=x.device)}
    o = sampler.run(x, w.params, u, hist=h, hist_len=w.hist_len, mask=m, outputs=out)
    torch.cuda.synchronize()
    for k in ("token", "row_flags", "kept_count"):
        np.testing.assert_array_equal(o[k].cpu().numpy(), g[k], err_msg=k)


@pytest.mark.parametrize("V,dtype,align", [(2053, "f32", 4), (30000, "f32", None), (30001, "bf16", 8), (30001, "f32", None)])
def test_rows_from_which_no_id_leaves(sampler, wl, V, dtype, align):
    """min-p and top-p that remove nothing, from rows whose numerators are all
    above 0, underflow to 0 though their logits are finite, or are masked out;
    kept sets of thousands by top-p and by min-p beside them; the write-back."""
    # (knobs, sigma of the logits)
    rows = [(dict(min_p=1e-12), 1.0), (dict(min_p=1e-45), 60.0), (dict(min_p=1e-45, top_p=0.9999999), 60.0),
            (dict(top_p=0.9999999), 1.0), (dict(top_p=0.9), 0.3), (dict(min_p=0.3), 0.2),
            (dict(top_p=0.95, min_p=0.3), 0.2), (dict(min_p=1e-12), 1.0)]
    plist = [wl.identity_params(temperature=0.9, **k) for k, _ in rows]
    w = _wl(wl, V, len(rows), plist, seed=V, sigma=[s for _, s in rows])
    w.logits[1:3, 100:103] = 400.0        # fl(1/S) below a half: the threshold rounds to 0
    w = _as(wl, w, dtype)
    w.mask = np.full((len(rows), (V + 31) // 32), 0xFFFFFFFF, np.uint32)
    w.mask[7, ::3] = 0x0FF0F0F1
    g = run_gpu(sampler, w, set_cap=V, row_align=align)
    assert compare_rows(w, g) == len(rows)
    assert int(g["kept_count"][0]) == int(g["kept_count"][1]) == V and int(g["kept_count"][7]) < V
    assert 512 < min(int(g["kept_count"][r]) for r in (4, 5, 6))
    _without_sets(sampler, w, g, align)
    if dtype == "f32":
        g = run_gpu(sampler, w, writeback=True, set_cap=V, row_align=align)
        assert compare_rows(w, g, writeback=True) == len(rows)


@pytest.mark.parametrize("V,dtype,align", [(30001, "f32", 4), (30001, "bf16", 8), (30001, "f32", None)])
def test_nan_logits_in_top_p_and_min_p_rows(hs, sampler, wl, V, dtype, align):
    """NaN logits count as -inf and flag the row, also where the transformed
    row is not kept: the outputs are those of the row with the NaN ids masked
    out (checked against the oracle), but for the flag."""
    knobs = [(dict(top_p=0.9), 2.0), (dict(top_p=0.9), 0.2), (dict(min_p=0.05), 2.0), (dict(min_p=0.3), 0.2),
             (dict(min_p=1e-12), 1.0), (dict(top_p=0.9, min_p=1e-45), 60.0), (dict(min_p=1e-45), 60.0)]
    n = len(knobs)
    w = _wl(wl, V, n, [wl.identity_params(temperature=0.8, **k) for k, _ in knobs], seed=9, sigma=[s for _, s in knobs])
    w.logits[5:, 100:110] = 400.0
    w = _as(wl, w, dtype)
    at = [0, 5, 512, 2047, V - 1] + [int(i) for r in range(n) for i in np.argsort(w.logits_f32()[r])[-3:]]
    w.mask = np.full((n, (V + 31) // 32), 0xFFFFFFFF, np.uint32)
    for i in at:
        w.mask[:, i // 32] &= np.uint32(0xFFFFFFFF) ^ np.uint32(1 << (i % 32))
    want = run_gpu(sampler, w, set_cap=V, row_align=align)
    assert compare_rows(w, want) == n
    w.mask = None
    x = w.logits_f32().copy()
    x[:, at] = np.nan
    w.logits = x if dtype == "f32" else wl.to_bf16_bits(np.where(np.isnan(x), np.float32(0), x))
    if dtype == "bf16":
        w.logits[:, at] = 0x7FC0
    got = run_gpu(sampler, w, set_cap=V, row_align=align)
    for r in range(n):
        c = int(want["kept_count"][r])
        assert int(got["token"][r]) == int(want["token"][r]) and int(got["kept_count"][r]) == c, r
        np.testing.assert_array_equal(got["kept_idx"][r][:c], want["kept_idx"][r][:c])
        np.testing.assert_array_equal(got["kept_prob"][r][:c].view(np.uint32), want["kept_prob"][r][:c].view(np.uint32))
        assert int(got["row_flags"][r]) == int(want["row_flags"][r]) | hs.ROW_NAN, r
    _without_sets(sampler, w, got, align)


def test_full_vocab_draw_without_sets(sampler, wl):
    """With no kept set asked for, rows whose top-p or min-p removed ids take
    the draw's window sums from the numerators alone and their kept count from
    the stages' own counts: token, row flags and kept count must equal those of
    the run that writes the sets (checked against the oracle). Rows: cfg3's
    spike rows (the cut splits ids of equal p at the top) and flat rows, top-p
    and min-p knobs, and min_p 2 (every id removed: the uniform draw)."""
    import torch
    V = 151936
    w3 = wl.config(3, seed=11, rows=4)
    knobs = [dict(temperature=0.8, top_p=0.5), dict(temperature=1.2, min_p=0.05),
             dict(temperature=0.7, top_p=0.95, min_p=0.02), dict(temperature=1.5, min_p=2.0)]
    wk = _wl(wl, V, len(knobs), [wl.identity_params(**k) for k in knobs], seed=19)
    for w in (w3, wk):
        g = run_gpu(sampler, w, set_cap=V)
        assert compare_rows(w, g) == w.rows
        from gpu_helpers import to_device
        x, u, h, m = to_device(w)
        out = {"kept_count": torch.empty(w.rows, dtype=torch.int32, device=x.device)}
        o = sampler.run(x, w.params, u, hist=h, hist_len=w.hist_len, mask=m, outputs=out)
        torch.cuda.synchronize()
        for k in ("token", "row_flags", "kept_count"):
            assert np.array_equal(o[k].cpu().numpy(), g[k]), (w.name, k)
