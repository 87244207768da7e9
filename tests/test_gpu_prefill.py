"""GPU parity of chunked-prefill attention (MFMA) against the oracle's
flash_attn_f32 restatement driven per query row (causal: keys 0..position).
bf16 tolerance |got - ref| <= 1e-2 + 2e-3 |ref|; softmax accumulates in fp32.
The chunk's own K/V are appended through the cache's append kernel first,
exactly as a caller of the chunked-prefill path does."""
import numpy as np
import pytest

import oracle as orc
from kvutil import assert_close, from_dev, kv_values, random_tables, slots_for, to_dev, widen

pytestmark = pytest.mark.gpu

RTOL, ATOL = 2e-3, 1e-2


def _setup(dt, hq, hkv, ctx, q_lens, seed, nb=None, bs=16, D=128, k_gain=None, mb=None):
    """Paged cache holding every position of every sequence (cached prefix
    and chunk), the chunk's queries, and the tables.  k_gain(pos) scales the
    K row at position pos (then rounded to the cache dtype)."""
    import torch
    from infer_train_amd.kv import PagedKvCache

    ctx = np.asarray(ctx, np.int32)
    q_lens = np.asarray(q_lens, np.int32)
    mb = max(int((ctx.max() + bs - 1) // bs), mb or 0)
    need = int(sum((int(c) + bs - 1) // bs for c in ctx))
    nb = nb or need + 3
    tables = random_tables(seed, ctx, bs, nb, mb)
    seqs, pos = [], []
    for b, c in enumerate(ctx):
        seqs += [b] * int(c)
        pos += list(range(int(c)))
    slots = slots_for(tables, seqs, pos, bs)
    n = len(slots)
    k = kv_values(seed + 1, n * hkv * D, dt).reshape(n, hkv, D)
    if k_gain is not None:
        g = np.array([k_gain(p) for p in pos], np.float32)[:, None, None]
        kf = widen(k, dt) * g
        k = orc.f32_to_bf16(kf) if dt == orc.BF16 else orc.f32_to_f16(kf)
    v = kv_values(seed + 2, n * hkv * D, dt).reshape(n, hkv, D)
    ref = orc.Cache(nb, bs, hkv, D, dt)
    ref.append(k, v, slots)
    dev = PagedKvCache(nb, bs, hkv, D, dt)
    td = torch.bfloat16 if dt == orc.BF16 else torch.float16
    dev.append(to_dev(k.view(np.int16), td), to_dev(v.view(np.int16), td), to_dev(slots))
    cu = np.concatenate([[0], np.cumsum(q_lens)]).astype(np.int32)
    q = kv_values(seed + 3, int(cu[-1]) * hq * D, dt).reshape(int(cu[-1]), hq, D)
    return dev, ref, tables, ctx, cu, q, td


def _run(dev, tables, ctx, cu, q, td, hq, causal=True, out_f32=True, scale=None):
    import torch

    D = q.shape[2]
    if scale is None:
        scale = float(np.float32(1.0) / np.sqrt(np.float32(D)))
    dq = to_dev(q.view(np.int16), td)
    max_q = int(np.max(np.diff(cu)))
    out = dev.prefill(dq, to_dev(cu), max_q, to_dev(tables), to_dev(ctx), scale=scale, causal=causal,
                      out_dtype=torch.float32 if out_f32 else td)
    dev.check()
    return out, scale


@pytest.mark.parametrize("dt", [orc.BF16, orc.F16])
@pytest.mark.parametrize("hq,hkv", [(8, 2), (4, 4), (6, 3), (16, 2), (6, 2), (5, 1), (7, 1)])
def test_prefill_small_causal(dt, hq, hkv):
    """Ragged chunks: partial 32-row query blocks and 64-key blocks, chunk
    lengths 1 and whole-context, GQA groups 4, 1, 2, 8, 3, 5, 7 (workgroups
    of 8, 8, 8, 8, 6, 5, 7 waves)."""
    ctx = [100, 37, 64, 1, 200]
    q_lens = [45, 37, 1, 1, 70]
    dev, ref, tables, ctx, cu, q, td = _setup(dt, hq, hkv, ctx, q_lens, seed=11 + hq)
    out, scale = _run(dev, tables, ctx, cu, q, td, hq)
    want = ref.prefill(widen(q, dt), hq, cu, tables, ctx, scale, causal=True)
    assert_close(from_dev(out), want, RTOL, ATOL, what=f"prefill dt={dt} hq={hq} hkv={hkv}")


def test_prefill_longest_first_order_with_tail_workgroups():
    """Workgroup ids are dealt to XCDs as 8 ranges; an XCD holding whole
    (sequence, KV head) pairs takes its query blocks longest first.  Here 9
    sequences x 2 KV heads x 2 query blocks of 64 rows = 36 workgroups:
    ranges of 4 (2 pairs each, so the remap is not the identity), and 4 tail
    workgroups past the last full set of 8 keep their ids.  Every row of
    every sequence against the oracle."""
    ctx = [128 + 16 * i for i in range(9)]
    q_lens = [128] * 9
    dev, ref, tables, ctx, cu, q, td = _setup(orc.BF16, 8, 2, ctx, q_lens, seed=71)
    out, scale = _run(dev, tables, ctx, cu, q, td, 8)
    want = ref.prefill(widen(q, orc.BF16), 8, cu, tables, ctx, scale, causal=True)
    assert_close(from_dev(out), want, RTOL, ATOL, what="prefill, 36 workgroups")


def test_prefill_non_causal_and_bf16_out():
    hq, hkv = 8, 2
    dev, ref, tables, ctx, cu, q, td = _setup(orc.BF16, hq, hkv, [130, 77], [33, 77], seed=5)
    out, scale = _run(dev, tables, ctx, cu, q, td, hq, causal=False, out_f32=False)
    want = ref.prefill(widen(q, orc.BF16), hq, cu, tables, ctx, scale, causal=False)
    assert_close(widen(from_dev(out), orc.BF16), want, RTOL, ATOL, what="prefill non-causal bf16 out")


@pytest.mark.parametrize("scale", [-0.0883883, 0.0, 0.25])
def test_prefill_scale_values(scale):
    """A negative scale (the max is taken over scaled scores), a zero scale
    (uniform weights over the visible keys) and a large one."""
    hq, hkv = 8, 2
    dev, ref, tables, ctx, cu, q, td = _setup(orc.BF16, hq, hkv, [150, 70], [90, 70], seed=21)
    out, scale = _run(dev, tables, ctx, cu, q, td, hq, scale=scale)
    want = ref.prefill(widen(q, orc.BF16), hq, cu, tables, ctx, scale, causal=True)
    assert_close(from_dev(out), want, RTOL, ATOL, what=f"prefill scale={scale}")


@pytest.mark.parametrize("dt", [orc.BF16, orc.F16])
def test_prefill_rising_scores(dt):
    """K rows grow with position, so each 64-key block raises the running
    max by several times the lazy-rescale threshold (2^8) and the
    accumulators are rescaled mid-context; also a falling ramp (the max is
    set by the first block and never rescaled)."""
    hq, hkv = 8, 2
    for gain in (lambda p: 1.0 + p / 24.0, lambda p: 8.0 / (1.0 + p / 24.0)):
        dev, ref, tables, ctx, cu, q, td = _setup(dt, hq, hkv, [600, 333], [200, 333], seed=31, k_gain=gain)
        out, scale = _run(dev, tables, ctx, cu, q, td, hq)
        want = ref.prefill(widen(q, dt), hq, cu, tables, ctx, scale, causal=True)
        assert_close(from_dev(out), want, RTOL, ATOL, what=f"prefill rising/falling dt={dt}")


@pytest.mark.parametrize("bs", [8, 32, 64])
def test_prefill_block_sizes(bs):
    """Pages of 8, 32 and 64 tokens: a 64-key block spans 8, 2 or 1 pages
    (each 4-row load stays inside one page)."""
    hq, hkv = 8, 2
    ctx, q_lens = [333, 200], [150, 200]
    dev, ref, tables, ctx, cu, q, td = _setup(orc.BF16, hq, hkv, ctx, q_lens, seed=71 + bs, bs=bs)
    out, scale = _run(dev, tables, ctx, cu, q, td, hq)
    want = ref.prefill(widen(q, orc.BF16), hq, cu, tables, ctx, scale, causal=True)
    assert_close(from_dev(out), want, RTOL, ATOL, what=f"prefill bs={bs}")


def test_prefill_wide_table_scalar_page_ids():
    """A block table wider than fits beside the K/V rings in LDS (13,000
    entries per row): page ids come from scalar loads of the table instead
    of the workgroup's LDS copy."""
    hq, hkv = 8, 2
    ctx, q_lens = [400, 150], [130, 150]
    dev, ref, tables, ctx, cu, q, td = _setup(orc.BF16, hq, hkv, ctx, q_lens, seed=81, mb=13000)
    assert tables.shape[1] == 13000
    out, scale = _run(dev, tables, ctx, cu, q, td, hq)
    want = ref.prefill(widen(q, orc.BF16), hq, cu, tables, ctx, scale, causal=True)
    assert_close(from_dev(out), want, RTOL, ATOL, what="prefill wide table")


def test_prefill_config3_rows():
    """Config 3: Hq 32, Hkv 8, D 128, bs 16; 8 sequences with 2048 cached
    tokens append a 512-token chunk; table = a permutation of a 4096-block
    pool.  Against the oracle (on the host's threads): every row of every
    sequence (4096 rows x 32 heads).  Every row: finite, and each output
    element inside the range of the V rows it attends (keys 0 .. its
    position of its KV head), as a convex combination must be."""
    import os

    hq, hkv, D = 32, 8, 128
    ctx = [2560] * 8
    q_lens = [512] * 8
    dev, ref, tables, ctx, cu, q, td = _setup(orc.BF16, hq, hkv, ctx, q_lens, seed=3, nb=4096)
    out, scale = _run(dev, tables, ctx, cu, q, td, hq)
    got = from_dev(out)
    assert np.isfinite(got).all()
    qf = widen(q, orc.BF16)
    threads = max(1, min(16, len(os.sched_getaffinity(0))))
    for s in range(8):
        want = ref.prefill(qf, hq, cu, tables, ctx, scale, causal=True, rows=(s, 0, 512), threads=threads)
        rows = slice(int(cu[s]), int(cu[s]) + 512)
        assert_close(got[rows], want[rows], RTOL, ATOL, what=f"config3 seq {s}, all 512 rows")
    # Convex hull: running min / max of V over positions, per KV head and dim.
    n = ctx.astype(np.int64)
    cu_tok = np.concatenate([[0], np.cumsum(n)[:-1]]).astype(np.int64)
    _, gv = ref.gather(tables, ctx, None, cu_tok, int(n.sum()))
    vrows = widen(gv.view(np.uint16), orc.BF16).reshape(-1, D)
    G = hq // hkv
    for s in range(8):
        V = vrows[int(cu_tok[s]) * hkv:(int(cu_tok[s]) + int(n[s])) * hkv].reshape(hkv, int(n[s]), D)
        hi = np.maximum.accumulate(V, axis=1)
        lo = np.minimum.accumulate(V, axis=1)
        pos = int(ctx[s]) - 512 + np.arange(512)
        o = got[int(cu[s]):int(cu[s + 1])].reshape(512, hkv, G, D)
        up = hi[:, pos, :].transpose(1, 0, 2)[:, :, None, :]
        dn = lo[:, pos, :].transpose(1, 0, 2)[:, :, None, :]
        assert np.all(o <= up + 1e-4) and np.all(o >= dn - 1e-4), f"config3 seq {s}: outside the V hull"


@pytest.mark.parametrize("n_seqs,hq,hkv,causal", [(2, 7, 1, True), (24, 8, 1, True), (25, 8, 1, True), (63, 8, 1, True),
                                                  (64, 4, 2, False), (65, 8, 1, True)])
def test_prefill_unit_order_ragged(n_seqs, hq, hkv, causal):
    """Workgroups find their unit in the longest-first order over up to 64
    sequences (searched one way up to 24, another way past them; more than 64
    take ids in pair order): batches at those edges, with empty chunks, chunk
    lengths of one row, whole prompts and long cached prefixes.  Every row against the oracle, so every unit is
    computed, and by nobody else (a unit missed leaves its rows unwritten)."""
    rng = np.random.RandomState(n_seqs)
    q_lens = rng.choice([0, 1, 31, 32, 33, 65, 100], n_seqs)
    q_lens[0] = 97
    ctx = q_lens + rng.choice([0, 1, 63, 64, 200], n_seqs)
    ctx[0] += 300
    dev, ref, tables, ctx, cu, q, td = _setup(orc.BF16, hq, hkv, ctx, q_lens, seed=500 + n_seqs)
    out, scale = _run(dev, tables, ctx, cu, q, td, hq, causal=causal)
    want = ref.prefill(widen(q, orc.BF16), hq, cu, tables, ctx, scale, causal=causal)
    assert_close(from_dev(out), want, RTOL, ATOL, what=f"prefill order n_seqs={n_seqs}")


@pytest.mark.parametrize("n_seqs,hq,hkv,equal,causal", [
    (16, 32, 4, False, True),   # 256 workgroups: one per CU, ids in pair order
    (22, 24, 3, False, True),   # 264: searched 64 block counts at a time
    (24, 24, 3, False, False), (25, 24, 3, False, True), (64, 14, 2, False, True),
    (24, 24, 3, True, True),    # equal sequences: pairs dealt to the XCDs in runs
    (25, 24, 3, True, True),    # 75 pairs: one by one
])
def test_prefill_unit_order_past_one_round(n_seqs, hq, hkv, equal, causal):
    """Grids of more than 256 workgroups take the longest-first order, smaller
    ones do not: both sides of the line and of the order's own branches.  Every
    row against the oracle."""
    rng = np.random.RandomState(700 + n_seqs)
    q_lens = np.full(n_seqs, 97) if equal else rng.choice([0, 1, 31, 32, 33, 65, 100], n_seqs)
    q_lens[0] = 97
    ctx = q_lens + (63 if equal else rng.choice([0, 1, 63, 64, 200], n_seqs))
    assert (4 * n_seqs * hkv > 256) == (n_seqs != 16)  # four query blocks of 32 rows (hq / hkv of 7 or 8)
    dev, ref, tables, ctx, cu, q, td = _setup(orc.BF16, hq, hkv, ctx, q_lens, seed=700 + n_seqs)
    out, scale = _run(dev, tables, ctx, cu, q, td, hq, causal=causal)
    want = ref.prefill(widen(q, orc.BF16), hq, cu, tables, ctx, scale, causal=causal)
    assert_close(from_dev(out), want, RTOL, ATOL, what=f"prefill order n_seqs={n_seqs} equal={equal}")


def _expected_cuts(hq, hkv, ctx, q_lens, causal, tiles):
    """The number of cuts the device prices from a call's lengths (blocks of 64
    keys, a cut costs five, at least eight a cut, 256 workgroups at once)."""
    group = hq // hkv
    rows = 32 * (1 if group >= 8 else 8 // group)
    blocks = lambda keys: max((keys + 63) // 64, 0)  # noqa: E731
    units = work = most = 0
    for c, q in zip(ctx, q_lens):
        n = -(-q // rows)
        if n == 0:
            continue
        first, last = (blocks(c - q + (min(q, x) if causal else q)) for x in (rows, n * rows))
        units += n * hkv
        work += n * (first + last) // 2
        most = max(most, last)
    if most < 16 or units == 0 or 2 * units > tiles:
        return 1
    mean, best = hkv * work * 16 // units, None
    for cuts in range(1, 17):
        if cuts > 1 and (units * cuts > tiles or most < 8 * cuts):
            break
        extra = 80 if cuts > 1 else 0
        cost = max(-(-units * cuts // 256) * (mean // cuts + extra), 16 * most // cuts + extra)
        cost -= cost // 10 if cuts == 1 else 0
        if best is None or cost < best[0]:
            best = cost, cuts
    return best[1]


@pytest.mark.parametrize("dt,hq,hkv,ctx,q_lens,causal,mb,cuts", [
    (orc.BF16, 8, 2, [2100], [70], True, 260, 4),          # one long context, few rows: 33 key blocks
    (orc.F16, 7, 1, [4096, 130], [33, 1], True, 260, 8),   # 7 waves; a unit too short to cut beside long ones
    (orc.BF16, 5, 1, [2049, 0, 3000], [1, 0, 129], True, 260, 5),  # 5 waves, an empty sequence, the diagonal inside the last cut
    (orc.BF16, 2, 2, [2111], [300], False, 260, 4),        # 8 query tiles a workgroup, every key visible
    (orc.BF16, 8, 1, [1100, 1023], [64, 64], True, 260, 2),  # at the edge: 18 and 16 key blocks
    (orc.BF16, 8, 2, [2100, 1500], [70, 40], True, 13000, 4),  # a table too wide for LDS: block ids by scalar loads
    (orc.F16, 6, 2, [5000], [33], False, 7200, 9),
])
def test_prefill_units_cut_over_keys(dt, hq, hkv, ctx, q_lens, causal, mb, cuts):
    """Launches of few units divide each unit's key blocks among several
    workgroups and merge their partial (m, l, O).  Against the oracle, and
    against the same call without a workspace (no cuts): the two differ by
    the rounding of the 16-bit probabilities to different maxima.  The number of
    cuts the device took is the one priced here."""
    import torch
    from infer_train_amd import lib

    gain = lambda p: 1.0 + (p % 700) / 300.0  # noqa: E731  cuts with different maxima
    raw_ctx, raw_q = list(ctx), list(q_lens)
    dev, ref, tables, ctx, cu, q, td = _setup(dt, hq, hkv, ctx, q_lens, seed=900 + hq, mb=mb, k_gain=gain)
    need = lib.it_paged_prefill_workspace(hq, hkv, len(ctx), int(max(q_lens)), mb, 16)
    waves = hq // hkv * (1 if hq // hkv >= 8 else 8 // (hq // hkv))
    assert _expected_cuts(hq, hkv, raw_ctx, raw_q, causal, (need - 256) // (waves * 64 * 264)) == cuts
    out, scale = _run(dev, tables, ctx, cu, q, td, hq, causal=causal)
    want = ref.prefill(widen(q, dt), hq, cu, tables, ctx, scale, causal=causal)
    got = from_dev(out)
    assert_close(got, want, RTOL, ATOL, what=f"prefill cut dt={dt} hq={hq}")
    dq, plain = to_dev(q.view(np.int16), td), torch.empty(q.shape, dtype=torch.float32, device="cuda")
    dcu, dt_, dctx = to_dev(cu), to_dev(tables), to_dev(ctx)
    assert lib.it_paged_prefill(dev.handle, dq.data_ptr(), dev.dtype, hq, dcu.data_ptr(), int(max(q_lens)), dt_.data_ptr(),
                                mb, dctx.data_ptr(), len(ctx), scale, int(causal), plain.data_ptr(), 0,
                                torch.cuda.current_stream().cuda_stream) == 0
    assert_close(got, from_dev(plain), RTOL, ATOL, what="cut against uncut")
    ws, own = torch.empty(need, dtype=torch.uint8, device="cuda"), torch.empty_like(plain)
    assert lib.it_paged_prefill_ws(dev.handle, dq.data_ptr(), dev.dtype, hq, dcu.data_ptr(), int(max(q_lens)), dt_.data_ptr(),
                                   mb, dctx.data_ptr(), len(ctx), scale, int(causal), ws.data_ptr(), need, own.data_ptr(), 0,
                                   torch.cuda.current_stream().cuda_stream) == 0
    np.testing.assert_array_equal(from_dev(own), got)
    assert int(ws[:4].view(torch.int32).item()) == cuts  # the main kernel leaves the number there for the merge


@pytest.mark.parametrize("dt,n_seqs,hq,hkv,equal,mb,causal", [
    (orc.BF16, 5, 16, 2, False, 260, True),    # few workgroups: the order without a search
    (orc.F16, 5, 7, 1, True, 260, True),       # equal sequences
    (orc.BF16, 22, 24, 3, False, 260, True),   # 264 workgroups: searched
    (orc.BF16, 24, 24, 3, True, 260, True),
    (orc.BF16, 3, 10, 2, False, 13000, False),  # block ids by scalar loads
])
def test_prefill_short_contexts_in_wide_tables(dt, n_seqs, hq, hkv, equal, mb, causal):
    """Tables wide enough that contexts may be long, over contexts that are
    short: the call takes a workspace and cuts nothing.  With a bound on the
    contexts it takes none.  Both give the oracle's rows and the same bits, and
    the bounded call allocates its output alone."""
    import torch
    from infer_train_amd import lib

    rng = np.random.RandomState(40 + n_seqs)
    q_lens = np.full(n_seqs, 97) if equal else rng.choice([0, 1, 31, 33, 65, 100], n_seqs)
    q_lens[0] = 97
    ctx = q_lens + (63 if equal else rng.choice([0, 1, 63, 64, 200], n_seqs))
    dev, ref, tables, ctx, cu, q, td = _setup(dt, hq, hkv, ctx, q_lens, seed=40 + n_seqs, mb=mb)
    assert lib.it_paged_prefill_workspace(hq, hkv, n_seqs, 97 if equal else int(max(q_lens)), mb, 16) > 0
    out, scale = _run(dev, tables, ctx, cu, q, td, hq, causal=causal)
    want = ref.prefill(widen(q, dt), hq, cu, tables, ctx, scale, causal=causal)
    assert_close(from_dev(out), want, RTOL, ATOL, what=f"wide table n_seqs={n_seqs}")
    args = to_dev(q.view(np.int16), td), to_dev(cu), int(max(q_lens)), to_dev(tables), to_dev(ctx)
    torch.cuda.synchronize()
    before = torch.cuda.memory_allocated()
    torch.cuda.reset_peak_memory_stats()
    bounded = dev.prefill(*args, scale=scale, causal=causal, out_dtype=torch.float32, max_ctx_len=int(ctx.max()))
    assert torch.cuda.max_memory_allocated() - before <= bounded.numel() * 4 + 512
    np.testing.assert_array_equal(from_dev(bounded), from_dev(out))


def test_prefill_bound_of_long_contexts_changes_nothing():
    """A bound that leaves room for cuts: the call is the one without it."""
    import torch

    dev, ref, tables, ctx, cu, q, td = _setup(orc.BF16, 16, 2, [2100], [1100], seed=61, mb=260)
    out, scale = _run(dev, tables, ctx, cu, q, td, 16)  # 70 units of 8 waves, 3 cuts: more merges than the combine has workgroups
    want = ref.prefill(widen(q, orc.BF16), 16, cu, tables, ctx, scale, causal=True, threads=8)
    assert_close(from_dev(out), want, RTOL, ATOL, what="cut prefill of 70 units")
    again = dev.prefill(to_dev(q.view(np.int16), td), to_dev(cu), 1100, to_dev(tables), to_dev(ctx), scale=scale,
                        out_dtype=torch.float32, max_ctx_len=np.int64(2100))
    np.testing.assert_array_equal(from_dev(again), from_dev(out))


def test_prefill_without_memory_for_its_workspace():
    """A device too full for the workspace: the call runs without one, with
    the bits of a call that never asked for it."""
    import torch
    from infer_train_amd import lib

    dev, ref, tables, ctx, cu, q, td = _setup(orc.BF16, 16, 2, [2100], [1100], seed=62, mb=260)
    need = lib.it_paged_prefill_workspace(16, 2, 1, 1100, 260, 16)
    assert need > 32 << 20
    scale = 0.0884
    dq, dcu, dtab, dctx = to_dev(q.view(np.int16), td), to_dev(cu), to_dev(tables), to_dev(ctx)
    out, plain = (torch.empty(q.shape, dtype=torch.float32, device="cuda") for _ in range(2))
    assert lib.it_paged_prefill(dev.handle, dq.data_ptr(), dev.dtype, 16, dcu.data_ptr(), 1100, dtab.data_ptr(), 260,
                                dctx.data_ptr(), 1, scale, 1, plain.data_ptr(), 0,
                                torch.cuda.current_stream().cuda_stream) == 0
    torch.cuda.synchronize()
    torch.cuda.empty_cache()
    total = torch.cuda.get_device_properties(0).total_memory
    torch.cuda.set_per_process_memory_fraction(torch.cuda.memory_reserved() / total)
    try:
        with pytest.raises(torch.OutOfMemoryError):
            torch.empty(need, dtype=torch.uint8, device="cuda")
        dev.prefill(dq, dcu, 1100, dtab, dctx, scale=scale, out=out)
    finally:
        torch.cuda.set_per_process_memory_fraction(1.0)
    np.testing.assert_array_equal(from_dev(out), from_dev(plain))
