"""MFMA prefill (ragged causal over the paged cache) and HiDream DiT
attention on the GPU against the CPU oracle."""
import numpy as np
import pytest
import torch

import omni_attn as oa
import workloads as W
from gpu_util import assert_close, dev_bits, dev_i32, host_bits
from refs import bits_to_f64

pytestmark = pytest.mark.gpu


def run_prefill(c, exact_p=False):
    pf = oa.prefill_plan(c.rows, c.hq, c.hk, c.page, c.seq, c.pos, exact_p=exact_p)
    out = torch.zeros(c.rows, c.hq * 128, dtype=torch.bfloat16, device="cuda")
    oa.prefill_run(pf, dev_bits(c.qkv), dev_bits(c.kv), dev_i32(c.pos), dev_i32(c.seq), dev_i32(c.indptr),
                   dev_i32(c.pages), out, c.scale)
    torch.cuda.synchronize()
    return host_bits(out)


def oracle_paged(oracle, c, threads=16):
    return oracle.paged_attend(c.qkv, c.kv, c.pos, c.seq, c.ragged, c.indptr, c.pages, c.page, c.hq, c.hk, c.scale,
                               nthreads=threads)


@pytest.mark.parametrize("hq,hk", [(32, 8), (16, 16), (16, 8), (64, 8)])
def test_prefill_parity(oracle, hq, hk):
    c = W.ragged_prefill_case(3, hq, hk, 1, 300, 0, 200, seed=hq + hk)
    assert_close(run_prefill(c), oracle_paged(oracle, c), what=f"prefill {hq}/{hk}")


@pytest.mark.parametrize("page", [3, 12, 24, 48, 80])
def test_prefill_any_page(oracle, page):
    """Pages that are not powers of two: 48 and 80 (multiples of a wave's 16
    tile rows) take the one-page-id-per-wave loader with a multiply-high
    division, 3, 12 and 24 the per-key loader."""
    c = W.ragged_prefill_case(3, 32, 8, 1, 300, 0, 200, page=page, seed=page, slack_pages=3)
    assert_close(run_prefill(c), oracle_paged(oracle, c), what=f"prefill page {page}")


def test_prefill_single_rows_and_odd_lengths(oracle):
    c = W.ragged_prefill_case(6, 32, 8, 1, 3, 0, 70, seed=3)
    assert_close(run_prefill(c), oracle_paged(oracle, c), what="short")


def test_prefill_matches_decode_kernel(oracle):
    """The same rows through the split-K decode kernel: two kernels, one answer."""
    c = W.ragged_prefill_case(4, 32, 8, 50, 200, 0, 300, seed=4)
    a = run_prefill(c)
    plan = oa.decode_plan(c.rows, 32, 8, 16, int(c.pos.max()) + 1, 128)
    out = torch.zeros(c.rows, 32 * 128, dtype=torch.bfloat16, device="cuda")
    oa.qwen3_attend(dev_bits(c.qkv), dev_bits(c.kv), dev_i32(c.pos), dev_i32(c.seq), 1, dev_i32(c.indptr),
                    dev_i32(c.pages), 16, out, 32, 8, c.scale, plan, oa.workspace_for(plan))
    torch.cuda.synchronize()
    assert_close(a, host_bits(out), what="prefill vs decode")


def test_prefill_config4_subset(oracle):
    """Config 4's construction (new U[512,4096], cached U[0,1024]) on 2 requests."""
    c = W.ragged_prefill_case(2, 32, 8, 512, 4096, 0, 1024, seed=4000)
    assert_close(run_prefill(c), oracle_paged(oracle, c), what="config4 subset")


def test_prefill_config4_own_draw(oracle):
    """Config 4's own seeded draw (B = 8, seed 4000: 25,499 rows, up to 4,563
    keys), the workload bench.py times, so its work-list order (longest tiles
    first, XCD ranges, the 8 sequences' items) is the one checked: every row
    against the oracle (about 895 GFLOP, 10-20 s on 16 host threads), and
    every row against the split-K decode kernel (the reference's f32 P)."""
    c = W.config_case(4)
    assert c.rows == 25499 and len(c.extra["new"]) == 8
    got = run_prefill(c)
    want = oracle_paged(oracle, c)
    mx, mn = assert_close(got, want, what=f"config4 all {c.rows} rows vs oracle")
    print(f"config4 vs oracle: max-abs {mx:.3g} mean-abs {mn:.3g}")
    plan = oa.decode_plan(c.rows, c.hq, c.hk, c.page, int(c.pos.max()) + 1)
    out = torch.zeros(c.rows, c.hq * 128, dtype=torch.bfloat16, device="cuda")
    oa.qwen3_attend(dev_bits(c.qkv), dev_bits(c.kv), dev_i32(c.pos), dev_i32(c.seq), 1, dev_i32(c.indptr),
                    dev_i32(c.pages), c.page, out, c.hq, c.hk, c.scale, plan, oa.workspace_for(plan))
    torch.cuda.synchronize()
    assert_close(got, host_bits(out), what="config4 prefill vs decode, every row")
    # The plan's exact_p (P as bf16 hi + lo, the reference's f32-P numerics):
    # every row against the oracle and, nearly bit for bit, the decode kernel.
    ex = run_prefill(c, exact_p=True)
    mx, mn = assert_close(ex, want, what=f"config4 exact_p all {c.rows} rows vs oracle")
    print(f"config4 exact_p vs oracle: max-abs {mx:.3g} mean-abs {mn:.3g}")
    same = float(np.mean(ex == host_bits(out)))
    assert same >= 0.99, f"exact_p prefill and the f32-P decode kernel agree on {same:.4f} of elements"


def run_dense(c, b_all=True):
    q, k, v = dev_bits(c.q), dev_bits(c.k), dev_bits(c.v)
    out = torch.zeros(c.batch, c.q_len, c.hq * 128, dtype=torch.bfloat16, device="cuda")
    kvl = dev_i32(np.array([c.kv_len], np.int32))
    if c.batch == 1:
        oa.hidream_attend(q, k, v, out, c.q_len, kvl, c.q_stride, c.causal, c.scale_log2, c.hq, c.hk)
    else:
        oa.hidream_attend_batched(q, k, v, out, c.q_len, kvl, c.q_stride, c.causal, c.scale_log2, c.hq, c.hk, c.batch,
                                  c.q_len * c.q_stride, c.kv_len * c.hk * 128, c.q_len * c.hq * 128)
    torch.cuda.synchronize()
    return host_bits(out)


def oracle_dense(oracle, c, b=0, kv_len=None):
    return oracle.dense_attend(np.ascontiguousarray(c.q[b]), np.ascontiguousarray(c.k[b]),
                               np.ascontiguousarray(c.v[b]), c.q_len, kv_len or c.kv_len, c.q_stride, c.hq, c.hk,
                               c.causal, c.scale_log2, nthreads=16)


def dit_path(hq, hk, q_len, batch=1, ws=False):
    """How a DiT call runs its 256-row tiles (a mirror of the library's rule):
    whole; all as row quarters; those past whole rounds as row halves, or, with a
    workspace, as (count of) key chunks."""
    cus = torch.cuda.get_device_properties(0).multi_processor_count
    items = -(-q_len // (256 * hk // hq)) * hk * batch
    rem = items % cus
    if ws and 0 < rem <= cus // 2:
        chunks = min(cus // rem, max(2, -(-q_len // 128) // 4))
        if items >= cus or chunks >= (4 if items * 4 <= cus else 3):
            return f"{chunks} chunks"
    return "quarters" if items * 4 <= cus else "halves" if 0 < rem <= cus // 2 else "whole"


# On 256 CUs. (16, 8, 65) and (4, 4, 1) have quarters with few and no rows, (8, 8,
# 2049) and (32, 4, 520) last tiles of a few rows.
@pytest.mark.parametrize("hq,hk,q_len,kv_len,causal,path", [
    (32, 8, 300, 300, 1, "quarters"), (32, 8, 257, 333, 0, "quarters"), (8, 8, 100, 130, 0, "quarters"),
    (4, 4, 1, 1, 0, "quarters"), (16, 8, 65, 64, 1, "quarters"), (32, 4, 40, 500, 0, "quarters"),
    (8, 8, 2049, 400, 1, "halves"), (16, 8, 1100, 300, 0, "halves"), (32, 8, 600, 520, 1, "halves"),
    (32, 4, 520, 200, 0, "halves"), (32, 8, 1100, 300, 1, "whole"), (16, 16, 2200, 150, 0, "whole"),
])
def test_dit_parity(oracle, hq, hk, q_len, kv_len, causal, path):
    assert dit_path(hq, hk, q_len) == path
    c = W.dense_case(hq, hk, q_len, kv_len, causal, seed=q_len)
    assert_close(run_dense(c)[0], oracle_dense(oracle, c), what=f"dit {hq}/{hk} {q_len}x{kv_len} c{causal}")


def test_dit_kv_len_read_from_device(oracle):
    c = W.dense_case(32, 8, 200, 400, 0, seed=7)
    q, k, v = dev_bits(c.q), dev_bits(c.k), dev_bits(c.v)
    out = torch.zeros(c.q_len, c.hq * 128, dtype=torch.bfloat16, device="cuda")
    kvl = dev_i32(np.array([259], np.int32))
    oa.hidream_attend(q, k, v, out, c.q_len, kvl, c.q_stride, 0, c.scale_log2, c.hq, c.hk)
    torch.cuda.synchronize()
    assert_close(host_bits(out), oracle_dense(oracle, c, kv_len=259), what="kv_len 259")


def test_dit_batched_pair(oracle):
    c = W.dense_case(32, 8, 130, 130, 0, batch=2, seed=8)
    got = run_dense(c)
    for b in range(2):
        assert_close(got[b], oracle_dense(oracle, c, b), what=f"batch {b}")


def test_dit_config5_subset(oracle):
    """Config 5's shape (4352 keys, 32q/8kv, RMS-normed q/k) on the first 256 queries."""
    c = W.dense_case(32, 8, 4352, 4352, 0, seed=5000)
    got = run_dense(c)[0]
    sub = W.DenseCase(hq=32, hk=8, q_len=256, kv_len=4352, causal=0, q_stride=c.q_stride, q=c.q, k=c.k, v=c.v)
    want = oracle_dense(oracle, sub)
    assert_close(got[:256], want, what="config5 first 256 rows")


def run_dense_ws(c, kv_len=None):
    q, k, v = dev_bits(c.q), dev_bits(c.k), dev_bits(c.v)
    out = torch.zeros(c.batch, c.q_len, c.hq * 128, dtype=torch.bfloat16, device="cuda")
    kvl = dev_i32(np.array([kv_len or c.kv_len], np.int32))
    ws = oa.hidream_workspace()
    ws.fill_(0xFF)  # stale partials must not matter
    oa.hidream_attend_ws(q, k, v, out, c.q_len, kvl, c.q_stride, c.causal, c.scale_log2, c.hq, c.hk, c.batch,
                         c.q_len * c.q_stride, c.kv_len * c.hk * 128, c.q_len * c.hq * 128, ws)
    torch.cuda.synchronize()
    return host_bits(out)


@pytest.mark.parametrize("hq,hk,q_len,kv_len,causal,batch", [
    (8, 2, 256, 256, 0, 1), (32, 8, 300, 700, 1, 2), (32, 8, 1000, 1000, 0, 1), (4, 4, 1, 1, 0, 1),
])
def test_dit_small_calls_with_a_workspace(oracle, hq, hk, q_len, kv_len, causal, batch):
    """Calls of less than a round (8, 80, 128 and 4 tiles) that could be split in
    fewer than four chunks: the workspace stays unused."""
    assert dit_path(hq, hk, q_len, batch, ws=True) == dit_path(hq, hk, q_len, batch)
    c = W.dense_case(hq, hk, q_len, kv_len, causal, batch=batch, seed=q_len + kv_len)
    got = run_dense_ws(c)
    for b in range(batch):
        assert_close(got[b], oracle_dense(oracle, c, b), what=f"ws dit {hq}/{hk} {q_len}x{kv_len} c{causal} b{b}")


# Every G, with more chunks than key tiles in some (chunks without a key).
SPLITS = [
    (8, 8, 8200, 300, 1, 16),    # 264 tiles, the last 8 split; 3 key tiles
    (16, 8, 4100, 700, 1, 8),    # 264; 6 key tiles
    (32, 8, 2049, 130, 1, 4),    # 264; 2 key tiles, the last query tile one position
    (32, 8, 1100, 1500, 2, 2),   # 288
    (32, 4, 2060, 520, 1, 4),    # 260; 5 key tiles
    (32, 32, 257, 300, 5, 2),    # 320
    (8, 1, 1921, 1000, 1, 4),    # 61 tiles, all split
    (8, 8, 2049, 600, 1, 3),     # 72, all split
]


@pytest.mark.parametrize("causal", [0, 1])
@pytest.mark.parametrize("hq,hk,q_len,kv_len,batch,chunks", SPLITS)
def test_dit_tail_split_parity(oracle, hq, hk, q_len, kv_len, batch, chunks, causal):
    """Tiles past whole rounds as key chunks with a workspace and as row halves
    (61 tiles: quarters) without one: every row of the first and last problem
    against the oracle in both forms."""
    assert dit_path(hq, hk, q_len, batch, ws=True) == f"{chunks} chunks" and splits_by_keys(hq, hk, q_len, batch)
    assert dit_path(hq, hk, q_len, batch) == ("quarters" if hk == 1 else "halves")
    c = W.dense_case(hq, hk, q_len, kv_len, causal, batch=batch, seed=q_len + kv_len)
    split, rows = run_dense_ws(c), run_dense(c)
    for b in {0, batch - 1}:
        want = oracle_dense(oracle, c, b)
        assert_close(split[b], want, what=f"chunks {hq}/{hk} {q_len}x{kv_len} c{causal} b{b}")
        assert_close(rows[b], want, what=f"row parts {hq}/{hk} {q_len}x{kv_len} c{causal} b{b}")


@pytest.mark.parametrize("hk,seed", [(8, 5000), (32, 5032)])
def test_dit_config5_full_size(oracle, hk, seed):
    """Config 5 at its full size, the CFG pair of 4352 queries and keys, 32
    q heads over hk = 8 (the reference's shape) and hk = 32 (the MHA variant
    bench.py also times). On a 256-CU GPU its 1088 items run as 1024 whole
    and 64 split into 4 key chunks with a workspace (the kernels bench.py
    times), and as row halves without one. Every row of both batch halves
    meets the oracle in both forms (2 x 310 GFLOP, about 10 s on 16 host
    threads), and the two forms agree on every row."""
    c = W.dense_case(32, hk, 4352, 4352, 0, batch=2, seed=seed)
    got, ref = run_dense_ws(c), run_dense(c)
    for b in range(2):
        want = oracle_dense(oracle, c, b)
        mx, mn = assert_close(got[b], want, what=f"config5 hk {hk} batch {b} (workspace) vs oracle")
        print(f"config5 hk {hk} batch {b} vs oracle: max-abs {mx:.3g} mean-abs {mn:.3g}")
        assert_close(ref[b], want, what=f"config5 hk {hk} batch {b} (no workspace) vs oracle")
        assert_close(got[b], ref[b], what=f"config5 hk {hk} batch {b}: workspace vs row halves")


@pytest.mark.parametrize("causal", [0, 1])
def test_dit_row_halves_match_split(oracle, causal):
    """544 items: on a 256-CU GPU the last 32 (kv head 7, queries 2304..)
    run as row halves without a workspace and as 8 key chunks with one. Both
    agree with each other everywhere and with the oracle on the last 128
    queries (whole tiles for heads 0..27, halves for 28..31)."""
    c = W.dense_case(32, 8, 4352, 1024, causal, seed=31 + causal)
    got, split = run_dense(c)[0], run_dense_ws(c)[0]
    assert_close(got, split, what="halves vs split")
    # Queries 4224.. see all 1024 keys, causal or not.
    want = oracle.dense_attend(np.ascontiguousarray(c.q[0, -128:]), np.ascontiguousarray(c.k[0]),
                               np.ascontiguousarray(c.v[0]), 128, 1024, c.q_stride, 32, 8, 0, c.scale_log2,
                               nthreads=16)
    assert_close(got[-128:], want, what=f"halves tail vs oracle c{causal}")


@pytest.mark.parametrize("causal", [0, 1])
@pytest.mark.parametrize("q_len,paths", [
    (65, ("quarters", "quarters", "quarters")), (300, ("quarters", "halves", "halves")),
    (1100, ("whole", "halves", "2 chunks")), (2049, ("halves", "halves", "4 chunks")),
])
def test_dit_no_key_gives_nan(oracle, causal, q_len, paths):
    """*kv_len_at = 0 (hidream.cu:337-346: l = 0, so O * (1 / l) = NaN): every
    output element is NaN through the plain call, the batched call and the
    workspace call (key chunks, all empty), each running its tiles as `paths`
    says, as the oracle gives; a second call with keys overwrites them with
    finite values."""
    assert (dit_path(32, 8, q_len), dit_path(32, 8, q_len, 2), dit_path(32, 8, q_len, 2, ws=True)) == paths
    c = W.dense_case(32, 8, q_len, 300, causal, batch=2, seed=41 + causal)
    want = oracle.dense_attend(np.ascontiguousarray(c.q[0]), np.ascontiguousarray(c.k[0]), np.ascontiguousarray(c.v[0]),
                               c.q_len, 0, c.q_stride, c.hq, c.hk, causal, c.scale_log2, nthreads=16)
    assert np.isnan(bits_to_f64(want)).all()
    q, k, v = dev_bits(c.q), dev_bits(c.k), dev_bits(c.v)
    zero = dev_i32(np.array([0], np.int32))
    bs = (c.q_len * c.q_stride, c.kv_len * c.hk * 128, c.q_len * c.hq * 128)
    outs = [torch.zeros(c.batch, c.q_len, c.hq * 128, dtype=torch.bfloat16, device="cuda") for _ in range(3)]
    oa.hidream_attend(q, k, v, outs[0], c.q_len, zero, c.q_stride, causal, c.scale_log2, c.hq, c.hk)
    oa.hidream_attend_batched(q, k, v, outs[1], c.q_len, zero, c.q_stride, causal, c.scale_log2, c.hq, c.hk, 2, *bs)
    oa.hidream_attend_ws(q, k, v, outs[2], c.q_len, zero, c.q_stride, causal, c.scale_log2, c.hq, c.hk, 2, *bs,
                         oa.hidream_workspace())
    torch.cuda.synchronize()
    assert np.isnan(bits_to_f64(host_bits(outs[0][0]))).all(), "plain call"
    assert np.isnan(bits_to_f64(host_bits(outs[1]))).all(), "batched call"
    assert np.isnan(bits_to_f64(host_bits(outs[2]))).all(), "workspace call"
    # The same buffers with keys again: finite and equal to the oracle.
    oa.hidream_attend_ws(q, k, v, outs[2], c.q_len, dev_i32(np.array([c.kv_len], np.int32)), c.q_stride, causal,
                         c.scale_log2, c.hq, c.hk, 2, *bs, oa.hidream_workspace())
    torch.cuda.synchronize()
    assert_close(host_bits(outs[2])[1], oracle_dense(oracle, c, 1), what="keys again")


def test_dit_empty_query_launch_is_a_no_op():
    """q_len = 0 (and batch = 0) returns OK and writes nothing."""
    c = W.dense_case(32, 8, 4, 4, 0, seed=43)
    q, k, v = dev_bits(c.q), dev_bits(c.k), dev_bits(c.v)
    out = torch.full((4, c.hq * 128), 3.0, dtype=torch.bfloat16, device="cuda")
    kvl = dev_i32(np.array([4], np.int32))
    oa.hidream_attend(q, k, v, out, 0, kvl, c.q_stride, 0, c.scale_log2, c.hq, c.hk)
    oa.hidream_attend_ws(q, k, v, out, 0, kvl, c.q_stride, 0, c.scale_log2, c.hq, c.hk, 1, 0, 0, 0,
                         oa.hidream_workspace())
    oa.hidream_attend_batched(q, k, v, out, 4, kvl, c.q_stride, 0, c.scale_log2, c.hq, c.hk, 0, 0, 0, 0)
    torch.cuda.synchronize()
    assert bool((out == 3.0).all())


@pytest.mark.parametrize("page", [1, 2, 4, 8, 64])
def test_prefill_page_sizes(oracle, page):
    """The paged tile loader at pages below a wave's 16 rows of a tile (one
    page id per key row) and from 16 up (one scalar page id per wave and tile)."""
    c = W.ragged_prefill_case(3, 32, 8, 40, 260, 0, 150, page=page, seed=page)
    assert_close(run_prefill(c), oracle_paged(oracle, c), what=f"prefill page {page}")


BF16_NAN = 0x7FC0


def test_prefill_reads_no_slot_past_its_keys(oracle):
    """Every cache slot no row may see holds NaN, including the rest of each
    sequence's last page: the tail tile must not read them into P.V."""
    c = W.ragged_prefill_case(4, 32, 8, 30, 300, 0, 150, seed=21)
    seen = np.zeros(c.kv.shape[0], bool)
    for s in range(len(c.indptr) - 1):
        rows = c.seq == s
        if not rows.any():
            continue
        keys = np.arange(int(c.pos[rows].max()) + 1)
        pg = c.pages[c.indptr[s]:c.indptr[s + 1]]
        seen[pg[keys // c.page] * c.page + keys % c.page] = True
    assert (~seen).any() and any((int(c.pos[c.seq == s].max()) + 1) % 64 for s in np.unique(c.seq))
    c.kv = c.kv.copy()
    c.kv[~seen] = BF16_NAN
    assert_close(run_prefill(c), oracle_paged(oracle, c), what="prefill with NaN past the keys")


@pytest.mark.parametrize("causal", [0, 1])
def test_dit_reads_no_key_past_kv_len(oracle, causal):
    """K and V rows past *kv_len_at hold NaN; the partial last key tile must
    not read them into P.V."""
    c = W.dense_case(32, 8, 200, 400, causal, seed=22)
    c.k, c.v = c.k.copy(), c.v.copy()
    c.k[:, 259:] = BF16_NAN
    c.v[:, 259:] = BF16_NAN
    q, k, v = dev_bits(c.q), dev_bits(c.k), dev_bits(c.v)
    out = torch.zeros(c.q_len, c.hq * 128, dtype=torch.bfloat16, device="cuda")
    kvl = dev_i32(np.array([259], np.int32))
    oa.hidream_attend(q, k, v, out, c.q_len, kvl, c.q_stride, causal, c.scale_log2, c.hq, c.hk)
    torch.cuda.synchronize()
    assert_close(host_bits(out), oracle_dense(oracle, c, kv_len=259), what=f"kv_len 259 with NaN past it, c{causal}")


@pytest.mark.parametrize("layout", ["gaps", "interleaved"])
def test_prefill_runs_split_at_gaps_and_interleaving(oracle, layout):
    """Rows whose positions jump inside a sequence, or whose sequences
    alternate row by row: the plan cuts them into separate runs (single rows
    when interleaved), and each row still sees keys 0..pos of its sequence."""
    base = W.ragged_prefill_case(3, 32, 8, 150, 300, 20, 200, seed=77)
    rng = np.random.default_rng(78)
    if layout == "gaps":
        keep = np.sort(rng.choice(base.rows, size=base.rows * 2 // 3, replace=False))  # drop a third of the rows
    else:
        per_seq = [np.flatnonzero(base.seq == s) for s in range(3)]
        n = min(len(x) for x in per_seq)
        keep = np.stack([x[:n] for x in per_seq], axis=1).reshape(-1)  # seq 0, 1, 2, 0, 1, 2, ...
    c = W.PagedCase(hq=32, hk=8, page=base.page, pos=base.pos[keep], seq=base.seq[keep], ragged=1,
                    indptr=base.indptr, pages=base.pages, num_pages=base.num_pages, qkv=base.qkv[keep], kv=base.kv)
    pf = oa.prefill_plan(c.rows, 32, 8, c.page, c.seq, c.pos)
    assert pf.plan.tiles > (c.rows + 63) // 64  # really cut into more, shorter runs
    assert_close(run_prefill(c), oracle_paged(oracle, c), what=f"prefill {layout}")


def test_prefill_long_sequence(oracle):
    """One sequence of 6000 new rows over 3000 cached keys: 94 tiles per kv
    head. The oracle checks the first and last 96 rows (rows are independent)."""
    c = W.ragged_prefill_case(1, 32, 8, 6000, 6000, 3000, 3000, seed=79)
    got = run_prefill(c)
    pick = np.r_[0:96, c.rows - 96:c.rows]
    sub = W.PagedCase(hq=32, hk=8, page=c.page, pos=c.pos[pick], seq=c.seq[pick], ragged=1, indptr=c.indptr,
                      pages=c.pages, num_pages=c.num_pages, qkv=c.qkv[pick], kv=c.kv)
    assert_close(got[pick], oracle_paged(oracle, sub), what="long prefill, first and last rows")


@pytest.mark.parametrize("exact_p", [False, True])
@pytest.mark.parametrize("rows,cached,hq,hk", [
    # with 256 CUs: 64 (tile, kv head) items or fewer run as four workgroups per
    # tile, 128 or fewer as two, more as one
    (16, 0, 32, 8), (17, 200, 32, 8), (513, 5, 32, 8),  # four: a quarter tile, one row more, 72 items -> two
    (512, 31, 16, 8), (1024, 0, 16, 8), (2048, 127, 16, 8), (2049, 0, 16, 8),  # 32, 64 (four), 128 (two), 136 items
    (40, 8500, 16, 8), (200, 8300, 64, 8), (700, 8200, 32, 8),  # more than 64 key tiles: page ids reloaded
])
def test_prefill_workgroups_per_tile(oracle, rows, cached, hq, hk, exact_p):
    """One request either side of each choice of workgroups per tile, with
    rows that end inside a quarter or half of a tile; unread slots hold NaN.
    The oracle checks up to 64 rows spread over the request."""
    c = W.ragged_prefill_case(1, hq, hk, rows, rows, cached, cached, seed=rows + cached, slack_pages=3)
    kv = c.kv.reshape(c.num_pages, 16, -1)
    used = np.zeros((c.num_pages, 16), bool)
    t = np.arange(rows + cached)
    used[c.pages[t // 16], t % 16] = True
    kv[~used] = 0x7FC0
    got = run_prefill(c, exact_p=exact_p)
    pick = np.unique(np.r_[0, rows - 1, np.linspace(0, rows - 1, 62).astype(int)])
    sub = W.PagedCase(hq=hq, hk=hk, page=c.page, pos=c.pos[pick], seq=c.seq[pick], ragged=1, indptr=c.indptr,
                      pages=c.pages, num_pages=c.num_pages, qkv=c.qkv[pick], kv=c.kv)
    assert_close(got[pick], oracle_paged(oracle, sub), what=f"{rows} rows over {cached}")


@pytest.mark.parametrize("causal", [0, 1])
@pytest.mark.parametrize("q_len,kv_len,batch,path", [
    (16, 40, 1, "quarters"), (512, 700, 1, "quarters"), (513, 600, 1, "halves"), (1024, 1000, 1, "halves"),
    (1025, 1102, 1, "whole"), (520, 520, 2, "whole"), (1100, 1024, 2, "halves"),
])
def test_dit_workgroups_per_tile(oracle, q_len, kv_len, batch, path, causal):
    """DiT calls either side of each choice (64 and 72 tiles, 128 and 136, 144, 288
    = a round and 32) against the oracle on every row of the last problem."""
    assert dit_path(32, 8, q_len, batch) == path
    c = W.dense_case(32, 8, q_len, kv_len, causal, batch=batch, seed=q_len + kv_len)
    assert_close(run_dense(c)[-1], oracle_dense(oracle, c, batch - 1), what=f"{q_len}x{kv_len} c{causal}")


@pytest.mark.parametrize("new", [100, 300, 900])  # 32, 80 and 240 items: quarters, halves, whole tiles
@pytest.mark.parametrize("page", [16, 12])
def test_prefill_item_ranges_follow_the_lists_header(new, page):
    """The work list's header bounds the items that run: ranges moved between
    XCDs run the same items, and an item left out of them stays unwritten."""
    c = W.ragged_prefill_case(2, 32, 8, new, new, 0, 100, page=page, seed=new)
    pf = oa.prefill_plan(c.rows, 32, 8, page, c.seq, c.pos)
    head, items = pf.work[:9].cpu().numpy(), pf.plan.tiles * 8
    assert head[0] == 0 and head[8] == items and pf.plan.workgroups == items  # ranges of items / 8 each

    def run(header):
        out = torch.zeros(c.rows, 32 * 128, dtype=torch.bfloat16, device="cuda")
        work = pf.work.clone()
        work[:9] = dev_i32(header)
        oa.prefill_run(oa.Prefill(pf.plan, work), dev_bits(c.qkv), dev_bits(c.kv), dev_i32(c.pos), dev_i32(c.seq),
                       dev_i32(c.indptr), dev_i32(c.pages), out, c.scale)
        torch.cuda.synchronize()
        return host_bits(out)

    whole = run(head)
    body = pf.work[16:].view(-1, 4).cpu().numpy()
    cut = head.copy()
    cut[8] -= 1  # the last item is in no range
    got, (_, first, n, h) = run(cut), body[items - 1]
    left = np.zeros((c.rows, 32, 128), bool)
    left[first:first + n, 4 * h:4 * h + 4] = True
    left = left.reshape(c.rows, -1)
    assert np.array_equal(got[~left], whole[~left]) and not got[left].any() and whole[left].any()
    moved = head.copy()
    moved[1:8] -= 1  # range 0 loses its last item, 1..6 begin one earlier, 7's last item is left out
    moved[8] -= 1
    assert np.array_equal(run(moved), got)


@pytest.mark.parametrize("exact_p", [False, True])
@pytest.mark.parametrize("hq,hk,rows,cached", [(16, 8, 187, 0), (32, 8, 150, 700), (16, 16, 40, 300), (64, 8, 33, 1000)])
def test_prefill_row_bits_do_not_depend_on_the_call(hq, hk, rows, cached, exact_p):
    """A request's rows alone (few tiles: row halves), beside others that still
    leave CUs idle, and in a call of more tiles than CUs (whole tiles): the same
    bits every time, since each row is computed the same way in all of them."""
    per = 256 * hk // hq
    c = W.ragged_prefill_case(2, hq, hk, rows, rows, cached, cached, seed=rows)
    alone, both = np.flatnonzero(c.seq == 0), np.arange(c.rows)
    # Sequence 1's rows pushed again and again: `many` more tiles per head.
    many = 256 // hk + 1
    tiled = np.r_[alone, np.tile(np.flatnonzero(c.seq == 1), many)]
    bits = []
    for keep in (alone, both, tiled):
        sub = W.PagedCase(hq=hq, hk=hk, page=c.page, pos=c.pos[keep], seq=c.seq[keep], ragged=1, indptr=c.indptr,
                          pages=c.pages, num_pages=c.num_pages, qkv=c.qkv[keep], kv=c.kv)
        pf = oa.prefill_plan(sub.rows, hq, hk, sub.page, sub.seq, sub.pos)
        assert (pf.plan.tiles * hk > 256) == (keep is tiled) and pf.plan.tiles >= -(-rows // per)
        bits.append(run_prefill(sub, exact_p=exact_p)[:rows])
    assert np.array_equal(bits[0], bits[1]), f"{np.sum(bits[0] != bits[1])} elements differ beside another request"
    assert np.array_equal(bits[0], bits[2]), f"{np.sum(bits[0] != bits[2])} elements differ in a large call"


def splits_by_keys(hq, hk, q_len, batch=1):
    """Whether hidream_attend_ws splits this shape by keys: a call with a
    workspace of 16 bytes is refused exactly then."""
    st = (hq + 2 * hk) * 128
    q = torch.zeros(batch, q_len, st, dtype=torch.bfloat16, device="cuda")
    k = torch.zeros(batch, 8, hk * 128, dtype=torch.bfloat16, device="cuda")
    out = torch.zeros(batch, q_len, hq * 128, dtype=torch.bfloat16, device="cuda")
    try:
        oa.hidream_attend_ws(q, k, k, out, q_len, dev_i32(np.array([8], np.int32)), st, 0, 0.1, hq, hk, batch,
                             q_len * st, 8 * hk * 128, q_len * hq * 128,
                             torch.zeros(16, dtype=torch.uint8, device="cuda"))
    except oa.OmniAttnError as e:
        assert e.code == oa.EWORKSPACE
        return True
    finally:
        torch.cuda.synchronize()
    return False


@pytest.mark.parametrize("hq,hk,q_len,batch,split", [
    # below one round (256 CUs): by rows, unless at least four chunks of four key tiles fit, three past 64 tiles
    (32, 8, 65, 1, False), (32, 8, 1000, 1, False), (8, 1, 1920, 1, False), (8, 1, 1921, 1, True), (4, 1, 4000, 1, True),
    (8, 8, 1920, 1, False), (8, 8, 2049, 1, True), (8, 8, 2560, 1, True), (8, 8, 2561, 1, False),  # 64, 72, 80 tiles: three chunks; 88: two
    (8, 2, 4000, 1, False),  # 126 items: two chunks
    # past a round: the remainder, if at most half a round
    (32, 8, 1100, 2, True), (32, 8, 2049, 1, True), (32, 8, 3000, 1, True), (32, 8, 3100, 1, False),
])
def test_dit_split_rule(hq, hk, q_len, batch, split):
    """Which shapes a workspace call splits by keys."""
    assert splits_by_keys(hq, hk, q_len, batch) == split


@pytest.mark.parametrize("causal", [0, 1])
@pytest.mark.parametrize("hq,hk,q_len,kv_len", [(32, 8, 257, 334), (32, 8, 130, 900), (16, 8, 65, 64), (8, 8, 300, 300)])
def test_dit_row_bits_do_not_depend_on_the_call(hq, hk, q_len, kv_len, causal):
    """Without a workspace a problem's rows have the same bits alone (row halves),
    as the first of a batch of one round of tiles (whole), and as the last of a
    batch with a short last round (halved)."""
    G, n = hq // hk, 256 // hk
    tiles = -(-q_len * G // 256)
    one = W.dense_case(hq, hk, q_len, kv_len, causal, seed=q_len)
    want = run_dense(one)[0]
    for batch in (-(-n // tiles), n // tiles + 1):
        c = W.DenseCase(hq=hq, hk=hk, q_len=q_len, kv_len=kv_len, causal=causal, q_stride=one.q_stride,
                        q=np.repeat(one.q, batch, 0), k=np.repeat(one.k, batch, 0), v=np.repeat(one.v, batch, 0),
                        batch=batch)
        got = run_dense(c)
        for b in range(batch):
            assert np.array_equal(got[b], want), f"batch {batch}, problem {b}: {np.sum(got[b] != want)} elements differ"


@pytest.mark.parametrize("hq,hk,page", [(32, 8, 16), (16, 16, 16), (16, 8, 12), (64, 8, 16), (8, 4, 3)])
def test_prefill_exact_p_parity(oracle, hq, hk, page):
    """The plan's exact_p (P carried as two bf16 terms through P.V) on every
    query-head group, paged through powers of two and not, against the oracle."""
    c = W.ragged_prefill_case(3, hq, hk, 1, 300, 0, 200, page=page, seed=hq + hk + page)
    assert_close(run_prefill(c, exact_p=True), oracle_paged(oracle, c), what=f"prefill exact_p {hq}/{hk} page {page}")


@pytest.mark.parametrize("seed", [29, 31])
def test_prefill_exact_p_is_the_f32_p_kernel(seed):
    """With exact_p the MFMA prefill keeps P to 16 significant bits (hi + lo
    bf16), the precision qwen3_attend(ragged = 1)'s f32 P reaches in its
    bf16 output: it agrees bit for bit with the split-K decode kernel (f32 P)
    on >= 99% of elements, differs by at most one bf16 ulp (or 2^-15 near zero)
    elsewhere, and its
    error against f64 SDPA is the decode kernel's (mean within 5%), below the
    bf16-P prefill's."""
    from refs import paged_truth
    from gpu_util import bits_f32

    c = W.ragged_prefill_case(2, 32, 8, 300, 700, 0, 200, seed=seed)
    ex, pre = run_prefill(c, exact_p=True), run_prefill(c)
    plan = oa.decode_plan(c.rows, c.hq, c.hk, c.page, int(c.pos.max()) + 1)
    out = torch.zeros(c.rows, c.hq * 128, dtype=torch.bfloat16, device="cuda")
    oa.qwen3_attend(dev_bits(c.qkv), dev_bits(c.kv), dev_i32(c.pos), dev_i32(c.seq), 1, dev_i32(c.indptr),
                    dev_i32(c.pages), c.page, out, c.hq, c.hk, c.scale, plan, oa.workspace_for(plan))
    torch.cuda.synchronize()
    dec = host_bits(out)
    assert np.mean(ex == dec) >= 0.99
    fe, fd = bits_f32(ex).astype(np.float64), bits_f32(dec).astype(np.float64)
    from refs import bf16_ulp
    # Beyond the rounding step the two f32 results differ by summation order
    # and P's 17th bit, a few 2^-24 of sum p |v| / l (< 1): 2^-15 absolute
    # covers outputs near zero, where one ulp is smaller than that.
    assert np.all(np.abs(fe - fd) <= bf16_ulp(np.maximum(np.abs(fe), np.abs(fd))) + 2.0 ** -15)
    truth = paged_truth(c).reshape(c.rows, -1)
    e_ex, e_dec = np.abs(fe - truth), np.abs(fd - truth)
    e_pre = np.abs(bits_f32(pre).astype(np.float64) - truth)
    assert e_ex.mean() <= 1.05 * e_dec.mean(), (e_ex.mean(), e_dec.mean())
    assert e_ex.mean() < e_pre.mean(), (e_ex.mean(), e_pre.mean())


def test_prefill_error_against_f64_truth_is_near_the_f32_p_kernels():
    """The MFMA prefill rounds P to bf16 (an MFMA operand) where
    qwen3_attend(ragged = 1) keeps it in f32 (qwen3.cu:123-208). Against f64
    SDPA its error stays within 2.5x the mean and 2x the max of the split-K
    decode kernel (f32 P) on the same rows."""
    from refs import paged_truth
    from gpu_util import bits_f32

    c = W.ragged_prefill_case(2, 32, 8, 300, 700, 0, 200, seed=29)
    pre = run_prefill(c)
    plan = oa.decode_plan(c.rows, c.hq, c.hk, c.page, int(c.pos.max()) + 1)
    out = torch.zeros(c.rows, c.hq * 128, dtype=torch.bfloat16, device="cuda")
    oa.qwen3_attend(dev_bits(c.qkv), dev_bits(c.kv), dev_i32(c.pos), dev_i32(c.seq), 1, dev_i32(c.indptr),
                    dev_i32(c.pages), c.page, out, c.hq, c.hk, c.scale, plan, oa.workspace_for(plan))
    torch.cuda.synchronize()
    truth = paged_truth(c).reshape(c.rows, -1)
    e_pre = np.abs(bits_f32(pre).astype(np.float64) - truth)
    e_dec = np.abs(bits_f32(host_bits(out)).astype(np.float64) - truth)
    assert e_pre.mean() <= 2.5 * e_dec.mean(), (e_pre.mean(), e_dec.mean())
    assert e_pre.max() <= 2.0 * e_dec.max(), (e_pre.max(), e_dec.max())
    assert e_pre.max() < 2e-2 / 4 and e_pre.mean() < 2e-3 / 4
