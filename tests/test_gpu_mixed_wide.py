"""Wide launches of the mixed kernel (enough prefill rows to fill the chip) against the oracle.

Every case here asserts from its plan that the launch is wide.  It is compared
with the fp32 oracle, planned and unplanned (which must agree bit for bit), at
the edges of the tiles: lengths of a whole tile (16 * floor(8 / G) rows), one row
more and less, chunks of one and two column tiles a wave, items of half the
columns, sequences that split their keys and decode rows beside them."""
import pytest
import torch

from custom_inference_engine_amd import kv_append_tokens, mixed_gqa_attention, mixed_plan
from oracle import inputs
from tests.conftest import assert_attn_close
from tests.gpu_helpers import DEV, bits, err_word, note, oracle_mixed

pytestmark = pytest.mark.gpu


def _word(plan):
    """Header word 6 of a mixed plan: 16 * column tiles an item + 16-row blocks a tile, 0 if not wide."""
    return int(plan[6])


def _most_chunks(plan):
    """The most chunks that a query tile of the plan has."""
    n, (ct, m) = int(plan[0]), divmod(_word(plan), 16)
    items = plan[8:8 + 8 * n].view(n, 8).cpu()
    _, count = torch.unique(items[:, 0] * (1 << 20) + items[:, 1], return_counts=True)
    g = int(plan[4]) // int(plan[5])
    return int(count.max()) // (2 if m * g > ct else 1)


def _run(case, h_q, max_seqlen=None, poison=False, rows=slice(None), bad_v=(), chunks=1,
         half=False):
    c = case.to(DEV)
    kp, vp = c.k_pool.clone(), c.v_pool.clone()
    if poison:  # pool rows past each sequence's end hold NaN (as uninitialised memory may)
        used = torch.zeros(kp.shape[0], kp.shape[2], dtype=torch.bool)
        for b in range(case.B):
            n = int(case.kv_lens[b] + case.new_lens[b])
            pg = case.block_table[int(case.slot_ids[b])]
            pos = torch.arange(n)
            used[pg[pos // case.page_size], pos % case.page_size] = True
        kp.transpose(1, 2)[~used.to(DEV)] = float("nan")
        vp.transpose(1, 2)[~used.to(DEV)] = float("nan")
    err = err_word()
    kv_append_tokens(kp, vp, c.k_new, c.v_new, c.pages, c.offsets, err=err)
    for b, j in bad_v:  # V of new row j of sequence b
        pos = int(case.kv_lens[b]) + j
        row = vp[int(case.block_table[int(case.slot_ids[b]), pos // case.page_size]), :, pos % case.page_size]
        row[:, 0::2], row[:, 1::2] = float("inf"), float("nan")
    ms = max_seqlen or int(case.new_lens.max())
    plan = mixed_plan(kp, c.cu_seqlens, c.kv_lens, c.slot_ids, c.block_table, ms, case.T, h_q, err=err)
    assert _word(plan) // 16 == (4 if half else 8), "not the items that this case is for"
    assert _most_chunks(plan) >= chunks
    o = [mixed_gqa_attention(c.q, kp, vp, ms, c.cu_seqlens, c.kv_lens, c.slot_ids, c.block_table, err=err,
                             plan=p) for p in (plan, None)]
    torch.cuda.synchronize()
    # (rows that are not computed hold what torch.empty_like left there)
    assert torch.equal(bits(o[0][0, rows]), bits(o[1][0, rows])), "planned and unplanned differ"
    return o[0][0].float().cpu(), int(err.item())


CASES = {
    # h_q, h_kv, d, page_size, prior, new
    "d128": (14, 2, 128, 16, [0, 700, 33, 0, 5, 90, 3000], [320, 17, 250, 16, 1, 1, 200]),
    "d128-g4-ps32": (32, 8, 128, 32, [0, 1000, 40, 7], [31, 1, 33, 400]),
    "d128-g1": (8, 8, 128, 16, [0, 500, 0], [127, 1, 1500]),
    "d128-g8": (16, 2, 128, 16, [100, 2], [700, 300]),
    "d64-g1": (8, 8, 64, 16, [0, 3, 200, 64], [900, 129, 1100, 16]),
    "d64-g2": (8, 4, 64, 32, [0, 31, 1500], [2000, 65, 2200]),
    "d64-g7": (14, 2, 64, 16, [0, 15, 600, 40, 1000], [2100, 15, 1990, 1, 1]),
    "d64-g5": (20, 4, 64, 16, [10, 0], [17, 2500]),
    "d64-g3": (24, 8, 64, 16, [10, 0], [33, 2100]),
    "d64-g4": (16, 4, 64, 16, [0, 100], [3000, 257]),
    "d64-g6": (24, 4, 64, 16, [0, 100], [2100, 33]),
    "d64-g8": (32, 4, 64, 16, [0, 100], [1570, 17]),
    "d128-g3": (24, 8, 128, 16, [0, 100, 9], [300, 33, 70]),
    "d128-g6": (24, 4, 128, 16, [0, 100, 9], [300, 33, 70]),
    # items of half the columns: one long prompt makes most of few columns
    "d128-g7-half": (14, 2, 128, 16, [0, 700, 33, 90], [630, 17, 16, 1]),
    "d128-g1-half": (8, 8, 128, 16, [0, 500, 0, 7], [1100, 1, 63, 65]),
    "d128-g2-half": (16, 8, 128, 32, [30, 500], [550, 33]),
    "d128-g3-half": (12, 4, 128, 16, [30, 500], [750, 17]),
    "d128-g5-half": (10, 2, 128, 16, [30, 500], [900, 16]),
    "d128-g8-half": (16, 2, 128, 16, [30, 500], [600, 2]),
}


@pytest.mark.parametrize("name", CASES)
def test_wide_launch_matches_the_oracle(native_lib, name):
    h_q, h_kv, d, ps, prior, new = CASES[name]
    case = inputs.make_case(prior, new, h_q=h_q, h_kv=h_kv, d=d, page_size=ps, seed=91)
    note(f"wide {name}")
    o, err = _run(case, h_q, poison=True, half=name.endswith("half"))
    assert err == 0
    want, written = oracle_mixed(case)
    assert_attn_close(o[written], want[written], what=name)


# h_q, h_kv, d, rows, max_seqlen (None: the rows), column tiles an item (0: 16-row tiles)
LINES = [
    (8, 8, 64, 1536, None, 0), (8, 8, 64, 1537, None, 8),
    (16, 8, 64, 2048, None, 0), (16, 8, 64, 2049, None, 8),
    (24, 8, 64, 2048, None, 0), (24, 8, 64, 2049, None, 8),
    (14, 2, 64, 3510, None, 0), (14, 2, 64, 3511, None, 8),
    (32, 8, 128, 256, None, 0), (32, 8, 128, 257, None, 8),
    (14, 2, 128, 585, None, 0), (14, 2, 128, 586, None, 4), (14, 2, 128, 586, 256, 8),
    (14, 2, 128, 877, None, 4), (14, 2, 128, 878, None, 8),
    (19, 19, 128, 500, None, 4), (20, 4, 128, 410, None, 8),
]


@pytest.mark.parametrize("h_q,h_kv,d,rows,max_seqlen,ct", LINES)
def test_wide_lines(native_lib, h_q, h_kv, d, rows, max_seqlen, ct):
    """The launches on either side of each line: columns (rows x q heads) a launch is wide
    from, and those up to which few heads' items hold half the columns."""
    pages = -(-rows // 16)
    pool = torch.zeros(pages, h_kv, 16, d, dtype=torch.float16, device=DEV)
    i64 = dict(dtype=torch.int64, device=DEV)
    plan = mixed_plan(pool, torch.tensor([0, rows], **i64), torch.zeros(1, **i64), torch.zeros(1, **i64),
                      torch.arange(pages, **i64)[None], max_seqlen or rows, rows, h_q)
    g = h_q // h_kv
    assert _word(plan) == (ct * 16 + max(1, ct // g) if ct else 0)


def test_wide_launch_splits_long_tiles(native_lib):
    """One long chunk over a long prefix beside short ones: its tiles are far above
    the average share of keys and split; with no partials budget the same
    tiles run whole, and both match the oracle."""
    case = inputs.make_case([6000, 0, 0], [300, 200, 300], d=128, seed=92)
    note("wide split")
    o, err = _run(case, 14, chunks=2)
    assert err == 0
    want, written = oracle_mixed(case)
    assert_attn_close(o[written], want[written], what="split")
    c = case.to(DEV)
    kp, vp = (t.to(DEV) for t in case.appended_pools())
    whole = mixed_gqa_attention(c.q, kp, vp, 300, c.cu_seqlens, c.kv_lens, c.slot_ids, c.block_table,
                                partials_bytes=0)
    assert_attn_close(whole[0].float().cpu()[written], want[written], what="whole")


def test_wide_launch_of_many_sequences(native_lib):
    """More than 64 sequences (the block plan), most of them decode rows."""
    new = [1 if i % 3 else 29 for i in range(100)]
    case = inputs.make_case([(i * 37) % 400 for i in range(100)], new, d=128, seed=93)
    note("wide block plan")
    o, err = _run(case, 14)
    assert err == 0
    want, written = oracle_mixed(case)
    assert_attn_close(o[written], want[written], what="many")


def test_wide_launch_past_max_seqlen(native_lib):
    """Rows past max_seqlen (rounded up to 16) are reported and not computed, the others are."""
    case = inputs.make_case([0, 100], [500, 500], d=128, seed=94)
    note("wide max_seqlen")
    rows = torch.cat([torch.arange(208), 500 + torch.arange(208)])
    o, err = _run(case, 14, max_seqlen=200, rows=rows)
    assert err == 2  # CIE_ERRBIT_LEN
    want, _ = oracle_mixed(case)
    assert_attn_close(o[rows], want[rows], what="max_seqlen")


SPLITS = {
    # few rows over long prefixes: tiles of up to 8 chunks, the partial last tile among them
    "d128-g7": (14, 2, 128, [9000, 6001, 0, 1500], [900, 30, 17, 1]),
    "d128-g7-half": (14, 2, 128, [9000, 6001, 0, 1500], [670, 30, 17, 1]),
    "d128-g1-half": (8, 8, 128, [9000, 6001, 0], [1200, 3, 17]),
    "d128-g4": (32, 8, 128, [8015, 700, 3000], [290, 3, 1]),
    "d64-g1": (8, 8, 64, [7000, 0, 2000], [1801, 70, 1]),
}


@pytest.mark.parametrize("name", SPLITS)
def test_wide_launch_of_long_prefixes(native_lib, name):
    """Tiles of several chunks, under the default partials budget, a third of it
    (fewer, longer chunks) and none: every one matches the oracle."""
    h_q, h_kv, d, prior, new = SPLITS[name]
    case = inputs.make_case(prior, new, h_q=h_q, h_kv=h_kv, d=d, seed=95)
    note(f"wide long prefixes {name}")
    o, err = _run(case, h_q, chunks=3, half=name.endswith("half"))
    assert err == 0
    want, written = oracle_mixed(case)
    assert_attn_close(o[written], want[written], what=name)
    c = case.to(DEV)
    kp, vp = (t.to(DEV) for t in case.appended_pools())
    full = native_lib.cie_mixed_default_partials_bytes(case.T, max(new), h_q, h_kv, d)
    for nbytes in (full // 3, 0):
        o = mixed_gqa_attention(c.q, kp, vp, max(new), c.cu_seqlens, c.kv_lens, c.slot_ids, c.block_table,
                                partials_bytes=nbytes)
        assert_attn_close(o[0].float().cpu()[written], want[written], what=f"{name}, {nbytes} bytes")


MASKED = {  # h_q, h_kv, d, prior, new
    "d64-g1": (8, 8, 64, [0, 37, 2000], [700, 500, 420]),
    "d64-g2": (16, 8, 64, [0, 37, 2000], [700, 600, 800]),
    "d64-g3": (24, 8, 64, [0, 37, 2000], [900, 700, 500]),
    "d128-g1": (8, 8, 128, [0, 37, 3000], [900, 700, 500]),
    "d128-g2": (16, 8, 128, [0, 37, 3000], [400, 300, 200]),
    "d128-g4": (32, 8, 128, [0, 37, 3000], [200, 170, 130]),
    "d128-g3": (24, 8, 128, [0, 37, 3000], [200, 170, 130]),
    "d128-g7": (14, 2, 128, [0, 37, 3000], [500, 450, 300]),
    "d128-g1-half": (8, 8, 128, [0, 37, 3000], [900, 300, 100]),
}


@pytest.mark.parametrize("name", MASKED)
def test_wide_launch_keeps_masked_values_out(native_lib, name):
    """Inf and NaN in the V row of a new token reach no row of an earlier 16-row block of
    its sequence: those rows are bit for bit what they are with finite values there."""
    h_q, h_kv, d, prior, new = MASKED[name]
    case = inputs.make_case(prior, new, h_q=h_q, h_kv=h_kv, d=d, seed=96)
    m = 8 // (h_q // h_kv)
    # the last block of a wide tile, the second block of one (its first row), the last row
    first = [16 * m - 1 + 16 * m, 16 if m > 1 else 32, new[2] - 1]
    note(f"wide masked {name}")
    half = name.endswith("half")
    clean, err = _run(case, h_q, half=half)
    assert err == 0
    bad, err = _run(case, h_q, bad_v=list(enumerate(first)), half=half)
    assert err == 0
    for b, j in enumerate(first):
        t0 = int(case.cu_seqlens[b])
        before = slice(t0, t0 + j // 16 * 16)
        assert torch.equal(bits(bad[before]), bits(clean[before])), (name, b)
        assert not torch.isfinite(bad[t0 + j]).any(), (name, b)


OWN_PLANS = {  # heads (G = 1), d, workgroups a kv head on 256 CUs, prior, new
    "d64": (256, 64, 3, [i % 9 for i in range(200)], [200 if i == 70 else 1 + i % 3 for i in range(200)]),
    "d128": (256, 128, 2, [i % 9 for i in range(135)], [200 if i == 70 else 1 + i % 3 for i in range(135)]),
}


@pytest.mark.parametrize("name", OWN_PLANS)
def test_wide_launch_plans_a_workgroups_rounds_in_parts(native_lib, name):
    """Unplanned wide launches make the descriptors of 64 rounds of a workgroup at a time:
    with few workgroups a kv head, a large batch has more rounds than that."""
    h, d, slots, prior, new = OWN_PLANS[name]
    case = inputs.make_case(prior, new, h_q=h, h_kv=h, d=d, seed=97)
    assert len(new) > 64 * slots  # an item at least for each sequence
    note(f"wide own plan {name}")
    o, err = _run(case, h)
    assert err == 0
    want, written = oracle_mixed(case)
    assert_attn_close(o[written], want[written], what=name)
