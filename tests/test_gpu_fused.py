"""GPU parity of the fused mixed-batch paged_attention against the CPU
oracle, and its agreement with the decode and prefill operators on the rows
they share.

Tolerances (the contract of this path): bf16 atol/rtol 2e-2, fp16 atol/rtol
5e-3, outputs compared in float32.
"""

from __future__ import annotations

import numpy as np
import pytest
import torch

import proxy_attention_lab as pal
from gpu_util import DEV, announce, dev_bits, dev_index, host_bits, host_f32
from oracle import pal_oracle as orc
from pal_cases import assert_close, extreme_query_bits, make_fused_case, make_paged_case, make_prefill_case, randn_bits
from proxy_attention_lab import _lib

pytestmark = pytest.mark.gpu
DTYPES = ["f16", "bf16"]


def _fused_gpu(case, q, q2seq, q_off, stream=None):
    out = pal.paged_attention(dev_bits(q, case.dtype), dev_bits(case.k_pool, case.dtype),
                              dev_bits(case.v_pool, case.dtype), dev_index(case.page_table, torch.uint32),
                              dev_index(case.seq_lens), dev_index(q2seq, torch.uint32), dev_index(q_off), stream)
    torch.cuda.synchronize()
    return out


def _check_fused(fc, what):
    c = fc.case
    announce(f"fused {what} R={len(fc.q2seq)} S={c.num_seqs} Hq={c.num_q_heads} Hkv={c.num_kv_heads} "
             f"HD={c.head_dim} TPP={c.tokens_per_page} {c.dtype}")
    out = host_f32(_fused_gpu(c, fc.queries, fc.q2seq, fc.q_offset))
    assert out.shape == fc.queries.shape
    ref = orc.paged_attention(fc.queries, c.k_pool, c.v_pool, c.page_table, c.seq_lens, fc.q2seq, fc.q_offset,
                              c.dtype)
    assert_close(out, ref, c.dtype, what)
    return out


@pytest.mark.parametrize("dtype", DTYPES)
def test_fused_mixed_small(dtype):
    """A config-5-like batch in miniature: GQA 8:1, decode rows interleaved
    with blocks of three prefill chunks."""
    rng = np.random.default_rng(50)
    dec = rng.integers(1, 900, size=40)
    fc = make_fused_case(50, dec, [(0, 100), (130, 64), (500, 257)], 64, 8, 128, 16, dtype, block=40)
    _check_fused(fc, "mixed")


@pytest.mark.parametrize("hd", [32, 64, 96, 128, 256])
def test_fused_head_dims(hd):
    fc = make_fused_case(hd, [17, 300, 1], [(20, 33), (0, 5)], 8, 2, hd, 32 if hd == 64 else 16, "bf16")
    _check_fused(fc, f"hd{hd}")


@pytest.mark.parametrize("heads", [(1, 1), (4, 1), (32, 8), (40, 2), (32, 32)])
def test_fused_gqa_groups(heads):
    hq, hkv = heads
    fc = make_fused_case(hq + hkv, [100, 2000, 0, 16], [(64, 70), (3, 140)], hq, hkv, 64, 16, "f16", block=32)
    _check_fused(fc, f"heads{heads}")


def test_fused_decode_rows_equal_decode_op():
    lens = [1, 15, 16, 17, 511, 3000, 0, 40]
    case = make_paged_case(60, lens, 32, 8, 128, 16, "bf16")
    q = randn_bits(np.random.default_rng(60), (len(lens), 32, 128), "bf16")
    announce("fused decode rows vs decode op")
    fused = host_f32(_fused_gpu(case, q, np.arange(len(lens), dtype=np.uint32), case.seq_lens.copy()))
    dec = pal.paged_attention_decode(dev_bits(q, "bf16"), dev_bits(case.k_pool, "bf16"), dev_bits(case.v_pool, "bf16"),
                                     dev_index(case.page_table, torch.uint32), dev_index(case.seq_lens))
    torch.cuda.synchronize()
    assert_close(fused, host_f32(dec), "bf16", "fused vs decode")
    ref = orc.paged_attention_decode(q, case.k_pool, case.v_pool, case.page_table, case.seq_lens, "bf16")
    assert_close(fused, ref, "bf16", "fused vs oracle")


def test_fused_after_fill_equals_prefill_op():
    """fill_kv_pages writes the prompt into the pages; the fused op over the
    prompt rows then matches the reference-signature prefill (dense prompt)."""
    hist, plen, hq, hkv, hd, tpp = [37, 0, 64], 48, 16, 4, 128, 16
    case, qp, kp, vp = make_prefill_case(61, hist, plen, hq, hkv, hd, tpp, "f16")
    S = case.num_seqs
    # room for the prompt: extend each page row with fresh pages
    need = [(h + plen + tpp - 1) // tpp for h in hist]
    width = max(need)
    base = case.k_pool.shape[0]
    extra = sum(n - (h + tpp - 1) // tpp for n, h in zip(need, hist))
    k_pool = np.concatenate([case.k_pool, np.zeros((extra,) + case.k_pool.shape[1:], np.uint16)])
    v_pool = np.concatenate([case.v_pool, np.zeros((extra,) + case.v_pool.shape[1:], np.uint16)])
    pt = np.zeros((S, width), np.uint32)
    nxt = base
    for s in range(S):
        have = (hist[s] + tpp - 1) // tpp
        pt[s, :have] = case.page_table[s, :have]
        for j in range(have, need[s]):
            pt[s, j] = nxt
            nxt += 1
    announce("fused after fill vs prefill op")
    kd, vd = dev_bits(k_pool, "f16"), dev_bits(v_pool, "f16")
    ptd = dev_index(pt, torch.uint32)
    pos = np.concatenate([h + np.arange(plen) for h in hist]).astype(np.int32)
    q2s = np.repeat(np.arange(S), plen).astype(np.uint32)
    pal.fill_kv_pages(dev_bits(kp, "f16"), dev_bits(vp, "f16"), kd, vd, ptd, dev_index(pos),
                      dev_index(q2s, torch.uint32))
    lens_total = np.array(hist, np.int32) + plen
    fused = pal.paged_attention(dev_bits(qp, "f16"), kd, vd, ptd, dev_index(lens_total),
                                dev_index(q2s, torch.uint32), dev_index(pos + 1))
    pre = pal.paged_attention_prefill(dev_bits(qp, "f16"), dev_bits(kp, "f16"), dev_bits(vp, "f16"),
                                      dev_bits(case.k_pool, "f16"), dev_bits(case.v_pool, "f16"),
                                      dev_index(case.page_table, torch.uint32), dev_index(case.seq_lens))
    torch.cuda.synchronize()
    fused = host_f32(fused).reshape(-1, hd)
    assert_close(fused, host_f32(pre), "f16", "fused vs prefill")
    ref = orc.paged_attention_prefill(qp, kp, vp, case.k_pool, case.v_pool, case.page_table, case.seq_lens, "f16")
    assert_close(fused, ref, "f16", "fused vs oracle")


def test_fused_edge_rows():
    """Offsets of 0, negative and past the length; a row naming no sequence;
    a run longer than a tile; runs of two rows."""
    case = make_paged_case(62, [50, 300, 7], 8, 2, 64, 16, "bf16")
    rng = np.random.default_rng(62)
    q2seq = np.array([0, 0, 1, 2, 9, 1, 1, 1] + [1] * 150 + [2, 0], np.uint32)
    off = np.array([0, -3, 1000, 7, 5, 1, 2, 3] + list(range(4, 154)) + [1, 50], np.int32)
    q = randn_bits(rng, (len(q2seq), 8, 64), "bf16")
    announce("fused edge rows")
    out = host_f32(_fused_gpu(case, q, q2seq, off))
    ref = orc.paged_attention(q, case.k_pool, case.v_pool, case.page_table, case.seq_lens, q2seq, off, "bf16")
    assert_close(out, ref, "bf16", "edge rows")
    assert np.all(out[[0, 1, 4]] == 0)


def test_fused_many_rows_planner_chunks():
    """More than 1024 rows (the decode workers' row scan carries runs across
    its passes of 4096 rows): 1100 decode rows plus a 1500-row prompt run."""
    rng = np.random.default_rng(63)
    dec = rng.integers(0, 80, size=1100)
    fc = make_fused_case(63, dec, [(200, 1500)], 8, 1, 64, 16, "f16", block=1500, garbage_tail=False)
    _check_fused(fc, "many rows")


def test_fused_lone_rows_beyond_the_list():
    """More lone (decode) rows with keys than the fused kernel's in-LDS list
    holds (2048): the decode workers claim batches of 64 rows and compute each
    lone row whole.  Rows without keys and a prompt run interleave."""
    rng = np.random.default_rng(65)
    dec = rng.integers(0, 400, size=2300)
    fc = make_fused_case(65, dec, [(50, 300)], 8, 2, 64, 16, "bf16", block=100)
    assert int(np.count_nonzero(dec)) > 2048
    _check_fused(fc, "claiming mode")


def test_fused_deterministic_and_empty():
    fc = make_fused_case(64, [900, 3], [(100, 300)], 32, 8, 128, 16, "bf16", block=100)
    c = fc.case
    announce("fused determinism")
    a = host_bits(_fused_gpu(c, fc.queries, fc.q2seq, fc.q_offset))
    b = host_bits(_fused_gpu(c, fc.queries, fc.q2seq, fc.q_offset))
    assert np.array_equal(a, b)
    empty = pal.paged_attention(dev_bits(fc.queries[:0], "bf16"), dev_bits(c.k_pool, "bf16"),
                                dev_bits(c.v_pool, "bf16"), dev_index(c.page_table), dev_index(c.seq_lens),
                                dev_index(fc.q2seq[:0]), dev_index(fc.q_offset[:0]))
    assert empty.shape == (0, 32, 128)


@pytest.mark.parametrize("tpp", [16, 32])
def test_fused_long_history_window(tpp):
    """A prefill run over a cache longer than 8192 keys (window mode stages
    its page ids in chunks of 512 entries and rotates them), beside decode
    rows of similar length."""
    fc = make_fused_case(70 + tpp, [100, 30000], [(26000 if tpp == 16 else 38000, 64), (9000, 40)], 32, 8, 128,
                         tpp, "bf16", block=64)
    _check_fused(fc, f"long history window tpp{tpp}")


@pytest.mark.parametrize("dtype", DTYPES)
def test_fused_query_magnitudes(dtype):
    """A mixed batch whose query heads span the dtype's range (zeros, tiny,
    large, mixed, near the range ends), in its decode rows and its tiles
    (the large heads held to the tiles' exact range)."""
    fc = make_fused_case(74, [5, 300, 1200], [(0, 70), (200, 130)], 16, 4, 128, 16, dtype)
    fc.queries = extreme_query_bits(np.random.default_rng(74), fc.queries.shape, dtype, tiles=True)
    out = _check_fused(fc, f"query magnitudes {dtype}")
    assert np.isfinite(out).all()


# (query heads, kv heads, decode lengths, chunks, block).  From 1,200 (row, head
# of a group) per sequence on, tiles have a CU to themselves where no row is alone
# in its run (found on the device if there is more than one sequence): one side of
# that line and the other, with lone rows and without, tiles of one row group, of
# two, and more tiles than CUs (256) of either (claimed), windows that start and
# end inside a run
TILE_CASES = {
    "beside-decode": (32, 8, [300], [(100, 598)], 600),            # 599 rows * 4 < 1200 * 2
    "one-group": (32, 8, [300], [(100, 599)], 600),                # 600 rows * 4 = 1200 * 2, a lone row: half tiles
    "whole-one-group": (32, 8, [], [(100, 598), (50, 2)], 600),    # 152 tiles
    "whole-one-group-claimed": (104, 26, [], [(20, 590), (4, 12)], 590),  # 494 tiles of 32 rows, 260 of 64
    "whole-two-groups": (128, 8, [], [(37, 300), (500, 2)], 300),  # 304 tiles of 8 rows, 152 of 16
    "whole-two-groups-claimed": (256, 16, [], [(65, 401), (3, 5)], 401),  # 816 tiles of 8 rows, 416 of 16
    "whole-runs": (64, 4, [], [(20, 1700), (3, 40)], 33),          # several runs to a window
    "one-group-filled": (32, 32, [], [(0, 1400)], 1400),           # 352 tiles of 128 rows, 192 of 256: two groups
    "one-group-claimed": (130, 130, [], [(0, 300)], 300),          # 390 tiles of 128 rows, 260 of 256: two rounds either way
    "two-groups": (128, 8, [], [(37, 300), (500, 1)], 300),        # a lone row: half tiles
    "two-groups-claimed": (256, 16, [70], [(65, 401)], 401),       # a lone row
    "lone-rows": (64, 4, [900] * 20 + [0], [(20, 1700), (3, 40)], 33),  # interleaved with blocks of runs
}


@pytest.mark.parametrize("hd,tpp,dtype", [(32, 16, "f16"), (64, 32, "bf16"), (128, 16, "bf16"), (256, 16, "bf16")])
@pytest.mark.parametrize("name", TILE_CASES)
def test_fused_tile_sizes(name, hd, tpp, dtype):
    """Twice each: a call leaves the counters its tiles are claimed from as it
    found them, and the claim order does not show in the result."""
    hq, hkv, dec, chunks, block = TILE_CASES[name]
    fc = make_fused_case(hd + 77, dec, chunks, hq, hkv, hd, tpp, dtype, block=block)
    first = _check_fused(fc, name)
    again = host_f32(_fused_gpu(fc.case, fc.queries, fc.q2seq, fc.q_offset))
    assert np.array_equal(first, again)


@pytest.mark.parametrize("heads,rows", [((64, 32), 700), ((200, 100), 300)], ids=["by-place", "claimed"])
def test_fused_tile_claims_across_head_dims(heads, rows):
    """Head dims above and up to 128 claim tiles in kernels of different launch
    sequences, from the counters of one workspace.  700 rows of 32 kv heads make
    352 tiles of one row group, which head dim 256 claims, and 192 of two, all
    taken by place; 300 rows of 100 kv heads 500 or 300, claimed at every head dim."""
    for i, hd in enumerate([256, 64, 256, 32]):
        _check_fused(make_fused_case(90 + i, [], [(10, rows)], *heads, hd, 16, "bf16", block=rows), f"claims hd{hd}")


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("hd,tpp", [(32, 16), (64, 32), (128, 16), (256, 16)])
@pytest.mark.parametrize("decode,rows,heads", [([], 90, (16, 1)), ([], 2300, (8, 8)), ([300], 60, (8, 2))],
                         ids=["wide", "wide-more-rows", "beside-decode"])
def test_fused_nan_stays_in_its_rows(decode, rows, heads, hd, tpp, dtype):
    """A NaN in one query head of one row, or in a key that only the last row
    sees, leaves every other row's bits as they are without it."""
    fc = make_fused_case(hd + rows, decode, [(30, rows)], *heads, hd, tpp, dtype, block=rows)
    c = fc.case
    announce(f"NaN rows: fused R={len(fc.q2seq)} heads={heads} HD={hd} TPP={tpp} {dtype}")
    nan = 0x7FC0 if dtype == "bf16" else 0x7E00
    clean = host_bits(_fused_gpu(c, fc.queries, fc.q2seq, fc.q_offset))
    chunk = np.flatnonzero(fc.q2seq == len(decode))  # in position order

    q = fc.queries.copy()
    hit = chunk[[3, 40, len(chunk) - 1]]
    q[hit, 1, 5] = nan
    out = _fused_gpu(c, q, fc.q2seq, fc.q_offset)
    keep = np.ones(clean.shape[:2], bool)
    keep[hit, 1] = False
    assert np.isnan(host_f32(out)[hit, 1]).all()
    assert np.array_equal(host_bits(out)[keep], clean[keep])

    last = int(c.seq_lens[len(decode)]) - 1
    page = int(c.page_table[len(decode), last // tpp])
    c.k_pool[page, :, 0, last % tpp, 2] = nan
    out = _fused_gpu(c, fc.queries, fc.q2seq, fc.q_offset)
    keep = np.ones(len(clean), bool)
    keep[chunk[-1]] = False
    assert np.isnan(host_f32(out)[chunk[-1]]).all()
    assert np.array_equal(host_bits(out)[keep], clean[keep])


@pytest.mark.parametrize("hd", [64, 256])
@pytest.mark.parametrize("rows,heads,others", [(2200, (32, 32), None), (700, (64, 16), None), (2300, (128, 8), None),
                                               (2300, (128, 8), 30), (700, (64, 16), 1), (700, (32, 32), 1)],
                         ids=["one-group", "few", "two-groups", "two-sequences", "lone-row", "beside-decode"])
def test_fused_workspace_contract(rows, heads, others, hd):
    """Of the workspace, the four bytes at 64 are all that has to be zero before
    a call (head dim 64: 576 tiles of one row group on 256 CUs; 352 of one, 176
    of two; 2,304 / 1,152: claimed, all taken by place, claimed; the last again with
    a second sequence of 30 rows, so that the device decides for them, and batches
    with a lone row above and below that line), and are zero again after it."""
    hq, hkv = heads
    chunks = [(10, rows)] + ([(25, others)] if others else [])
    fc = make_fused_case(rows + hd, [], chunks, hq, hkv, hd, 16, "bf16", block=rows)
    c = fc.case
    announce(f"fused workspace contract rows={rows} heads={heads} HD={hd}")
    ref = host_bits(_fused_gpu(c, fc.queries, fc.q2seq, fc.q_offset))
    lib = _lib.lib()
    q, k, v = dev_bits(fc.queries, "bf16"), dev_bits(c.k_pool, "bf16"), dev_bits(c.v_pool, "bf16")
    pt, lens = dev_index(c.page_table, torch.uint32), dev_index(c.seq_lens)
    q2s, off = dev_index(fc.q2seq, torch.uint32), dev_index(fc.q_offset)
    n = len(fc.q2seq)
    size = lib.pal_paged_attention_workspace_size(_lib.DTYPE_BFLOAT16, n, hq, hkv, hd, 16)
    ws = torch.zeros(size, dtype=torch.uint8, device=DEV)
    ws[:256] = 0xA5
    ws[64:68] = 0
    for call in range(2):
        out = torch.full_like(q, 7.0)
        st = lib.pal_paged_attention(q.data_ptr(), k.data_ptr(), v.data_ptr(), pt.data_ptr(), lens.data_ptr(),
                                     q2s.data_ptr(), off.data_ptr(), out.data_ptr(), _lib.DTYPE_BFLOAT16, n, c.num_seqs,
                                     hq, hkv, hd, 16, int(c.k_pool.shape[0]), int(c.page_table.shape[1]), ws.data_ptr(),
                                     size, torch.cuda.current_stream().cuda_stream)
        assert st == 0, lib.pal_last_error()
        torch.cuda.synchronize()
        assert np.array_equal(host_bits(out), ref), f"call {call}"
        assert not ws[64:68].any(), f"call {call}"
