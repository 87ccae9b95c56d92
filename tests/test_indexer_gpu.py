"""GPU parity of the lightning indexer + top-k and of the indexer -> attention
pipeline, against the CPU oracle.

Scores must match the oracle bit for bit (the exact rounding order of
include/dsa_abi.h) and the selected positions must be the same sets, ties
going to the lower position.  Reference: solution/triton/indexer_kernel.py
:4-343 (score structure :185-275, intended selection :289-343) and the
BASELINE indexer workload (config 5).
"""
import ctypes
import math
import os

import numpy as np
import pytest
import torch

import oracle
from conftest import LSE_ATOL, LSE_RTOL, OUT_ATOL, OUT_RTOL, fill_lds_with_nan, mismatches
from dsa_amd import _lib, workloads
from dsa_amd.indexer_kernel import run_indexer_and_topk, run_sparse_attention_pipeline

pytestmark = pytest.mark.gpu

DEV = "cuda:0"
NTHREADS = min(16, os.cpu_count() or 1)


def _np(d):
    return {k: (v.numpy() if isinstance(v, torch.Tensor) and v.dtype != torch.bfloat16 else v)
            for k, v in d.items()}


def _gpu_indexer(d, topk, block_table=None, page_size=64, nan_lds=False):
    g = workloads.to_device(d, DEV)
    bt = None if block_table is None else block_table.to(DEV)
    if nan_lds:
        fill_lds_with_nan(DEV)
    out, scores = run_indexer_and_topk(g["q_idx"], g["k_idx"], g["k_scale"], g["weights"],
                                       g["causal_limit"], topk, block_table=bt,
                                       page_size=page_size, return_scores=True)
    torch.cuda.synchronize()
    return out.cpu().numpy(), scores.cpu().numpy()


def _oracle(d, topk):
    n = _np(d)
    sc = oracle.indexer_scores(n["q_idx"], n["k_idx"], n["k_scale"], n["weights"],
                               n["causal_limit"].astype(np.int64), NTHREADS)
    return oracle.topk(sc, n["causal_limit"].astype(np.int64), topk), sc


def _assert_same(got_idx, got_sc, ref_idx, ref_sc, label):
    bad = np.flatnonzero(got_sc.view(np.uint32) != ref_sc.view(np.uint32))
    assert bad.size == 0, (f"{label}: {bad.size} scores differ from the oracle, first at "
                           f"{np.unravel_index(bad[0], ref_sc.shape)}: {got_sc.flat[bad[0]]!r} vs "
                           f"{ref_sc.flat[bad[0]]!r}")
    for t in range(ref_idx.shape[0]):
        assert np.array_equal(np.sort(got_idx[t]), np.sort(ref_idx[t])), f"{label}: row {t} set differs"
        valid = got_idx[t][got_idx[t] >= 0]
        assert np.all(np.diff(valid) > 0), f"{label}: row {t} not in ascending position order"


def test_cfg5_indexer_full_bit_exact():
    d = workloads.indexer_inputs(seed=workloads.DEFAULT_SEED + 5)
    got_idx, got_sc = _gpu_indexer(d, 2048)
    ref_idx, ref_sc = _oracle(d, 2048)
    _assert_same(got_idx, got_sc, ref_idx, ref_sc, "cfg5")


@pytest.mark.parametrize("T,Hi,S,topk", [(5, 16, 1000, 64), (3, 32, 777, 300), (33, 48, 513, 17),
                                         (2, 64, 300, 512)])
def test_ragged_shapes(T, Hi, S, topk):
    d = workloads.indexer_inputs(T=T, Hi=Hi, S=S, seed=T * 1000 + S)
    got_idx, got_sc = _gpu_indexer(d, topk)
    ref_idx, ref_sc = _oracle(d, topk)
    _assert_same(got_idx, got_sc, ref_idx, ref_sc, f"T={T} Hi={Hi} S={S} k={topk}")


@pytest.mark.parametrize("T,Hi,S", [(22, 32, 3000), (5, 48, 2203), (9, 64, 4099), (1, 64, 900)])
def test_chunked_ranges_random_causal_limits(T, Hi, S):
    """Causal limits anywhere in a token's row.  The three-product path deals
    a range out in chunks of six blocks to the token's two waves; a limit
    cuts the last chunk after 1..6 blocks (with these shapes every remainder
    occurs), masks part of its last block and leaves later blocks at -inf.
    T not a multiple of 4 leaves workgroups with fewer tokens."""
    d = workloads.indexer_inputs(T=T, Hi=Hi, S=S, seed=T * 7919 + S)
    lim = np.random.default_rng(S).integers(-3, S, T)
    d["causal_limit"] = torch.from_numpy(lim.astype(np.int32))
    topk = min(256, S // 2)
    got_idx, got_sc = _gpu_indexer(d, topk)
    ref_idx, ref_sc = _oracle(d, topk)
    _assert_same(got_idx, got_sc, ref_idx, ref_sc, f"T={T} Hi={Hi} S={S}")


@pytest.mark.parametrize("scale,label", [(60.0, "third piece"), (28.0, "beyond the int32 combine")])
def test_one_wide_block_sends_its_range_to_the_general_paths(scale, label):
    """One block of 16 positions with large values: the position range that
    holds it takes the general paths (split between the token's two waves),
    every other range the three-product path."""
    T, Hi, S = 6, 64, 5000
    d = workloads.indexer_inputs(T=T, Hi=Hi, S=S, seed=99)
    g = torch.Generator().manual_seed(99)
    k = d["k_idx"].view(torch.float8_e4m3fn).float()
    k[592:608] = (torch.randn(16, 128, generator=g) * scale).clamp(-scale, scale)
    d["k_idx"] = workloads.e4m3(k)
    got_idx, got_sc = _gpu_indexer(d, 300)
    ref_idx, ref_sc = _oracle(d, 300)
    _assert_same(got_idx, got_sc, ref_idx, ref_sc, label)


def test_ties_go_to_lower_positions():
    d = workloads.indexer_inputs(T=4, Hi=16, S=600, seed=7)
    k = d["k_idx"].clone()
    k[300:600] = k[0:300]                      # exact duplicate rows ...
    sc = d["k_scale"].clone()
    sc[300:600] = sc[0:300]                    # ... with the same scales: tied scores
    d.update(k_idx=k, k_scale=sc)
    for topk in (1, 100, 333, 590):
        got_idx, got_sc = _gpu_indexer(d, topk)
        ref_idx, ref_sc = _oracle(d, topk)
        _assert_same(got_idx, got_sc, ref_idx, ref_sc, f"ties k={topk}")
    d["weights"] = torch.zeros_like(d["weights"])   # every score 0: the first k positions win
    got_idx, _ = _gpu_indexer(d, 50)
    assert np.array_equal(got_idx, np.tile(np.arange(50, dtype=np.int32), (4, 1)))


@pytest.mark.parametrize("n_tied,topk", [(40, 30), (150, 100), (300, 200), (150, 150)])
def test_tied_top_group_every_selection_path(n_tied, topk):
    """The top `n_tied` scores of each row are exactly equal (identical key
    rows) and the k-th largest lies among them: the register top-k then
    ranks up to 64 survivors with ballots, up to 256 pairwise, and more
    takes two further radix passes.  Every path must take the lowest
    positions of the tie."""
    g = torch.Generator().manual_seed(n_tied)
    T, Hi, S = 3, 16, 4096
    q = torch.ones(T, Hi, 128)
    k = torch.randn(S, 128, generator=g)
    k[:n_tied] = 2.0                                   # dot = 256 against ~N(0, 11)
    perm = torch.randperm(S, generator=g)             # spread the tied rows over the row
    k = k[perm]
    d = {"q_idx": workloads.e4m3(q), "k_idx": workloads.e4m3(k),
         "k_scale": torch.ones(S), "weights": torch.full((T, Hi), 1.0 / Hi),
         "causal_limit": torch.tensor([S - 1, S - 7, S - 1000], dtype=torch.int32)}
    got_idx, got_sc = _gpu_indexer(d, topk)
    ref_idx, ref_sc = _oracle(d, topk)
    _assert_same(got_idx, got_sc, ref_idx, ref_sc, f"tied group {n_tied}, k={topk}")
    tied_pos = np.sort(np.flatnonzero(np.isin(perm.numpy(), np.arange(n_tied))))
    for t in range(T):
        n = int(d["causal_limit"][t]) + 1
        want = tied_pos[tied_pos < n][:topk]           # the lowest tied positions win
        assert np.isin(want, got_idx[t]).all(), f"row {t}"
        if len(want) == topk:
            assert np.array_equal(got_idx[t], want), f"row {t}"


@pytest.mark.parametrize("topk", [1, 64, 1000])
def test_outlier_scores_crowd_the_linear_bins(topk):
    """A few huge scores stretch the row's score range, so the top-k's
    histogram of 2048 bins linear in the score puts nearly every key in a
    handful of bins and the k-th largest's bin is crowded: the selection
    must fall back to its radix passes and stay exact (rows 0-1); row 2 has
    an ordinary spread."""
    g = torch.Generator().manual_seed(71)
    T, Hi, S = 3, 16, 6000
    q = torch.ones(T, Hi, 128)
    q[2] = torch.randn(Hi, 128, generator=g)
    k = torch.randn(S, 128, generator=g)
    k[[17, 4000, 5999]] = 400.0                        # dot ~ 51200 against ~N(0, 11)
    d = {"q_idx": workloads.e4m3(q), "k_idx": workloads.e4m3(k),
         "k_scale": torch.ones(S), "weights": torch.full((T, Hi), 1.0 / Hi),
         "causal_limit": torch.tensor([S - 1, S - 2, S - 1], dtype=torch.int32)}
    print(f"outlier scores k={topk}", flush=True)
    got_idx, got_sc = _gpu_indexer(d, topk)
    ref_idx, ref_sc = _oracle(d, topk)
    _assert_same(got_idx, got_sc, ref_idx, ref_sc, f"outliers k={topk}")


def test_large_values_take_the_wide_paths():
    """|value| >= 32 needs the third 7-bit piece (fp64 combine), and large
    dots overflow the int32 fast combine; both must stay exact."""
    g = torch.Generator().manual_seed(11)
    T, Hi, S = 3, 16, 400
    q = (torch.randn(T, Hi, 128, generator=g) * 40).clamp(-440, 440)
    k = (torch.randn(S, 128, generator=g) * 40).clamp(-440, 440)
    q[0] = 1.0                                   # a token with only small values
    d = {"q_idx": workloads.e4m3(q), "k_idx": workloads.e4m3(k),
         "k_scale": torch.rand(S, generator=g) + 0.5,
         "weights": torch.randn(T, Hi, generator=g),
         "causal_limit": torch.tensor([S - 1, S - 50, 10], dtype=torch.int32)}
    got_idx, got_sc = _gpu_indexer(d, 128)
    ref_idx, ref_sc = _oracle(d, 128)
    _assert_same(got_idx, got_sc, ref_idx, ref_sc, "large values")
    # moderate values: no third piece, but products beyond the int32 fast path
    d2 = dict(d, q_idx=workloads.e4m3((q / 2).clamp(-31, 31)), k_idx=workloads.e4m3((k / 2).clamp(-31, 31)))
    got_idx, got_sc = _gpu_indexer(d2, 128)
    ref_idx, ref_sc = _oracle(d2, 128)
    _assert_same(got_idx, got_sc, ref_idx, ref_sc, "moderate values")


def test_short_rows_pad_with_minus_one():
    d = workloads.indexer_inputs(T=4, Hi=16, S=256, seed=3)
    d["causal_limit"] = torch.tensor([-1, 0, 9, 255], dtype=torch.int32)
    got_idx, got_sc = _gpu_indexer(d, 20)
    ref_idx, ref_sc = _oracle(d, 20)
    _assert_same(got_idx, got_sc, ref_idx, ref_sc, "short rows")
    assert (got_idx[0] == -1).all() and (got_idx[1][1:] == -1).all() and got_idx[1][0] == 0
    assert (got_idx[2][10:] == -1).all()


def test_block_table_maps_positions_to_slots():
    d = workloads.indexer_inputs(T=6, Hi=32, S=1024, seed=5)
    shared = torch.randperm(16, generator=torch.Generator().manual_seed(1)).to(torch.int32)
    per_tok = torch.stack([torch.randperm(16, generator=torch.Generator().manual_seed(t))
                           for t in range(6)]).to(torch.int32)
    ref_idx, _ = _oracle(d, 100)
    for bt in (shared, per_tok):
        got, _ = _gpu_indexer(d, 100, block_table=bt, page_size=64)
        for t in range(6):
            row = bt if bt.dim() == 1 else bt[t]
            want = workloads.positions_to_slots(torch.from_numpy(ref_idx[t]).long(), row, 64).numpy()
            assert np.array_equal(np.sort(got[t]), np.sort(want))


def test_cfg5_pipeline_end_to_end():
    d = workloads.cfg5()
    g = workloads.to_device(d, DEV)
    out, lse, slots = run_sparse_attention_pipeline(
        g["q_idx"], g["k_idx"], g["k_scale"], g["weights"], g["causal_limit"], g["block_table"],
        g["q_nope"], g["q_pe"], g["ckv_cache"], g["kpe_cache"], d["sm_scale"], topk=2048)
    torch.cuda.synchronize()
    ref_pos, _ = _oracle(d, 2048)
    ref_slots = workloads.positions_to_slots(torch.from_numpy(ref_pos).long(), d["block_table"], 64)
    got_slots = slots.cpu()
    for t in range(got_slots.shape[0]):
        assert torch.equal(torch.sort(got_slots[t]).values, torch.sort(ref_slots[t]).values)

    def bits(x):
        return x.contiguous().view(torch.int16).numpy().view(np.uint16)

    ref_out, ref_lse = oracle.attention(bits(d["q_nope"]), bits(d["q_pe"]), bits(d["ckv_cache"]),
                                        bits(d["kpe_cache"]), ref_slots.numpy(), d["sm_scale"],
                                        NTHREADS)
    assert mismatches(out.float().cpu().numpy(), oracle.bf16_bits_to_f32(ref_out), OUT_ATOL, OUT_RTOL) == 0
    assert mismatches(lse.cpu().numpy(), ref_lse, LSE_ATOL, LSE_RTOL) == 0


@pytest.mark.parametrize("T,Hi,S,topk", [(8, 64, 5000, 2048), (33, 48, 513, 17), (2, 16, 50000, 700),
                                         (2, 16, 70000, 700), (3, 64, 9000, 300)])
def test_after_nan_filled_lds(T, Hi, S, topk):
    """Scores and selections (register top-k of 16 and 64 keys per thread,
    the streaming top-k, rows shorter than top-k) right after a kernel that
    left NaN in every CU's LDS: every LDS location the indexer kernels read
    was written by them first, or the scores and sets would differ."""
    d = workloads.indexer_inputs(T=T, Hi=Hi, S=S, seed=9100 + S)
    ref_idx, ref_sc = _oracle(d, topk)
    for r in range(3):
        print(f"NaN-filled LDS indexer T={T} Hi={Hi} S={S} topk={topk} call {r}", flush=True)
        got_idx, got_sc = _gpu_indexer(d, topk, nan_lds=True)
        _assert_same(got_idx, got_sc, ref_idx, ref_sc, f"T={T} S={S} call {r}")


@pytest.mark.parametrize("S", [12000, 50000, 70000])
def test_long_rows_every_topk_variant(S):
    """Rows of 12000 / 50000 positions use the register top-k with 16 / 64
    keys per thread; 70000 positions the streaming top-k."""
    d = workloads.indexer_inputs(T=2, Hi=16, S=S, seed=S)
    d["causal_limit"] = torch.tensor([S - 1, S // 2], dtype=torch.int32)
    got_idx, got_sc = _gpu_indexer(d, 700)
    ref_idx, ref_sc = _oracle(d, 700)
    _assert_same(got_idx, got_sc, ref_idx, ref_sc, f"S={S}")


@pytest.mark.parametrize("S", [3000, 40000])
def test_causal_limit_extremes(S):
    """Limits at the ends of int32 (INT32_MAX: no limit; INT32_MIN: no
    candidate), around S and around 0, in the register top-k (S=3000) and the
    streaming one (S=40000), against the oracle (int64 limits)."""
    lims = [2**31 - 1, -2**31, S - 1, S, S - 2, -1, 0, 1]
    d = workloads.indexer_inputs(T=len(lims), Hi=16, S=S, seed=7 + S)
    d["causal_limit"] = torch.tensor(lims, dtype=torch.int32)
    print(f"causal limit extremes S={S}", flush=True)
    got_idx, got_sc = _gpu_indexer(d, 300)
    ref_idx, ref_sc = _oracle(d, 300)
    _assert_same(got_idx, got_sc, ref_idx, ref_sc, f"limit extremes S={S}")
    assert (got_idx[0] >= 0).all() and (got_idx[1] == -1).all()


def test_graph_replays_match_eager():
    d = workloads.indexer_inputs(T=8, Hi=64, S=5000, seed=21)
    g = workloads.to_device(d, DEV)
    args = (g["q_idx"], g["k_idx"], g["k_scale"], g["weights"], g["causal_limit"])
    eager = run_indexer_and_topk(*args, 256).clone()
    s = torch.cuda.Stream()
    s.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(s):
        run_indexer_and_topk(*args, 256)
    torch.cuda.current_stream().wait_stream(s)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = run_indexer_and_topk(*args, 256)
    for _ in range(3):
        out.fill_(-7)
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, eager)
        run_indexer_and_topk(*args, 100)   # eager work between replays
        torch.cuda.synchronize()


# ---- paged fp8 K cache ---------------------------------------------------

def _bf16_rows(g, n):
    """bf16 rows with a spread of magnitudes, a zero row, -0.0 and tiny rows."""
    k = torch.randn(n, 128, generator=g) * torch.exp2(torch.randint(-12, 12, (n, 1), generator=g).float())
    k[0] = 0.0
    k[1, 7] = -0.0
    k[2] *= 1e-30                                   # amax below the 1e-4 floor
    k[3, :64] = 3e4                                  # large, many equal magnitudes
    return k.to(torch.bfloat16)


def test_k_append_matches_oracle_bit_exact():
    """Quantise-on-append writes exactly the oracle's codes and fp32 scales to
    each slot's place in the page layout and leaves every other byte alone
    (negative and out-of-range slots are skipped)."""
    from dsa_amd import k_append
    g = torch.Generator().manual_seed(41)
    ps, pages, n = 64, 40, 1500
    k = _bf16_rows(g, n)
    slots = torch.randperm(pages * ps, generator=g)[:n].to(torch.int32)
    slots[10] = -1
    slots[11] = pages * ps + 5
    base = torch.randint(0, 256, (pages, ps * 132), generator=g, dtype=torch.uint8)
    cache = base.to(DEV)
    print("k_append n=1500 pages=40 ps=64", flush=True)
    k_append(k.to(DEV), slots.to(DEV), cache)
    torch.cuda.synchronize()
    codes, scale = oracle.quantize_k(k.float().numpy())
    want = oracle.pack_k_cache(base.numpy(), codes, scale, slots.numpy(), ps)
    got = cache.cpu().numpy()
    bad = np.flatnonzero(got != want)
    assert bad.size == 0, f"{bad.size} bytes differ, first at {np.unravel_index(bad[0], got.shape)}"
    # strided rows (a view of a wider tensor) give the same bytes
    wide = torch.zeros(n, 256, dtype=torch.bfloat16)
    wide[:, 64:192] = k
    cache2 = base.to(DEV)
    k_append(wide.to(DEV)[:, 64:192], slots.to(DEV), cache2)
    torch.cuda.synchronize()
    assert torch.equal(cache2.cpu(), cache.cpu())


def test_paged_indexer_equals_flat_bit_for_bit():
    """The indexer over a paged K cache (pages in a random order, appended by
    k_append) returns the same scores and slots as the flat call over the
    same codes and scales."""
    from dsa_amd import k_append, new_k_cache, run_indexer_and_topk_paged
    g = torch.Generator().manual_seed(42)
    T, Hi, S, ps, topk = 12, 64, 6000, 64, 512
    d = workloads.indexer_inputs(T=T, Hi=Hi, S=S, seed=43)
    k = torch.randn(S, 128, generator=g).to(torch.bfloat16)
    n_pages = -(-S // ps) + 3
    page_of = torch.randperm(n_pages, generator=g)[:-(-S // ps)].to(torch.int32)  # position page -> cache page
    pos = torch.arange(S)
    slots = (page_of[pos // ps] * ps + pos % ps).to(torch.int32)
    cache = new_k_cache(n_pages, ps, DEV)
    k_append(k.to(DEV), slots.to(DEV), cache)
    codes, scale = oracle.quantize_k(k.float().numpy())
    flat = dict(d, k_idx=torch.from_numpy(codes), k_scale=torch.from_numpy(scale))
    ref_idx, ref_sc = _gpu_indexer(flat, topk)
    gd = workloads.to_device(d, DEV)
    out, sc = run_indexer_and_topk_paged(gd["q_idx"], cache, page_of.to(DEV), S, gd["weights"],
                                         gd["causal_limit"], topk, return_scores=True)
    torch.cuda.synchronize()
    assert np.array_equal(sc.cpu().numpy().view(np.uint32), ref_sc.view(np.uint32))
    assert np.array_equal(out.cpu().numpy(), ref_idx)
    ora_idx, ora_sc = _oracle(flat, topk)
    _assert_same(ref_idx, ref_sc, ora_idx, ora_sc, "flat over the quantised K")


def test_pipeline_over_paged_k_cache_equals_flat():
    """cfg5's indexer K packed into a paged cache that shares the attention's
    block table: the pipeline gives the same slots, output and lse as over the
    flat K."""
    d = workloads.cfg5()
    g = workloads.to_device(d, DEV)
    ps = 64
    S = d["k_idx"].shape[0]
    bt = d["block_table"]
    assert bt.dim() == 1
    pos = torch.arange(S)
    slots = (bt[pos // ps].long() * ps + pos % ps).numpy()
    base = np.zeros((bt.numel(), ps * 132), np.uint8)
    cache = oracle.pack_k_cache(base, d["k_idx"].view(torch.uint8).numpy(), d["k_scale"].numpy(),
                                slots, ps)
    args = (g["q_nope"], g["q_pe"], g["ckv_cache"], g["kpe_cache"], d["sm_scale"])
    flat = run_sparse_attention_pipeline(g["q_idx"], g["k_idx"], g["k_scale"], g["weights"],
                                         g["causal_limit"], g["block_table"], *args, topk=2048)
    paged = run_sparse_attention_pipeline(g["q_idx"], None, None, g["weights"], g["causal_limit"],
                                          g["block_table"], *args, topk=2048,
                                          k_cache=torch.from_numpy(cache).to(DEV), num_positions=S)
    torch.cuda.synchronize()
    for a, b in zip(flat, paged):
        assert torch.equal(a, b)


def test_paged_indexer_unmapped_pages_read_as_zero_rows():
    """k_pages entries outside [0, pages) (a -1 or a stale id) read as zero
    codes with scale 0 -- score 0 -- and nothing outside the cache is read:
    the result equals the flat call with those positions zeroed."""
    from dsa_amd import k_append, new_k_cache, run_indexer_and_topk_paged
    g = torch.Generator().manual_seed(52)
    T, Hi, S, ps, topk = 6, 32, 1000, 64, 200
    d = workloads.indexer_inputs(T=T, Hi=Hi, S=S, seed=53)
    n_pages = -(-S // ps)
    k = torch.randn(S, 128, generator=g).to(torch.bfloat16)
    page_of = torch.arange(n_pages, dtype=torch.int32)
    cache = new_k_cache(n_pages, ps, DEV)
    pos = torch.arange(S)
    k_append(k.to(DEV), (page_of[pos // ps] * ps + pos % ps).to(torch.int32).to(DEV), cache)
    page_of[2] = -1
    page_of[5] = n_pages + 3
    page_of[7] = 2**31 - 1
    codes, scale = oracle.quantize_k(k.float().numpy())
    for pg in (2, 5, 7):
        codes[pg * ps:(pg + 1) * ps] = 0
        scale[pg * ps:(pg + 1) * ps] = 0.0
    flat = dict(d, k_idx=torch.from_numpy(codes), k_scale=torch.from_numpy(scale))
    ref_idx, ref_sc = _gpu_indexer(flat, topk)
    gd = workloads.to_device(d, DEV)
    print("paged indexer with unmapped pages", flush=True)
    out, sc = run_indexer_and_topk_paged(gd["q_idx"], cache, page_of.to(DEV), S, gd["weights"],
                                         gd["causal_limit"], topk, return_scores=True)
    torch.cuda.synchronize()
    assert np.array_equal(sc.cpu().numpy().view(np.uint32), ref_sc.view(np.uint32))
    assert np.array_equal(out.cpu().numpy(), ref_idx)
    ora_idx, ora_sc = _oracle(flat, topk)
    _assert_same(ref_idx, ref_sc, ora_idx, ora_sc, "flat with zeroed pages")


# ---- prepared K planes ---------------------------------------------------

def test_prepared_planes_give_the_same_bits():
    """Calls reading planes from prepare_k (capacity above the sequence
    length, the K tensors not passed) return the scores and sets of calls
    that prepare K themselves, and those match the oracle; one planes object
    serves several calls."""
    from dsa_amd import prepare_k
    d = workloads.cfg5()
    g = workloads.to_device(d, DEV)
    print("prepared planes cfg5", flush=True)
    planes = prepare_k(g["k_idx"], g["k_scale"], capacity=40000)
    assert planes.num_positions == d["k_idx"].shape[0]
    args = (g["q_idx"], g["k_idx"], g["k_scale"], g["weights"], g["causal_limit"])
    ref, ref_sc = run_indexer_and_topk(*args, 2048, return_scores=True)
    for topk in (2048, 77):
        out, sc = run_indexer_and_topk(g["q_idx"], None, None, g["weights"], g["causal_limit"],
                                       topk, return_scores=True, k_planes=planes)
        torch.cuda.synchronize()
        assert torch.equal(sc.view(torch.int32), ref_sc.view(torch.int32))
        if topk == 2048:
            assert torch.equal(out, ref)
    ora_idx, ora_sc = _oracle(d, 2048)
    _assert_same(ref.cpu().numpy(), ref_sc.cpu().numpy(), ora_idx, ora_sc, "cfg5 with planes")
    # the pipeline with planes gives the same slots, output and lse
    a = (g["q_nope"], g["q_pe"], g["ckv_cache"], g["kpe_cache"], d["sm_scale"])
    p1 = run_sparse_attention_pipeline(*args, g["block_table"], *a, topk=2048)
    p2 = run_sparse_attention_pipeline(g["q_idx"], None, None, g["weights"], g["causal_limit"],
                                       g["block_table"], *a, topk=2048, k_planes=planes)
    torch.cuda.synchronize()
    for x, y in zip(p1, p2):
        assert torch.equal(x, y)


def test_planes_refreshed_after_appends_match_a_full_preparation():
    """A paged K cache grows by appends of uneven lengths (some ending inside
    a 16-position block); after each append only the appended positions are
    re-prepared.  The planes then equal a full preparation byte for byte and
    the indexer over them equals the paged call without planes."""
    from dsa_amd import KPlanes, k_append, new_k_cache, prepare_k_paged, run_indexer_and_topk_paged
    gen = torch.Generator().manual_seed(61)
    T, Hi, ps, topk = 8, 64, 64, 300
    S_max = 3000
    n_pages = -(-S_max // ps) + 2
    page_of = torch.randperm(n_pages, generator=gen).to(torch.int32)
    k = torch.randn(S_max, 128, generator=gen).to(torch.bfloat16)
    pos = torch.arange(S_max)
    slots = (page_of[pos // ps].long() * ps + pos % ps).to(torch.int32)
    cache = new_k_cache(n_pages, ps, DEV)
    pages = page_of.to(DEV)
    planes = KPlanes(S_max, DEV)
    S = 0
    for n in (1000, 7, 9, 16, 1, 500, 1467):
        k_append(k[S:S + n].to(DEV), slots[S:S + n].to(DEV), cache)
        print(f"append {n} at {S}", flush=True)
        prepare_k_paged(cache, pages, S + n, planes=planes, first_position=S)
        S += n
        full = prepare_k_paged(cache, pages, S, capacity=S_max)
        torch.cuda.synchronize()
        # blocks past S hold whatever earlier refreshes left; compare the
        # regions the indexer reads for S positions
        nkb = (S + 15) // 16
        kpb = nkb * 6144
        kmax_off = (((S_max + 15) // 16) * 6144 + 255) // 256 * 256
        cs_off = kmax_off + ((((S_max + 15) // 16) * 4 + 255) // 256 * 256)
        for lo, hi in ((0, kpb), (kmax_off, kmax_off + nkb * 4), (cs_off, cs_off + S * 4)):
            assert torch.equal(planes.buf[lo:hi], full.buf[lo:hi]), (S, lo)
        assert _lib.load().dsa_indexer_k_planes_bytes(S_max) == planes.buf.numel()
        d = workloads.indexer_inputs(T=T, Hi=Hi, S=S, seed=62 + S)
        gd = workloads.to_device(d, DEV)
        ref, ref_sc = run_indexer_and_topk_paged(gd["q_idx"], cache, pages, S, gd["weights"],
                                                 gd["causal_limit"], topk, return_scores=True)
        out, sc = run_indexer_and_topk(gd["q_idx"], None, None, gd["weights"], gd["causal_limit"],
                                       topk, return_scores=True, k_planes=planes)
        torch.cuda.synchronize()
        assert torch.equal(sc.view(torch.int32), ref_sc.view(torch.int32)), S
        assert torch.equal(out, ref), S


def test_planes_in_graph_replays_match_eager():
    from dsa_amd import prepare_k
    d = workloads.indexer_inputs(T=8, Hi=64, S=5000, seed=63)
    g = workloads.to_device(d, DEV)
    planes = prepare_k(g["k_idx"], g["k_scale"])
    args = (g["q_idx"], None, None, g["weights"], g["causal_limit"])
    eager = run_indexer_and_topk(*args, 256, k_planes=planes).clone()
    s = torch.cuda.Stream()
    s.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(s):
        run_indexer_and_topk(*args, 256, k_planes=planes)
    torch.cuda.current_stream().wait_stream(s)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = run_indexer_and_topk(*args, 256, k_planes=planes)
    for _ in range(3):
        out.fill_(-7)
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, eager)


# ---- selection without scores: estimates, exact where they leave it open ---

def _select_both(d, topk, block_table=None):
    """The selection of the call that returns no scores (estimates, and exact
    scores of the positions those leave open) and of the call that computes
    every exact score, whose scores and sets the tests above compare with the
    oracle."""
    g = workloads.to_device(d, DEV)
    args = (g["q_idx"], g["k_idx"], g["k_scale"], g["weights"], g["causal_limit"], topk)
    got = run_indexer_and_topk(*args)
    want, _ = run_indexer_and_topk(*args, return_scores=True)
    torch.cuda.synchronize()
    return got.cpu().numpy(), want.cpu().numpy()


def _full_range(d, g):
    """q and K codes over the whole e4m3 range (rows quantised by their largest
    magnitude, as k_append does)."""
    T, Hi, _ = d["q_idx"].shape
    q, k = torch.randn(T, Hi, 128, generator=g), torch.randn(d["k_idx"].shape[0], 128, generator=g)
    qs, ks = (x.abs().amax(-1, keepdim=True) / 448.0 for x in (q, k))
    return dict(d, q_idx=workloads.e4m3(q / qs), k_idx=workloads.e4m3(k / ks), k_scale=ks[:, 0].contiguous(),
                weights=d["weights"] * qs[..., 0])


# S around the register top-k's sizes and the 16-position blocks, top-k next to 1
# and to the row length, token counts around the pairs and fours of the waves
@pytest.mark.parametrize("T,Hi,S,topk", [(1, 64, 65, 64), (2, 16, 8192, 2048), (3, 32, 8193, 1), (5, 48, 16384, 2048),
                                         (7, 64, 16385, 16000), (9, 64, 32768, 2048), (6, 16, 32751, 2047),
                                         (33, 64, 2049, 2048),
                                         # chunks and their lists: the shortest row, chunk ends inside a
                                         # block, 2 to 9 lists of 1024 to 4096 places, top-k above them
                                         (2, 64, 32769, 2048), (9, 32, 40007, 700), (3, 64, 131071, 2048),
                                         (2, 16, 262144, 2048), (2, 16, 262145, 512), (3, 16, 70000, 3584),
                                         (2, 16, 50000, 9000)])
@pytest.mark.parametrize("full_range", [False, True])
def test_selection_without_scores_matches_oracle(T, Hi, S, topk, full_range):
    gen = torch.Generator().manual_seed(S + T)
    d = workloads.indexer_inputs(T=T, Hi=Hi, S=S, seed=T * 31 + S)
    if full_range:
        d = _full_range(d, gen)
    lim = d["causal_limit"].clone()
    lim[0] = S - 1
    if T > 2:
        lim[1], lim[2] = S // 2, topk  # one candidate more than are taken
    d["causal_limit"] = lim
    print(f"select T={T} Hi={Hi} S={S} k={topk} full_range={full_range}", flush=True)
    got, want = _select_both(d, topk)
    ref, _ = _oracle(d, topk)
    for t in range(T):
        assert np.array_equal(np.sort(got[t]), np.sort(ref[t])), f"row {t} set differs from the oracle"
    assert np.array_equal(got, want)


def _hard(kind, T, Hi, S):
    gen = torch.Generator().manual_seed(len(kind) * 1000 + S)
    d = workloads.indexer_inputs(T=T, Hi=Hi, S=S, seed=17 + S)
    d["causal_limit"] = torch.full((T,), S - 1, dtype=torch.int32)
    k = d["k_idx"].view(torch.float8_e4m3fn).float()
    if kind == "many equal rows":         # more open positions than are ranked
        k = k[torch.randint(0, 3, (S,), generator=gen)]
        d["k_scale"] = torch.ones(S)
    elif kind == "nearly equal rows":     # scores apart by less than the estimate's error
        k = k[:1].expand(S, 128).clone()
        k[torch.arange(S), torch.randint(0, 128, (S,), generator=gen)] = 2.0 ** -9
        d["k_scale"] = 1.0 + torch.arange(S).float()[torch.randperm(S, generator=gen)] * 2.0 ** -23
    elif kind == "outlier rows":
        k[torch.rand(S, generator=gen) < 0.05] *= 8
    elif kind == "outlier scales":
        d["k_scale"][::97] *= 2.0 ** 20
        d["k_scale"][5::97] *= -1.0
    elif kind == "zero rows":
        k[torch.rand(S, generator=gen) < 0.7] = 0.0
    elif kind == "wide exponents":
        k *= torch.exp2(torch.randint(-9, 9, (S, 128), generator=gen).float())
    elif kind == "zero weights":
        d["weights"][::2] = 0.0
    elif kind == "zero queries":
        d["q_idx"] = d["q_idx"].clone()
        d["q_idx"][1::2] = 0
    elif kind == "tiny weights":
        d["weights"] *= 1e-30
        d["weights"][0] *= 1e-12          # subnormal products
    elif kind == "huge weights":
        d["weights"] *= 1e30              # the exact sum overflows
    elif kind == "weights not finite":
        d["weights"][0, 3], d["weights"][1, 0], d["weights"][2, 5] = float("inf"), float("nan"), -float("inf")
    elif kind == "scales not finite":
        d["k_scale"][[3, 700]] = float("inf")
        d["k_scale"][[44, 800]] = float("nan")
        d["k_scale"][[45, 900]] = -float("inf")
    d["k_idx"] = workloads.e4m3(k.clamp(-448, 448))
    if kind == "NaN codes":               # count as zeros in q and k
        d["k_idx"] = d["k_idx"].clone()
        d["k_idx"].view(-1)[torch.randint(0, S * 128, (S * 8,), generator=gen)] = 0x7F
        d["k_idx"][100:200, 5] = 0xFF
        d["q_idx"] = d["q_idx"].clone()
        d["q_idx"][:, ::3, 7] = 0xFF
    return d


@pytest.mark.parametrize("S", [6000, 20000, 40000])
@pytest.mark.parametrize("kind", ["many equal rows", "nearly equal rows", "outlier rows", "outlier scales", "zero rows",
                                  "wide exponents", "zero weights", "zero queries", "tiny weights", "huge weights",
                                  "weights not finite", "scales not finite", "NaN codes"])
def test_selection_without_scores_of_hard_rows(kind, S):
    """Rows whose estimates leave many positions open or whose error bound is
    not safe take exact scores for the whole row; codes, weights and scales
    at the ends of their formats."""
    d = _hard(kind, 4, 32, S)
    print(f"hard rows: {kind} S={S}", flush=True)
    for topk in (300, 2048):
        got, want = _select_both(d, topk)
        assert np.array_equal(got, want), kind


# every instantiation of the row kernel and of the list merge
@pytest.mark.parametrize("S,topk", [(3000, 512), (12000, 512), (32768, 512), (40000, 512), (140000, 1500), (262144, 2048)])
def test_padded_batch_rows_take_the_first_positions(S, topk):
    """Rows whose scores are all zero (padded rows of a batch: no weights or no
    queries) tie everywhere, so the first top-k positions win; rows between
    them are ordinary.  The rows' counts of open positions are cleared for a
    second selection only once every wave has read them."""
    T = 24
    d = workloads.indexer_inputs(T=T, Hi=32, S=S, seed=S)
    d["causal_limit"] = torch.full((T,), S - 1, dtype=torch.int32)
    d["weights"][::3] = 0.0
    d["q_idx"] = d["q_idx"].clone()
    d["q_idx"][1::3] = 0
    print(f"padded rows S={S}", flush=True)
    got, want = _select_both(d, topk)
    first = np.arange(topk, dtype=np.int32)
    for t in range(T):
        assert t % 3 == 2 or np.array_equal(got[t], first), t
    assert np.array_equal(got, want)
    g = workloads.to_device(d, DEV)
    for _ in range(5):
        again = run_indexer_and_topk(g["q_idx"], g["k_idx"], g["k_scale"], g["weights"], g["causal_limit"], topk)
        torch.cuda.synchronize()
        assert np.array_equal(again.cpu().numpy(), got)


def _crowded(kind, T, Hi, S):
    """Rows whose k-th score has many close to it."""
    gen = torch.Generator().manual_seed(len(kind) * 77 + S)
    d = workloads.indexer_inputs(T=T, Hi=Hi, S=S, seed=23 + S)
    d["causal_limit"] = torch.full((T,), S - 1, dtype=torch.int32)
    d["causal_limit"][-1] = S - 37
    shared = torch.randn(128, generator=gen)
    shared *= 128 ** 0.5 / shared.norm()
    q, k = torch.randn(T, Hi, 128, generator=gen), torch.randn(S, 128, generator=gen)
    w, scale = d["weights"].abs(), torch.ones(S)
    if kind.startswith("shared component"):   # one bin of the estimates holds hundreds to thousands
        q, k = q + 4 * shared, k + 4 * shared
        scale = 1.0 + 0.2 * torch.rand(S, generator=gen)
    elif kind == "no positive dot":           # every score 0, the estimates' bound is not
        q, k = q - 2 * shared, k + 2 * shared
    elif kind == "few positive dots":         # fewer positive scores than are selected
        q, k = q - 2 * shared, k + 2 * shared
        k[::50] *= -1
    elif kind == "a third one same row":
        same = torch.rand(S, generator=gen) < 0.33
        k[same] = k[0].clone()
        q[0] = q[0] * 0.2 + k[0]              # the same rows score high for one token
    if kind.endswith("full range"):
        qs, ks = (x.abs().amax(-1, keepdim=True) / 448.0 for x in (q, k))
        q, k, w, scale = q / qs, k / ks, w * qs[..., 0], scale * ks[:, 0]
    d.update(q_idx=workloads.e4m3(q), k_idx=workloads.e4m3(k), weights=w.contiguous(), k_scale=scale.contiguous())
    return d


CROWDED = ["shared component", "shared component, full range", "no positive dot", "few positive dots",
           "a third one same row"]


# every instantiation of the row kernel and of the list merge, lists that fit and that do not
@pytest.mark.parametrize("S,topk", [(6000, 300), (16000, 2048), (32768, 2048), (40000, 700), (140000, 1500),
                                    (262144, 2048)])
@pytest.mark.parametrize("kind", CROWDED)
def test_selection_without_scores_of_crowded_rows(kind, S, topk):
    d = _crowded(kind, 4, 64, S)
    print(f"crowded rows: {kind} S={S} k={topk}", flush=True)
    got, want = _select_both(d, topk)
    assert np.array_equal(got, want), kind


# a row in registers of each size, and in chunks and their lists
@pytest.mark.parametrize("S", [8000, 16000, 32768, 40000])
def test_selection_with_every_length_of_the_open_list(S):
    """Lists of open positions at the lengths where the selection goes another
    way: scored as they are up to 128, narrowed by ranking up to 256 (rows past
    8192 positions), by two more radix passes past that.  The top-k is chosen by how many scores share
    the 16-bit bin of the k-th."""
    d = _crowded("shared component", 1, 64, S)
    d["causal_limit"][:] = S - 1
    g = workloads.to_device(d, DEV)
    args = (g["q_idx"], g["k_idx"], g["k_scale"], g["weights"], g["causal_limit"])
    scores = run_indexer_and_topk(*args, 1, return_scores=True)[1].cpu().numpy()[0]
    desc = np.sort(scores)[::-1]
    assert desc[0] > 0
    bins, count = np.unique(desc.view(np.uint32) >> 16, return_counts=True)
    size = dict(zip(bins.tolist(), count.tolist()))
    share = np.array([size[b] for b in (desc.view(np.uint32) >> 16).tolist()])  # of the k-th score's bin
    taken = 0
    for lo, hi in ((1, 64), (65, 110), (135, 190), (190, 250), (262, 400), (400, 505), (520, 100000)):
        at = np.nonzero((share[:9000] >= lo) & (share[:9000] <= hi) & (desc[:9000] > 0))[0]
        for k in sorted({int(x) + 1 for x in (at[:1].tolist() + at[at.size // 2:at.size // 2 + 1].tolist() + at[-1:].tolist())}):
            print(f"open list S={S} k={k} bin {share[k - 1]}", flush=True)
            got = run_indexer_and_topk(*args, k).cpu().numpy()
            want = run_indexer_and_topk(*args, k, return_scores=True)[0].cpu().numpy()
            assert np.array_equal(got, want), (k, share[k - 1])
            taken += 1
    assert taken >= 12


def test_crowded_rows_cost_about_what_ordinary_ones_do():
    """Scores that share a large mean put hundreds of positions into the k-th
    one's bin, few of them within the estimates' bound of it: 64 rows take
    1.1 to 1.2 times an ordinary call (26 times when each such row's positions
    were all scored exactly by one workgroup)."""
    T, S, topk = 64, 32768, 2048
    times = {}
    for kind in ("ordinary", "shared component, full range"):
        d = _crowded(kind, T, 64, S)
        g = workloads.to_device(d, DEV)
        args = (g["q_idx"], g["k_idx"], g["k_scale"], g["weights"], g["causal_limit"], topk)
        for _ in range(5):
            run_indexer_and_topk(*args)
        best = math.inf
        for _ in range(10):
            a, b = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            a.record()
            for _ in range(10):
                run_indexer_and_topk(*args)
            b.record()
            torch.cuda.synchronize()
            best = min(best, a.elapsed_time(b) * 100)
        times[kind] = best
        print(f"{kind}: {best:.1f} us", flush=True)
    slow, fast = times["shared component, full range"], times["ordinary"]
    assert slow < 3 * fast, times


@pytest.mark.parametrize("T", [4, 9])  # K prepared by the estimate kernel, and before it
@pytest.mark.parametrize("S", [3000, 40000])
def test_selection_without_scores_of_subnormal_scales(T, S):
    """c_s = fl32(k_scale * 2^-18) is 0 or a few units of the smallest subnormal:
    every score is 0 and the first positions win, or scores differ only by
    that rounding."""
    d = workloads.indexer_inputs(T=T, Hi=32, S=S, seed=S + T)
    d["causal_limit"] = torch.full((T,), S - 1, dtype=torch.int32)
    scale = d["k_scale"]
    for name, k_scale in (("all zero", torch.full((S,), 1e-41)), ("spread", scale * 1e-41),
                          ("rounded", scale * 2.0 ** -130), ("among others", torch.where(scale > 1.5, scale, 1e-41))):
        print(f"subnormal scales: {name} T={T} S={S}", flush=True)
        got, want = _select_both(dict(d, k_scale=k_scale.float()), 300)
        assert np.array_equal(got, want), name
        if name in ("all zero", "spread"):
            assert np.array_equal(got, np.tile(np.arange(300, dtype=np.int32), (T, 1))), name


HARD = ["many equal rows", "nearly equal rows", "outlier rows", "outlier scales", "zero rows", "wide exponents",
        "zero weights", "zero queries", "tiny weights", "huge weights", "weights not finite", "scales not finite",
        "NaN codes"]


# K prepared on the estimate kernel's way (up to 8 tokens; a paged cache's long
# rows up to 4) and by its own kernel; rows in registers and in chunks; cache
# pages that end inside a 16-position block, or lie on one
@pytest.mark.parametrize("T,S,page", [(4, 7001, 20), (9, 7001, 64), (4, 40003, 64), (8, 40003, 64), (9, 40003, 12)])
@pytest.mark.parametrize("kind", HARD + CROWDED)
def test_selection_without_scores_over_every_k_source(kind, T, S, page):
    """Flat, paged and planes calls take the positions of the call that returns
    scores, for hard and crowded rows, with some pages unmapped (-1, ids past
    the cache): their positions are zero rows of scale 0."""
    from dsa_amd import prepare_k, prepare_k_paged, run_indexer_and_topk_paged
    d = (_hard if kind in HARD else _crowded)(kind, T, 64 if T == 9 else 32, S)
    gen = torch.Generator().manual_seed(S + page)
    n_pages = -(-S // page)
    page_of = torch.randperm(n_pages, generator=gen).to(torch.int32)
    pos = torch.arange(S)
    codes = torch.zeros(n_pages, page, 128, dtype=torch.uint8)
    scale = torch.zeros(n_pages, page)
    codes[page_of[pos // page].long(), pos % page] = d["k_idx"].view(torch.uint8)
    scale[page_of[pos // page].long(), pos % page] = d["k_scale"].float()
    cache = torch.cat([codes.view(n_pages, -1), scale.view(torch.uint8).view(n_pages, -1)], dim=1).contiguous()
    unmapped = [1, n_pages // 2, n_pages - 1]
    for pg, bad in zip(unmapped, (-1, n_pages, 2 ** 31 - 1)):
        page_of[pg] = bad
    gone = torch.isin(pos // page, torch.tensor(unmapped))
    k, ks = d["k_idx"].view(torch.uint8).clone(), d["k_scale"].float().clone()
    k[gone], ks[gone] = 0, 0.0
    g = workloads.to_device(dict(d, k_idx=k, k_scale=ks), DEV)
    cache, pages = cache.to(DEV).view(n_pages, -1), page_of.to(DEV)
    rest = (g["weights"], g["causal_limit"])
    flat_planes = prepare_k(g["k_idx"], g["k_scale"])
    paged_planes = prepare_k_paged(cache, pages, S)
    for topk in (300, 2048):
        print(f"K sources: {kind} T={T} S={S} page={page} k={topk}", flush=True)
        want, _ = run_indexer_and_topk(g["q_idx"], g["k_idx"], g["k_scale"], *rest, topk, return_scores=True)
        got = {"flat": run_indexer_and_topk(g["q_idx"], g["k_idx"], g["k_scale"], *rest, topk),
               "paged": run_indexer_and_topk_paged(g["q_idx"], cache, pages, S, *rest, topk),
               "planes of flat": run_indexer_and_topk(g["q_idx"], None, None, *rest, topk, k_planes=flat_planes),
               "planes of paged": run_indexer_and_topk(g["q_idx"], None, None, *rest, topk, k_planes=paged_planes)}
        torch.cuda.synchronize()
        for name, x in got.items():
            assert torch.equal(x, want), f"{kind}, {name}, k={topk}"


@pytest.mark.parametrize("Hi", [16, 32, 48, 64])
@pytest.mark.parametrize("T", [1, 2, 5, 8])
def test_paged_selection_without_scores_matches_oracle(T, Hi):
    """The estimate kernel reading a paged cache itself (up to 8 tokens), every
    head count, tokens below and at its pairs and fours, limits inside a page."""
    from dsa_amd import run_indexer_and_topk_paged
    S, ps, topk = 2500 + 100 * T, 64, 600
    d = _full_range(workloads.indexer_inputs(T=T, Hi=Hi, S=S, seed=Hi + T), torch.Generator().manual_seed(Hi * 10 + T))
    lim = torch.randint(topk - 5, S, (T,), generator=torch.Generator().manual_seed(T))
    d["causal_limit"] = lim.to(torch.int32)
    n_pages = -(-S // ps)
    page_of = torch.randperm(n_pages + 3, generator=torch.Generator().manual_seed(S))[:n_pages].to(torch.int32)
    pos = torch.arange(S)
    slots = (page_of[pos // ps].long() * ps + pos % ps).numpy()
    cache = oracle.pack_k_cache(np.zeros((n_pages + 3, ps * 132), np.uint8), d["k_idx"].view(torch.uint8).numpy(),
                                d["k_scale"].numpy(), slots, ps)
    g = workloads.to_device(d, DEV)
    print(f"paged selection T={T} Hi={Hi} S={S}", flush=True)
    got = run_indexer_and_topk_paged(g["q_idx"], torch.from_numpy(cache).to(DEV), page_of.to(DEV), S, g["weights"],
                                     g["causal_limit"], topk)
    torch.cuda.synchronize()
    ref, _ = _oracle(d, topk)
    assert np.array_equal(np.sort(got.cpu().numpy(), axis=1), np.sort(ref, axis=1))


# on both sides of the rule that says whether the estimate kernel prepares K itself
@pytest.mark.parametrize("T,Hi,S", [(2, 64, 32768), (2, 64, 32769), (4, 48, 16384), (4, 48, 16385), (5, 32, 21845),
                                    (6, 16, 21846), (8, 64, 16384), (8, 64, 16385), (7, 48, 16385), (4, 32, 40000)])
def test_selection_without_scores_where_k_is_prepared_ahead(T, Hi, S):
    """The same sets from a flat and a paged cache as from prepared planes."""
    from dsa_amd import prepare_k, run_indexer_and_topk_paged
    page, topk = 64, 1500
    d = _full_range(workloads.indexer_inputs(T=T, Hi=Hi, S=S, seed=Hi + T), torch.Generator().manual_seed(S))
    d["causal_limit"] = torch.arange(S - 40 * T, S, 40, dtype=torch.int32)
    d["causal_limit"][0] = topk + 3
    n_pages = -(-S // page)
    codes, scale = torch.zeros(n_pages * page, 128, dtype=torch.uint8), torch.zeros(n_pages * page)
    codes[:S], scale[:S] = d["k_idx"].view(torch.uint8), d["k_scale"]
    cache = torch.cat([codes.view(n_pages, -1), scale.view(n_pages, -1).view(torch.uint8)], dim=1).contiguous().to(DEV)
    pages = torch.arange(n_pages, dtype=torch.int32, device=DEV)
    g = workloads.to_device(d, DEV)
    rest = (g["weights"], g["causal_limit"], topk)
    print(f"K prepared ahead T={T} Hi={Hi} S={S}", flush=True)
    want = run_indexer_and_topk(g["q_idx"], None, None, *rest, k_planes=prepare_k(g["k_idx"], g["k_scale"]))
    flat = run_indexer_and_topk(g["q_idx"], g["k_idx"], g["k_scale"], *rest)
    paged = run_indexer_and_topk_paged(g["q_idx"], cache, pages, S, *rest)
    exact = run_indexer_and_topk(g["q_idx"], g["k_idx"], g["k_scale"], *rest, return_scores=True)[0]
    torch.cuda.synchronize()
    for name, x in (("flat", flat), ("paged", paged), ("exact", exact)):
        assert torch.equal(x, want), name


def _estimates(q, k, k_scale, w, topk):
    """What a call without scores leaves in its workspace: a row's estimates (its
    last T x S floats), except where exact scores took their place, which only
    rows with more than 512 positions close to the k-th have."""
    q, k, k_scale, w = (x.to(DEV).contiguous() for x in (q, k, k_scale, w))
    T, Hi, _ = q.shape
    S = k.shape[0]
    lim = torch.full((T,), S - 1, dtype=torch.int32, device=DEV)
    lib = _lib.load()
    n = lib.dsa_indexer_workspace_bytes(T, Hi, 128, S)
    ws = torch.zeros(n, dtype=torch.uint8, device=DEV)
    out = torch.empty((T, topk), dtype=torch.int32, device=DEV)
    a = _lib.IndexerArgs()
    a.q_idx, a.k_idx, a.k_scale, a.weights = q.data_ptr(), k.data_ptr(), k_scale.data_ptr(), w.data_ptr()
    a.causal_limit, a.out = lim.data_ptr(), out.data_ptr()
    a.num_tokens, a.num_heads, a.head_dim, a.num_positions, a.topk = T, Hi, 128, S, topk
    a.workspace, a.workspace_bytes = ws.data_ptr(), n
    _lib.check("dsa_indexer_topk",
               lib.dsa_indexer_topk(ctypes.byref(a), torch.cuda.current_stream().cuda_stream))
    torch.cuda.synchronize()
    first = n - (T * S * 4 + 255) // 256 * 256
    return ws[first:first + T * S * 4].view(torch.float32).view(T, S).double().cpu()


@pytest.mark.parametrize("T", [8, 16])  # K prepared by the estimate kernel, and before it
@pytest.mark.parametrize("at", [0, 7, 8, 40, 127])
def test_estimated_dots_of_directed_codes_stay_within_their_share_of_the_bound(T, at):
    """One large product at dim `at` beside 127 of every magnitude and sign: the
    sums' losses add up.  One head has weight 1, so an estimate is a dot.  16
    sums truncated to 24 bits lose at most 16 x 2^-23 of |q| |k|; the bound
    allows 2^-17."""
    levels = [2.0 ** e * (1 + m / 8) for e in range(-9, 9) for m in range(8) if 2.0 ** e * (1 + m / 8) <= 448]
    rows = []
    for big in (448.0, 416.0, 256.0, 288.0):
        for v in levels:
            for pattern in range(3):
                r = torch.full((128,), v if pattern != 1 else -v)
                if pattern == 2:
                    r[1::2] *= -1
                r[at] = big
                rows.append(r)
    top = torch.zeros(20, 128)      # the selected rows lie far above: the others are not near the k-th
    top[:, at] = 448.0
    k = workloads.e4m3(torch.cat([top, torch.stack(rows)]))
    k_scale = torch.ones(len(k))
    k_scale[:20] = 8.0
    w = torch.zeros(T, 16)
    w[torch.arange(T), torch.arange(T)] = 1.0
    worst = 0.0
    for small in (2.0 ** -9, 2.0 ** -6, 2.0 ** -4, 0.25, 1.0, 4.0):
        q = torch.zeros(T, 16, 128)
        for t in range(T):
            q[t, t] = small * (1 + (t % 8) / 8)
            q[t, t, at] = (448.0, 416.0, 384.0, 320.0, 256.0, 288.0, 352.0, 240.0)[t % 8]
        q = workloads.e4m3(q)
        est = _estimates(q, k, k_scale, w, 10)[:, 20:]
        qv = q.view(torch.float8_e4m3fn).double()[torch.arange(T), torch.arange(T)]
        kv = k.view(torch.float8_e4m3fn).double()[20:]
        err = (est - (qv @ kv.t()).clamp_min(0.0)).abs() / (qv.norm(dim=1)[:, None] * kv.norm(dim=1)[None])
        worst = max(worst, float(err.max()))
    print(f"largest loss at dim {at}, T={T}: 2^{math.log2(worst):.2f}", flush=True)
    assert worst <= 16 * 2.0 ** -23


@pytest.mark.parametrize("full_range", [False, True])
def test_estimates_of_ordinary_rows_stay_within_the_bound(full_range):
    T, Hi, S = 12, 64, 5000
    d = workloads.indexer_inputs(T=T, Hi=Hi, S=S, seed=404)
    if full_range:
        d = _full_range(d, torch.Generator().manual_seed(405))
    d["causal_limit"] = torch.full((T,), S - 1, dtype=torch.int32)
    est = _estimates(d["q_idx"], d["k_idx"], d["k_scale"], d["weights"], 300)
    g = workloads.to_device(d, DEV)
    _, sc = run_indexer_and_topk(g["q_idx"], g["k_idx"], g["k_scale"], g["weights"], g["causal_limit"], 300,
                                 return_scores=True)
    torch.cuda.synchronize()
    qn = d["q_idx"].view(torch.float8_e4m3fn).double().norm(dim=2)
    kn = (d["k_idx"].view(torch.float8_e4m3fn).double().norm(dim=1) * d["k_scale"].double().abs()).max()
    bound = 1.328125 * 2.0 ** -17 * (d["weights"].double().abs() * qn).sum(1) * kn
    assert ((est - sc.double().cpu()).abs() <= bound[:, None]).all()


def test_selection_without_scores_after_nan_filled_lds():
    for S in (20000, 45000):
        d = _full_range(workloads.indexer_inputs(T=5, Hi=64, S=S, seed=77), torch.Generator().manual_seed(78))
        ref, _ = _oracle(d, 2048)
        g = workloads.to_device(d, DEV)
        for r in range(3):
            fill_lds_with_nan(DEV)
            print(f"NaN-filled LDS selection S={S} call {r}", flush=True)
            out = run_indexer_and_topk(g["q_idx"], g["k_idx"], g["k_scale"], g["weights"], g["causal_limit"], 2048)
            torch.cuda.synchronize()
            assert np.array_equal(np.sort(out.cpu().numpy(), axis=1), np.sort(ref, axis=1))
