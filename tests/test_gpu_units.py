"""The partial kernel that spreads (sequence, split, KV head) units evenly over
the chip (GPU), forced with L20_PD_UNITS=1: output and LSE against the oracle at
the shapes where its schedule can go wrong -- units shared by 8, 4, 2 and 1 waves
(fewer units than waves, parts without blocks), several units per wave (the grid
capped), each with every cache type, pages of 16, 32 and 64 tokens, block tables and
page lists, draft rows and trees over one and two query tiles; lanes holding one and
several sequences, empty and one-token rows, splits that are not whole blocks, odd
head counts -- and the library's choice.  The entry points above it (tree
verification, the hook functions, strided caches, two streams, the allocation-free
entry) run on it in their own tests (PARTIAL_KERNELS).
"""

import zlib

import numpy as np
import pytest
import torch

import pd_helpers as H
from test_gpu_fused_split import _run as _run_call
from test_gpu_random_sweep import draw, run_case

pytestmark = pytest.mark.gpu

PDT = {"fp32": torch.float32, "fp16": torch.float16, "bf16": torch.bfloat16}


@pytest.fixture(autouse=True)
def _units(monkeypatch):
    monkeypatch.setenv("L20_PD_FUSED", "0")
    monkeypatch.setenv("L20_PD_FUSED_SPLIT", "0")
    monkeypatch.setenv("L20_PD_UNITS", "1")


@pytest.fixture
def no_queue():
    """The persistent kernel did not run: no call took a work-queue slot."""
    import l20_pd_cabi as cabi

    before = cabi.queue_launches()
    yield
    assert cabi.queue_launches() == before


@pytest.fixture
def kernels(monkeypatch):
    """The partial kernel of every call made through the C ABI, as the library names it."""
    import l20_pd_cabi as cabi

    ran, split_out = [], cabi.split_out

    def named(args, *rest):
        ran.append(cabi.partial_kernel(args))
        return split_out(args, *rest)

    monkeypatch.setattr(cabi, "split_out", named)
    return ran


def _run(inp, split, pdt, kernels, kernel="pd_units"):
    """One call through the C ABI, on ``kernel``."""
    out, lse, path = _run_call(inp, split, pdt)
    assert path == 0 and kernels[-1] == kernel
    return out, lse


CASES = [
    # name, batch, hq, hkv, d, lens, q_len, per_head, fp8, page, split, pdt, workgroups (0: the CUs)
    ("one_unit", 1, 8, 1, 128, [400], 1, False, "e4m3fn", 16, 512, "fp32", 0),
    ("empty_parts", 2, 8, 2, 128, [1, 90], 1, True, "e4m3fn", 16, 512, "fp32", 0),
    ("ragged_fp16", 5, 28, 4, 128, [1, 15, 1025, 2048, 600], 1, True, "e4m3fn", 16, 512, "fp16", 12),
    ("many_per_wave", 7, 16, 2, 128, [700, 1, 0, 64, 1300, 90, 513], 1, True, "e4m3fn", 16, 64, "fp32", 1),
    ("two_workgroups", 9, 12, 3, 128, [333, 5, 800, 64, 65, 0, 1, 1100, 127], 1, False, "e4m3fn", 16, 128, "bf16", 2),
    ("split80", 4, 8, 2, 128, [900, 81, 80, 79], 1, False, "e4m3fn", 16, 80, "fp32", 3),
    ("split1024", 3, 16, 2, 128, [3000, 1025, 70], 1, True, "e4m3fn", 16, 1024, "fp16", 2),
    ("d64", 6, 14, 2, 64, [1500, 64, 0, 900, 33, 512], 1, False, "e4m3fn", 16, 256, "fp32", 2),
    ("e5m2_pages32", 4, 16, 2, 128, [1, 1333, 2048, 64], 1, True, "e5m2", 32, 512, "fp16", 3),
    ("pages_64", 3, 28, 4, 128, [900, 31, 2500], 1, True, "e4m3fn", 64, 256, "fp16", 2),
    ("verify_2tiles", 5, 64, 8, 128, [1048, 17, 700, 4, 300], 4, False, "e4m3fn", 16, 256, "fp32", 2),
    ("verify_2tiles_p", 2, 64, 8, 128, [1048, 4], 4, False, "e4m3fn", 16, 512, "fp16", 0),
]


@pytest.mark.parametrize("case", CASES, ids=[c[0] for c in CASES])
def test_units_match_oracle(case, monkeypatch, kernels):
    name, batch, hq, hkv, d, lens, q_len, per_head, fp8, page, split, pdt, groups = case
    if groups:
        monkeypatch.setenv("L20_PD_MAX_WORKGROUPS", str(groups))
    inp = H.make_synthetic(batch, hq, hkv, d, lens, q_len=q_len, per_head=per_head, fp8=fp8, page=page,
                           seed=zlib.crc32(name.encode()) % 1000, garbage_tail=True)
    out, lse = _run(inp, split, PDT[pdt], kernels)
    H.compare(out, lse, *H.run_oracle(inp))


def _unit_count(lens, split, hkv):
    return hkv * sum(max(1, -(-x // split)) for x in lens)


def _groups(units, waves, tiles):
    """The smallest grid on which `waves` waves share a unit (at most half of the chip's
    waves with one query tile, all of them with two); 0: one workgroup for all units."""
    fill = 4 if tiles == 1 else 8
    return -(-units * waves // fill) if waves else 1


SHARED = [
    # name, hq, hkv, d, q_len, tree, cache, page, csr
    ("fp8", 8, 2, 128, 1, False, "e4m3fn", 16, False),
    ("fp8_d64", 8, 2, 64, 1, False, "e4m3fn", 32, False),
    ("e5m2_verify", 8, 2, 128, 4, False, "e5m2", 16, False),
    ("fp8_tree", 8, 2, 128, 4, True, "e4m3fn", 16, False),
    ("fp8_tree_2tiles", 16, 2, 128, 4, True, "e4m3fn", 16, False),
    ("fp8_tree_18cols", 12, 2, 128, 3, True, "e4m3fn", 64, False),
    ("e5m2_tree_2tiles_d64", 16, 2, 64, 4, True, "e5m2", 16, False),
    ("fp8_verify_2tiles_d64", 16, 2, 64, 4, False, "e4m3fn", 16, False),
    ("bf16", 8, 2, 128, 1, False, "bf16", 16, False),
    ("bf16_csr_pages32", 8, 2, 128, 1, False, "bf16", 32, True),
    ("fp16_tree_d64", 8, 2, 64, 4, True, "fp16", 64, False),
    ("bf16_tree_2tiles", 16, 2, 128, 4, True, "bf16", 16, False),
    ("fp16_tree_2tiles_csr", 16, 2, 128, 4, True, "fp16", 16, True),
    ("fp16_tree_18cols_d64", 12, 2, 64, 3, True, "fp16", 32, False),
    ("bf16_verify_2tiles_d64", 16, 2, 64, 4, False, "bf16", 64, False),
]


@pytest.mark.parametrize("waves", [8, 4, 2, 1, 0])
@pytest.mark.parametrize("case", SHARED, ids=[c[0] for c in SHARED])
def test_units_shared_by_waves(case, waves, monkeypatch, no_queue):
    """Every kind of call with 8, 4, 2 and 1 waves to a unit, and all units in one
    workgroup; ragged, so that the longest sequence's splits outnumber the others'."""
    name, hq, hkv, d, q_len, tree, cache, page, csr = case
    lens, split = [2000, 30, 545, 8, 64, 7], 512
    tiles = (hq // hkv * q_len + 15) // 16
    monkeypatch.setenv("L20_PD_MAX_WORKGROUPS", str(_groups(_unit_count(lens, split, hkv), waves, tiles)))
    seed = zlib.crc32(name.encode()) % 1000
    fp8 = cache in ("e4m3fn", "e5m2")
    if fp8:
        inp = H.make_synthetic(len(lens), hq, hkv, d, lens, q_len=q_len, per_head=True, fp8=cache, page=page,
                               seed=seed, garbage_tail=True)
    else:
        inp = H.make_synthetic16(len(lens), hq, hkv, d, lens, dtype=torch.float16 if cache == "fp16" else torch.bfloat16,
                                 q_len=q_len, page=page, seed=seed, garbage_tail=True, csr_pad=1)
    if tree:
        w = np.random.default_rng(seed).integers(0, 2**32, size=(len(lens), q_len), dtype=np.int64)
        inp["tree_mask"] = torch.from_numpy(np.where(w >= 2**31, w - 2**32, w).astype(np.int32)).cuda()
    if fp8:
        H.compare(*H.run_op(inp, split), *H.run_oracle(inp))
    else:
        H.compare(*H.run_op16(inp, split, csr=csr), *H.run_oracle16(inp, csr=csr))


@pytest.mark.parametrize("longest", [1, 15, 16, 17, 31, 32, 33, 63, 64, 65, 127, 128, 129])
@pytest.mark.parametrize("case", [SHARED[0], SHARED[4], SHARED[8], SHARED[11]],
                         ids=["fp8", "fp8_tree_2tiles", "bf16", "bf16_tree_2tiles"])
def test_units_shared_no_finer_than_blocks(case, longest, kernels):
    """One short split: the waves of a unit are as many as the longest sequence has whole
    blocks (32 tokens with fp8 caches, 16 with 16-bit ones), on both sides of each step."""
    _, hq, hkv, d, q_len, tree, cache, page, _ = case
    lens = [max(q_len, x) for x in (longest, longest // 2, longest, longest - 1)] * 3
    if cache == "e4m3fn":
        inp = H.make_synthetic(len(lens), hq, hkv, d, lens, q_len=q_len, per_head=True, page=page, seed=longest,
                               garbage_tail=True)
    else:
        inp = H.make_synthetic16(len(lens), hq, hkv, d, lens, dtype=torch.bfloat16, q_len=q_len, page=page,
                                 seed=longest, garbage_tail=True)
    if tree:
        w = np.random.default_rng(longest).integers(0, 2**31, size=(len(lens), q_len), dtype=np.int64)
        inp["tree_mask"] = torch.from_numpy(w.astype(np.int32)).cuda()
    if cache == "e4m3fn":
        (out, lse), (exp, exp_lse) = _run(inp, 512, torch.float32, kernels), H.run_oracle(inp)
    else:
        (out, lse), (exp, exp_lse) = H.run_op16(inp, 512), H.run_oracle16(inp)
    # A row that sees one or two keys is as large as a value row (up to ~5, where half a
    # bf16 step is 0.016): the output's own rounding, 2^-8 of it, is allowed on top.
    err = np.abs(out.float().cpu().numpy() - exp)
    assert (err <= H.OUT_ATOL + np.abs(exp) / 256).all(), err.max()
    np.testing.assert_allclose(lse.cpu().numpy(), exp_lse, rtol=H.LSE_RTOL, atol=H.LSE_RTOL)


@pytest.mark.parametrize("batch", [65, 256])
def test_units_many_sequences(batch, monkeypatch, kernels):
    """Lanes hold two and four sequences' lengths."""
    monkeypatch.setenv("L20_PD_MAX_WORKGROUPS", "11")
    rng = np.random.default_rng(batch)
    lens = [int(x) for x in rng.choice([0, 1, 63, 64, 65, 200, 400], size=batch)]
    inp = H.make_synthetic(batch, 4, 2, 64, lens, seed=batch, garbage_tail=True)
    out, lse = _run(inp, 64, torch.float32, kernels)
    H.compare(out, lse, *H.run_oracle(inp))


@pytest.mark.parametrize("groups", ["1", "5", "256"])
@pytest.mark.parametrize("case", range(32))
def test_units_random_shape(case, groups, monkeypatch, no_queue):
    monkeypatch.setenv("L20_PD_MAX_WORKGROUPS", groups)
    c = draw(case, seed_base=13000)
    print(case, c, flush=True)
    run_case(c)


def test_units_graph_replays_match_eager(kernels):
    inp = H.make_synthetic(6, 28, 4, 128, [900, 31, 1500, 0, 512, 77], seed=5)
    ref, _ = _run(inp, 256, torch.float32, kernels)
    q = inp["query"]
    po, pm, ps = H.workspace(inp, 256, torch.float32)
    out = torch.empty_like(q)
    ks, ksph = H._scales(inp["k_scale"])
    vs, vsph = H._scales(inp["v_scale"])

    def call():
        torch.ops.l20_stack.paged_decode_fp8_e4m3_split_out(
            q, inp["key_cache"], inp["value_cache"], inp["block_table"], inp["seq_lens"], po, pm, ps, out, ks, vs,
            inp["max_seq_len"], 256, inp["softmax_scale"], ksph, vsph)

    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        call()
    torch.cuda.current_stream().wait_stream(side)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        call()
    for _ in range(3):
        out.zero_()
        po.fill_(float("nan"))
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, ref)


def test_library_takes_the_units_kernel(monkeypatch, kernels):
    """By the library's own rule (no override), bitwise the forced call's result; a batch
    past the lengths a wave holds runs the persistent kernel, to the oracle all the same."""
    inp = H.make_synthetic(24, 16, 2, 128, [40 + 57 * i for i in range(24)], seed=3)
    forced, forced_lse = _run(inp, 256, torch.float32, kernels)
    for name in ("L20_PD_FUSED", "L20_PD_FUSED_SPLIT", "L20_PD_UNITS"):
        monkeypatch.delenv(name, raising=False)
    out, lse = _run(inp, 256, torch.float32, kernels)
    assert torch.equal(out, forced) and torch.equal(lse, forced_lse)
    big = H.make_synthetic(257, 4, 2, 64, [1 + 7 * (i % 90) for i in range(257)], seed=4)
    out, lse = _run(big, 64, torch.float32, kernels, kernel="pd_fp8_partial")
    H.compare(out, lse, *H.run_oracle(big))


def test_only_the_persistent_kernel_takes_a_queue_slot(monkeypatch):
    """Eager and captured calls of every path: a slot (16 for captured calls) goes to
    launches that have a work queue and to no other."""
    import l20_pd_cabi as cabi

    inp = H.make_synthetic(6, 28, 4, 128, [900, 31, 1000, 0, 512, 77], seed=5)
    exp = H.run_oracle(inp)
    q = inp["query"]
    work = H.workspace(inp, 256)
    out = torch.empty_like(q)
    ks, _ = H._scales(inp["k_scale"])
    vs, _ = H._scales(inp["v_scale"])

    def call():
        torch.ops.l20_stack.paged_decode_fp8_e4m3_split_out(
            q, inp["key_cache"], inp["value_cache"], inp["block_table"], inp["seq_lens"], *work, out, ks, vs,
            inp["max_seq_len"], 256, inp["softmax_scale"], None, None)

    for env, slots in (({"L20_PD_UNITS": "1"}, 0), ({"L20_PD_FUSED": "1"}, 0), ({"L20_PD_FUSED_SPLIT": "1"}, 0),
                       ({"L20_PD_UNITS": "0"}, 1)):
        with monkeypatch.context() as m:
            for name, value in env.items():
                m.setenv(name, value)
            before = cabi.queue_launches()
            call()
            assert cabi.queue_launches() == before + slots
            torch.cuda.synchronize()
            graph = torch.cuda.CUDAGraph()
            with torch.cuda.graph(graph):
                call()
            assert cabi.queue_launches() == before + 2 * slots
        for _ in range(3):
            out.zero_()
            graph.replay()
            torch.cuda.synchronize()
            H.compare(out, None, *exp, check_lse=False)
        assert cabi.queue_launches() == before + 2 * slots
