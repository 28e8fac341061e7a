"""Prefill entries split along their keys: short new turns over long cached
prefixes (and long prompts of one kv head), where a batch has too few units
for the chip.  The plan cuts their keys into parts, each part's units leave
fp32 partials in the workspace, and the merge joins them.  Checked against
the fp32 CPU oracle with the tolerances of tests/gpu_util.py; a batch that
should be split is also checked to have been (the plan header's count), and
the same batch in a workspace without room for the parts must agree."""
import numpy as np
import pytest
import torch

from nanovllm_self_amd import workloads as W
from nanovllm_self_amd.kv_cache import SeqSlice
from nanovllm_self_amd.layers import attention as LA
from oracle import attn_oracle as AO
from tests.gpu_util import bf16_to_np, compare, oracle_seq_rows, say
from tests.test_code_prefill_gpu import _oracle_with_holes

pytestmark = pytest.mark.gpu
N_LIST, N_SPLIT = 0, 12  # the plan header's words


def _workload(device, spec, Hkv, g, bs, kv, seed):
    lens = [p + n for p, n in spec]
    NB = sum((x + bs - 1) // bs for x in lens) + 2
    gen = torch.Generator().manual_seed(seed)
    tabs = W._tables(gen, lens, bs, NB)
    seqs = [SeqSlice(tabs[i], p, n) for i, (p, n) in enumerate(spec)]
    return W._assemble("parts", seqs, g * Hkv, Hkv, 128, bs, NB, kv, device, gen, seed=seed)


def _check(wl, got, spec, quant, what):
    """Rows of every sequence against the oracle: the first, the last and
    those around query-tile edges."""
    for i, (p, n) in enumerate(spec):
        for r0, r1 in ((0, min(n, 3)), (max(0, min(n, 65) - 3), min(n, 65)), (max(0, n - 2), n)):
            ref, rows = oracle_seq_rows(wl, i, r0, r1)
            compare(got[rows], ref, quant, f"{what} row {i} [{r0}, {r1})")


@pytest.mark.parametrize("Hkv,g,bs,kv,spec", [
    (8, 4, 256, "bf16", [(8192, 70), (2048, 3), (4352, 130)]),
    (8, 4, 256, "bf16", [(6400, 65), (300, 1), (9000, 1), (1000, 33)]),       # decode rows beside them
    (2, 8, 64, "fp8", [(4160, 40), (1111, 64), (64, 2)]),
    (2, 8, 64, "int8", [(3000, 1), (5056, 100)]),
    (1, 16, 128, "bf16", [(7040, 257)]),                                     # two head groups
    (2, 5, 64, "bf16", [(2752, 31), (1024, 2)]),                             # a head group not full
    (1, 1, 1024, "bf16", [(8192, 300)]),                                     # blocks of sixteen tiles
    (4, 3, 64, "fp16", [(3072, 129), (3000, 5)]),
])
def test_parts_match_oracle(device, monkeypatch, Hkv, g, bs, kv, spec):
    say(f"parts: Hkv={Hkv} g={g} block_size={bs} cache={kv} rows (cached, new)={spec}")
    wl = _workload(device, spec, Hkv, g, bs, kv, 11)
    out = wl.attn.forward(wl.q, wl.k, wl.v, wl.context)
    torch.cuda.synchronize()
    header = LA._workspaces[wl.q.device][:256].view(torch.int32).cpu()
    assert int(header[N_SPLIT]) > 0, "the batch was not split"
    got = bf16_to_np(out)
    _check(wl, got, spec, kv in ("int8", "fp8"), "parts")
    again = wl.attn.prefill_flashattn(wl.q, wl.k, wl.v, wl.context)
    torch.cuda.synchronize()
    assert torch.equal(out, again), "two identical calls differ"
    # No room for the parts: the whole entries, in another order of sums.
    monkeypatch.setattr(LA._lib.load(), "nvs_attention_split_bytes", lambda *a: 0)
    whole = wl.attn.prefill_flashattn(wl.q, wl.k, wl.v, wl.context)
    torch.cuda.synchronize()
    header = LA._workspaces[wl.q.device][:256].view(torch.int32).cpu()
    assert int(header[N_SPLIT]) == 0, "the batch was split without room"
    compare(got, bf16_to_np(whole), kv in ("int8", "fp8"), "parts vs whole")


@pytest.mark.parametrize("kv", ["bf16", "fp16"])
def test_local_prompt_parts_match_oracle(device, kv):
    """A long prompt of one kv head, nothing cached: its deep query tiles
    are cut into parts, its shallow ones (and the diagonal) are not."""
    spec = [(0, 3001), (0, 70)]
    say(f"local parts {kv} {spec}")
    wl = _workload(device, spec, 1, 8, 64, kv, 5)
    assert wl.context.block_tables is None
    out = wl.attn.forward(wl.q, wl.k, wl.v, wl.context)
    torch.cuda.synchronize()
    header = LA._workspaces[wl.q.device][:256].view(torch.int32).cpu()
    assert int(header[N_SPLIT]) > 0, "the batch was not split"
    ref = AO.attention_local(*(torch.from_numpy(bf16_to_np(x)) for x in (wl.q, wl.k, wl.v)),
                             wl.context.cu_seqlens_q.cpu(), 8, 1, 128)
    compare(bf16_to_np(out), ref.numpy(), False, f"local parts {kv}")


def test_parts_in_a_graph(device):
    """A captured call whose workspace has room for the parts, replayed over
    changed queries, equals the eager one; the captured workspace stays."""
    spec = [(4096, 40), (2048, 7), (500, 1)]
    say(f"parts in a graph {spec}")
    wl = _workload(device, spec, 8, 4, 256, "bf16", 3)
    args = (wl.q, wl.k, wl.v, wl.context)
    wl.attn.forward(*args)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = wl.attn.forward(*args)
    ws = LA._workspaces[wl.q.device]
    for step in range(3):
        wl.q.copy_(torch.randn_like(wl.q))
        graph.replay()
        torch.cuda.synchronize()
        replayed = out.clone()
        eager = wl.attn.forward(*args)
        torch.cuda.synchronize()
        assert torch.equal(replayed, eager), f"replay {step} differs"
    big = _workload(device, [(16384, 20), (16384, 30)], 8, 4, 256, "bf16", 4)
    big.attn.forward(big.q, big.k, big.v, big.context)
    torch.cuda.synchronize()
    need = LA._lib.load().nvs_attention_workspace_bytes(2, 30, 16384 + 30, 32, 8, 128, 0)
    assert ws.numel() < need or LA._workspaces[wl.q.device] is ws
    assert any(b is ws for b in LA._captured_workspaces[wl.q.device])
    assert np.all(np.isfinite(bf16_to_np(eager)))


@pytest.mark.parametrize("kv,bs", [("bf16", 64), ("bf16", 256), ("fp16", 64), ("fp8", 64), ("int8", 256)])
def test_parts_over_missing_blocks(device, kv, bs):
    """Parts whose tiles meet blocks that are missing (-1, outside the pool),
    and rows of more keys than their block-table row has blocks for, whose
    later parts start past its end: such blocks read as zero keys and values."""
    spec = [(5120, 40), (4096, 70), (6144, 33)]
    say(f"parts over missing blocks: {kv} block_size={bs}")
    wl = _workload(device, spec, 2, 4, bs, kv, 17)
    width = 2048 // bs  # every row has keys past it
    bt = wl.context.block_tables[:, :width].contiguous()
    bt[0, 512 // bs] = -1
    bt[1, 1024 // bs] = wl.num_blocks + 3
    wl.context.block_tables = bt
    wl.context.max_seqlen_k = 2048
    out = wl.attn.forward(wl.q, wl.k, wl.v, wl.context)
    torch.cuda.synchronize()
    header = LA._workspaces[wl.q.device][:256].view(torch.int32).cpu()
    assert int(header[N_SPLIT]) > 0, "the batch was not split"
    got = bf16_to_np(out)
    for i in range(len(spec)):
        row = [b if 0 <= b < wl.num_blocks else -1 for b in bt[i].tolist()]
        ref, rows = _oracle_with_holes(wl, i, row + [-1] * (len(wl.seqs[i].block_table) - width))
        compare(got[rows], ref, kv in ("int8", "fp8"), f"parts over missing blocks {kv} row {i}")


def test_parts_after_a_captured_decode(device, monkeypatch):
    """Follow-up turns after decode was captured in a graph (its workspace
    reserved for decode alone) are split all the same, and the graph replays
    over its own workspace."""
    for name in ("_workspaces", "_captured_workspaces"):
        monkeypatch.setattr(LA, name, {}, raising=False)
    say("parts after a captured decode")
    dec = _workload(device, [(3000 + 11 * i, 1) for i in range(40)], 8, 4, 256, "bf16", 21)
    LA.reserve_attention_workspace(40, 1, int(dec.context.max_seqlen_k), 32, device, 8)
    args = (dec.q, dec.k, dec.v, dec.context)
    dec.attn.forward(*args)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = dec.attn.forward(*args)
    spec = [(4096, 40), (2048, 70), (8192, 30)]
    turn = _workload(device, spec, 8, 4, 256, "bf16", 22)
    for step in range(3):
        got = turn.attn.forward(turn.q, turn.k, turn.v, turn.context)
        torch.cuda.synchronize()
        header = LA._workspaces[turn.q.device][:256].view(torch.int32).cpu()
        assert int(header[N_SPLIT]) > 0, "the batch was not split"
        if step == 0:
            _check(turn, bf16_to_np(got), spec, False, "turn after a captured decode")
        graph.replay()
        torch.cuda.synchronize()
        replayed = out.clone()
        assert torch.equal(replayed, dec.attn.forward(*args)), f"replay {step} differs"


@pytest.mark.parametrize("spec,bs", [([(3072, 40 + i) for i in range(4)], 256), ([(4160, 70), (2752, 9)], 64)])
def test_list_is_longest_first(device, spec, bs):
    """The list's records run from the longest part to the shortest, to a
    bucket of the plan's sort: each entry's short last part comes after the
    others' whole ones."""
    say(f"order of the parts {spec} block_size={bs}")
    wl = _workload(device, spec, 8, 4, bs, "bf16", 6)
    wl.attn.forward(wl.q, wl.k, wl.v, wl.context)
    torch.cuda.synchronize()
    ws = LA._workspaces[wl.q.device]
    header = ws[:256].view(torch.int32).cpu()
    assert int(header[N_SPLIT]) == len(spec) + sum(n > 64 for _, n in spec), "not every entry was split"
    at = LA._lib.load().nvs_attention_workspace_bytes(
        len(spec), max(n for _, n in spec), max(p + n for p, n in spec), 32, 8, 128, 0)
    at = (at + 255) // 256 * 256
    rec = ws[at:at + 64 * int(header[N_LIST])].view(torch.int32).cpu().reshape(-1, 16)
    tiles = rec[:, 9].tolist()
    assert sum(tiles) == sum((p + min(n, 64 * (t + 1)) + 63) // 64 for p, n in spec for t in range((n + 63) // 64))
    slack = max(tiles) // 16 + 1
    assert all(a + slack > b for a, b in zip(tiles, tiles[1:])), tiles
    assert max(tiles) - min(tiles) > slack  # else every order would do


@pytest.mark.parametrize("spec,Hkv,g", [
    ([(1536, 40 + i) for i in range(12)], 8, 4),   # a unit on every third work-group, shallow
    ([(1536, 200 + i) for i in range(24)], 1, 8),  # even rows, most work-groups busy
    ([(2048, 200 + i) for i in range(20)], 2, 4),
])
def test_even_batches_keep_the_row_order(device, spec, Hkv, g):
    """Batches whose rows are alike and keep the chip busy gain nothing by
    parts or another order: whole entries, row by row, deepest first."""
    say(f"row order: Hkv={Hkv} g={g} {len(spec)} rows from {spec[0]}")
    wl = _workload(device, spec, Hkv, g, 256, "bf16", 8)
    out = wl.attn.forward(wl.q, wl.k, wl.v, wl.context)
    torch.cuda.synchronize()
    ws = LA._workspaces[wl.q.device]
    header = ws[:256].view(torch.int32).cpu()
    assert int(header[N_SPLIT]) == 0
    at = LA._lib.load().nvs_attention_workspace_bytes(
        len(spec), max(n for _, n in spec), max(p + n for p, n in spec), g * Hkv, Hkv, 128, 0)
    at = (at + 255) // 256 * 256
    rec = ws[at:at + 64 * int(header[N_LIST])].view(torch.int32).cpu().reshape(-1, 16)
    pos = 256 // (1 << min(3, g.bit_length() - 1))
    want = [(b, pos * t) for b, (_, n) in enumerate(spec) for t in reversed(range((n + pos - 1) // pos))]
    assert [(r[13], r[8]) for r in rec.tolist()] == want
    assert all(r[0] == -1 for r in rec.tolist())
    _check(wl, bf16_to_np(out), spec[:2] if len(spec) > 2 else spec, False, "row order")


def test_local_prompts_in_order_without_parts(device):
    """Several prompts of more than a round of units, nothing cached: put
    longest first, whole (no slots, no merge launch)."""
    lens = [150, 90] * 6 + [2700, 2400, 2600]
    say(f"local prompts longest first {lens}")
    wl = _workload(device, [(0, n) for n in lens], 8, 1, 64, "bf16", 12)
    assert wl.context.block_tables is None
    out = wl.attn.forward(wl.q, wl.k, wl.v, wl.context)
    torch.cuda.synchronize()
    ws = LA._workspaces[wl.q.device]
    header = ws[:256].view(torch.int32).cpu()
    assert int(header[N_SPLIT]) == 0
    n = sum((x + 255) // 256 for x in lens)
    assert int(header[N_LIST]) == n
    at = 256 + (4 * len(lens) * ((max(lens) + 255) // 256) + 255) // 256 * 256  # behind the header and the list
    tiles = ws[at:at + 64 * n].view(torch.int32).cpu().reshape(-1, 16)[:, 9].tolist()
    assert sorted(tiles) == sorted((min(x, 256 * (t + 1)) + 63) // 64 for x in lens for t in range((x + 255) // 256))
    assert all(a + max(tiles) // 16 + 1 > b for a, b in zip(tiles, tiles[1:])), tiles
    ref = AO.attention_local(*(torch.from_numpy(bf16_to_np(x)) for x in (wl.q, wl.k, wl.v)),
                             wl.context.cu_seqlens_q.cpu(), 8, 8, 128)
    compare(bf16_to_np(out), ref.numpy(), False, "local prompts longest first")


@pytest.mark.parametrize("Hkv,g,kv", [(8, 4, "bf16"), (2, 16, "fp16"), (1, 4, "int8")])
def test_parts_into_a_strided_output(device, Hkv, g, kv):
    """Split entries and decode rows into output rows and heads further apart
    than they are long: the values of a contiguous output, nothing beside them."""
    from nanovllm_self_amd import _lib
    spec = [(6144, 67), (5000, 1), (4096, 20)]
    say(f"parts into a strided output: heads {g * Hkv}/{Hkv} cache={kv}")
    wl = _workload(device, spec, Hkv, g, 256, kv, 14)
    want = wl.attn.forward(wl.q, wl.k, wl.v, wl.context)
    torch.cuda.synchronize()
    ws = LA._workspaces[wl.q.device]
    assert int(ws[:256].view(torch.int32).cpu()[N_SPLIT]) > 0, "the batch was not split"
    Hq, T, ctx, attn = g * Hkv, wl.q.shape[0], wl.context, wl.attn
    room = torch.full((T, Hq + 3, 144), 7.0, dtype=wl.q.dtype, device=device)
    out = room[:, 1:Hq + 1, :128]
    _lib.check(_lib.load().nvs_paged_attention(
        wl.q.data_ptr(), wl.q.stride(0), wl.q.stride(1), attn.k_cache.data_ptr(), attn.v_cache.data_ptr(),
        _lib.nvs_dtype(attn.k_cache.dtype), _lib.ptr(attn.k_scale_cache), _lib.ptr(attn.v_scale_cache),
        ctx.cu_seqlens_q.data_ptr(), ctx.cu_seqlens_k.data_ptr(), ctx.block_tables.data_ptr(), ctx.block_tables.size(1),
        len(spec), T, int(ctx.max_seqlen_q), int(ctx.max_seqlen_k), Hq, Hkv, 128, 256, wl.num_blocks, 128 ** -0.5,
        out.data_ptr(), out.stride(0), out.stride(1), ws.data_ptr(), ws.numel(), _lib.stream_of(wl.q)),
        "paged_attention")
    torch.cuda.synchronize()
    assert int(ws[:256].view(torch.int32).cpu()[N_SPLIT]) > 0, "the batch was not split"
    assert torch.equal(out, want)
    room[:, 1:Hq + 1, :128] = 7.0
    assert bool((room == 7.0).all()), "written outside the output"
