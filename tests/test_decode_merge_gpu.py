"""Decode rows split across few, several and very many groups, so that the
merge of their partials takes each of its routes: one wave alone (up to sixteen
partials), a team of four, eight or sixteen waves, and several rounds of
teams, for one, a few and all sixteen query heads a kv head, in a decode call
and in a call with prefill rows (where the merge follows another launch).
Checked against the fp32 CPU oracle with the tolerances of
tests/gpu_util.py."""
import pytest
import torch

from nanovllm_self_amd import workloads as W
from nanovllm_self_amd.kv_cache import SeqSlice
from tests.gpu_util import bf16_to_np, compare, oracle_paged, say

pytestmark = pytest.mark.gpu

# rows' cached tokens: one row over every group; two and three long rows
# beside short ones; rows of about 5, 9 and 20 partials
_ROWS = {
    "one": [6001],
    "two": [9000, 3, 4001, 40],
    "three": [5000, 7003, 6500, 130, 0],
    "some": [1300 + 7 * i for i in range(24)],
    "few": [300 + 11 * i for i in range(60)],
    # the longest rows that a launch without teams serves, and a tile more
    "edge_one_pass": [1951, 5, 1951], "past_one_pass": [1952, 1980],
    # rows just past a wave's own beside shorter ones
    "mixed_2000": [2000 + 7 * i for i in range(6)], "mixed_1000": [1000 + 7 * i for i in range(12)],
    "edge_two_passes": [1471, 927], "past_two_passes": [1472, 1500],
}


@pytest.mark.parametrize("rows", list(_ROWS))
@pytest.mark.parametrize("Hkv,g,kv", [(1, 8, "bf16"), (2, 1, "int8"), (2, 16, "bf16"), (4, 5, "fp8"), (8, 4, "fp16")])
@pytest.mark.parametrize("prefill", [False, True])
def test_split_rows_match_oracle(device, rows, Hkv, g, kv, prefill):
    spec = [(p, 1) for p in _ROWS[rows]] + ([(64, 5)] if prefill else [])
    say(f"split rows {rows}: Hkv={Hkv} g={g} cache={kv} prefill={prefill}")
    lens = [p + n for p, n in spec]
    NB = sum((n + 63) // 64 for n in lens) + 2
    gen = torch.Generator().manual_seed(7)
    tabs = W._tables(gen, lens, 64, NB)
    seqs = [SeqSlice(tabs[i], p, n) for i, (p, n) in enumerate(spec)]
    wl = W._assemble("split", seqs, g * Hkv, Hkv, 128, 64, NB, kv, device, gen, seed=7)
    out = wl.attn.forward(wl.q, wl.k, wl.v, wl.context)
    torch.cuda.synchronize()
    ref, at = oracle_paged(wl, list(range(len(spec))))
    compare(bf16_to_np(out)[at], ref, kv in ("int8", "fp8"), f"split rows {rows}")
