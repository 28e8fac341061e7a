"""The write of the step's k / v that a prefill call makes in its planning
launch, or in a launch of its own where it is long: caches and scales equal,
byte for byte, those of nvs_store_kvcache alone, on both sides of the size
where the route changes, with padding slots (-1), slots outside the pool,
strided k / v and head counts that leave the last work-group partly empty."""
import pytest
import torch

from nanovllm_self_amd import workloads as W
from nanovllm_self_amd.kv_cache import SeqSlice
from tests.gpu_util import say

pytestmark = pytest.mark.gpu

_SPECS = {
    "local_small": [(0, 5), (0, 70)],
    "local_edge": [(0, 64)] * 128,              # 8192 tokens of 8 heads: 1024 work-groups
    "local_past": [(0, 64)] * 127 + [(0, 65)],
    "paged": [(128, 33), (64, 2), (300, 1), (17, 1)],
    "paged_edge": [(64, 64)] * 127 + [(64, 63), (500, 1)],
    "paged_past": [(64, 64)] * 128 + [(500, 1)],
}


@pytest.mark.parametrize("what", list(_SPECS))
@pytest.mark.parametrize("kv,Hkv,g", [("bf16", 8, 1), ("fp16", 8, 2), ("fp8", 8, 1), ("int8", 8, 4), ("bf16", 3, 2),
                                      ("int8", 1, 5)])
def test_prefill_call_writes_as_the_store_alone(device, what, kv, Hkv, g):
    spec = _SPECS[what]
    say(f"write in a prefill call: {what} cache={kv} heads {g * Hkv}/{Hkv}")
    lens = [p + n for p, n in spec]
    NB = sum((n + 63) // 64 for n in lens) + 2
    gen = torch.Generator().manual_seed(31)
    tabs = W._tables(gen, lens, 64, NB)
    seqs = [SeqSlice(tabs[i], p, n) for i, (p, n) in enumerate(spec)]
    wl = W._assemble("store", seqs, g * Hkv, Hkv, 128, 64, NB, kv, device, gen, seed=31)
    attn, ctx = wl.attn, wl.context
    both = torch.cat([wl.k, wl.v], dim=1)  # k and v as slices of one buffer
    k, v = both[:, :Hkv], both[:, Hkv:]
    slots = ctx.slot_mapping.clone()
    slots[1], slots[-2] = -1, NB * 64 + 3
    ctx.slot_mapping = slots
    caches = [c for c in (attn.k_cache, attn.v_cache, attn.k_scale_cache, attn.v_scale_cache) if c is not None]
    before = [c.clone() for c in caches]
    assert attn._store_in_prefill(wl.q, k, v, ctx)
    attn.forward(wl.q, k, v, ctx)
    torch.cuda.synchronize()
    called = [c.clone() for c in caches]
    for c, b in zip(caches, before):
        c.copy_(b)
    attn.write_kv_cache(k, v, slots)
    torch.cuda.synchronize()
    changed = False
    for c, d, b in zip(caches, called, before):
        assert torch.equal(c.view(torch.uint8), d.view(torch.uint8))
        changed = changed or not torch.equal(c.view(torch.uint8), b.view(torch.uint8))
    assert changed
