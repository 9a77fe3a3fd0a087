"""The balanced prefill's wave-pair kernel (head_dim 256: 192-row units, 32-key tiles, a score wave
one step ahead of its output wave, tiles loaded two steps ahead) at the edges of its pipeline: runs
of one, two and three tiles, units of one tile behind each other, chunks and contexts just below, at
and above a tile, wave pairs without rows or without a visible key, groups that give a workgroup 192,
16 or 3 tokens, and page ids outside the cache, all against the oracle within the repository's
prefill tolerance (P and the output are rounded to 16 bits, as in the oracle)."""
import pytest
import torch

from helpers import ATOL, RTOL, bits, say
from oracle.ref_torch import ref_gqa_prefill_paged
from tileinfer_amd.kernels import fused_sigmoid_mul, gqa_prefill_paged_fn
from tileinfer_amd.workloads import prefill_step

pytestmark = pytest.mark.gpu


def run(step, dev, causal=True, **kw):
    return gqa_prefill_paged_fn(step.q.to(dev), step.k_cache.to(dev), step.v_cache.to(dev),
                                step.block_table.to(dev), step.cu_seqlens_q.to(dev),
                                step.seqlen_k.to(dev), step.max_seqlen_q, step.page_size,
                                causal=causal, schedule="balanced", **kw)


def both(step, dev, causal=True):
    out = run(step, dev, causal)
    ref = ref_gqa_prefill_paged(step.q, step.k_cache, step.v_cache, step.block_table,
                                step.cu_seqlens_q, step.seqlen_k, step.page_size, causal)
    return out, ref


@pytest.mark.parametrize("hq,hkv", [(24, 4), (2, 2), (12, 1), (64, 1)])
@pytest.mark.parametrize("q_lens,kv_lens", [
    ([1], [1]), ([31], [31]), ([32], [32]), ([33], [33]), ([1], [65]), ([32, 33], [96, 64]),
    ([1] * 70, [1] * 70),                        # one-tile units behind each other
    ([3, 1, 40, 0, 5], [3, 33, 129, 7, 0]),      # an empty chunk, a chunk without context
    ([200], [231]), ([64, 1, 1], [64, 900, 32]),
])
def test_pipeline_edges_vs_oracle(q_lens, kv_lens, hq, hkv, dev):
    say(f"prefill pairs q={q_lens} kv={kv_lens} heads={hq}/{hkv}")
    step = prefill_step(q_lens, kv_lens, seed=51, hq=hq, hkv=hkv)
    for causal in (True, False):
        out, ref = both(step, dev, causal)
        torch.testing.assert_close(out.float().cpu(), ref.float(), atol=ATOL, rtol=RTOL)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("q_lens,kv_lens", [
    ([1], [1]), ([33], [33]), ([1] * 70, [1] * 70), ([3, 1, 40, 0, 5], [3, 33, 129, 7, 0]),
    ([200, 31, 64], [700, 31, 900]),             # cut units: gated by the merge
])
def test_gate_is_applied_to_the_rounded_rows(q_lens, kv_lens, dtype, dev):
    """The gated call gives the bits of the plain call followed by the gate, for gate rows of their
    own and for rows that lie a stride apart, and changes no row of its operands."""
    say(f"prefill pairs gated q={q_lens} kv={kv_lens} {dtype}")
    step = prefill_step(q_lens, kv_lens, seed=53, dtype=dtype)
    plain = run(step, dev)
    gate = 3 * torch.randn(plain.shape, generator=torch.Generator().manual_seed(5))
    gate = gate.to(dtype).to(dev)
    apart = torch.empty(gate.shape[0], 2, *gate.shape[1:], dtype=dtype, device=dev)[:, 1].copy_(gate)
    want = fused_sigmoid_mul(plain, gate)
    for g in (gate, apart):
        assert torch.equal(bits(run(step, dev, gate=g)), bits(want))
    assert torch.equal(bits(apart), bits(gate))


def test_values_outside_every_mask_stay_out(dev):
    """Non-finite K and V at positions that no query of the call may see leave the output as it is:
    tokens behind the context in its last page, and tokens that only later query blocks see."""
    step = prefill_step([400], [470], seed=52)
    clean, _ = both(step, dev)
    for first in (470, 448):  # past the context; the last tile, seen by tokens 378.. of the chunk
        kc, vc = step.k_cache.clone(), step.v_cache.clone()
        for pos in range(first, 480 if first == 470 else 470):
            page, row = int(step.block_table[0, pos // 16]), pos % 16
            kc[page, row] = float("nan")
            vc[page, row] = float("inf")
        out = gqa_prefill_paged_fn(step.q.to(dev), kc.to(dev), vc.to(dev), step.block_table.to(dev),
                                   step.cu_seqlens_q.to(dev), step.seqlen_k.to(dev), 400, 16,
                                   schedule="balanced")
        keep = 400 if first == 470 else 352  # whole query blocks of 32 tokens before position 448
        assert torch.equal(bits(out[:keep]), bits(clean[:keep])), first


@pytest.mark.parametrize("page", [16, 8, 4])
def test_page_ids_outside_the_cache(page, dev):
    """Ids outside the cache inside a context are absent keys, in cut units too (a few chunks over long
    contexts: every unit is cut between workgroups): the rows are the attention over the other keys,
    in 64 bits within the prefill tolerance."""
    q_lens, kv_lens, hq, hkv, d = [20, 9], [3000, 1700], 4, 2, 256
    step = prefill_step(q_lens, kv_lens, seed=54, hq=hq, hkv=hkv, page=page)
    say(f"prefill pairs absent pages, page={page}")
    nb = step.k_cache.shape[0]
    for b, at, bad in ((0, 0, -1), (0, 1000, nb), (0, 1016, 10 ** 8), (0, 2999, -7), (1, 640, 2 ** 31 - 1)):
        step.block_table[b, at // page] = bad
    out = run(step, dev).cpu()
    k, v = (c.reshape(-1, hkv, d).double() for c in (step.k_cache, step.v_cache))
    at = 0
    for b, (n, c) in enumerate(zip(q_lens, kv_lens)):
        pos = torch.arange(c)
        ids = step.block_table[b, pos // page].long()
        pos = pos[(ids >= 0) & (ids < nb)]
        rows = step.block_table[b, pos // page].long() * page + pos % page
        assert len(pos) < c
        seen = pos[None] <= c - n + torch.arange(n)[:, None]
        for h in range(hq):
            s = step.q[at:at + n, h].double() @ k[rows, h // (hq // hkv)].T / d ** 0.5
            want = torch.softmax(s.masked_fill(~seen, float("-inf")), -1) @ v[rows, h // (hq // hkv)]
            torch.testing.assert_close(out[at:at + n, h].double(), want, atol=ATOL, rtol=RTOL)
        at += n
