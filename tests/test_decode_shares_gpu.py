"""The stream decode's shares, prefix sums, packed queries and dense addressing at their
edges, on the MI355X (``-m gpu``), against the oracles at the repository's tolerances."""

from __future__ import annotations

import random

import pytest
import torch

from conftest import ATTN_ATOL, assert_max_abs
from mini_vllm.workloads import build_batch
from oracle.dense_attention import dense_attention as dense_oracle
from oracle.paged_attention import paged_attention as oracle

pytestmark = pytest.mark.gpu

F8 = torch.float8_e4m3fn


def check(extension, b, dtype, options=None):
    got = extension.paged_attention(*b.args(), k_scale=b.k_scale, v_scale=b.v_scale,
                                    plan_options=options)
    scales = {"k_scale": b.k_scale, "v_scale": b.v_scale} if b.k_scale is not None else {}
    want = oracle(b.q, b.key_pool, b.value_pool, b.block_tables, b.cu_seqlens_q, b.context_lens,
                  b.scale, **scales)
    assert_max_abs(got.float(), want, ATTN_ATOL[dtype])
    return got


@pytest.mark.parametrize("seqs", [1, 2, 63, 64, 65, 130])
@pytest.mark.parametrize("dtype,kv_dtype", [(torch.float32, None), (torch.bfloat16, None),
                                            (torch.float16, F8)])
def test_sequence_counts_and_smallest_shares(extension, device, dtype, kv_dtype, seqs):
    """One lane per sequence up to 64, LDS beyond; contexts of 1 to a few shares of the
    smallest size (8, 16 and 32 keys), so shares begin and end at sequence edges."""
    rng = random.Random(seqs)
    contexts = [rng.choice([1, 7, 8, 9, 15, 16, 17, 31, 32, 33, 100]) for _ in range(seqs)]
    b = build_batch(contexts, [1] * seqs, dtype=dtype, kv_dtype=kv_dtype, num_q_heads=16,
                    num_kv_heads=8, head_dim=128, seed=seqs, device="cuda")
    check(extension, b, kv_dtype or dtype)


@pytest.mark.parametrize("seqs,kv_heads", [(66, 1), (257, 1), (512, 8), (513, 8), (2049, 2), (4096, 8)])
def test_prefix_sums_of_many_sequences(extension, device, seqs, kv_heads):
    """Past 64 sequences each wave of a workgroup (one per kv head here) sums a run of them:
    runs that end within 64, empty last ones, up to the most sequences a launch takes, prompt
    chunks, which have no decode keys, among them."""
    rng = random.Random(seqs)
    lens = [3 if i % 97 == 50 else 1 for i in range(seqs)]
    contexts = [rng.choice([3, 16, 17, 31, 40]) for _ in range(seqs)]
    b = build_batch(contexts, lens, dtype=torch.bfloat16, num_q_heads=2 * kv_heads,
                    num_kv_heads=kv_heads, head_dim=128, seed=seqs, device="cuda")
    check(extension, b, torch.bfloat16)


@pytest.mark.parametrize("wgs_per_cu", [1, 3, 300])
@pytest.mark.parametrize("contexts", [[5000], [1, 4999], [4099, 2, 8191], [17] * 40])
def test_share_division(extension, device, contexts, wgs_per_cu):
    """Key counts that the share count does not divide, shares of one key too many and
    more workgroups than the 16-bit share limit allows (300 per CU)."""
    b = build_batch(contexts, [1] * len(contexts), dtype=torch.bfloat16, num_q_heads=16,
                    num_kv_heads=8, head_dim=128, seed=1, device="cuda")
    one = check(extension, b, torch.bfloat16, {"decode_wgs_per_cu": wgs_per_cu})
    again = check(extension, b, torch.bfloat16, {"decode_wgs_per_cu": wgs_per_cu})
    assert torch.equal(one, again)


@pytest.mark.parametrize("dtype,kv_dtype", [(torch.bfloat16, None), (torch.float16, None),
                                            (torch.bfloat16, F8), (torch.float16, F8)])
def test_queries_at_any_element(extension, device, dtype, kv_dtype):
    """q starting two bytes past a 16-byte boundary: the same bits as an aligned copy."""
    b = build_batch([300, 40], [1, 1], dtype=dtype, kv_dtype=kv_dtype, num_q_heads=16,
                    num_kv_heads=8, head_dim=128, seed=3, device="cuda")
    want = check(extension, b, kv_dtype or dtype)
    room = torch.empty(b.q.numel() + 8, dtype=dtype, device="cuda")
    b.q = room[1:1 + b.q.numel()].view(b.q.shape).copy_(b.q)
    assert b.q.data_ptr() % 16 == 2
    assert torch.equal(check(extension, b, kv_dtype or dtype), want)


@pytest.mark.parametrize("batch,keys,room", [(1, 1, 1), (3, 17, 40), (70, 33, 33), (2, 4097, 5000)])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_dense_decode_without_metadata(extension, device, dtype, batch, keys, room):
    gen = torch.Generator().manual_seed(keys)
    q = torch.randn(batch, 16, 1, 128, generator=gen).to(dtype).cuda()
    k, v = (torch.randn(batch, 8, room, 128, generator=gen).to(dtype).cuda()[:, :, :keys]
            for _ in range(2))
    got = extension.decode_attention(q, k, v, 128 ** -0.5)
    want = dense_oracle(q.cpu(), k.cpu(), v.cpu())
    assert_max_abs(got.float(), torch.as_tensor(want), ATTN_ATOL[dtype])
