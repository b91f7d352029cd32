"""The pair prefill kernel (GQA pairs, D = 128) at the edges of its tiles, its blocks of page
ids and its split schedule, on the MI355X (``-m gpu``), against the fp32 oracle at the
repository's tolerances (tests/conftest.py)."""

from __future__ import annotations

import pytest
import torch

from mini_vllm.workloads import build_batch
from oracle.paged_attention import paged_attention as oracle
from conftest import ATTN_ATOL, assert_max_abs

pytestmark = pytest.mark.gpu

F8 = torch.float8_e4m3fn
WHOLE = {"prefill_schedule": "grid", "prefill_pieces": 1}
CUT = {"prefill_schedule": "stream", "prefill_share_tiles": 1}


def check(extension, contexts, lens, dtype, kv_dtype, options, hq=16):
    b = build_batch(contexts, lens, dtype=dtype, kv_dtype=kv_dtype, num_q_heads=hq,
                    num_kv_heads=8, head_dim=128, seed=len(contexts), device="cuda")
    got = extension.paged_attention(*b.args(), k_scale=b.k_scale, v_scale=b.v_scale,
                                    plan_options=options)
    want = oracle(b.q, b.key_pool, b.value_pool, b.block_tables, b.cu_seqlens_q, b.context_lens,
                  b.scale, **({"k_scale": b.k_scale, "v_scale": b.v_scale} if kv_dtype else {}))
    assert_max_abs(got.float(), want, ATTN_ATOL[kv_dtype or dtype], f"{contexts} {lens}")
    return got


@pytest.mark.parametrize("options", [WHOLE, CUT], ids=["whole", "cut"])
@pytest.mark.parametrize("dtype,kv_dtype", [(torch.bfloat16, None), (torch.float16, None),
                                            (torch.bfloat16, F8)])
def test_tile_edges(extension, device, dtype, kv_dtype, options):
    """Query and key counts one below, at and one past the 64-row tiles, one to three key
    tiles, a wave with no rows, rows that see a tile's first key only."""
    lens = [2, 31, 32, 33, 63, 64, 65, 127, 129]
    contexts = [2, 64, 65, 33, 128, 127, 192, 193, 129]
    check(extension, contexts, lens, dtype, kv_dtype, options)


@pytest.mark.parametrize("options", [WHOLE, CUT], ids=["whole", "cut"])
@pytest.mark.parametrize("kv_dtype", [None, F8], ids=["bf16", "fp8"])
def test_page_id_blocks(extension, device, kv_dtype, options):
    """A wave holds its page ids 64 tiles at a time: contexts ending around tiles 63-66 and
    127-129, where the next block is taken up a step or two before it is used."""
    contexts = [64 * n + d for n, d in ((63, 0), (63, 1), (64, 0), (64, 1), (65, 1), (66, 0), (128, 5))]
    check(extension, contexts, [5] * 7, torch.bfloat16, kv_dtype, options)


@pytest.mark.parametrize("tokens", [64 * 31, 64 * 32 + 1])
def test_fp8_workgroups_of_either_size(extension, device, tokens):
    """Around the token count where fp8 pools take 128-position workgroups (256 of them)."""
    lens = [tokens - 3 * 500, 500, 500, 500]
    check(extension, [n + 77 for n in lens], lens, torch.bfloat16, F8, WHOLE, hq=32)


def test_cut_items_of_many_sequences(extension, device):
    """More than 64 sequences (the schedule's lanes hold 64 at a time), chunks among decode
    rows, one far longer than the rest and cut into many pieces; three calls, the same bits."""
    contexts = [40 + 7 * i for i in range(150)]
    lens = [1 if i % 3 else 1 + i % 90 for i in range(150)]
    contexts[99], lens[99] = 5000, 66
    lens = [min(n, c) for n, c in zip(lens, contexts)]
    check(extension, contexts, lens, torch.bfloat16, None, CUT)
    b = build_batch([3000, 64], [70, 64], dtype=torch.bfloat16, num_q_heads=16, num_kv_heads=8,
                    head_dim=128, seed=2, device="cuda")
    outs = [extension.paged_attention(*b.args(), plan_options=CUT) for _ in range(3)]
    assert torch.equal(outs[0], outs[1]) and torch.equal(outs[0], outs[2])


def test_the_default_cuts_a_lone_long_chunk(extension, device):
    """No options: 63 tokens after 6393 keys (8 items on 256 CUs)."""
    check(extension, [6456], [63], torch.bfloat16, None, None)


# (chunk lengths, keys before each, decode rows, their contexts' bound, heads, pool, item, listed)
ROUTES = {
    "whole, last query tiles first": ([129, 64, 2, 200, 65], [0, 100, 62, 57, 191], 20, 300, 16, None, 64, 1),
    "whole, by sequence": ([256, 255, 257], [2400, 2345, 2000], 5, 900, 32, None, 64, 1),
    "whole, a few holes": ([512, 300, 201, 449], [0, 65, 500, 127], 0, 300, 32, None, 64, 1),
    "whole, fp8 items of 128": ([390, 385, 388, 384], [500, 0, 127, 64], 6, 700, 32, F8, 128, 1),
    "cut, items of 128": ([130, 257, 65, 500], [4870, 4000, 4800, 4500], 3, 900, 16, None, 128, 64),
    "cut, fp8 items of 128": ([130, 257, 65, 500], [3870, 3000, 3800, 3500], 3, 900, 16, F8, 128, 64),
    "whole, more than 64 sequences": ([100, 33], [0, 64], 66, 200, 16, None, 64, 0),
    "cut, more than 64 sequences": ([63, 3], [6000, 900], 70, 200, 16, None, 64, 64),
    "cut, fp8, more than 64 sequences": ([300, 200], [5000, 4000], 68, 200, 16, F8, 128, 64),
}


@pytest.mark.parametrize("route", ROUTES)
def test_the_planner_s_own_routes(extension, device, route):
    """Ragged chunks among decode rows, every query tile and key tile edge somewhere in them,
    by each way the planner runs a batch when no option forces one; the same bits again."""
    chunks, before, decodes, bound, hq, kv_dtype, item, listed = ROUTES[route]
    gen = torch.Generator().manual_seed(len(route))
    rows = [(int(c), 1) for c in torch.randint(1, bound, (decodes,), generator=gen)]
    rows += [(n + b, n) for n, b in zip(chunks, before)]
    rows = [rows[i] for i in torch.randperm(len(rows), generator=gen).tolist()]
    contexts, lens = [c for c, _ in rows], [n for _, n in rows]
    plan = extension.paged_attention_plan(sum(lens), len(lens), hq, 8, 128, 16, max(lens), max(contexts),
                                          torch.bfloat16, kv_dtype or torch.bfloat16)
    if torch.cuda.get_device_properties(0).multi_processor_count == 256:
        assert (plan["prefill_item"], plan["prefill_listed"]) == (item, listed)
    first, again = (check(extension, contexts, lens, torch.bfloat16, kv_dtype, None, hq) for _ in range(2))
    assert torch.equal(first, again)


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("context,tokens", [(128, 64), (400, 100), (600, 61)])
def test_whole_short_items_err_no_more_than_single_tiles(extension, device, dtype, context, tokens):
    """An item of a few tiles run whole against one cut into single tiles, whose probabilities
    are all taken against their tile's own maximum (the largest is 1 and not rounded): the
    same products are rounded, so the error against 64 bits is the same but for which way
    single outputs round (their share of the error's square is about 1 / sqrt(outputs), below
    1%). Against one maximum per item it is 1.4% to 4% larger."""
    b = build_batch([context], [tokens], dtype=dtype, num_q_heads=16, num_kv_heads=8,
                    head_dim=128, seed=11, device="cuda")
    ids = b.block_tables[0, : -(-context // 16)].long()
    k, v = (p[ids].double().reshape(-1, 8, 128)[:context].repeat_interleave(2, dim=1).transpose(0, 1)
            for p in (b.key_pool, b.value_pool))
    scores = b.q.double().transpose(0, 1) @ k.transpose(1, 2).contiguous() * b.scale
    hidden = torch.ones(tokens, context, dtype=torch.bool, device="cuda").triu(context - tokens + 1)
    want = (scores.masked_fill(hidden, -torch.inf).softmax(dim=-1) @ v).transpose(0, 1)
    whole, single = ((extension.paged_attention(*b.args(), plan_options=o).double() - want).norm()
                     for o in (WHOLE, CUT))
    assert whole <= 1.01 * single
