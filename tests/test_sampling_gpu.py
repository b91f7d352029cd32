"""The sampling distribution's kernels (``ops.sampling_probabilities``) on the MI355X
(``-m gpu``), against the float64 oracle: the kept sets exactly, the probabilities within
fp32 rounding: the scaled logit x and its distance from the maximum m are each rounded once
(2^-24 of their size, an absolute error of the exponent), expf, the sum and the division add
a few 2^-24, and the sum's own terms err as much again."""

from __future__ import annotations

import pytest
import torch

from torch.overrides import TorchFunctionMode
from torch.utils._python_dispatch import TorchDispatchMode

from mini_vllm.kernels import ops
from mini_vllm.sampler import SamplingParams, sampling_probabilities
from oracle import sampler as oracle

pytestmark = pytest.mark.gpu

PARAMS = [SamplingParams(0.7, 0, 0.9), SamplingParams(0.0), SamplingParams(1.3, 5, 1.0),
          SamplingParams(1.0), SamplingParams(0.9, 40, 0.6), SamplingParams(1.0, 0, 1e-6),
          SamplingParams(2.0, 3000, 0.999)]


def check(logits, rows):
    got = ops.sampling_probabilities(logits, rows, use_cuda=True)
    assert got is not None and got.dtype == torch.float32 and got.shape == logits.shape
    want = torch.from_numpy(oracle.sampling_probabilities(
        logits.float().cpu().numpy(), [torch.tensor(r.temperature).item() for r in rows],
        [r.top_k for r in rows], [torch.tensor(r.top_p).item() for r in rows]))
    got = got.double().cpu()
    tiny = want < 1e-30  # fp32 exponentials end there
    assert torch.equal(got[~tiny] > 0, want[~tiny] > 0), "kept sets differ"
    x = logits.float().cpu()
    x = x / torch.tensor([r.temperature or 1.0 for r in rows])[:, None]
    size = x[x.isfinite()].abs().max().item()
    assert torch.allclose(got, want, rtol=2 * (3 * size + 8) * 2.0 ** -24, atol=1e-30)


@pytest.mark.parametrize("dtype", [torch.float32, torch.float16, torch.bfloat16])
@pytest.mark.parametrize("vocab", [1, 3, 8, 511, 16384, 16385, 50257, 151936])
def test_matches_the_oracle(device, vocab, dtype):
    """Vocabularies around a chunk, a segment and several, aligned and not, rows of every
    kind in one call; 16-bit logits tie often."""
    gen = torch.Generator().manual_seed(vocab)
    logits = (torch.randn(len(PARAMS), vocab, generator=gen) * 2.5).to(dtype).to(device)
    check(logits, PARAMS)


@pytest.mark.parametrize("rows,vocab", [
    (256, 4096), (257, 4096), (128, 4097), (7, 32768), (32, 32769), (51, 40960), (52, 40960),
    (3, 524288), (4, 524289), (14, 151936)])
def test_segment_lengths(device, rows, vocab):
    """Both sides of each line where the segments' length changes, and of a segment's end."""
    gen = torch.Generator(device=device).manual_seed(rows)
    logits = torch.randn(rows, vocab, generator=gen, device=device) * 2.5
    check(logits.to(torch.bfloat16), [PARAMS[i % len(PARAMS)] for i in range(rows)])


@pytest.mark.parametrize("vocab", [700, 151936])
def test_many_tokens_at_the_boundary(device, vocab):
    """Flat rows: every token in one bin, all equal (kept by index) or apart by less than
    a bin, so the selection narrows thousands of tokens; a row far below its one peak."""
    flat = torch.full((vocab,), 1.5)
    close = torch.linspace(0.0, 0.05, vocab)[torch.randperm(vocab)]
    peak = torch.full((vocab,), -200.0)
    peak[vocab // 2] = 10.0
    rows = [SamplingParams(1.0, 0, 0.37), SamplingParams(1.0, vocab // 3, 1.0),
            SamplingParams(0.5, 0, 0.37), SamplingParams(1.0, vocab // 2, 0.9),
            SamplingParams(1.0, 600, 1.0), SamplingParams(1.0, 0, 0.5)]
    check(torch.stack([flat, flat, close, close, peak, peak]).to(device), rows)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("vocab", [513, 20000, 151936, 1048576])
def test_the_boundary_among_most_of_the_vocabulary(device, vocab, dtype):
    """Rows whose last kept token lies among most of the vocabulary's: one value everywhere,
    negative ones, values of both signs far below one peak, two interleaved values, and rows
    of which all but a few tokens are masked, with -inf or the type's lowest, while top_k asks
    for more of them."""
    gen = torch.Generator().manual_seed(vocab)
    x = torch.randn(8, vocab, generator=gen)
    allowed = torch.randperm(vocab, generator=gen)[:30]
    x[0] = -3.25
    x[1] *= 1e-3
    x[2, 77] = 25.0
    x[3] = torch.tensor([2.0, -2.0]).repeat(-(-vocab // 2))[:vocab]
    x[3, 5] = 40.0
    for row, mask in ((4, -torch.inf), (5, torch.finfo(dtype).min)):
        kept = x[row, allowed].clone()
        x[row] = mask
        x[row, allowed] = kept
    x[6] = -x[6].abs() - 20.0
    x[6, -1] = 1.0
    x[7] = 5.0 - torch.arange(vocab) * 2.0 ** -14
    rows = [SamplingParams(0.7, 0, 0.61), SamplingParams(1.0, vocab // 3, 1.0),
            SamplingParams(1.0, 50, 1.0), SamplingParams(1.0, vocab // 2 + 9, 1.0),
            SamplingParams(1.0, 50, 1.0), SamplingParams(0.6, 50, 0.999),
            SamplingParams(1.0, 501, 1.0), SamplingParams(1.3, vocab - 1, 0.9)]
    check(x.to(dtype).to(device), rows)


def test_no_row_costs_many_times_another(device):
    """A call's time on rows whose boundary lies among the whole vocabulary, against a call on
    ordinary rows beside it: the selection's few passes over one row's tokens (3 to 6 times,
    measured), not its steps for every token one after another (20 to 80 times)."""
    gen = torch.Generator(device=device).manual_seed(4)
    x = torch.randn(1, 151936, generator=gen, device=device)

    def fastest(logits, params):
        best = float("inf")
        for _ in range(8):
            start, end = (torch.cuda.Event(enable_timing=True) for _ in range(2))
            start.record()
            for _ in range(10):
                ops.sampling_probabilities(logits, params, use_cuda=True)
            end.record()
            end.synchronize()
            best = min(best, start.elapsed_time(end))
        return best
    params = [SamplingParams(1.0, 50, 1.0)]
    ordinary = fastest(x, params)
    peaked, masked = x.clone(), torch.full_like(x, -torch.inf)
    peaked[0, 9] = 25.0
    masked[0, :30] = x[0, :30]
    for odd in (torch.full_like(x, 1.5), peaked, masked):
        assert fastest(odd, params) < 12 * ordinary


def test_strided_rows_many_rows_and_signed_zeros(device):
    base = torch.randn(300, 1203, device=device)
    base[:, ::2] = 0.0
    base[:, 1::4] = -0.0
    rows = [PARAMS[i % len(PARAMS)] for i in range(300)]
    check(base[:, 3:1003], rows)


def test_non_finite_rows(device):
    """-inf tokens have no mass; a row holding NaN or +inf, or nothing but -inf, is all NaN
    (as softmax gives it); its neighbours are untouched."""
    x = torch.randn(6, 20000)
    x[0, 7:] = float("-inf")
    x[1, 19999] = float("nan")
    x[2, 3] = float("inf")
    x[3] = float("-inf")
    rows = [SamplingParams(0.8, 4, 0.95), SamplingParams(0.8, 4, 0.95), SamplingParams(1.0),
            SamplingParams(1.0, 0, 0.9), SamplingParams(0.0), SamplingParams(1.0, 2)]
    got = ops.sampling_probabilities(x.to(device), rows, use_cuda=True).cpu()
    assert bool(got[1:4].isnan().all())
    keep = [0, 4, 5]
    check(x[keep].to(device), [rows[i] for i in keep])
    assert torch.equal(got[keep], ops.sampling_probabilities(
        x[keep].to(device), [rows[i] for i in keep], use_cuda=True).cpu())


@pytest.mark.parametrize("temperature", [1e30, 1e38, 2.5e38])
def test_quotients_below_the_normal_range(device, temperature):
    """Temperatures so large that the scaled logits are subnormal: many tie, and the kept ones
    are still the first of the order by value, then index. (All are 1 / k: their differences
    are far below fp32.) Many top_k, so that tokens of the last kept value whose approximate
    quotient is off are among them."""
    x = torch.rand(1, 20000, generator=torch.Generator().manual_seed(1)) * 1e-4 + 0.0499
    ks = range(150, 19500, 151)
    got = ops.sampling_probabilities(x.expand(len(ks), -1).contiguous().to(device),
                                     [SamplingParams(temperature, k, 1.0) for k in ks], use_cuda=True)
    order = (x / temperature).sort(dim=-1, descending=True, stable=True).indices
    for row, k in zip(got.cpu(), ks):
        want = torch.zeros(20000).scatter_(0, order[0, :k], 1.0 / k)
        assert torch.equal(row > 0, want > 0)
        assert torch.allclose(row, want, rtol=1e-6)


def test_what_stays_on_the_torch_path(device):
    """Autograd, float64 and parameters outside float32 keep the torch path and its
    results."""
    x = torch.randn(2, 50, device=device)
    rows = [SamplingParams(0.7, 5, 0.9), SamplingParams()]
    grad = x.clone().requires_grad_()
    p = sampling_probabilities(grad, rows[:1] * 2)
    assert p.requires_grad
    assert torch.allclose(p.detach(), sampling_probabilities(x, rows[:1] * 2), rtol=1e-5)
    assert ops.sampling_probabilities(x.double(), rows, use_cuda=True) is None
    for odd in (SamplingParams(1e-40), SamplingParams(1e39), SamplingParams(1.0, 0, 1e-40)):
        assert ops.sampling_probabilities(x, [odd, odd], use_cuda=True) is None


def test_modes_and_traces_see_the_torch_path(device):
    """A dispatch or function mode and a trace see every step, as they did before there were
    kernels; the mode that only picks new tensors' device hides none."""
    class Dispatch(TorchDispatchMode):
        seen = 0

        def __torch_dispatch__(self, func, types, args=(), kwargs=None):
            self.seen += 1
            return func(*args, **(kwargs or {}))

    class Function(TorchFunctionMode):
        seen = 0

        def __torch_function__(self, func, types, args=(), kwargs=None):
            self.seen += 1
            return func(*args, **(kwargs or {}))
    x = torch.randn(3, 500, device=device)
    rows = [SamplingParams(0.7, 5, 0.9), SamplingParams(), SamplingParams(1.0, 0, 0.8)]
    want = sampling_probabilities(x, rows)
    for mode in (Dispatch(), Function()):
        with mode:
            assert ops.sampling_probabilities(x, rows, use_cuda=True) is None
            got = sampling_probabilities(x, rows)
        assert mode.seen > 5 and torch.allclose(got, want, rtol=1e-5)
    with torch.device(device):
        assert torch.equal(ops.sampling_probabilities(x, rows, use_cuda=True), want)
    traced = torch.jit.trace(lambda t: sampling_probabilities(t, rows), (x,), check_trace=False)
    y = torch.randn_like(x)
    assert torch.allclose(traced(y), sampling_probabilities(y, rows), rtol=1e-5)
