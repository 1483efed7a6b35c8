"""HIP graphs: a whole layer step (forward and backward, bf16 masters quantized
per call, top-8 routing so that the gathered GEMMs run), a decode step and a
GEMM whose last round is split. Every replay gives the eager step's results bit
for bit, with eager steps and synchronizations between the replays (a captured
memset or a library call that writes differently on replay would show here)."""

import math

import pytest
import torch

import mlops_amd
from mlops_amd import kernels as K

pytestmark = pytest.mark.gpu


def test_layer_step_replays_bitwise_in_a_graph(device):
    g = torch.Generator().manual_seed(11)
    tokens, hidden, inter, experts, top_k = 512, 512, 256, 16, 8
    x = torch.randn(tokens, hidden, generator=g).to(torch.bfloat16).to(device)
    res = torch.randn(tokens, hidden, generator=g).to(torch.bfloat16).to(device)
    dy = torch.randn(tokens, hidden, generator=g).to(torch.bfloat16).to(device)
    wr = (torch.randn(experts, hidden, generator=g) / math.sqrt(hidden)).to(device)
    w13 = (torch.randn(experts, 2 * inter, hidden, generator=g) * 0.02).to(torch.bfloat16).to(device)
    w2 = (torch.randn(experts, hidden, inter, generator=g) * 0.02).to(torch.bfloat16).to(device)
    leaves = [t.requires_grad_(True) for t in (x, wr, w13, w2)]
    daux = torch.full((), 0.01, device=device)
    holder = {}

    def step():
        for t in leaves:
            t.grad = None
        out, aux, _, _ = mlops_amd.moe(x, res, wr, w13, w2, top_k=top_k,
                                       routing_mode="topk_then_softmax",
                                       compute_precision="fp8_block")
        torch.autograd.backward([out, aux], [dy, daux])
        holder["out"] = out.detach()

    def results():
        return [holder["out"].clone()] + [t.grad.clone() for t in leaves]

    for _ in range(2):
        step()
    torch.cuda.synchronize()
    want = results()

    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        step()
    torch.cuda.current_stream().wait_stream(side)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        step()
    # The graph's own output tensors (an eager step below rebinds .grad).
    captured = [holder["out"]] + [t.grad for t in leaves]
    for _ in range(3):
        graph.replay()
        torch.cuda.synchronize()
        for got, ref in zip(captured, want):
            assert torch.equal(got, ref)
        step()
        torch.cuda.synchronize()
        for got, ref in zip(results(), want):
            assert torch.equal(got, ref)


def _replays_as_eager(step):
    """Captures ``step`` (a tuple of tensors), clears what it wrote before each
    of three replays, and holds them and eager steps between them against the
    eager result, bit for bit."""
    step()
    want = [t.clone() for t in step()]
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        step()
    torch.cuda.current_stream().wait_stream(side)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        captured = step()
    for _ in range(3):
        for t in captured:
            t.zero_()
        graph.replay()
        torch.cuda.synchronize()
        for got, ref in zip(captured, want, strict=True):
            assert torch.equal(got, ref)
        for got, ref in zip(step(), want, strict=True):
            assert torch.equal(got, ref)


@pytest.mark.parametrize("precision", ["fp8_block", "fp8_current"])
def test_few_token_forward_replays_bitwise_in_a_graph(device, precision):
    """A decode step: the routing of few tokens in two launches, small tiles."""
    g = torch.Generator().manual_seed(13)
    tokens, hidden, inter, experts, top_k = 24, 512, 256, 16, 8
    x = torch.randn(tokens, hidden, generator=g).to(torch.bfloat16).to(device)
    res = torch.randn(tokens, hidden, generator=g).to(torch.bfloat16).to(device)
    wr = (torch.randn(experts, hidden, generator=g) / math.sqrt(hidden)).to(device)
    w13 = (torch.randn(experts, 2 * inter, hidden, generator=g) * 0.02).to(torch.bfloat16).to(device)
    w2 = (torch.randn(experts, hidden, inter, generator=g) * 0.02).to(torch.bfloat16).to(device)
    if precision == "fp8_current":
        w13 = mlops_amd.RowFP8Weight.quantize(w13, interleaved=True)
        w2 = mlops_amd.RowFP8Weight.quantize(w2)
    else:
        w13, w2 = mlops_amd.BlockFP8Weight.quantize(w13), mlops_amd.BlockFP8Weight.quantize(w2)
    assert K._native.query("mi355x_moe_route_tokens_workspace_size", tokens, experts, top_k,
                           K.ROUTING_MODES["topk_then_softmax"], 1, 1, hidden) > 0

    def step():
        with torch.no_grad():
            return mlops_amd.moe(x, res, wr, w13, w2, top_k=top_k,
                                 routing_mode="topk_then_softmax")

    _replays_as_eager(step)


def test_split_last_round_replays_bitwise_in_a_graph(device):
    """Both launches of a GEMM whose last round of tiles is split over K, by
    itself and inside the down sequence, with their scratch from the graph's
    pool."""
    g = torch.Generator(device=device).manual_seed(17)
    counts, hidden, inter = [500, 400, 300, 500], 4096, 8192
    offsets = torch.tensor([0, *counts], device=device).cumsum(0).to(torch.int32)
    rows, experts = sum(counts), len(counts)
    assert K._native.query("mi355x_gemm_tail_workspace_size", rows, experts, hidden, inter) > 0

    def normal(*shape, std=1.0):
        return (torch.randn(*shape, generator=g, device=device) * std).to(torch.bfloat16)

    w2, w2_scale = K.quantize_weight_blocks(normal(experts, hidden, inter, std=0.02))
    h13, residual = normal(rows, 2 * inter), normal(rows, hidden)
    act, act_scale = K.swiglu_quantize(h13)
    slots = torch.arange(rows, dtype=torch.int32, device=device).view(rows, 1)
    weights = torch.ones(rows, 1, device=device)

    def step():
        return (K.gemm(act, act_scale, w2, w2_scale, offsets),
                K.moe_down(h13, w2, w2_scale, offsets, slots, weights, residual))

    _replays_as_eager(step)
