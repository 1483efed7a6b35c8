"""Kernel-level parity of the HIP entry points against the CPU oracle.

Bar: bit-exact for routing ids, the permutation (order / offsets / slots /
counts), every e4m3 byte and fp32 scale of the quantizers; GEMMs within
1e-2 worst-relative (per expert) of the fp64 product of the same
dequantized operands (the reference's own bound,
tests/test_block_fp8_transpose_gemm.py:486-531); fp32 router math within
1e-5 relative.
"""

import numpy as np
import pytest
import torch

from mlops_amd import kernels as K
from oracle import moe_oracle as O
from tests.conftest import frob_rel, max_rel, worst_cell_rel

pytestmark = pytest.mark.gpu


def _bytes(t):
    return t.detach().cpu().view(torch.uint8)


def _zipf_ids(tokens, top_k, experts, s, seed):
    rng = np.random.default_rng(seed)
    p = 1.0 / np.arange(1, experts + 1) ** s
    p /= p.sum()
    ids = np.stack([rng.choice(experts, size=top_k, replace=False, p=p) for _ in range(tokens)])
    return torch.from_numpy(ids.astype(np.int32))


# ------------------------------------------------------------------ router
@pytest.mark.parametrize("mode", ["topk_then_softmax", "softmax_then_topk", "sigmoid_noaux_tc"])
@pytest.mark.parametrize("experts,top_k", [(128, 8), (8, 2), (300, 6), (256, 8), (512, 32), (64, 1),
                                            (128, 16), (128, 17), (16, 16), (100, 3)])
def test_router_topk_matches_oracle(device, mode, experts, top_k):
    g = torch.Generator().manual_seed(experts + top_k)
    logits = torch.randn(1000, experts, generator=g)
    logits[3] = 0.0          # all tied
    logits[4, 1] = logits[4, experts - 1] = 4.0  # tie at the top
    w, ids = K.router_topk(logits.to(device), top_k, mode, routed_scaling=1.3)
    ow, oids = O.route(logits, top_k, mode, routed_scaling=1.3)
    assert torch.equal(ids.cpu(), oids)
    assert max_rel(w.cpu(), ow) < 1e-5


@pytest.mark.parametrize("mode", ["topk_then_softmax", "sigmoid_noaux_tc"])
@pytest.mark.parametrize("experts,top_k", [(128, 8), (300, 6)])
def test_router_topk_nan_and_signed_zero(device, mode, experts, top_k):
    """torch.sort's order on the awkward values: NaN ahead of every number,
    -0 equal to +0 (ties to the lower id), -inf last among numbers."""
    g = torch.Generator().manual_seed(5)
    logits = torch.randn(64, experts, generator=g)
    logits[0, 7] = float("nan")
    logits[1, [3, 9]] = float("nan")
    logits[2] = float("-inf")
    logits[2, 11] = 0.5
    logits[3] = 0.0
    logits[3, ::2] = -0.0
    logits[4, : experts - 2] = float("-inf")
    _, ids = K.router_topk(logits.to(device), top_k, mode)
    _, oids = O.route(logits, top_k, mode)
    assert torch.equal(ids.cpu(), oids)


def test_router_topk_group_limited(device):
    g = torch.Generator().manual_seed(11)
    logits = torch.randn(777, 64, generator=g)
    bias = torch.randn(64, generator=g) * 0.05
    w, ids = K.router_topk(logits.to(device), 6, "sigmoid_noaux_tc", bias=bias.to(device),
                           n_group=8, topk_group=3, routed_scaling=2.5)
    ow, oids = O.route(logits, 6, "sigmoid_noaux_tc", bias=bias, n_group=8, topk_group=3,
                       routed_scaling=2.5)
    assert torch.equal(ids.cpu(), oids)
    assert max_rel(w.cpu(), ow) < 1e-5


def test_router_forced_ids(device):
    g = torch.Generator().manual_seed(12)
    logits = torch.randn(50, 16, generator=g)
    forced = torch.stack([torch.randperm(16, generator=g)[:4] for _ in range(50)]).int()
    for mode in ("topk_then_softmax", "softmax_then_topk", "sigmoid_noaux_tc"):
        w, ids = K.router_topk(logits.to(device), 4, mode, forced_ids=forced.to(device))
        ow, oids = O.route(logits, 4, mode, forced_ids=forced)
        assert torch.equal(ids.cpu(), forced)
        assert max_rel(w.cpu(), ow) < 1e-5


@pytest.mark.parametrize("mode,lengths,experts,top_k", [
    ("topk_then_softmax", None, 32, 4),
    ("softmax_then_topk", None, 32, 4),
    ("topk_then_softmax", (300, 200), 32, 4),         # softmax aux over all segments
    ("sigmoid_noaux_tc", (100, 37, 363), 32, 4),
    ("softmax_then_topk", (77, 250, 173), 512, 8),   # 8 logits per lane, odd segments
    ("sigmoid_noaux_tc", (201, 299), 512, 6),
    ("topk_then_softmax", None, 64, 32),               # top_k near the lane limit
    ("sigmoid_noaux_tc", (13, 487), 64, 32),
    ("topk_then_softmax", None, 128, 8),               # two expert slots per lane
    ("softmax_then_topk", (250, 250), 200, 8),         # four slots per lane, masked tail
    ("sigmoid_noaux_tc", None, 256, 8),
])
def test_router_stats_and_backward(device, mode, lengths, experts, top_k):
    g = torch.Generator().manual_seed(13 + experts + top_k)
    tokens = 500
    lengths = (tokens,) if lengths is None else lengths
    logits = torch.randn(tokens, experts, generator=g)
    w, ids = O.route(logits, top_k, mode)
    aux, psum, seg_counts, seg_offsets = K.router_stats(logits.to(device), ids.to(device), top_k,
                                                        mode, lengths)
    oaux, ocounts, opsum = O.routing_statistics(logits, ids, mode, lengths, experts)
    assert abs(aux.item() - oaux.item()) <= 1e-5 * max(1.0, abs(oaux.item()))
    assert max_rel(psum.cpu(), opsum) < 1e-5
    assert torch.equal(seg_counts.cpu().sum(0).long(), ocounts)
    # backward: route-weight cotangent arrives as per-sorted-row dscore
    order, offsets, slots = O.sort_assignments(ids, experts)
    dscore = torch.randn(tokens * top_k, generator=g)
    gw = dscore[slots.reshape(-1).long()].view(tokens, top_k)
    ga = torch.tensor(0.3)
    gps = torch.randn(experts, generator=g)
    grad = K.router_backward(logits.to(device), w.to(device), ids.to(device), dscore.to(device),
                             slots.to(device), mode, grad_aux=ga.to(device),
                             grad_prob_sum=gps.to(device), offsets=offsets.to(device),
                             seg_offsets=seg_offsets, seg_counts=seg_counts)
    want = O.routing_gradient(ga, gps, gw, w, ids, logits, mode, lengths)
    assert max_rel(grad.cpu(), want) < 1e-5
    # the split form: [hi | mid] bf16 pieces of the same fp32 gradient, as
    # torch's casts make them
    pieces = K.router_backward(logits.to(device), w.to(device), ids.to(device),
                               dscore.to(device), slots.to(device), mode, grad_aux=ga.to(device),
                               grad_prob_sum=gps.to(device), offsets=offsets.to(device),
                               seg_offsets=seg_offsets, seg_counts=seg_counts, pieces=True).cpu()
    hi = grad.cpu().to(torch.bfloat16)
    assert torch.equal(pieces[:, :experts], hi)
    assert torch.equal(pieces[:, experts:], (grad.cpu() - hi.float()).to(torch.bfloat16))


@pytest.mark.parametrize("tokens,experts,hidden", [
    (16384, 128, 2048),   # C3's router
    (1000, 32, 256),      # ragged last step
    (37, 8, 512),         # one step, most expert rows masked
    (700, 200, 768),      # E not a multiple of the 128-row tile
    (513, 256, 256),      # two expert tiles
    (0, 16, 256),         # no tokens: zeros
])
def test_router_weight_grad_matches_fp64(device, tokens, experts, hidden):
    """dW = hi^T x + mid^T x (bf16 pieces, fp32 sums) against fp64 on the same
    bf16 operands, and equal to the pieces' fp32 cotangent within the bf16
    split's resolution."""
    g = torch.Generator().manual_seed(tokens + experts)
    grad = torch.randn(tokens, experts, generator=g) * 1e-3
    hi = grad.to(torch.bfloat16)
    mid = (grad - hi.float()).to(torch.bfloat16)
    pieces = torch.cat([hi, mid], 1)
    x = torch.randn(tokens, hidden, generator=g).to(torch.bfloat16)
    got = K.router_weight_grad(pieces.to(device), x.to(device)).cpu()
    want = hi.double().t() @ x.double() + mid.double().t() @ x.double()
    assert got.dtype == torch.float32 and got.shape == (experts, hidden)
    if tokens == 0:
        assert torch.count_nonzero(got) == 0
        return
    assert (got.double() - want).abs().max() <= 1e-5 * want.abs().max()
    # the split carries the fp32 cotangent to ~2^-16 relative
    exact = grad.double().t() @ x.double()
    assert (got.double() - exact).abs().max() <= 1e-4 * exact.abs().max()


# ------------------------------------------------------------------ permute
@pytest.mark.parametrize("tokens,top_k,experts,kind", [
    (16384, 8, 128, "uniform"),      # Qwen3-30B-A3B routing shape
    (4096, 8, 32, "zipf"),           # skewed, some experts empty
    (1, 3, 4, "uniform"),
    (777, 2, 1, "uniform"),          # one expert
    (5000, 1, 512, "uniform"),       # max experts
])
def test_permute_plan_bit_exact(device, tokens, top_k, experts, kind):
    if kind == "zipf":
        ids = _zipf_ids(tokens, top_k, experts, 1.2, seed=tokens)
    else:
        g = torch.Generator().manual_seed(tokens + experts)
        if top_k <= experts:
            ids = torch.stack([torch.randperm(experts, generator=g)[:top_k] for _ in range(tokens)]).int() \
                if tokens < 5000 else torch.randint(0, experts, (tokens, top_k), generator=g).int()
        else:
            ids = torch.randint(0, experts, (tokens, top_k), generator=g).int()
    counts, offsets, order, slots = K.permute_plan(ids.to(device), experts)
    oorder, ooffsets, oslots = O.sort_assignments(ids, experts)
    assert torch.equal(order.cpu(), oorder)
    assert torch.equal(offsets.cpu(), ooffsets)
    assert torch.equal(slots.cpu(), oslots)
    assert torch.equal(counts.cpu(), torch.bincount(ids.reshape(-1).long(), minlength=experts))


def test_permute_quantize_bit_exact(device):
    g = torch.Generator().manual_seed(14)
    tokens, width, top_k, experts = 700, 1024, 4, 16
    x = (torch.randn(tokens, width, generator=g) * 2).to(torch.bfloat16)
    x[7, :128] = 0  # zero group
    x[8, 5] = 300.0  # outlier
    ids = torch.stack([torch.randperm(experts, generator=g)[:top_k] for _ in range(tokens)]).int()
    order, offsets, slots = O.sort_assignments(ids, experts)
    q, s = K.permute_quantize(x.to(device), slots.to(device))
    oq, os_ = O.quantize_rows_1x128(x[order.long() // top_k])
    assert torch.equal(_bytes(q), oq.view(torch.uint8))
    assert torch.equal(s.cpu(), os_)


@pytest.mark.parametrize("mode", ["topk_then_softmax", "softmax_then_topk", "sigmoid_noaux_tc"])
@pytest.mark.parametrize("tokens,experts,top_k", [
    (1, 128, 8), (1, 1, 1), (16, 16, 2), (17, 33, 16), (63, 127, 5), (64, 128, 16),
    (65, 128, 8),            # two statistics chunks: the separate kernels
    (64, 129, 4), (64, 128, 17),
])
def test_route_in_one_launch_equals_separate_kernels(device, mode, tokens, experts, top_k):
    """Top-k, statistics and plan fused for few tokens, at the edges of its
    range: bitwise the separate kernels, with a bias, NaN, infinities and ties
    among the logits, and forced ids."""
    g = torch.Generator().manual_seed(tokens * experts + top_k)
    logits = torch.randn(tokens, experts, generator=g)
    logits[:, experts // 2] = logits[:, 0]
    logits[0, experts - 1] = float("inf") if top_k < experts else 0.0
    if tokens > 2:
        logits[1, 0] = -float("inf")
        logits[2] = 0.0
    if tokens > 16:
        logits[16, experts // 3] = float("nan")
    logits = logits.to(device)
    bias = (torch.randn(experts, generator=g) * 0.1).to(device)
    forced = torch.stack([torch.randperm(experts, generator=g)[:top_k]
                          for _ in range(tokens)]).to(torch.int32).to(device)
    for forced_ids in (None, forced):
        options = dict(bias=bias if mode == "sigmoid_noaux_tc" else None, routed_scaling=2.5,
                       forced_ids=forced_ids)
        got = K.route(logits, top_k, mode, (tokens,), **options)
        weights, ids = K.router_topk(logits, top_k, mode, **options)
        aux, prob_sum, _, _ = K.router_stats(logits, ids, top_k, mode, (tokens,))
        want = (weights, ids, *K.permute_plan(ids, experts), aux, prob_sum)
        for a, b in zip(got, want, strict=True):
            assert a.dtype == b.dtype and torch.equal(_bytes(a.reshape(-1)), _bytes(b.reshape(-1)))


@pytest.mark.parametrize("assignments,experts", [(1, 1), (1024, 300), (1025, 1024), (6144, 128),
                                                 (6145, 128)])
def test_permute_plan_around_the_one_block_size(device, assignments, experts):
    """The plan in one block (up to 6144 assignments) and in three kernels
    against the oracle's stable sort, with an overloaded and an empty expert."""
    g = torch.Generator().manual_seed(assignments)
    ids = torch.randint(0, experts, (assignments, 1), generator=g)
    ids[torch.rand(assignments, generator=g) < 0.3] = 0
    ids[ids == experts - 1] = 0
    ids = ids.to(torch.int32)
    counts, offsets, order, slots = K.permute_plan(ids.to(device), experts)
    want_order, want_offsets, want_slots = O.sort_assignments(ids, experts)
    assert torch.equal(order.cpu(), want_order) and torch.equal(offsets.cpu(), want_offsets)
    assert torch.equal(slots.cpu(), want_slots)
    assert torch.equal(counts.cpu(), torch.bincount(ids.reshape(-1).long(), minlength=experts))


@pytest.mark.parametrize("gate_up", [False, True])
def test_quantize_rows_bit_exact(device, gate_up):
    g = torch.Generator().manual_seed(15)
    x = (torch.randn(333, 1536, generator=g) * 0.1).to(torch.bfloat16)
    q, s = K.quantize_rows(x.to(device), gate_up=gate_up)
    src = x[:, O.gate_up_columns(1536)] if gate_up else x
    oq, os_ = O.quantize_rows_1x128(src)
    assert torch.equal(_bytes(q), oq.view(torch.uint8))
    assert torch.equal(s.cpu(), os_)


@pytest.mark.parametrize("limit", [None, 0.5])
def test_swiglu_quantize(device, limit):
    g = torch.Generator().manual_seed(16)
    h = torch.randn(257, 2 * 768, generator=g).to(torch.bfloat16)
    q, s = K.swiglu_quantize(h.to(device), limit)
    act = O.swiglu(h, limit)
    oq, os_ = O.quantize_rows_1x128(act)
    # exp() differs in the last ulp between libraries: scales agree to 1e-6,
    # bytes agree except where a value sits on a rounding boundary.
    assert max_rel(s.cpu(), os_) < 1e-6
    same = (_bytes(q) == oq.view(torch.uint8)).float().mean().item()
    assert same > 0.999
    assert max_rel(O.dequantize_rows(q.cpu(), s.cpu()), O.dequantize_rows(oq, os_)) < 0.07


@pytest.mark.parametrize("shape,dtype", [((4, 256, 384), torch.bfloat16),
                                         ((3, 208, 144), torch.float32)])
def test_quantize_weight_blocks_bit_exact(device, shape, dtype):
    g = torch.Generator().manual_seed(17)
    w = (torch.randn(*shape, generator=g) * 0.02).to(dtype)
    w[0, :128, :128] = 0
    w[1, 0, 0] = 2.0 ** 14 * 0.02
    data, scale, data_t = K.quantize_weight_blocks(w.to(device), transposed=True)
    od, os_ = O.quantize_blocks(w)
    assert torch.equal(_bytes(data), od.view(torch.uint8))
    assert torch.equal(scale.cpu(), os_)
    assert torch.equal(_bytes(data_t), od.transpose(1, 2).contiguous().view(torch.uint8))
    assert torch.equal(_bytes(K.transpose_fp8(data)), _bytes(data_t))


@pytest.mark.parametrize("gather,gate_up", [(False, False), (True, False), (False, True)])
def test_quantize_transpose_bit_exact(device, gather, gate_up):
    g = torch.Generator().manual_seed(18)
    experts, top_k, tokens, width = 6, 2, 400, 512
    ids = torch.stack([torch.randperm(experts, generator=g)[:top_k] for _ in range(tokens)]).int()
    ids[ids == 4] = 5  # expert 4 empty
    order, offsets, slots = O.sort_assignments(ids, experts)
    if gather:
        src = torch.randn(tokens, width, generator=g).to(torch.bfloat16)
        rows = src[order.long() // top_k]
        qt, st, padded = K.quantize_transpose(src.to(device), offsets.to(device), tokens * top_k,
                                              gather=order.to(device), gather_div=top_k)
    else:
        rows = torch.randn(tokens * top_k, width, generator=g).to(torch.bfloat16)
        src = rows
        qt, st, padded = K.quantize_transpose(rows.to(device), offsets.to(device), tokens * top_k,
                                              gate_up=gate_up)
    if gate_up:
        rows = rows[:, O.gate_up_columns(width)]
    oq, os_, total = O.quantize_transpose_padded(rows, offsets, padded)
    assert torch.equal(_bytes(qt)[:, :total], oq.view(torch.uint8)[:, :total])
    assert torch.equal(st.cpu()[: total // 128], os_[: total // 128])


# ------------------------------------------------------------------- GEMMs
def _ragged(counts):
    offs = [0]
    for c in counts:
        offs.append(offs[-1] + c)
    return torch.tensor(offs, dtype=torch.int32)


def _block_factors(g, shape, exponents):
    """A power of two per 128x128 block of a ``[E, R, C]`` weight, 2**e with e
    uniform over ``exponents``, and one all-zero block (the last expert's
    last block row, first block column), as the reference's block-weight
    helper builds them (tests/test_block_fp8_transpose_gemm.py:431-444)."""
    experts, r, c = shape
    lo, hi = exponents
    blocks = (experts, -(-r // 128), -(-c // 128))
    e = torch.randint(lo, hi + 1, blocks, generator=g).double()
    f = torch.exp2(e).float()
    if f.numel() > 1:
        f[-1, -1, 0] = 0.0
    return f.repeat_interleave(128, 1).repeat_interleave(128, 2)[:, :r, :c]


def _gemm_case(device, counts, n, k, *, seed, transposed=False, interleave=False,
               exponents=(-3, 3), addend=False, lora_rank=0):
    g = torch.Generator().manual_seed(seed)
    experts = len(counts)
    offsets = _ragged(counts)
    rows = int(offsets[-1])
    x = torch.randn(rows, k, generator=g).to(torch.bfloat16)
    wshape = (experts, k, n) if transposed else (experts, n, k)
    # Block scales a few powers of two apart (or 2^-14..2^14), so every
    # block's scale shows in every output cell.
    w = torch.randn(*wshape, generator=g) * 0.02 * _block_factors(g, wshape, exponents)
    xq, xs = K.quantize_rows(x.to(device))
    if transposed:
        wd, ws, wt = K.quantize_weight_blocks(w.to(device), transposed=True)
        wq_kernel = wt
    else:
        wd, ws = K.quantize_weight_blocks(w.to(device))
        wq_kernel = wd
    c = torch.randn(rows, n, generator=g).to(torch.bfloat16) if addend else None
    lora = None
    if lora_rank:
        zz = (torch.randn(rows, lora_rank, generator=g) * 0.5).to(torch.bfloat16)
        bb = (torch.randn(experts, n, lora_rank, generator=g) * 0.1).to(torch.bfloat16)
        lora = (zz.to(device), bb.to(device))
    out = K.gemm(xq, xs, wq_kernel, ws, offsets.to(device), transposed_scale=transposed,
                 interleave=interleave, addend=None if c is None else c.to(device), lora=lora)
    want = O.grouped_gemm(xq.cpu(), xs.cpu(), wd.cpu(), ws.cpu(), offsets, transposed=transposed,
                          interleave=interleave)
    if c is not None:
        want = want + c.double()
    if lora_rank:
        # The rank term in weight-row order (gate rows, then up rows), then
        # in the output's column order.
        term = torch.zeros(rows, n, dtype=torch.float64)
        for e in range(experts):
            lo, hi = int(offsets[e]), int(offsets[e + 1])
            term[lo:hi] = zz[lo:hi].double() @ bb[e].double().t()
        if interleave:
            term = term.view(rows, 2, n // 2).transpose(1, 2).reshape(rows, n)
        want = want + term
    return out.cpu(), want, offsets


COUNTS = [0, 70, 131, 15, 260]  # an empty expert, partial row tiles (reference COUNTS)


@pytest.mark.parametrize("case", [
    dict(counts=COUNTS, n=256, k=512),                                  # block scales 2^-3..2^3
    dict(counts=COUNTS, n=384, k=1024, exponents=(-14, 14)),            # extreme scales, zero block
    dict(counts=COUNTS, n=256, k=1024, exponents=(-14, 14), transposed=True),
    dict(counts=COUNTS, n=512, k=1024, exponents=(-14, 14), interleave=True),
    dict(counts=[129, 64, 257], n=256, k=384, interleave=True),         # gate/up interleaved output
    dict(counts=[100, 200, 0, 33], n=256, k=512, transposed=True),      # input-gradient orientation
    dict(counts=[90, 190], n=128, k=256, addend=True),                  # LoRA-style addend
    dict(counts=COUNTS, n=256, k=512, lora_rank=16),                    # rank term, empty expert
    dict(counts=[129, 64, 257], n=512, k=384, interleave=True, lora_rank=32),  # gate/up order
    dict(counts=[100, 200, 0, 33], n=256, k=512, transposed=True, lora_rank=16),  # input gradient
])
def test_grouped_gemm_matches_fp64(device, case):
    """Worst relative Frobenius error over (expert, 128-column) cells < 1e-2,
    the reference's GEMM metric (tests/test_block_fp8_transpose_gemm.py:
    390-406), so a block 2^28 times smaller than its neighbours is still
    checked at its own magnitude."""
    out, want, offsets = _gemm_case(device, seed=sum(case["counts"]) + case["k"], **case)
    assert torch.isfinite(out).all()
    assert worst_cell_rel(out, want, offsets.tolist()) < 1e-2



@pytest.mark.parametrize("tokens,width,experts,top_k,mode,dtype,quantize", [
    (1, 128, 1, 1, "topk_then_softmax", torch.float32, None),        # the smallest call
    (17, 2048, 128, 8, "topk_then_softmax", torch.float32, "blocks"),
    (64, 4224, 40, 5, "sigmoid_noaux_tc", torch.bfloat16, "rows"),   # a last K part of 128
    (33, 640, 9, 4, "softmax_then_topk", torch.bfloat16, "blocks"),
    (64, 7168, 128, 16, "softmax_then_topk", torch.float32, "rows"),
])
def test_route_tokens_against_separate_calls(device, tokens, width, experts, top_k, mode, dtype,
                                             quantize):
    """The logits against the fp64 product of the bf16 operands (fp32 sums of
    `width` products in chains of 32: 2^-24 * (32 + width / 32) of the sum of
    magnitudes bounds them), the routing of those logits and the quantized rows
    bitwise against the kernels called one at a time."""
    g = torch.Generator(device=device).manual_seed(tokens + width)
    x = torch.randn(tokens, width, generator=g, device=device).to(torch.bfloat16)
    w = (torch.randn(experts, width, generator=g, device=device) / width ** 0.5).to(dtype)
    bias = None
    if mode == "sigmoid_noaux_tc":
        bias = torch.randn(experts, generator=g, device=device) * 0.1
    options = dict(bias=bias, routed_scaling=2.5 if bias is not None else 1.0)
    logits, rows, routing = K.route_tokens(x, w, top_k, mode, (tokens,), quantize=quantize,
                                           **options)
    xd, wd = x.double(), w.to(torch.bfloat16).double()
    bound = xd.abs() @ wd.abs().t() * 2.0 ** -24 * (32 + width / 32)
    assert ((logits.double() - xd @ wd.t()).abs() <= bound).all()
    for a, b in zip(routing, K.route(logits, top_k, mode, (tokens,), **options), strict=True):
        assert torch.equal(a, b)
    if quantize is not None:
        q, s = (K.quantize_token_rows if quantize == "blocks" else K.quantize_rows_current)(x)
        assert torch.equal(_bytes(rows[0]), _bytes(q)) and torch.equal(rows[1], s)
    # Outside the range: more tokens, a group limit, sequences, an unaligned or
    # strided operand.
    assert K.route_tokens(x.expand(65, -1, -1)[:, 0].contiguous(), w, top_k, mode, (65,)) is None
    assert K.route_tokens(x.repeat(2, 1), w, top_k, mode, (tokens, tokens)) is None
    assert K.route_tokens(x, w.double(), top_k, mode, (tokens,)) is None
    if experts > 1:
        assert K.route_tokens(x, w.t().contiguous().t(), top_k, mode, (tokens,)) is None


# Row counts and N that reach each tile size of the grouped GEMM: 64-row tiles
# (few rows a group; 1 to 3 K steps, shorter than the copy pipeline), 128-row
# tiles (a 256 x 256 grid that fills less than half the CUs), the 256 x 256
# tiles, and 256 x 128 tiles (N an odd multiple of 128 over many row blocks).
TILE_CASES = [
    ([1, 63, 64, 65, 0, 17], 512, 128),
    ([1, 63, 64, 65, 0, 17], 768, 256),
    ([1, 63, 64, 65, 0, 17], 384, 384),
    ([3], 256, 1024),
    ([129, 160, 256, 1, 250], 512, 128),
    ([129, 160, 256, 1, 250], 256, 640),
    ([129, 160, 256, 1, 250], 384, 384),
    ([300, 511, 0, 900], 4096, 256),
    # 256 x 256 tiles with 1 to 4 of their 64-row groups in use, around each edge.
    ([257, 64, 321, 128, 129, 448, 705, 0, 255], 4096, 384),
    ([300, 511, 0, 900], 12416, 128),
]


@pytest.mark.parametrize("counts,n,k", TILE_CASES)
def test_grouped_gemm_forms_at_every_tile_size(device, counts, n, k):
    _every_form(device, counts, n, k)


# More tiles than the 2 x 256 workgroups of the 64- and 128-row tiles, so each
# walks several: its issue pointer and its two gathered-row tables cross tile
# borders, at K steps below, at and above the depth of the copy pipeline (3
# stages for 64 rows, 2 for 128), experts of no rows among them.
WALKED_64 = [(7 * e * e + 3) % 71 for e in range(24)] + [0]
WALKED_128 = [129, 10, 0, 256, 1, 9, 140, 0, 257, 30, 2, 127, 5, 0, 17, 33]


@pytest.mark.parametrize("tile,counts,n,k", [
    (64, WALKED_64, 4096, 128),
    (64, WALKED_64, 4096, 256),
    (64, WALKED_64, 4096, 384),
    (64, WALKED_64, 3072, 640),
    (128, WALKED_128, 8192, 128),
    (128, WALKED_128, 8192, 256),
    (128, WALKED_128, 8192, 384),
])
def test_grouped_gemm_forms_over_several_tiles(device, tile, counts, n, k):
    rows_per_expert = sum(counts) // len(counts)
    assert rows_per_expert <= 48 if tile == 64 else 48 < rows_per_expert <= 64
    tiles = sum(-(-c // tile) for c in counts) * (n // 128)
    assert tiles > 2 * torch.cuda.get_device_properties(device).multi_processor_count
    _every_form(device, counts, n, k)


def _every_form(device, counts, n, k):
    """Every operand form at each tile size against the fp64 product of the
    dequantized operands. Bound: one bf16 rounding of the result is 2^-9 of
    each element, fp32 sums of K / 128 block partials add 1e-6, and a 128
    column cell averages them: 4e-3 is twice the worst rounding. Forms that
    read the same operands another way are bitwise equal."""
    for options in (dict(), dict(transposed=True), dict(interleave=True), dict(addend=True),
                    dict(lora_rank=16), dict(lora_rank=32, interleave=True)):
        if options.get("lora_rank") and n % 256:
            continue  # the rank forms take N in multiples of 256
        out, want, offsets = _gemm_case(device, counts, n, k, seed=n + k, **options)
        assert torch.isfinite(out).all(), options
        assert worst_cell_rel(out, want, offsets.tolist()) < 4e-3, options
    if n % 256:
        return
    g = torch.Generator().manual_seed(n * k)
    offsets = _ragged(counts).to(device)
    rows, experts, tokens = int(offsets[-1]), len(counts), 37
    slots = torch.randint(0, 3 * tokens, (rows,), generator=g).to(torch.int32).to(device)
    x = torch.randn(tokens, k, generator=g).to(torch.bfloat16).to(device)
    routed = x[(slots // 3).long()]
    tq, ts = K.quantize_token_rows(x)
    xq, xs = K.quantize_rows(routed)
    w = (torch.randn(experts, n, k, generator=g) * 0.02).to(device)
    wq, ws = K.quantize_weight_blocks(w)
    for interleave in (False, True):
        assert torch.equal(
            K.gemm_gathered(tq, ts, slots, wq, ws, offsets, interleave=interleave, rows_div=3),
            K.gemm(xq, xs, wq, ws, offsets, interleave=interleave))
    kq, ks = K.quantize_weight_blocks(w.transpose(1, 2).contiguous())
    want = K.gemm(xq, xs, K.transpose_fp8(kq), ks, offsets, transposed_scale=True)
    assert torch.equal(K.gemm_kmajor(xq, xs, kq, ks, offsets), want)
    assert torch.equal(K.gemm_gathered(tq, ts, slots, kq, ks, offsets, kmajor=True, rows_div=3),
                       want)
    h, act, act_s = K.gemm_swiglu(xq, xs, wq, ws, offsets)
    assert torch.equal(h, K.gemm(xq, xs, wq, ws, offsets, interleave=True))
    q_ref, s_ref = K.swiglu_quantize(h)
    assert torch.equal(_bytes(act), _bytes(q_ref)) and torch.equal(act_s, s_ref)
    rq, _, rs, _ = K.quantize_weights_current(w)
    cq, cs = K.quantize_rows_current(routed)
    out = K.gemm_rowwise(cq, cs, rq, rs, offsets)
    want = O.rowwise_gemm(cq.cpu(), cs.cpu(), rq.cpu(), rs.cpu(), offsets.cpu())
    assert worst_cell_rel(out.cpu(), want, offsets.tolist()) < 4e-3
    ctq, cts = K.quantize_rows_current(x)
    assert torch.equal(K.gemm_rowwise_gathered(ctq, cts, slots, rq, rs, offsets, rows_div=3), out)
    z = (torch.randn(rows, 16, generator=g) * 0.5).to(torch.bfloat16)
    b = (torch.randn(experts, n, 16, generator=g) * 0.1).to(torch.bfloat16)
    out = K.gemm_rowwise(cq, cs, rq, rs, offsets, lora=(z.to(device), b.to(device)))
    for e, (lo, hi) in enumerate(zip(offsets.tolist(), offsets.tolist()[1:])):
        want[lo:hi] += z[lo:hi].double() @ b[e].double().t()
    assert worst_cell_rel(out.cpu(), want, offsets.tolist()) < 4e-3


@pytest.mark.parametrize("counts,n,k,rows", [
    ([1, 63, 64, 65, 0, 300, 17], 4096, 128, 2304),   # 64-row tiles; nk = 1
    ([1, 63, 64, 65, 0, 300, 17], 4096, 384, 2304),   # nk < 8: the full rotation
    ([1, 63, 64, 65, 0, 300, 17], 4096, 1024, 2304),  # nk >= 8: three starts
    ([1, 63, 64, 65, 0, 300, 17], 4096, 6144, 2304),  # the large weight's order: no rotation
    ([129, 600, 1, 0, 70], 4096, 640, 2304),          # 128-row tiles
    ([500, 520, 500, 530, 0, 510, 1, 515], 512, 1152, 16384),  # wide grid too small
])
def test_small_tiles_sum_in_the_wide_tiles_order(device, monkeypatch, counts, n, k, rows):
    """A launch on smaller tiles gives the bytes of the 256 x 256 tiles. The
    rows of the operand, not those the offsets cover, decide the tiles, so the
    same groups with ``rows`` operand rows run on the wide ones."""
    monkeypatch.setattr(K, "_TAIL_MIN_K", 1 << 30)  # whole tiles on both sides
    g = torch.Generator(device=device).manual_seed(n + k)
    offsets = _ragged(counts).to(device)
    used, experts, tokens = int(offsets[-1]), len(counts), 211
    slots = torch.randint(0, 3 * tokens, (rows,), generator=g, device=device).to(torch.int32)
    x = torch.randn(tokens, k, generator=g, device=device).to(torch.bfloat16)
    w = (torch.randn(experts, n, k, generator=g, device=device) * 0.02).to(torch.bfloat16)
    tq, ts = K.quantize_token_rows(x)
    ctq, cts = K.quantize_rows_current(x)
    wq, ws = K.quantize_weight_blocks(w)
    kq, ks = K.quantize_weight_blocks(w.transpose(1, 2).contiguous())
    rq, _, rs, _ = K.quantize_weights_current(w)
    b = (torch.randn(experts, n, 16, generator=g, device=device) * 0.1).to(torch.bfloat16)
    z = (torch.randn(rows, 16, generator=g, device=device) * 0.5).to(torch.bfloat16)

    def forms(count):
        routed = x[(slots[:count] // 3).long()]
        xq, xs = K.quantize_rows(routed)
        cq, cs = K.quantize_rows_current(routed)
        return dict(
            plain=K.gemm(xq, xs, wq, ws, offsets),
            interleaved=K.gemm(xq, xs, wq, ws, offsets, interleave=True),
            rank=K.gemm(xq, xs, wq, ws, offsets, lora=(z[:count], b)),
            gathered=K.gemm_gathered(tq, ts, slots[:count], wq, ws, offsets, rows_div=3),
            kmajor=K.gemm_kmajor(xq, xs, kq, ks, offsets),
            kmajor_gathered=K.gemm_gathered(tq, ts, slots[:count], kq, ks, offsets, kmajor=True,
                                            rows_div=3),
            rows=K.gemm_rowwise(cq, cs, rq, rs, offsets),
            rows_rank=K.gemm_rowwise(cq, cs, rq, rs, offsets, lora=(z[:count], b)),
            rows_gathered=K.gemm_rowwise_gathered(ctq, cts, slots[:count], rq, rs, offsets,
                                                  rows_div=3),
        )

    small, wide = forms(used), forms(rows)
    for name, out in small.items():
        assert torch.equal(out, wide[name][:used]), name


@pytest.mark.parametrize("counts,n,k", [
    ([300, 511, 0, 900, 130], 8192, 4096),  # a full round, then 4 tiles an XCD in 4 parts
    ([500, 400, 300, 500], 4096, 8192),  # fewer tiles than CUs: 16 an XCD in 2 parts
    ([1000, 900, 800, 700, 600, 620], 4096, 8192),  # a full round, then 10 an XCD in 3
])
def test_grouped_gemm_last_round_split_over_k(device, monkeypatch, counts, n, k):
    """Every form whose last round of tiles is split over K against the whole
    tiles' result, and the plain ones against the fp64 product. Both results
    are one bf16 rounding (2^-9 of each element) of fp32 sums that agree to
    1e-6, so they differ by at most 2 * 2^-9 < 4e-3 of a cell's norm."""
    g = torch.Generator(device=device).manual_seed(n + k)
    offsets = _ragged(counts).to(device)
    bounds = offsets.tolist()
    rows, experts, tokens = bounds[-1], len(counts), 301
    assert K._native.query("mi355x_gemm_tail_workspace_size", rows, experts, n, k) > 0

    def normal(*shape, std=1.0):
        return (torch.randn(*shape, generator=g, device=device) * std).to(torch.bfloat16)

    def product(a, w):
        out = torch.empty(rows, n, dtype=torch.float64, device=device)
        for e, (lo, hi) in enumerate(zip(bounds, bounds[1:])):
            out[lo:hi] = a(lo, hi) @ w(e).t()
        return out

    slots = torch.randint(0, 3 * tokens, (rows,), generator=g, device=device).to(torch.int32)
    x = normal(tokens, k)
    routed = x[(slots // 3).long()]
    w = normal(experts, n, k, std=0.02)
    xq, xs = K.quantize_rows(routed)
    tq, ts = K.quantize_token_rows(x)
    wq, ws = K.quantize_weight_blocks(w)
    kq, ks = K.quantize_weight_blocks(w.transpose(1, 2).contiguous())
    kt = K.transpose_fp8(kq)
    rq, _, rs, _ = K.quantize_weights_current(w)
    cq, cs = K.quantize_rows_current(routed)
    ctq, cts = K.quantize_rows_current(x)
    c, z, b = normal(rows, n), normal(rows, 16, std=0.5), normal(experts, n, 16, std=0.1)
    forms = dict(
        plain=lambda: K.gemm(xq, xs, wq, ws, offsets),
        gathered=lambda: K.gemm_gathered(tq, ts, slots, wq, ws, offsets, rows_div=3),
        interleaved=lambda: K.gemm(xq, xs, wq, ws, offsets, interleave=True),
        swiglu=lambda: K.gemm_swiglu(xq, xs, wq, ws, offsets)[0],
        addend=lambda: K.gemm(xq, xs, wq, ws, offsets, addend=c),
        rank=lambda: K.gemm(xq, xs, wq, ws, offsets, lora=(z, b)),
        transposed=lambda: K.gemm(xq, xs, kt, ks, offsets, transposed_scale=True),
        kmajor=lambda: K.gemm_kmajor(xq, xs, kq, ks, offsets),
        kmajor_gathered=lambda: K.gemm_gathered(tq, ts, slots, kq, ks, offsets, kmajor=True,
                                                rows_div=3),
        rows=lambda: K.gemm_rowwise(cq, cs, rq, rs, offsets),
        rows_gathered=lambda: K.gemm_rowwise_gathered(ctq, cts, slots, rq, rs, offsets,
                                                      rows_div=3),
        rows_rank=lambda: K.gemm_rowwise(cq, cs, rq, rs, offsets, lora=(z, b)),
    )
    split = {name: form() for name, form in forms.items()}
    for name, form in forms.items():
        assert torch.equal(split[name], form()), name  # the parts are added in a fixed order
    for name, same in (("plain", "gathered"), ("interleaved", "swiglu"),
                       ("transposed", "kmajor"), ("kmajor", "kmajor_gathered"),
                       ("rows", "rows_gathered")):
        assert torch.equal(split[name], split[same]), same
    monkeypatch.setattr(K, "_TAIL_MIN_K", 1 << 30)
    for name, form in forms.items():
        whole = form()
        if not name.startswith("rows"):  # (unscaled e4m3 products add up exactly)
            assert not torch.equal(split[name], whole), name  # the split did run
        assert worst_cell_rel(split[name], whole, bounds) < 4e-3, name
    xd = xq.double() * xs.t().double().repeat_interleave(128, 1)
    wd = lambda e: wq[e].double() * ws[e].double().repeat_interleave(128, 0).repeat_interleave(128, 1)
    assert worst_cell_rel(split["plain"], product(lambda lo, hi: xd[lo:hi], wd), bounds) < 4e-3
    cd = cq.double() * cs.double()[:, None]
    rd = lambda e: rq[e].double() * rs[e].double()[:, None]
    assert worst_cell_rel(split["rows"], product(lambda lo, hi: cd[lo:hi], rd), bounds) < 4e-3


@pytest.mark.parametrize("rows,experts,n,k,wanted", [
    (4096, 8, 4096, 14336, True),    # 40 tiles an XCD expected: 8 in the last round
    (16384, 32, 4096, 7168, True),   # 160 expected, a full round; a block more leaves 2
    (2048, 8, 4096, 14336, False),   # 24 expected, 22 to 26 likely: no half-empty round
    (16384, 32, 7168, 2048, False),  # K too short to split
    (640, 8, 4096, 14336, False),    # smaller tiles
    (2304, 16, 4096, 8192, True),    # 144 rows an expert: wide ones, 2 of 34 an XCD left over
    (0, 8, 4096, 14336, False),
])
def test_gemm_tail_workspace_where_a_short_last_round_is_likely(device, rows, experts, n, k,
                                                                wanted):
    size = K._native.query("mi355x_gemm_tail_workspace_size", rows, experts, n, k)
    assert (size > 0) == wanted


@pytest.mark.parametrize("tokens,top_k,experts,k,n,form", [
    (2000, 4, 16, 512, 512, "up"),           # gate/up interleave, partial row tiles
    (1000, 3, 8, 128, 256, "plain"),         # one K step: the next tile's rows at once
    (777, 2, 5, 1024, 768, "kmajor"),        # input gradient through a K-major weight
    (16384, 8, 128, 2048, 1536, "up"),       # C3's up projection
    (16384, 8, 128, 2048, 768, "kmajor"),    # C3's input gradient through W2
    (600, 16, 64, 256, 512, "up"),           # top-16: slot order / 16 in the kernel
])
def test_grouped_gemm_gathered_matches_permuted_copy(device, tokens, top_k, experts, k, n, form):
    """Token rows quantized once and read through the routed rows' tokens
    (a_rows = order // top_k) give the same bytes as the routed-row GEMM on
    the permuted copy; the per-token quantization equals the permuted one."""
    g = torch.Generator().manual_seed(tokens + k + n)
    logits = torch.randn(tokens, experts, generator=g)
    logits[:, 1] -= 30.0  # expert 1 empty
    x = torch.randn(tokens, k, generator=g).to(torch.bfloat16).to(device)
    _, ids = K.router_topk(logits.to(device), top_k, "topk_then_softmax")
    _, offsets, order, slots = K.permute_plan(ids, experts)
    a_rows = (order // top_k).to(torch.int32)
    xq, xs = K.permute_quantize(x, slots)
    tq, ts = K.quantize_token_rows(x)
    assert torch.equal(_bytes(tq[a_rows.long()]), _bytes(xq))
    assert torch.equal(ts[a_rows.long()].t().cpu(), xs.cpu())
    w = (torch.randn(experts, n, k, generator=g) * 0.02).to(torch.bfloat16).to(device)
    if form == "kmajor":
        wk = w.transpose(1, 2).contiguous()              # [E, K, N] as stored
        wq, ws = K.quantize_weight_blocks(wk)
        want = K.gemm_kmajor(xq, xs, wq, ws, offsets)
        got = K.gemm_gathered(tq, ts, a_rows, wq, ws, offsets, kmajor=True)
        # The plan's slot order itself, divided by top_k in the kernel.
        got_slots = K.gemm_gathered(tq, ts, order, wq, ws, offsets, kmajor=True, rows_div=top_k)
    else:
        wq, ws = K.quantize_weight_blocks(w)
        inter = form == "up"
        want = K.gemm(xq, xs, wq, ws, offsets, interleave=inter)
        got = K.gemm_gathered(tq, ts, a_rows, wq, ws, offsets, interleave=inter)
        got_slots = K.gemm_gathered(tq, ts, order, wq, ws, offsets, interleave=inter,
                                    rows_div=top_k)
    assert torch.equal(got.cpu(), want.cpu())
    assert torch.equal(got_slots.cpu(), want.cpu())


@pytest.mark.parametrize("form", ["up", "kmajor"])
def test_grouped_gemm_gathered_matches_fp64(device, form):
    """The gathered GEMMs on the C3 hot path (the interleaved up projection
    and r = dy @ W2 through the K-major weight) checked directly against the
    fp64 product of the dequantized operands, under the reference's metric
    (worst relative Frobenius error over (expert, 128-column) cells < 1e-2,
    tests/test_block_fp8_transpose_gemm.py:390-406): weight block scales
    2^-14..2^14 with an all-zero block, an empty expert, partial row blocks,
    and one token row scaled by 2^12 (its 1x128 scales ~4096 times its
    neighbours', read token-major through each of its routed rows)."""
    tokens, top_k, experts = 700, 4, 6
    k, n = (512, 768) if form == "up" else (1024, 512)
    g = torch.Generator().manual_seed(41 + k)
    logits = torch.randn(tokens, experts, generator=g)
    logits[:, 2] -= 30.0  # expert 2 empty
    x = torch.randn(tokens, k, generator=g)
    x[17] *= 2.0 ** 12
    x = x.to(torch.bfloat16).to(device)
    _, ids = K.router_topk(logits.to(device), top_k, "topk_then_softmax")
    _, offsets, order, _ = K.permute_plan(ids, experts)
    a_rows = (order // top_k).to(torch.int32)
    tq, ts = K.quantize_token_rows(x)
    wshape = (experts, k, n) if form == "kmajor" else (experts, n, k)
    w = torch.randn(*wshape, generator=g) * 0.02 * _block_factors(g, wshape, (-14, 14))
    wq, ws = K.quantize_weight_blocks(w.to(device))
    got = K.gemm_gathered(tq, ts, a_rows, wq, ws, offsets, interleave=form == "up",
                          kmajor=form == "kmajor").cpu()
    rows = a_rows.long().cpu()
    xq, xs = tq.cpu()[rows], ts.cpu()[rows].t().contiguous()
    want = O.grouped_gemm(xq, xs, wq.cpu(), ws.cpu(), offsets.cpu(),
                          transposed=form == "kmajor", interleave=form == "up")
    bounds = offsets.cpu().tolist()
    assert bounds[3] == bounds[2]  # the empty expert
    assert torch.isfinite(got).all()
    assert worst_cell_rel(got, want, bounds) < 1e-2


@pytest.mark.parametrize("tokens,top_k,experts,k,n", [
    (1500, 4, 16, 512, 512),
    (16384, 8, 128, 2048, 1536),             # C3's up projection at fp8_current
])
def test_rowwise_gemm_gathered_matches_permuted_copy(device, tokens, top_k, experts, k, n):
    """The row-scaled GEMM on token rows read through the routed rows equals
    the one on the permuted copy bit for bit (per-row descales in the epilogue
    taken from the tokens)."""
    g = torch.Generator().manual_seed(tokens + n)
    logits = torch.randn(tokens, experts, generator=g)
    logits[:, 2] -= 30.0
    x = torch.randn(tokens, k, generator=g).to(torch.bfloat16).to(device)
    _, ids = K.router_topk(logits.to(device), top_k, "topk_then_softmax")
    _, offsets, order, slots = K.permute_plan(ids, experts)
    a_rows = (order // top_k).to(torch.int32)
    xq, xs = K.permute_quantize_current(x, slots)
    tq, ts = K.quantize_rows_current(x)
    assert torch.equal(_bytes(tq[a_rows.long()]), _bytes(xq))
    assert torch.equal(ts[a_rows.long()].cpu(), xs.cpu())
    w = (torch.randn(experts, n, k, generator=g) * 0.02).to(torch.bfloat16).to(device)
    wq, _, wsc, _ = K.quantize_weights_current(w)
    want = K.gemm_rowwise(xq, xs, wq, wsc, offsets)
    got = K.gemm_rowwise_gathered(tq, ts, a_rows, wq, wsc, offsets)
    assert torch.equal(got.cpu(), want.cpu())
    got_slots = K.gemm_rowwise_gathered(tq, ts, order, wq, wsc, offsets, rows_div=top_k)
    assert torch.equal(got_slots.cpu(), want.cpu())


@pytest.mark.parametrize("counts,k,n", [
    (COUNTS, 512, 256),                      # empty expert, partial row tiles
    ([300, 0, 520, 45], 1536, 2048),         # C3's input gradient through W13 (K = 2I)
    ([129, 64, 257], 2048, 768),             # C3's input gradient through W2 (N = I)
    ([40, 700], 14336, 4096),                # Mixtral's K, the large-weight tile order
])
def test_grouped_gemm_kmajor_matches_transposed_copy(device, counts, k, n):
    """The input-gradient GEMM on the weight as stored ([E, K, N], fragments
    through ds_read_b64_tr_b8) is bitwise the GEMM on its transposed copy
    (same products, same MFMA K grouping), including extreme block scales and
    a zero block."""
    g = torch.Generator().manual_seed(k + n + sum(counts))
    offsets = _ragged(counts)
    rows, experts = int(offsets[-1]), len(counts)
    x = torch.randn(rows, k, generator=g).to(torch.bfloat16).to(device)
    w = (torch.randn(experts, k, n, generator=g) * 0.02)
    w[0, :128, :128] *= 2.0 ** 12
    w[-1, 128:256, :128] = 0.0
    xq, xs = K.quantize_rows(x)
    wq, ws, wt = K.quantize_weight_blocks(w.to(device), transposed=True)
    off = offsets.to(device)
    want = K.gemm(xq, xs, wt, ws, off, transposed_scale=True)
    got = K.gemm_kmajor(xq, xs, wq, ws, off)
    assert torch.equal(got, want)


def test_grouped_gemm_baseline_config2_row_blocks(device):
    """The BASELINE single-GEMM config (E=8, K=4096, N=2048, M_e ~ U{256..4096}
    step 128) under the reference's per-cell metric: each expert's first and
    last full 256-row blocks (every output column of them) against fp64,
    worst relative Frobenius error over (block, 128-column) cells < 1e-2."""
    rng = np.random.default_rng(2)
    counts = (rng.integers(2, 33, size=8) * 128).tolist()
    g = torch.Generator().manual_seed(3)
    offsets = _ragged(counts)
    rows = int(offsets[-1])
    x = torch.randn(rows, 4096, generator=g).to(torch.bfloat16).to(device)
    w = (torch.randn(8, 2048, 4096, generator=g) * 0.02).to(device)
    xq, xs = K.quantize_rows(x)
    wq, ws = K.quantize_weight_blocks(w)
    out = K.gemm(xq, xs, wq, ws, offsets.to(device)).cpu()
    a = O.dequantize_rows(xq.cpu(), xs.cpu()).double()
    wd = O.dequantize_blocks(wq.cpu(), ws.cpu()).double()
    worst = 0.0
    for e in range(8):
        lo, hi = int(offsets[e]), int(offsets[e + 1])
        for start in sorted({lo, hi - 256}):
            sel = slice(start, start + 256)
            want = a[sel] @ wd[e].t()
            worst = max(worst, worst_cell_rel(out[sel], want, [0, 256]))
    assert worst < 1e-2


@pytest.mark.parametrize("interleave", [False, True])
def test_grouped_gemm_large_weight_tile_order(device, interleave):
    """Experts whose weight is 24 MB or more (N x K e4m3 bytes) run in the
    grouped tile order: 8 N tiles x all the expert's row blocks, unrotated.
    N = 6400 gives groups of 8, 8, 8 and 1 N tiles; an empty expert and
    partial row blocks are included. Every output element is checked
    against the dequantized oracle operands multiplied in fp32."""
    counts, n, k = [300, 0, 520, 45], 6400, 4096
    assert n * k >= 24 << 20
    g = torch.Generator().manual_seed(17)
    offsets = _ragged(counts)
    rows = int(offsets[-1])
    x = torch.randn(rows, k, generator=g).to(torch.bfloat16).to(device)
    w = (torch.randn(len(counts), n, k, generator=g) * 0.02).to(torch.bfloat16).to(device)
    xq, xs = K.quantize_rows(x)
    wq, ws = K.quantize_weight_blocks(w)
    out = K.gemm(xq, xs, wq, ws, offsets.to(device), interleave=interleave)
    a = O.dequantize_rows(xq.cpu(), xs.cpu()).float().to(device)
    for e, count in enumerate(counts):
        lo, hi = int(offsets[e]), int(offsets[e + 1])
        if hi == lo:
            continue
        wd = O.dequantize_blocks(wq[e:e + 1].cpu(), ws[e:e + 1].cpu())[0].float().to(device)
        want = a[lo:hi] @ wd.t()
        if interleave:  # output columns 2j, 2j + 1 = gate j, up j
            want = want.view(hi - lo, 2, n // 2).transpose(1, 2).reshape(hi - lo, n)
        assert max_rel(out[lo:hi].float(), want) < 1e-2, e
        assert worst_cell_rel(out[lo:hi], want, [0, hi - lo]) < 1e-2, e


def test_rowwise_gemm_large_weight_tile_order(device):
    """The row-scaled kernel in the grouped tile order (same shape rule)."""
    counts, n, k = [0, 260, 700], 6400, 4096
    g = torch.Generator().manual_seed(19)
    offsets = _ragged(counts)
    rows = int(offsets[-1])
    x = torch.randn(rows, k, generator=g).to(torch.bfloat16).to(device)
    w = (torch.randn(len(counts), n, k, generator=g) * 0.02).to(torch.bfloat16).to(device)
    xq, xs = K.quantize_rows_current(x)
    wq, _, wsc, _ = K.quantize_weights_current(w)
    out = K.gemm_rowwise(xq, xs, wq, wsc, offsets.to(device))
    a = xq.float() * xs[:, None]
    for e, count in enumerate(counts):
        lo, hi = int(offsets[e]), int(offsets[e + 1])
        if hi == lo:
            continue
        want = a[lo:hi] @ (wq[e].float() * wsc[e][:, None]).t()
        assert max_rel(out[lo:hi].float(), want) < 1e-2, e


# Both on the 128 x 128 tiles, (256, 384) outside the widths of the wide ones.
@pytest.mark.parametrize("features", [(256, 384), (512, 768)])
@pytest.mark.parametrize("out_dtype", [torch.float32, torch.bfloat16])
def test_wgrad_matches_fp64(device, out_dtype, features):
    g = torch.Generator().manual_seed(19)
    counts = [0, 300, 50, 129]
    offsets = _ragged(counts)
    rows = int(offsets[-1])
    p_rows = torch.randn(rows, features[0], generator=g).to(torch.bfloat16)
    q_rows = torch.randn(rows, features[1], generator=g).to(torch.bfloat16)
    p_rows[7] *= 1e4  # spread the per-block scales over many binades
    q_rows[:, 5] *= 1e-5
    pt, pts, padded = K.quantize_transpose(p_rows.to(device), offsets.to(device), rows)
    qt, qts, _ = K.quantize_transpose(q_rows.to(device), offsets.to(device), rows, padded=padded)
    out = K.wgrad(pt, pts, qt, qts, offsets.to(device), out_dtype=out_dtype).cpu()
    want = O.wgrad(pt.cpu(), pts.cpu(), qt.cpu(), qts.cpu(), offsets)
    assert torch.all(out[0] == 0)
    tol = 1e-4 if out_dtype == torch.float32 else 1e-2  # fp32 accumulation order
    for e in range(1, 4):
        assert max_rel(out[e], want[e]) < tol, e
        # per (128-row, 128-column) cell, as the reference measures GEMMs
        assert worst_cell_rel(out[e], want[e], list(range(0, features[0] + 1, 128))) < tol, e


@pytest.mark.parametrize("counts,features", [
    ([0, 1, 128, 129, 0], (128, 384)),                 # 128 x 128 tiles, odd multiples of 128
    ([40, 300, 0, 257], (384, 640)),                   # several K blocks, an empty expert
    ([3] * 31 + [0], (1024, 512)),                     # 256 tiles of 256 x 256: the wide kernel
    ([130] * 7 + [0] * 18 + [1] * 7, (512, 1024)),
    # Several tiles a workgroup (1440 on 512, 384 on 256), and with them the wait
    # that leaves the last tile's stores in flight: experts of no rows at the
    # start, in the middle and at the end, of one row and of many K blocks.
    ([0, 1, 300, 129, 0, 0, 1, 700, 128, 1, 0, 513, 2, 40, 1, 0], (1280, 1152)),
    ([0, 1, 300, 129, 0, 0, 1, 700, 128, 1, 0, 513, 2, 40, 1, 0], (1024, 1536)),
])
@pytest.mark.parametrize("out_dtype", [torch.float32, torch.bfloat16])
def test_wgrad_at_both_tile_sizes(device, out_dtype, counts, features):
    """Both tile sizes and output types against the fp64 sums. fp32: the matrix
    core aligns the 128 products of one instruction to the largest before it
    adds them, dropping bits below about 2^-22 of it: 128 such losses against a
    sum of about sqrt(128) products are at most 128 / sqrt(128) 2^-22 = 3e-6
    per unit of the largest product over the typical one, which is up to 20
    for normal operands, 6e-5 of a cell (1e-4 in the test above); bf16: one
    rounding, 2^-9 of each element (4e-3 of a cell, twice the worst)."""
    g = torch.Generator().manual_seed(sum(counts))
    offsets = _ragged(counts)
    rows = int(offsets[-1])
    p_rows = torch.randn(rows, features[0], generator=g).to(torch.bfloat16)
    q_rows = torch.randn(rows, features[1], generator=g).to(torch.bfloat16)
    pt, pts, padded = K.quantize_transpose(p_rows.to(device), offsets.to(device), rows)
    qt, qts, _ = K.quantize_transpose(q_rows.to(device), offsets.to(device), rows, padded=padded)
    out = K.wgrad(pt, pts, qt, qts, offsets.to(device), out_dtype=out_dtype).cpu()
    want = O.wgrad(pt.cpu(), pts.cpu(), qt.cpu(), qts.cpu(), offsets)
    tol = 6e-5 if out_dtype == torch.float32 else 4e-3
    for e, n in enumerate(counts):
        if n == 0:
            assert torch.all(out[e] == 0)
            continue
        assert worst_cell_rel(out[e], want[e], list(range(0, features[0] + 1, 128))) < tol, e


@pytest.mark.parametrize("features", [(128, 384), (256, 640), (384, 512)])
@pytest.mark.parametrize("out_dtype", [torch.float32, torch.bfloat16])
def test_wgrad_applies_any_scale_at_odd_widths(device, out_dtype, features):
    """Descales that are no powers of two, and zeros, at widths outside the
    256 x 256 tiles, against the fp64 sums; the bounds of
    test_wgrad_at_both_tile_sizes hold (the fold of a step is one more fp32
    rounding of its product, 2^-24). Some steps keep power-of-two scales, so
    one tile's sum mixes both ways of applying them."""
    counts = [300, 0, 1, 513]
    g = torch.Generator().manual_seed(sum(features))
    offsets = _ragged(counts)
    rows = int(offsets[-1])
    padded = K.wgrad_padded_rows(rows, len(counts))
    operands = []
    for width in features:
        x = torch.randn(rows, width, generator=g).to(torch.bfloat16).to(device)
        q, s, _ = K.quantize_transpose(x, offsets.to(device), rows, padded=padded)
        factor = torch.rand(s.shape, generator=g) + 0.5
        factor[1] = 1.0
        factor[3, ::7] = 0.0
        operands += [q, s * factor.to(device)]
    out = K.wgrad(*operands, offsets.to(device), out_dtype=out_dtype).cpu()
    want = O.wgrad(*(t.cpu() for t in operands), offsets)
    tol = 6e-5 if out_dtype == torch.float32 else 4e-3
    for e, n in enumerate(counts):
        if n == 0:
            assert torch.all(out[e] == 0)
            continue
        assert worst_cell_rel(out[e], want[e], list(range(0, features[0] + 1, 128))) < tol, e


def test_wgrad_rows_beyond_32_bit_offsets(device):
    """A padded row count whose feature rows lie further apart than a 32-bit
    offset spans (two operands of 20 GB, their first two row blocks filled)
    gives the bytes of the same rows in a short layout."""
    features, padded, rows = (128, 128), 160_000_000, 200
    offsets = torch.tensor([0, rows], dtype=torch.int32, device=device)
    g = torch.Generator().manual_seed(29)
    short, far = [], []
    for width in features:
        x = torch.randn(rows, width, generator=g).to(torch.bfloat16).to(device)
        q, s, _ = K.quantize_transpose(x, offsets, rows, padded=256)
        wide_q = torch.empty(width, padded, dtype=K.FP8, device=device)
        wide_s = torch.empty(padded // 128, width, dtype=torch.float32, device=device)
        wide_q.view(torch.uint8)[:, :256] = q.view(torch.uint8)
        wide_s[:2] = s
        short += [q, s]
        far += [wide_q, wide_s]
    want = K.wgrad(*short, offsets, out_dtype=torch.float32)
    assert torch.equal(K.wgrad(*far, offsets, out_dtype=torch.float32), want)


@pytest.mark.parametrize("out_dtype", [torch.float32, torch.bfloat16])
def test_wgrad_small_tiles_sum_in_the_wide_tiles_order(device, out_dtype):
    """The 128 x 128 tiles give the bytes of the 256 x 256 ones where both
    serve the widths. Empty experts behind the others add tiles, and with them
    the wide kernel, without moving a row."""
    counts, m, n, more = [1200, 0, 130, 1, 700, 384], 512, 768, 60
    g = torch.Generator().manual_seed(23)
    offsets = _ragged(counts)
    rows = int(offsets[-1])
    many = torch.cat([offsets, offsets[-1:].expand(more)]).contiguous().to(device)
    padded = K.wgrad_padded_rows(rows, len(counts) + more)
    operands = []
    for width in (m, n):
        x = torch.randn(rows, width, generator=g).to(torch.bfloat16).to(device)
        operands += K.quantize_transpose(x, offsets.to(device), rows, padded=padded)[:2]
    small = K.wgrad(*operands, offsets.to(device), out_dtype=out_dtype)
    wide = K.wgrad(*operands, many, out_dtype=out_dtype)
    assert torch.equal(small, wide[:len(counts)])


def test_combine_and_token_sum(device):
    g = torch.Generator().manual_seed(20)
    tokens, top_k, width, experts = 300, 3, 768, 8
    ids = torch.stack([torch.randperm(experts, generator=g)[:top_k] for _ in range(tokens)]).int()
    order, offsets, slots = O.sort_assignments(ids, experts)
    y = torch.randn(tokens * top_k, width, generator=g).to(torch.bfloat16)
    w = torch.rand(tokens, top_k, generator=g)
    res = torch.randn(tokens, width, generator=g).to(torch.bfloat16)
    out = K.combine(y.to(device), slots.to(device), w.to(device), res.to(device)).cpu()
    want = O.combine(y, slots, w, res)
    # one fp32 sum rounded once; summation order may move the last bf16 bit
    assert max_rel(out.float(), want.float()) < 1e-2
    assert (out == want).float().mean().item() > 0.99
    s = K.unpermute_sum(y.to(device), slots.to(device)).cpu()
    assert (s == O.unpermute_sum(y, slots)).float().mean().item() > 0.99


@pytest.mark.parametrize("limit", [None, 0.7])
def test_routed_swiglu_backward(device, limit):
    g = torch.Generator().manual_seed(21)
    rows, width, tokens, top_k = 256, 384, 128, 2
    r = torch.randn(rows, width, generator=g).to(torch.bfloat16)
    h = torch.randn(rows, 2 * width, generator=g).to(torch.bfloat16)
    weights = torch.rand(tokens, top_k, generator=g)
    order = torch.randperm(rows, generator=g).int()
    dh, ap, ds = K.routed_swiglu_backward(r.to(device), h.to(device), weights.reshape(-1).to(device),
                                          order.to(device), limit)
    score = weights.reshape(-1)[order.long()]
    ods, odh, oap = O.routed_swiglu_backward(r, h, score, limit)
    assert max_rel(ds.cpu(), ods) < 1e-4
    assert max_rel(dh.cpu().float(), odh) < 1e-2
    assert max_rel(ap.cpu().float(), oap) < 1e-2


@pytest.mark.parametrize("limit", [None, 0.7])
@pytest.mark.parametrize("rows,width", [(256, 384), (37, 1152), (1, 128)])
def test_routed_swiglu_backward_rows_matches_unfused(device, limit, rows, width):
    """The routed backward with dh row-quantized in the same pass writes the
    plain kernel's dh, a' and dscore, and the row quantizer's bytes and scales
    on that dh (widths past one 1024-column chunk, ragged row counts)."""
    g = torch.Generator().manual_seed(rows + width)
    r = torch.randn(rows, width, generator=g).to(torch.bfloat16).to(device)
    h = torch.randn(rows, 2 * width, generator=g).to(torch.bfloat16).to(device)
    h[0] *= 40.0
    weights = torch.rand(rows, generator=g).to(device)
    order = torch.randperm(rows, generator=g).int().to(device)
    dh, ap, ds, dhq, dhs = K.routed_swiglu_backward_rows(r, h, weights, order, limit)
    dh_ref, ap_ref, ds_ref = K.routed_swiglu_backward(r, h, weights, order, limit)
    q_ref, s_ref = K.quantize_rows(dh_ref, gate_up=True)
    assert torch.equal(dh, dh_ref) and torch.equal(ap, ap_ref) and torch.equal(ds, ds_ref)
    assert torch.equal(_bytes(dhq), _bytes(q_ref))
    assert torch.equal(dhs, s_ref)


@pytest.mark.parametrize("limit", [None, 0.7])
def test_swiglu_bwd_quantize_matches_unfused(device, limit):
    """The fused kernel's outputs are, byte for byte, the unfused kernels'
    (routed SwiGLU backward -> bf16 dh / a' -> row and transposing quantizers),
    which the tests above pin to the oracle. dscore too: both kernels sum the
    score dot in the same order (per 128-column block, blocks in order)."""
    g = torch.Generator().manual_seed(33)
    experts, top_k, tokens, width = 6, 2, 700, 384
    ids = torch.stack([torch.randperm(experts, generator=g)[:top_k] for _ in range(tokens)]).int()
    ids[ids == 3] = 4  # an empty expert
    order, offsets, slots = O.sort_assignments(ids, experts)
    rows = tokens * top_k
    r = torch.randn(rows, width, generator=g).to(torch.bfloat16).to(device)
    h = torch.randn(rows, 2 * width, generator=g).to(torch.bfloat16).to(device)
    h[5] *= 50.0  # a row past the clamp limit
    weights = torch.rand(tokens * top_k, generator=g).to(device)
    order_d, offsets_d = order.to(device), offsets.to(device)
    dhq, dhs, dht, dhts, apt, apts, ds, padded = K.swiglu_bwd_quantize(
        r, h, weights, order_d, offsets_d, limit=limit)
    dh, ap, ds_ref = K.routed_swiglu_backward(r, h, weights, order_d, limit)
    q_ref, s_ref = K.quantize_rows(dh, gate_up=True)
    assert torch.equal(_bytes(dhq), _bytes(q_ref))
    assert torch.equal(dhs, s_ref)
    t_ref, ts_ref, _ = K.quantize_transpose(dh, offsets_d, rows, gate_up=True, padded=padded)
    a_ref, as_ref, _ = K.quantize_transpose(ap, offsets_d, rows, padded=padded)
    total = O.padded_layout(offsets)[1]
    assert torch.equal(_bytes(dht)[:, :total], _bytes(t_ref)[:, :total])
    assert torch.equal(dhts[: total // 128], ts_ref[: total // 128])
    assert torch.equal(_bytes(apt)[:, :total], _bytes(a_ref)[:, :total])
    assert torch.equal(apts[: total // 128], as_ref[: total // 128])
    assert torch.equal(ds, ds_ref)
    # Transposed outputs skipped: the row outputs are unchanged.
    dhq2, dhs2, dht2, _, apt2, _, _, _ = K.swiglu_bwd_quantize(
        r, h, weights, order_d, offsets_d, limit=limit, transposed_dh=False, transposed_ap=False)
    assert dht2 is None and apt2 is None
    assert torch.equal(_bytes(dhq2), _bytes(dhq)) and torch.equal(dhs2, dhs)
    # The bf16 form (fp8_current's backward): dh exactly as the routed SwiGLU
    # backward writes it (h's interleaved order), the same transposed
    # operands and dscore.
    blocks = K.padded_row_blocks(offsets_d, padded)
    dh3, dht3, dhts3, apt3, apts3, ds3 = K.swiglu_bwd_bf16(
        r, h, weights, order_d, offsets_d, padded=padded, row_blocks=blocks, limit=limit)
    assert torch.equal(dh3, dh)
    assert torch.equal(_bytes(dht3)[:, :total], _bytes(t_ref)[:, :total])
    assert torch.equal(dhts3[: total // 128], ts_ref[: total // 128])
    assert torch.equal(_bytes(apt3)[:, :total], _bytes(a_ref)[:, :total])
    assert torch.equal(apts3[: total // 128], as_ref[: total // 128])
    assert torch.equal(ds3, ds_ref)


def test_padded_row_blocks_table(device):
    """(first row, valid rows) of every padded 128-row block, from the oracle's
    padded layout; zeros past the last expert's blocks."""
    counts = [0, 300, 128, 1, 0, 257]
    offsets = _ragged(counts)
    starts, total = O.padded_layout(offsets)
    padded = total + 3 * 128
    blocks = K.padded_row_blocks(offsets.to(device), padded).cpu()
    want = torch.zeros(padded // 128, 2, dtype=torch.int32)
    for e, start in enumerate(starts):
        n = counts[e]
        for j in range(-(-n // 128)):
            want[start // 128 + j] = torch.tensor([int(offsets[e]) + 128 * j, min(128, n - 128 * j)])
    assert torch.equal(blocks, want)


@pytest.mark.parametrize("limit", [None, 0.9])
@pytest.mark.parametrize("inter", [256, 384])  # 2I = 512: pipelined epilogue; 768: GEMM then SwiGLU pass
def test_gemm_swiglu_fused_matches_separate_pass(device, limit, inter):
    """The up projection's fused SwiGLU output equals swiglu_quantize of its
    own h bit for bit; h equals the plain gate/up GEMM's."""
    g = torch.Generator().manual_seed(41)
    counts = [300, 0, 77, 512, 129]
    offsets = _ragged(counts)
    rows, hidden = int(offsets[-1]), 256
    x = torch.randn(rows, hidden, generator=g).to(torch.bfloat16).to(device)
    w = (torch.randn(len(counts), 2 * inter, hidden, generator=g) * 0.3).to(device)
    xq, xs = K.quantize_rows(x)
    wq, ws = K.quantize_weight_blocks(w)
    h, act, act_s = K.gemm_swiglu(xq, xs, wq, ws, offsets.to(device), limit=limit)
    h_ref = K.gemm(xq, xs, wq, ws, offsets.to(device), interleave=True)
    assert torch.equal(h, h_ref)
    q_ref, s_ref = K.swiglu_quantize(h, limit)
    assert torch.equal(_bytes(act), _bytes(q_ref))
    assert torch.equal(act_s, s_ref)


@pytest.mark.parametrize("counts,k,rank", [
    ([0, 37, 5, 0, 150, 16], 512, 16),   # empty experts, blocks spanning boundaries
    ([300, 1, 200], 1536, 32),
    ([64], 96, 48),                      # K % 128 != 0: the register-operand form
    ([64, 129, 0, 31], 384, 48),         # the LDS-staged form at each rank
    ([1000, 0, 33, 700], 1024, 64),
    ([257, 0, 40, 511, 3, 0, 90, 200], 4096, 16),   # C5's K (hidden) at its rank
    ([130, 0, 17, 250], 14336, 16),                  # C5's K (intermediate)
])
def test_rank_product_matches_fp32(device, counts, k, rank):
    g = torch.Generator().manual_seed(sum(counts) + k)
    offsets = _ragged(counts)
    rows, experts = int(offsets[-1]), len(counts)
    a = torch.randn(rows, k, generator=g).to(torch.bfloat16)
    bt = (torch.randn(experts, rank, k, generator=g) * 0.05).to(torch.bfloat16)
    out = K.rank_product(a.to(device), bt.to(device), offsets.to(device)).cpu()
    want = torch.zeros(rows, rank)
    for e in range(experts):
        lo, hi = int(offsets[e]), int(offsets[e + 1])
        want[lo:hi] = a[lo:hi].float() @ bt[e].float().t()
    # fp32 sums of exact bf16 products, one bf16 rounding of the result
    assert max_rel(out.float(), want) < 1e-2
    assert frob_rel(out.float(), want) < 4e-3


def test_rank_grad_row_weight_without_gather(device):
    """Routed rows of big (no gather) with small scaled by weight[order[j]]:
    dA2 = sum_j (score_j u2_j) a_j^T, against fp64 on the same operands."""
    g = torch.Generator().manual_seed(5)
    tokens, top_k, experts, m, rank = 250, 2, 5, 392, 16
    ids = torch.stack([torch.randperm(experts, generator=g)[:top_k] for _ in range(tokens)]).int()
    order, offsets, _ = O.sort_assignments(ids, experts)
    rows = tokens * top_k
    big = torch.randn(rows, m, generator=g).to(torch.bfloat16)
    small = (torch.randn(rows, rank, generator=g) * 0.3).to(torch.bfloat16)
    weight = torch.rand(rows, generator=g)
    out = K.rank_grad(big.to(device), small.to(device), offsets.to(device), transposed=True,
                      weight=weight.to(device), weight_index=order.to(device)).cpu()
    scaled = (small.float() * weight[order.long()][:, None]).to(torch.bfloat16)
    for e in range(experts):
        lo, hi = int(offsets[e]), int(offsets[e + 1])
        want = (big[lo:hi].double().t() @ scaled[lo:hi].double()).t()
        assert (out[e].double() - want).abs().max() <= 1e-5 * want.abs().max() + 1e-6, e


@pytest.mark.parametrize("splits", [1, 3, 7])
def test_rank_product_k_splits(device, splits):
    """K split over several blocks (fp32 partials added in split order, uneven
    chunk ranges) against fp32, and each split count repeatable bit for bit."""
    g = torch.Generator().manual_seed(90 + splits)
    offsets = _ragged([300, 0, 77, 650])
    rows, experts, k, rank = int(offsets[-1]), 4, 1152, 32
    a = torch.randn(rows, k, generator=g).to(torch.bfloat16)
    bt = (torch.randn(experts, rank, k, generator=g) * 0.05).to(torch.bfloat16)
    args = (a.to(device), bt.to(device), offsets.to(device))
    out = K.rank_product(*args, splits=splits).cpu()
    want = torch.zeros(rows, rank)
    for e in range(experts):
        lo, hi = int(offsets[e]), int(offsets[e + 1])
        want[lo:hi] = a[lo:hi].float() @ bt[e].float().t()
    assert max_rel(out.float(), want) < 1e-2
    assert frob_rel(out.float(), want) < 4e-3
    assert torch.equal(out, K.rank_product(*args, splits=splits).cpu())


@pytest.mark.parametrize("counts,m,rank,transposed,chunk", [
    ([0, 37, 5, 0, 150, 16], 512, 16, False, None),     # empty experts, short experts
    ([700, 1, 1300], 1544, 32, True, 256),              # several chunks per expert, M % 2048
    ([300, 0, 900], 3072, 48, False, 128),              # three rank passes, chunk tails
    ([2048, 1024, 4096, 0, 512, 100, 90, 80], 14336, 16, True, None),  # C5-like widths
])
def test_rank_grad_matches_fp64(device, counts, m, rank, transposed, chunk):
    """``sum_j big[j]^T small[j]`` per expert (the LoRA factor gradients)
    against an fp64 product of the same bf16 operands."""
    g = torch.Generator().manual_seed(sum(counts) + m + rank)
    offsets = _ragged(counts)
    rows = int(offsets[-1])
    big = torch.randn(rows, m, generator=g).to(torch.bfloat16)
    small = (torch.randn(rows, rank, generator=g) * 0.3).to(torch.bfloat16)
    out = K.rank_grad(big.to(device), small.to(device), offsets.to(device),
                      transposed=transposed, chunk=chunk).cpu()
    for e in range(len(counts)):
        lo, hi = int(offsets[e]), int(offsets[e + 1])
        want = big[lo:hi].double().t() @ small[lo:hi].double()
        if transposed:
            want = want.t()
        got = out[e].double()
        if hi == lo:
            assert torch.all(got == 0)
            continue
        # fp32 sums of exact bf16 products
        assert (got - want).abs().max() <= 1e-5 * want.abs().max() + 1e-6, e
    again = K.rank_grad(big.to(device), small.to(device), offsets.to(device),
                        transposed=transposed, chunk=chunk).cpu()
    assert torch.equal(out, again)  # fixed summation order


@pytest.mark.parametrize("weighted", [False, True])
@pytest.mark.parametrize("transposed", [False, True])
def test_rank_grad_gathered_token_rows(device, weighted, transposed):
    """The token-side form: row j of big is the token row big[order[j] // k],
    and small's row j is scaled by weight[order[j]] * alpha (rounded to bf16
    once), against an fp64 product of the same operands. An empty expert and
    ragged counts come from the routing."""
    g = torch.Generator().manual_seed(7 + 2 * weighted + transposed)
    tokens, top_k, experts, m, rank = 300, 2, 6, 264, 16
    ids = torch.stack([torch.randperm(experts, generator=g)[:top_k] for _ in range(tokens)]).int()
    ids[ids == 2] = 3  # expert 2 gets no rows
    order, offsets, _ = O.sort_assignments(ids, experts)
    rows = tokens * top_k
    big = torch.randn(tokens, m, generator=g).to(torch.bfloat16)
    small = (torch.randn(rows, rank, generator=g) * 0.3).to(torch.bfloat16)
    weight = torch.rand(rows, generator=g) if weighted else None
    alpha = 1.5 if weighted else 1.0
    out = K.rank_grad(big.to(device), small.to(device), offsets.to(device),
                      transposed=transposed, gather=order.to(device), gather_div=top_k,
                      weight=None if weight is None else weight.to(device),
                      weight_index=order.to(device), alpha=alpha).cpu()
    tok = order.long() // top_k
    scaled = small
    if weighted:
        scaled = (small.float() * (weight[order.long()] * alpha)[:, None]).to(torch.bfloat16)
    for e in range(experts):
        lo, hi = int(offsets[e]), int(offsets[e + 1])
        want = big[tok[lo:hi]].double().t() @ scaled[lo:hi].double()
        if transposed:
            want = want.t()
        got = out[e].double()
        if hi == lo:
            assert torch.all(got == 0)
            continue
        assert (got - want).abs().max() <= 1e-5 * want.abs().max() + 1e-6, e
