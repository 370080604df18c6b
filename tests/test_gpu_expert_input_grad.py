"""The expert GEMM's input gradient on the weights as they are (transposing LDS
reads) against the product from explicitly transposed weights (``wt=``): the
same products in the same order, so the same bits.  Which of the two a call
takes is set here, so that the first is compared whatever the rule says, and
which entry points ran is checked."""
import importlib

import pytest
import torch

pytestmark = pytest.mark.gpu

et_api = importlib.import_module("peer-review-agents_amd.expert_threshold")


@pytest.fixture
def direct(monkeypatch):
    """Input gradients without wt= take the weights as they are; the entry
    points called, in order."""
    calls, call = [], et_api._call
    monkeypatch.setattr(et_api, "_transpose_first", lambda *a: False)
    monkeypatch.setattr(et_api, "_call", lambda fn, *a: (calls.append(fn), call(fn, *a))[1])
    return calls


def _case(et, dev, N, K, counts, ints=False):
    E, S, T = len(counts), sum(counts), 400
    g = torch.Generator(device=dev).manual_seed(N * 31 + K)
    eo = torch.tensor([0] + counts).cumsum(0).to(torch.int32).to(dev)
    tok = torch.randint(0, T, (S,), generator=g, device=dev, dtype=torch.int32)
    if ints:    # every product and sum exact
        gate = torch.exp2(torch.randint(-3, 3, (S,), generator=g, device=dev).float())
        w = torch.randint(-2, 3, (E, N, K), generator=g, device=dev).to(torch.bfloat16)
        dy = torch.randint(-2, 3, (T, N), generator=g, device=dev).to(torch.bfloat16)
    else:
        gate = torch.rand(S, generator=g, device=dev)
        w = (torch.randn(E, N, K, generator=g, device=dev) * N ** -0.5).to(torch.bfloat16)
        dy = torch.randn(T, N, generator=g, device=dev).to(torch.bfloat16)
    plan = et.RoutingPlan(torch.tensor(counts, dtype=torch.int32, device=dev), eo,
                          torch.zeros(T + 1, dtype=torch.int32, device=dev), tok, gate, tok, T, E, S, S)
    return plan, w, dy


def _bits(t):
    return t.view(torch.int16)


# the sum's length on both sides of the k-step and the 64-row chunk (one chunk,
# two, many), columns off the 256-wide tile, slots below and above a tile
SHAPES = [(8, 8, [1, 0, 3]), (56, 264, [130, 17]), (64, 256, [300]), (72, 520, [0, 5, 256]), (128, 1032, [257, 600]),
          (200, 40, [64, 1000]), (1096, 776, [33, 513, 20]), (3072, 512, [700, 90])]


@pytest.mark.parametrize("N,K,counts", SHAPES)
def test_input_grad_equals_product_of_transposed_weights(et, dev, direct, N, K, counts):
    print(f"input_grad N={N} K={K} counts={counts}", flush=True)
    plan, w, dy = _case(et, dev, N, K, counts)
    S, tok, gate, eo = plan.rows, plan.sorted_token, plan.slot_gate, plan.expert_offsets
    wt = torch.empty(len(counts), K, N, dtype=torch.bfloat16, device=dev)
    for gather, dc in ((True, dy), (False, dy[tok.long()].contiguous())):
        for scale in (None, gate):
            out = torch.full((S, K), 9.0, dtype=torch.bfloat16, device=dev)
            del direct[:]
            da = et.expert_gemm_input_grad(dc, w, plan, gather=gather, row_scale=scale, out=out)
            assert direct == ["et_expert_input_grad_impl"]
            want = et.expert_gemm_input_grad(dc, w, plan, gather=gather, row_scale=scale, wt=wt)
            assert direct[1:] == ["et_expert_weight_transpose", "et_expert_gemm_impl"]
            assert torch.equal(_bits(da), _bits(want))
    ref = torch.cat([dy.double()[tok[eo[e]:eo[e + 1]].long()] @ w[e].double() for e in range(len(counts))])
    assert float((da.double() - ref * gate.double()[:, None]).norm() / ref.norm()) < 4e-3   # bf16 rounding


@pytest.mark.parametrize("N,K,counts", SHAPES)
def test_direct_input_grad_exact_on_integers_and_within_the_capacity(et, dev, direct, N, K, counts):
    """Integer operands: the float64 product rounded once; with a capacity above
    the slots (the rest untouched) and below them (the first rows)."""
    print(f"input_grad integers N={N} K={K} counts={counts}", flush=True)
    plan, w, dy = _case(et, dev, N, K, counts, ints=True)
    S, tok, eo = plan.rows, plan.sorted_token, plan.expert_offsets
    ref = torch.cat([dy.double()[tok[eo[e]:eo[e + 1]].long()] @ w[e].double() for e in range(len(counts))])
    want = _bits(ref.float().to(torch.bfloat16))
    dc = dy[tok.long()].contiguous()
    plan.num_slots = None
    for cap in (S, S + 9, max(1, S - 3)):
        n = min(S, cap)
        plan.capacity = cap
        plan.sorted_token = torch.cat([tok, tok[:1].expand(9)])[:cap].contiguous()
        for gather, d in ((True, dy), (False, torch.cat([dc, dc[:1].expand(9, N)])[:cap].contiguous())):
            out = torch.full((cap, K), 7.0, dtype=torch.bfloat16, device=dev)
            et.expert_gemm_input_grad(d, w, plan, gather=gather, out=out)
            assert torch.equal(_bits(out[:n]), want[:n]) and bool((out[n:] == 7.0).all())
    assert set(direct) == {"et_expert_input_grad_impl"}


def test_direct_input_grad_replays_in_a_graph(et, dev, direct):
    plan, w, dy = _case(et, dev, 1096, 776, [33, 513, 20])
    out = torch.empty(plan.rows, 776, dtype=torch.bfloat16, device=dev)
    s = torch.cuda.Stream()
    with torch.cuda.stream(s):
        et.expert_gemm_input_grad(dy, w, plan, gather=True, row_scale=plan.slot_gate, out=out)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=s):
        et.expert_gemm_input_grad(dy, w, plan, gather=True, row_scale=plan.slot_gate, out=out)
    for i in range(3):
        dy.mul_(-1.5 if i else 1.0)
        want = et.expert_gemm_input_grad(dy, w, plan, gather=True, row_scale=plan.slot_gate)
        out.fill_(9.0)
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(_bits(out), _bits(want)), i
    assert set(direct) == {"et_expert_input_grad_impl"}
