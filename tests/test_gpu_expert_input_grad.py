"""The expert GEMM's input gradient on the weights as they are (transposing LDS
reads) against the product from explicitly transposed weights (``wt=``): the
same products in the same order, so the same bits."""
import pytest
import torch

pytestmark = pytest.mark.gpu


# the sum's length on both sides of the k-step and the 64-row chunk (one chunk,
# two, many), columns off the 256-wide tile, slots below and above a tile
@pytest.mark.parametrize("N,K,counts", [(8, 8, [1, 0, 3]), (56, 264, [130, 17]), (64, 256, [300]), (72, 520, [0, 5, 256]),
                                        (128, 1032, [257, 600]), (200, 40, [64, 1000]), (1096, 776, [33, 513, 20]),
                                        (3072, 512, [700, 90])])
def test_input_grad_equals_product_of_transposed_weights(et, dev, N, K, counts):
    print(f"input_grad N={N} K={K} counts={counts}", flush=True)
    E, S, T = len(counts), sum(counts), 400
    g = torch.Generator(device=dev).manual_seed(N * 31 + K)
    eo = torch.tensor([0] + counts).cumsum(0).to(torch.int32).to(dev)
    tok = torch.randint(0, T, (S,), generator=g, device=dev, dtype=torch.int32)
    gate = torch.rand(S, generator=g, device=dev)
    plan = et.RoutingPlan(torch.tensor(counts, dtype=torch.int32, device=dev), eo,
                          torch.zeros(T + 1, dtype=torch.int32, device=dev), tok, gate, tok, T, E, S, S)
    w = (torch.randn(E, N, K, generator=g, device=dev) * N ** -0.5).to(torch.bfloat16)
    dy = torch.randn(T, N, generator=g, device=dev).to(torch.bfloat16)
    wt = torch.empty(E, K, N, dtype=torch.bfloat16, device=dev)
    for gather, dc in ((True, dy), (False, dy[tok.long()].contiguous())):
        for scale in (None, gate):
            out = torch.full((S, K), 9.0, dtype=torch.bfloat16, device=dev)
            da = et.expert_gemm_input_grad(dc, w, plan, gather=gather, row_scale=scale, out=out)
            want = et.expert_gemm_input_grad(dc, w, plan, gather=gather, row_scale=scale, wt=wt)
            assert torch.equal(da.view(torch.int16), want.view(torch.int16))
    ref = torch.cat([dy.double()[tok[eo[e]:eo[e + 1]].long()] @ w[e].double() for e in range(E)])
    assert float((da.double() - ref * gate.double()[:, None]).norm() / ref.norm()) < 4e-3   # bf16 rounding
