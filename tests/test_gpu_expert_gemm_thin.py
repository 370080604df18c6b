"""Expert grouped GEMM at the slot counts where its kernel and tile height
change (one to 128 slots per thin tile, 64-slot tiles for small calls, experts
split between the thin and the 256-row kernel in one call).

Integer operands make every product and sum exact in binary32, so each output
must be the float64 product rounded once (torch's cast); random operands give
the same bits whichever kernel an expert's slot count selects, because both sum
the same k-steps in the same order.
"""
import pytest
import torch

pytestmark = pytest.mark.gpu

F8 = torch.float8_e4m3fn
# per-expert slots on both sides of every tile's edge
EDGES = [0, 1, 15, 16, 17, 32, 33, 64, 0, 65, 96, 97, 127, 128, 129, 200]
# a few heavy experts beside many light ones: both kernels run, each on its experts
MIXED = [2000, 20, 20, 20, 20, 20, 20, 20, 20, 20] * 4


def _plan(et, dev, counts, T, seed):
    """A plan with these slots per expert (only the arrays the GEMM reads)."""
    g = torch.Generator().manual_seed(seed)
    S, E = sum(counts), len(counts)
    eo = torch.tensor([0] + counts, dtype=torch.int64).cumsum(0).to(torch.int32).to(dev)
    tok = torch.randint(0, T, (S,), generator=g, dtype=torch.int32).to(dev)
    gate = torch.exp2(torch.randint(-3, 3, (S,), generator=g).float()).to(dev)
    return et.RoutingPlan(torch.tensor(counts, dtype=torch.int32, device=dev), eo,
                          torch.zeros(T + 1, dtype=torch.int32, device=dev), tok, gate, tok, T, E, S, S)


def _reference(a, w, plan):
    eo = plan.expert_offsets.tolist()
    ref = torch.zeros(plan.rows, w.shape[1], dtype=torch.float64, device=a.device)
    for e in range(plan.num_experts):
        ref[eo[e]:eo[e + 1]] = a[eo[e]:eo[e + 1]].double() @ w[e].double().T
    return ref


def _ints(shape, seed, dev, lim=2):
    g = torch.Generator(device=dev).manual_seed(seed)
    return torch.randint(-lim, lim + 1, shape, generator=g, device=dev).to(torch.bfloat16)


def _bits(t):
    return t.view(torch.int16)


# K off the k-step and the chunk (and above one ring turn), N off the wave's and
# the block's rows, one with more 64-slot tiles than CUs
@pytest.mark.parametrize("counts,K,N", [(EDGES, 8, 8), (EDGES, 40, 16), (EDGES, 264, 136), (EDGES, 776, 272),
                                        (EDGES, 520, 2064), (MIXED, 72, 3072), ([3], 4104, 48), ([130], 1040, 4112)])
def test_thin_tiles_exact_on_integer_inputs(et, orc, dev, counts, K, N):
    import numpy as np
    print(f"thin expert_gemm K={K} N={N} counts={counts[:16]}", flush=True)
    T = 90
    plan = _plan(et, dev, counts, T, K + N)
    x, w = _ints((T, K), 1, dev), _ints((len(counts), N, K), 2, dev)
    xp = x[plan.sorted_token.long()].contiguous()
    ref = _reference(xp, w, plan)
    want = _bits(ref.float().to(torch.bfloat16))
    scaled = _bits((ref * plan.slot_gate.double()[:, None]).float().to(torch.bfloat16))
    for gather, a in ((True, x), (False, xp)):
        assert torch.equal(_bits(et.expert_gemm(a, w, plan, gather=gather)), want)
        assert torch.equal(_bits(et.expert_gemm(a, w, plan, gather=gather, epilogue="row_scale",
                                                row_scale=plan.slot_gate)), scaled)
        if N % 16 == 0:
            h = et.expert_gemm(a, w, plan, gather=gather, epilogue="swiglu")
            gate, up = (ref[:, i * (N // 2):(i + 1) * (N // 2)].float().cpu().numpy() for i in (0, 1))
            assert np.array_equal(_bits(h).cpu().numpy(), orc.f32_to_bf16(orc.swiglu(gate, up)).view(np.int16))


@pytest.mark.parametrize("counts,K,N", [(EDGES, 16, 8), (EDGES, 272, 200), (EDGES, 528, 1040), (MIXED, 80, 3072),
                                        ([3], 4112, 48)])
def test_thin_fp8_tiles_exact_on_integer_inputs(et, orc, dev, counts, K, N):
    import numpy as np
    print(f"thin expert_gemm_fp8 K={K} N={N} counts={counts[:16]}", flush=True)
    T, E = 90, len(counts)
    plan = _plan(et, dev, counts, T, K + N)
    x, w = _ints((T, K), 3, dev).to(F8), _ints((E, N, K), 4, dev).to(F8)
    g = torch.Generator(device=dev).manual_seed(5)
    sa = torch.exp2(torch.randint(-3, 3, (T,), generator=g, device=dev).float())
    sw = torch.exp2(torch.randint(-3, 3, (E, N), generator=g, device=dev).float())
    tok = plan.sorted_token.long()
    xp, sp = x.float()[tok].to(F8), sa[tok].contiguous()
    ref = _reference(xp.float(), w.float(), plan) * sp.double()[:, None]
    eo = plan.expert_offsets.tolist()
    for e in range(E):
        ref[eo[e]:eo[e + 1]] *= sw[e].double()
    want = _bits(ref.float().to(torch.bfloat16))
    for gather, a, s in ((True, x, sa), (False, xp, sp)):
        assert torch.equal(_bits(et.expert_gemm_fp8(a, s, w, sw, plan, gather=gather)), want)
        if N % 16 == 0:
            h = et.expert_gemm_fp8(a, s, w, sw, plan, gather=gather, epilogue="swiglu")
            gate, up = (ref[:, i * (N // 2):(i + 1) * (N // 2)].float().cpu().numpy() for i in (0, 1))
            assert np.array_equal(_bits(h).cpu().numpy(), orc.f32_to_bf16(orc.swiglu(gate, up)).view(np.int16))


@pytest.mark.parametrize("n", [1, 16, 31, 64, 90, 128])
def test_thin_and_256_row_tiles_give_the_same_bits(et, dev, n):
    """The first n slots alone (thin tiles) and followed by 40000 others of the
    same expert (256-row tiles): the same rows, bit for bit."""
    T, K, N = 200, 1096, 272
    g = torch.Generator(device=dev).manual_seed(n)
    x = torch.randn(T, K, generator=g, device=dev).to(torch.bfloat16)
    w = (torch.randn(1, N, K, generator=g, device=dev) * K ** -0.5).to(torch.bfloat16)
    many = _plan(et, dev, [n + 40000], T, 6)
    few = _plan(et, dev, [n], T, 6)
    few.sorted_token = many.sorted_token[:n].contiguous()
    for epilogue in ("none", "swiglu"):
        assert torch.equal(_bits(et.expert_gemm(x, w, few, epilogue=epilogue)),
                           _bits(et.expert_gemm(x, w, many, epilogue=epilogue)[:n]))
    q, wq = (x * 4).to(F8)[:, :1088].contiguous(), (w * 16).to(F8)[:, :, :1088].contiguous()
    sa, sw = torch.rand(T, generator=g, device=dev) + 0.5, torch.rand(1, N, generator=g, device=dev) + 0.5
    for epilogue in ("none", "swiglu"):
        assert torch.equal(_bits(et.expert_gemm_fp8(q, sa, wq, sw, few, epilogue=epilogue)),
                           _bits(et.expert_gemm_fp8(q, sa, wq, sw, many, epilogue=epilogue)[:n]))


@pytest.mark.parametrize("T,counts,cap", [(1, [1, 0, 1], 3), (64, [64, 0, 3] * 40, 64 * 120), (65, [65, 0, 3] * 40, 65 * 120),
                                          (8, [300, 0, 129] * 40, 429 * 40)])
def test_slot_major_product_of_a_small_batch(et, dev, T, counts, cap):
    """Up to 64 tokens the thin kernel alone takes the call, above it the device
    decides; the last plan holds more slots per expert than it names tokens."""
    print(f"slot-major expert_gemm T={T} cap={cap}", flush=True)
    K, N = 264, 2064
    plan = _plan(et, dev, counts, T, T)
    S, plan.capacity, plan.num_slots = plan.rows, cap, None
    a = _ints((cap, K), 7, dev)
    w = _ints((len(counts), N, K), 8, dev)
    c = torch.full((cap, N), 7.0, device=dev, dtype=torch.bfloat16)
    et.expert_gemm(a, w, plan, gather=False, out=c)
    assert torch.equal(_bits(c[:S]), _bits(_reference(a, w, plan)[:S].float().to(torch.bfloat16)))
    assert (c[S:] == 7.0).all()


@pytest.mark.parametrize("counts", [[20] * 40, [390, 400, 0, 410] * 10, [2000] + [20] * 9 + [1] * 10 + [2000] + [129] * 9 + [0] * 10])
def test_device_decides_from_the_slot_counts(et, dev, counts):
    """A slot count that was not read back: both kernels are launched, and light
    experts, heavy ones or each take the one or the other; the same rows as of
    the exact plan."""
    E, T, K, N, S = len(counts), 4000, 1040, 3072, sum(counts)
    print(f"expert_gemm decided on the device S={S}", flush=True)
    exact = _plan(et, dev, counts, T, 11)
    cap = S + 7
    pad = torch.zeros(7, dtype=torch.int32, device=dev)
    plan = et.RoutingPlan(exact.counts, exact.expert_offsets, exact.token_offsets, torch.cat([exact.sorted_token, pad]),
                          torch.cat([exact.slot_gate, pad.float()]), exact.token_slot, T, E, cap)
    for fp8, epi in ((0, 0), (0, 2)):
        assert et.lib().et_expert_gemm_route_impl(fp8, epi, 1, E, K, N, cap, 0, T, 256) == 2
    x, w = _ints((T, K), 12, dev), _ints((E, N, K), 13, dev)
    want = _bits(_reference(x[exact.sorted_token.long()], w, exact).float().to(torch.bfloat16))
    xp = torch.cat([x[exact.sorted_token.long()], x[:7]]).contiguous()
    for gather, a in ((True, x), (False, xp)):
        c = torch.full((cap, N), 7.0, device=dev, dtype=torch.bfloat16)
        et.expert_gemm(a, w, plan, gather=gather, out=c)
        assert torch.equal(_bits(c[:S]), want) and bool((c[S:] == 7.0).all())
        h = et.expert_gemm(a, w, plan, gather=gather, epilogue="swiglu")
        assert torch.equal(_bits(h[:S]), _bits(et.expert_gemm(a[:S] if not gather else a, w, exact, gather=gather,
                                                              epilogue="swiglu")))
    q, wq = x.to(F8), w.to(F8)
    sa, sw = torch.ones(T, device=dev), torch.ones(E, N, device=dev)
    for epilogue in ("none", "swiglu"):
        assert torch.equal(_bits(et.expert_gemm_fp8(q, sa, wq, sw, plan, epilogue=epilogue)[:S]),
                           _bits(et.expert_gemm_fp8(q, sa, wq, sw, exact, epilogue=epilogue)))
