"""Router logits of few tokens (one wave per tile of 16 or 32 tokens x 16, 32 or
64 experts) against the same rows of a large batch (the tiled kernel): a
logit's bits depend on its row, d and floor(t / 256) mod 4 only."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("E,d", [(1, 8), (16, 264), (17, 1000), (64, 2048), (100, 1032), (128, 1096), (200, 520),
                                 (256, 776)])
def test_small_batches_equal_rows_of_a_large_one(et, dev, E, d):
    g = torch.Generator(device=dev).manual_seed(E * 8191 + d)
    x = torch.randn(70000, d, generator=g, device=dev).to(torch.bfloat16)
    w = (torch.randn(E, d, generator=g, device=dev) * d ** -0.5).to(torch.bfloat16)
    whole = et.router_logits(x, w)
    # on both sides of every tile's edge and of every change of the wave tile
    for T in (1, 15, 16, 17, 255, 257, 512, 513, 1023, 1025, 2049, 4096, 4097, 8191, 8193):
        print(f"router_logits small T={T} d={d} E={E}", flush=True)
        guard = torch.full((T + 1, E), 7.0, device=dev)
        out = et.router_logits(x[:T], w, out=guard[:T])
        assert torch.equal(out.view(torch.int32), whole[:T].view(torch.int32))
        assert bool((guard[T] == 7.0).all())
