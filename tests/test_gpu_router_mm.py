"""Router logits of many tokens on the fp32 matrix cores: the documented order bit for bit (CPU oracle), and equal to the
vector kernel for what the oracle's entry does not cover (the shared gate's logit row)."""
import numpy as np
import pytest
import torch

from helpers import np_u16, orc

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("T,E,d", [
    (192, 128, 2048),    # the first call on the matrix cores at E = 128
    (1537, 16, 64),      # one group of lanes, a ragged token block
    (3100, 8, 320),      # half a row tile, chunks end inside the first 64 lanes
    (801, 32, 2880),     # lanes with five and with six chunks
    (250, 100, 576),     # a ragged row tile; chunks past 64 for the first lanes only
    (4096, 128, 512),    # two token tiles per wave
    (2085, 257, 192),    # the same, ragged in both
])
@pytest.mark.parametrize("scale", [1.0, 1e-20])
def test_logits_bit_exact(T, E, d, scale):
    from moelab_amd import router
    g = torch.Generator(device=DEV).manual_seed(T + E + d)
    x = (torch.randn((T, d), generator=g, device=DEV) * scale).to(torch.bfloat16)
    wr = (torch.randn((E, d), generator=g, device=DEV) * 0.02 * scale).to(torch.bfloat16)   # 1e-20: subnormal sums
    b = torch.randn(E, generator=g, device=DEV) if scale == 1.0 else None
    print(f"case logits T={T} E={E} d={d} {scale}", flush=True)
    idx, _, logits = router.route(x, wr, min(E, 4), bias=b, return_logits=True)
    want = orc.router_logits(np_u16(x), np_u16(wr), None if b is None else b.cpu().numpy())
    np.testing.assert_array_equal(logits.cpu().numpy().view(np.uint32), want.view(np.uint32))
    np.testing.assert_array_equal(idx.cpu().numpy(), orc.topk(want, min(E, 4))[0])


def test_gate_row_and_grouping_equal_the_vector_kernel(monkeypatch):
    """Shared experts with a gate (one more logit row, E + 1 = 17) in a layer call, with the grouping behind it."""
    from moelab_amd import experts
    from moelab_amd.problem import baseline_int4_layer
    from moelab_amd.shapes import MoEShape
    T, d, f, E, k = 1500, 192, 64, 16, 3
    s = baseline_int4_layer(MoEShape("t", d=d, f=f, E=E, k=k), seed=5, device=DEV)
    wr = s.pop("wr")
    s["shared"] = baseline_int4_layer(MoEShape("t", d=d, f=f, E=1, k=1), seed=6, device=DEV, router=False)
    s["shared_gate"] = (torch.randn(d, device=DEV) * 0.05).to(torch.bfloat16)
    s = experts.merge_shared(s)
    x = torch.randn((T, d), device=DEV).to(torch.bfloat16)
    got = []
    for least in ("1000000000", "1"):
        monkeypatch.setenv("MOE_ROUTER_MM_MIN", least)
        got.append(experts.run_routed(s, x, wr, k, out_dtype=torch.float32))
    for a, b in zip(*got):
        assert torch.equal(a, b)
