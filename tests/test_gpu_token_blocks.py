"""Calls whose h passes 32-bit byte offsets (4 GiB a plane) run as blocks of tokens: rows of the first and the last block, and
of both sides of the old limit, equal the same rows in a small call bit for bit."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("fmt,entry", [("int4", "given"), ("int4", "routed"), ("mxfp4", "given")])
def test_h_past_4_gib(monkeypatch, fmt, entry):
    from moelab_amd import _lib, experts
    from moelab_amd.problem import baseline_int4_layer, baseline_mxfp4_layer
    from moelab_amd.shapes import MoEShape
    monkeypatch.setattr(_lib, "_WS", {})           # the 9 GB workspace goes with the test
    monkeypatch.setenv("MOE_DENSE_KSPLIT", "1")    # the down's sums in one order whatever the size of the call
    d, F, E, k, T = 64, 16384, 8, 2, 65600         # T k F 2 = 2^32 + 2^22
    shape = MoEShape("t", d=d, f=F, E=E, k=k)
    s = baseline_int4_layer(shape, seed=1, device=DEV) if fmt == "int4" else \
        baseline_mxfp4_layer(shape, seed=1, device=DEV, biases=False)
    wr = s.pop("wr")
    g = torch.Generator(device=DEV).manual_seed(T)
    x = torch.randn((T, d), generator=g, device=DEV).to(torch.bfloat16)
    res = torch.randn((T, d), generator=g, device=DEV)
    idx = torch.rand((T, E), generator=g, device=DEV).topk(k, dim=1).indices.to(torch.int32)
    wts = torch.rand((T, k), generator=g, device=DEV)
    print(f"case h past 4 GiB {fmt} {entry}", flush=True)

    def call(rows):
        if entry == "routed":
            return experts.run_routed(s, x[rows], wr, k, residual=res[rows], out_dtype=torch.float32)
        return (experts.run_experts(s, x[rows], idx[rows].contiguous(), wts[rows].contiguous(), residual=res[rows],
                                    out_dtype=torch.float32),)
    whole = call(slice(0, T))
    assert torch.isfinite(whole[0]).all()
    for a in (0, 31000, T - 2048):                 # 32800 is the blocks' border; 65536 tokens fill the 32 bits
        rows = slice(a, a + 2048)
        for u, v in zip(whole, call(rows)):
            assert torch.equal(u[rows], v), (fmt, entry, a)
