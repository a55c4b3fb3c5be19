"""The two-launch grouping of calls with many slots (chunk counts, then one placing workgroup per chunk) against the
one-workgroup grouping: the same stable order, so the layer's outputs are equal bit for bit."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _layer(fmt, d, f, E, S, seed):
    from moelab_amd import experts
    from moelab_amd.problem import baseline_int4_layer, baseline_mxfp4_layer
    from moelab_amd.shapes import MoEShape
    make = baseline_int4_layer if fmt == "int4" else baseline_mxfp4_layer
    kw = {} if fmt == "int4" else {"biases": False}
    s = make(MoEShape("t", d=d, f=f, E=E, k=1), seed=seed, device=DEV, **kw)
    wr = s.pop("wr")
    if S:
        s["shared"] = make(MoEShape("t", d=d, f=f, E=S, k=1), seed=seed + 1, device=DEV, router=False, **kw)
        s = experts.merge_shared(s)
    return s, wr


@pytest.mark.parametrize("T,E,k,S,fmt", [
    (129, 16, 16, 0, "int4"),     # 2064 slots: nine chunks of 16 tokens, the last with one
    (2048, 8, 1, 0, "int4"),      # 16 slots per chunk, one placing wave
    (700, 60, 4, 2, "int4"),      # shared experts in the slot lists
    (4097, 128, 2, 0, "int4"),    # more than 256 chunks of 16 tokens: 32 tokens each
    (257, 130, 8, 0, "mxfp4"),    # three chunks of 64 experts, term records from the tails
    (300, 700, 8, 0, "int4"),     # more experts than half the workgroup
])
@pytest.mark.parametrize("entry", ["routed", "given", "skewed"])
def test_split_grouping_equals_one_workgroup(monkeypatch, T, E, k, S, fmt, entry):
    from moelab_amd import experts
    d, f = 128, 64
    s, wr = _layer(fmt, d, f, E, S, seed=T + E)
    g = torch.Generator(device=DEV).manual_seed(T)
    x = torch.randn((T, d), generator=g, device=DEV).to(torch.bfloat16)
    bias = torch.where(torch.arange(E, device=DEV) < k, 50.0, 0.0) if entry == "skewed" else None
    idx = torch.randint(-1, E + 1, (T, k), generator=g, device=DEV, dtype=torch.int32)   # some join no group
    wts = torch.rand((T, k), generator=g, device=DEV)
    got = []
    for least in ("1000000000", "1024"):
        monkeypatch.setenv("MOE_GROUP_SPLIT_MIN", least)
        print(f"case T={T} E={E} k={k} S={S} {fmt} {entry} least={least}", flush=True)
        if entry == "given":
            y = experts.run_layer(s, x, idx, wts, out_dtype=torch.float32)
            got.append((y,))
        else:
            got.append(experts.run_routed(s, x, wr, k, bias=bias, out_dtype=torch.float32))
        torch.cuda.synchronize()
    assert torch.isfinite(got[0][0]).all()
    for a, b in zip(*got):
        assert torch.equal(a, b)


def test_split_grouping_replays_in_a_graph():
    """Captured and replayed with the program's own work between the replays."""
    from moelab_amd import backend, experts
    T, E, k = 520, 32, 4
    s, wr = _layer("int4", 128, 64, E, 0, seed=3)
    x = torch.randn((T, 128), device=DEV).to(torch.bfloat16)
    experts.reserve(s, T, k)
    graph, out = backend.capture(lambda: experts.run_routed(s, x, wr, k, out_dtype=torch.float32))
    for i in range(4):
        x.copy_(torch.randn((T, 128), device=DEV).to(torch.bfloat16))
        want = experts.run_routed(s, x, wr, k, out_dtype=torch.float32)
        graph.replay()
        torch.cuda.synchronize()
        for a, b in zip(out, want):
            assert torch.equal(a, b)
