"""The two-launch grouping of calls with many slots (chunk counts, then one placing workgroup per chunk): the layer's
outputs equal those of the one-workgroup grouping bit for bit, and the lists that either leaves in the workspace (an output
shows neither the order within an expert nor the active list and the bad-id count) equal a stable sort of the ids."""
import numpy as np
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
    (129, 16, 16, 0, "int4"),     # 2064 slots: nine chunks of 16 tokens, the last with one; 17 of 128 given slots
    (2048, 8, 1, 0, "int4"),      # 16 slots per chunk, one placing wave
    (700, 60, 4, 2, "int4"),      # shared experts in the slot lists
    (4097, 128, 2, 0, "int4"),    # 86 chunks of 48 tokens from the router's tails, 65 of 128 slots from given ids
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


def _workspace_lists(ws, E, d, F, T, k):
    """The grouping's lists out of an experts workspace: moe_api.hip's layout, whose total must be the size query's."""
    n = T * k
    passes = lambda P: (n + P - 1) // P + min(n, E)   # noqa: E731
    parts = [("h", n * F * 2), ("h2", n * F * 2), ("xp", 3 * T * d * 2), ("yp", n * d * 16), ("x16", T * d * 2),
             ("xexp", T * 4), ("counts", E * 4), ("offsets", (E + 1) * 4), ("sorted", n * 4), ("active", E * 4), ("meta", 16),
             ("items", passes(16) * 12), ("items2", passes(64) * 12)]
    out, off = {}, 0
    for name, size in parts:
        out[name] = (off, size)
        off += (size + 255) // 256 * 256
    return off, {m: ws[o:o + z].view(torch.int32).cpu().numpy() for m, (o, z) in out.items()
                 if m not in ("h", "h2", "xp", "yp", "x16", "xexp")}


def _expected_lists(ids, E, P, P2):
    flat = ids.reshape(-1)
    valid = np.flatnonzero((flat >= 0) & (flat < E))
    counts = np.bincount(flat[valid], minlength=E)
    act = np.flatnonzero(counts)
    items = lambda p: np.array([(e, q, -(-counts[e] // p)) for e in act for q in range(-(-counts[e] // p))])   # noqa: E731
    out = {"counts": counts, "offsets": np.concatenate([[0], np.cumsum(counts)]),
           "sorted": valid[np.argsort(flat[valid], kind="stable")], "active": np.concatenate([act, -np.ones(E - len(act))]),
           "items": items(P).reshape(-1)}
    meta = [len(act), len(flat) - len(valid), len(items(P))]
    if P2:
        out["items2"] = items(P2).reshape(-1)
        meta.append(len(items(P2)))
    return dict(out, meta=np.array(meta))


LISTS = [
    (129, 16, 16, 0, "int4", 128, 64, 0),     # the last chunk with one token
    (2048, 8, 1, 0, "int4", 64, 64, 0),       # one placing wave's worth of slots per chunk
    (700, 60, 4, 2, "int4", 64, 64, 0),       # shared experts in the slot lists
    (256, 40, 4, 0, "int4", 64, 32, 64),      # two pass lists; given: 8 chunks of the smallest call that splits
    (257, 130, 8, 0, "mxfp4", 64, 64, 0),     # three chunks of 64 experts
    (300, 700, 8, 0, "int4", 64, 16, 0),      # more experts than half the workgroup
    (4097, 128, 8, 0, "int4", 64, 64, 0),     # 384 slots per chunk: a placing wave's cursors go through two steps
    (9000, 16, 8, 0, "int4", 64, 64, 0),      # 640 (given) and 768: three steps, cursors of few experts
    (1025, 1024, 1, 0, "int4", 64, 16, 0),    # routed: 65 rows of 1024 counts pass the scratch, one workgroup groups
    (300, 2100, 4, 0, "int4", 64, 16, 0),     # more experts than the placing workgroup's LDS holds: one workgroup groups
]


@pytest.mark.parametrize("entry,T,E,k,S,fmt,d,P,P2", [(e, *c) for e in ("routed", "given", "skewed") for c in LISTS
                                                       if e == "given" or c[1] <= 1024])   # the router's limit
def test_grouping_lists(monkeypatch, entry, T, E, k, S, fmt, d, P, P2):
    from moelab_amd import _lib, experts
    F = 64
    s, wr = _layer(fmt, d, F, E, S, seed=T + E)
    monkeypatch.setenv("MOE_DENSE", "1")
    g = torch.Generator(device=DEV).manual_seed(T)
    x = torch.randn((T, d), generator=g, device=DEV).to(torch.bfloat16)
    bias = torch.where(torch.arange(E, device=DEV) < k, 50.0, 0.0) if entry == "skewed" else None
    idx = torch.randint(-1, E + 1, (T, k), generator=g, device=DEV, dtype=torch.int32)
    wts = torch.rand((T, k), generator=g, device=DEV)
    monkeypatch.setattr(_lib, "_WS", {})
    ws = _lib.workspace(x.device, _lib.lib().moe_layer_shared_workspace_bytes(experts._desc(s), S, T, k) if S else
                        _lib.lib().moe_layer_workspace_bytes(experts._desc(s), T, k))
    for least in ("1000000000", "1024"):
        monkeypatch.setenv("MOE_GROUP_SPLIT_MIN", least)
        print(f"case lists T={T} E={E} k={k} S={S} {fmt} {entry} least={least}", flush=True)
        ws.fill_(0xEE)
        if entry == "given":
            experts.run_layer(s, x, idx, wts, out_dtype=torch.float32)
            ids = idx.cpu().numpy()
        else:
            ids = experts.run_routed(s, x, wr, k, bias=bias, out_dtype=torch.float32)[1].cpu().numpy()
        if S:
            ids = np.concatenate([np.where((ids >= 0) & (ids < E), ids, -1), np.tile(np.arange(E, E + S), (T, 1))], 1)
        total, got = _workspace_lists(ws, E + S, d, F, T, k + S)
        assert total == _lib.lib().moe_experts_workspace_bytes(experts._desc(s), T, k + S, _lib.PATH_GROUPED)
        for name, want in _expected_lists(ids, E + S, P, P2).items():
            np.testing.assert_array_equal(got[name][:len(want)], want, err_msg=f"{name} least={least}")


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
