"""int4 dense tiles at the edges of their token tiles: counts per expert around multiples of 16, 32 and 64 (both token-tile
sizes, one and several passes), ragged last row blocks, inputs that end at half a slice, one to many K slices, every GLU,
fp16 and bf16 activations, against the CPU oracle at the dense tiles' gate."""
import numpy as np
import pytest
import torch

from helpers import assert_close, oracle_y

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _run(d, F, counts, act, dtype, seed):
    """Experts with the given slot counts (k = 1), in shuffled token order."""
    from moelab_amd import _lib, experts
    from moelab_amd.problem import baseline_int4_layer
    from moelab_amd.shapes import MoEShape
    E, T = len(counts), sum(counts)
    s = baseline_int4_layer(MoEShape("t", d=d, f=F, E=E, k=1), seed=seed, device=DEV, router=False)
    rng = np.random.default_rng(seed)
    idx = torch.from_numpy(rng.permutation(np.repeat(np.arange(E, dtype=np.int32), counts))[:, None].copy()).to(DEV)
    wts = torch.from_numpy(rng.random((T, 1), dtype=np.float32)).to(DEV)
    x = torch.from_numpy(rng.standard_normal((T, d), dtype=np.float32)).to(DEV).to(dtype)
    print(f"case dense i4 d={d} F={F} counts={counts} act={act} {dtype}", flush=True)
    y = experts.run_experts(s, x, idx, wts, act=act, path=_lib.PATH_GROUPED, out_dtype=torch.float32)
    # fp16 weights and activations: 2^-12 per operand, a few thousand terms: well inside 5e-3 of the RMS
    assert_close(y, oracle_y(s, x, idx, wts, act=act), tol=5e-3, what=(d, F, counts, act))


@pytest.mark.parametrize("counts", [[47, 33, 48, 32, 1, 64, 65, 49], [31, 16, 17, 63, 15, 80, 81, 60],        # avg <= 48
                                    [128, 129, 127, 64, 65, 33, 96, 1], [200, 1, 0, 191, 193, 63, 0, 97]])   # avg > 48
@pytest.mark.parametrize("d,F,act,dtype", [(192, 320, 0, torch.bfloat16), (128, 64, 1, torch.float16),
                                           (1088, 192, 2, torch.bfloat16)])
def test_token_tile_edges(monkeypatch, counts, d, F, act, dtype):
    monkeypatch.setenv("MOE_DENSE", "1")
    _run(d, F, counts, act, dtype, seed=sum(counts) + d)


def test_large_and_small_h_beside_ordinary_tokens(monkeypatch):
    """h beyond fp16 and below 2^-8 (per-chunk exponents, the epilogue's scaled branch) beside ordinary tokens in one pass, in
    passes with dead tokens (100 and 50 slots): every row against its class's own size, so that no row takes another's
    exponent or values. (Dead tokens repeat the expert's last slot: what they would store is that slot's own row.)"""
    from moelab_amd import _lib, experts
    from moelab_amd.problem import baseline_int4_layer
    from moelab_amd.shapes import MoEShape
    monkeypatch.setenv("MOE_DENSE", "1")
    d, F, E, T = 256, 192, 2, 150
    s = baseline_int4_layer(MoEShape("t", d=d, f=F, E=E, k=1), seed=9, device=DEV, router=False)
    x = torch.randn((T, d), generator=torch.Generator(device=DEV).manual_seed(9), device=DEV).to(torch.bfloat16)
    x[::7] *= 3e3      # |h| to ~1e8
    x[3::7] *= 1e-3    # chunks below 2^-8
    idx = (torch.arange(T, device=DEV, dtype=torch.int32) % 3 == 0).to(torch.int32)[:, None].contiguous()
    wts = torch.ones((T, 1), device=DEV)
    y = experts.run_experts(s, x, idx, wts, path=_lib.PATH_GROUPED, out_dtype=torch.float32)
    want = oracle_y(s, x, idx, wts)
    for r in range(7):
        assert_close(y[r::7], want[r::7], tol=1e-2, what=r)
    # row by row too, in norms (fp16 operands: 2^-12 each, about 3.5e-4 of the norm)
    off = np.linalg.norm(y.cpu().numpy() - want, axis=1) / np.linalg.norm(want, axis=1)
    assert off.max() < 2e-3, (int(off.argmax()), float(off.max()))


@pytest.mark.parametrize("F", [64, 192, 1088, 4096])   # 4096: a wave per slot
def test_slot_exponents_brought_together(monkeypatch, F):
    """Slots whose 32-row chunks need different exponents (W_up rows at very different scales), mixed with slots that need
    none and zero rows, over more slots than one workgroup takes, the last one partly filled."""
    from moelab_amd import _lib, experts, formats
    monkeypatch.setenv("MOE_DENSE", "1")
    d, E, T = 128, 2, 137
    g = torch.Generator(device=DEV).manual_seed(F)
    gate, up, down = (formats.random_int4(E, n, k, generator=g, device=DEV) for n, k in ((F, d), (F, d), (d, F)))
    grow = torch.ones(F, device=DEV)
    grow[:32] = 2.0 ** 14          # the first chunk of every h row far above the others
    up = (up[0], (up[1].float() * grow[None, :, None]).to(torch.bfloat16), (up[2].float() * grow[None, :, None]).to(torch.bfloat16))
    s = experts.make_state("int4", gate, up, down)
    x = torch.randn((T, d), generator=g, device=DEV).to(torch.bfloat16)
    x[::5] *= 2.0 ** -12           # nothing to bring together here
    x[7] = 0
    idx = (torch.arange(T, device=DEV, dtype=torch.int32) % 2)[:, None].contiguous()
    y = experts.run_experts(s, x, idx, torch.ones((T, 1), device=DEV), path=_lib.PATH_GROUPED, out_dtype=torch.float32)
    want = oracle_y(s, x, idx, torch.ones((T, 1), device=DEV))
    assert (y[7] == 0).all()
    for rows in (slice(0, None, 5), slice(1, None, 5), slice(3, None, 5)):
        assert_close(y[rows], want[rows], tol=5e-3, what=(F, rows))


@pytest.mark.parametrize("d,F,dtype", [(128, 64, torch.bfloat16), (192, 320, torch.float16), (1088, 192, torch.bfloat16),
                                       (64, 128, torch.bfloat16), (2048, 64, torch.float16)])
@pytest.mark.parametrize("counts", [[32, 31, 33, 1, 24, 40, 16, 21], [64, 65, 0, 1, 0, 33, 31, 2]])
def test_exact_weight_gate_up(monkeypatch, counts, d, F, dtype):
    """21 to 32 slots per expert: the dense gate/up on exact weights, whose group biases go in as a product of their own.
    Biases of every size (a wrong group-sum term is an O(1) error), inputs and scales spread over powers of two, against
    the oracle and against the wave tiles' exact codes: both round h to the same fp16, so they differ by the h16 values on
    which 1e-6 of h decides the rounding (a few in ten thousand, 2^-11 each): far below rounding weights to fp16 (2e-4)."""
    from moelab_amd import _lib, experts, formats
    monkeypatch.setenv("MOE_DENSE", "1")
    E, T = len(counts), sum(counts)
    assert 20 < (T + E - 1) // E <= 32
    g = torch.Generator(device=DEV).manual_seed(T + d)

    def proj(N, K):
        codes, scales, _ = formats.random_int4(E, N, K, generator=g, device=DEV)
        scales = (scales.float() * torch.exp2(torch.randint(-3, 4, scales.shape, generator=g, device=DEV).float())).to(torch.bfloat16)
        return codes, scales, (torch.randn(scales.shape, generator=g, device=DEV) * 0.1).to(torch.bfloat16)
    s = experts.make_state("int4", proj(F, d), proj(F, d), proj(d, F))
    x = torch.randn((T, d), generator=g, device=DEV) * torch.exp2(torch.randint(-6, 7, (T, 1), generator=g, device=DEV).float())
    x[3] = 0
    x = x.to(dtype)
    rng = np.random.default_rng(T)
    idx = torch.from_numpy(rng.permutation(np.repeat(np.arange(E, dtype=np.int32), counts))[:, None].copy()).to(DEV)
    wts = torch.ones((T, 1), device=DEV)
    print(f"case exact gate/up d={d} F={F} {dtype} {counts}", flush=True)
    got = {}
    for least in ("20", "100"):
        monkeypatch.setenv("MOE_DENSE_EX_MIN_AVG", least)
        got[least] = experts.run_experts(s, x, idx, wts, path=_lib.PATH_GROUPED, out_dtype=torch.float32).double()
    # In norms, row by row too: the rows' sizes span 2^24 (h grows with x^2) and single outputs have a heavy tail where few
    # terms dominate. h and W_down each carry fp16's rounding, at most 2^-12 per term: sqrt(2) 2^-12 = 3.5e-4 of the norm
    # (rows of few terms: four times that); the wave tiles' result carries the same.
    want = torch.from_numpy(oracle_y(s, x, idx, wts)).to(DEV).double()
    off, off_wave = ((got[k] - want).norm() / want.norm() for k in ("20", "100"))
    assert off < 5e-4 and off < 1.25 * off_wave + 1e-6
    assert ((got["20"] - want).norm(dim=1) <= 1.5e-3 * want.norm(dim=1)).all()
    assert float((got["20"] - got["100"]).norm() / got["100"].norm()) < 5e-5


@pytest.mark.parametrize("T,E,k,d", [(150, 16, 3, 192), (61, 8, 4, 2112), (340, 16, 3, 128), (1100, 8, 2, 320)])
def test_router_writes_the_fp16_rows(T, E, k, d, monkeypatch):
    """A layer call whose router writes x16 (beside the tails of one-workgroup groupings, with the split tails otherwise;
    with the group sums at 21 to 32 slots per expert) against routing first and calling the experts on the ids: the same
    bits."""
    from moelab_amd import experts, router
    from moelab_amd.problem import baseline_int4_layer
    from moelab_amd.shapes import MoEShape
    monkeypatch.setenv("MOE_DENSE", "1")
    s = baseline_int4_layer(MoEShape("t", d=d, f=128, E=E, k=k), seed=T, device=DEV)
    wr = s.pop("wr")
    x = (torch.randn((T, d), device=DEV) * torch.exp2(torch.randint(-12, 20, (T, 1), device=DEV).float())).to(torch.bfloat16)
    y, idx, wts = experts.run_routed(s, x, wr, k, out_dtype=torch.float32)
    i2, w2 = router.route(x, wr, k)
    assert torch.equal(idx, i2) and torch.equal(wts, w2)
    assert torch.equal(y, experts.run_experts(s, x, idx, wts, out_dtype=torch.float32))


@pytest.mark.parametrize("d,F,E,T,k", [(512, 1024, 32, 400, 2),    # gate/up blocks for the chip, 25 slots per expert
                                       (1024, 64, 24, 480, 1),     # at the edge: 224 down blocks in 128-token passes, 256 in 64
                                       (64, 8192, 8, 88, 2)])
def test_exact_down_where_its_grid_is_small(monkeypatch, d, F, E, T, k):
    """17 to 32 slots per expert and a down projection of few blocks: both stages stay on exact codes and two planes of h,
    whatever the gate/up's grid. h = hi + lo keeps 2^-17 per term, so 1e-4 of the RMS is above 10 standard errors; the fp16
    weights and h of the dense down (2^-12 per operand) miss it by ten times."""
    from moelab_amd import _lib, experts
    from moelab_amd.problem import baseline_int4_layer
    from moelab_amd.shapes import MoEShape
    monkeypatch.delenv("MOE_DENSE", raising=False)
    assert 16 < (T * k + E - 1) // E <= 32
    s = baseline_int4_layer(MoEShape("t", d=d, f=F, E=E, k=k), seed=d + T, device=DEV, router=False)
    g = torch.Generator(device=DEV).manual_seed(T)
    x = torch.randn((T, d), generator=g, device=DEV).to(torch.bfloat16)
    idx = torch.rand((T, E), generator=g, device=DEV).topk(k, dim=1).indices.to(torch.int32)
    wts = torch.rand((T, k), generator=g, device=DEV)
    print(f"case small down d={d} F={F} E={E} T={T} k={k}", flush=True)
    y = experts.run_experts(s, x, idx, wts, path=_lib.PATH_GROUPED, out_dtype=torch.float32)
    assert_close(y, oracle_y(s, x, idx, wts), tol=1e-4, what=(d, F, E, T, k))
