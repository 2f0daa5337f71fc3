"""Non-finite activations: a NaN or Inf in row m of x makes every output of row m non-finite,
as Light's F32 arithmetic does (kernels/cpu/quant_matmul.go: the dequantized dot of that row),
and leaves every other row bit-identical to the call without it.  The int8 paths quantize x
per 32-block, where a max that ignores NaN would otherwise hide it behind finite codes."""
import pytest
import torch

from light_amd import hipq, synth

pytestmark = pytest.mark.gpu


def _rows_check(y_bad, y_ok):
    assert not torch.isfinite(y_bad[0]).any(), "row 0 holds a non-finite x but has finite outputs"
    assert torch.equal(y_bad[1:], y_ok[1:]), "other rows changed"


@pytest.mark.parametrize("dt,K", [(hipq.Q4_K, 2048), (hipq.Q4_K, 4096), (hipq.Q4_K, 14336), (hipq.Q5_K, 4096),
                                  (hipq.Q8_0, 4096), (hipq.Q8_0, 1024), (hipq.Q6_K, 4096), (hipq.Q4_0, 12288),
                                  (hipq.Q5_0, 2048)])
@pytest.mark.parametrize("M", [2, 3, 16])
@pytest.mark.parametrize("bad", [float("nan"), float("inf"), float("-inf")])
def test_matmul_q_nonfinite_row(dev, dt, K, M, bad):
    print(f"[case] nonfinite matmul_q dt={hipq.NAMES[dt]} K={K} M={M} x={bad}", flush=True)
    g = synth.rng(K + M + dt)
    N = 96
    w = torch.from_numpy(synth.gguf_weight(dt, N, K, g)).to(dev)
    x = torch.randn(M, K, device=dev)
    ok = hipq.matmul_q(x, w, N, K, dt)
    x[0, 37] = bad
    _rows_check(hipq.matmul_q(x, w, N, K, dt), ok)
    act = hipq.quantize_act(x)
    y = hipq.matmul_q_act(act, w, M, N, K, dt)
    assert not torch.isfinite(y[0]).any()
    assert torch.isfinite(y[1:]).all()


@pytest.mark.parametrize("M", [1, 2, 16])
def test_gated_and_mlp_nonfinite_row(dev, M):
    print(f"[case] nonfinite gated/mlp M={M}", flush=True)
    g = synth.rng(90 + M)
    H, I = 1024, 2816
    t = lambda a: torch.from_numpy(a).to(dev)
    wg, wu, wd = (t(synth.gguf_weight(hipq.Q4_K, r, c, g)) for r, c in ((I, H), (I, H), (H, I)))
    x = torch.randn(max(M, 2), H, device=dev)
    ok_g = hipq.matmul_q_gated(x, wg, wu, I, H, hipq.Q4_K)
    ok_m = hipq.mlp_q(x, wg, wu, wd, H, I, hipq.Q4_K)
    x[0, 5] = float("nan")
    _rows_check(hipq.matmul_q_gated(x, wg, wu, I, H, hipq.Q4_K), ok_g)
    _rows_check(hipq.mlp_q(x, wg, wu, wd, H, I, hipq.Q4_K), ok_m)


@pytest.mark.parametrize("M", [2, 16, 64])
@pytest.mark.parametrize("xdt", [torch.float32, torch.float16])
def test_int4_nonfinite_row(dev, M, xdt):
    print(f"[case] nonfinite int4 M={M} x={xdt}", flush=True)
    gen = torch.Generator(device="cpu").manual_seed(M)
    N, K, G = 200, 2048, 128
    codes = torch.randint(0, 2 ** 31, (N, K // 8), dtype=torch.int32, generator=gen).to(dev)
    s = (torch.rand(N, K // G, generator=gen) * 0.02 + 1e-3).to(dev)
    z = torch.randint(0, 16, (N, K // G), generator=gen).float().to(dev)
    x = torch.randn(M, K, generator=gen).to(dev)
    ok = hipq.int4_matmul(x.to(xdt), codes, s, z, G)
    x[0, 100] = float("nan")
    _rows_check(hipq.int4_matmul(x.to(xdt), codes, s, z, G), ok)


def _same_class(y, want):
    """Every output is NaN, +Inf or -Inf where float64 on the dequantized weight has it so."""
    want = want.to(torch.float32)
    assert torch.equal(torch.isnan(y), torch.isnan(want))
    inf = torch.isinf(want)
    assert torch.equal(torch.isinf(y), inf) and torch.equal(torch.sign(y[inf]), torch.sign(want[inf]))


def _plant(x):
    """Row 0: one Inf; row 1: two of one sign far apart; row 2: Inf and -Inf; the last: a NaN beside an Inf
    (with three rows, the last is row 2)."""
    K, x = x.shape[1], x.clone()
    x[0, 37] = float("-inf")
    x[1, 5], x[1, K - 3] = float("inf"), float("inf")
    x[2, K // 2], x[2, K // 2 + 9] = float("inf"), float("-inf")
    x[-1, K - 1], x[-1, 0] = float("nan"), float("inf")
    return x


# 3 to 8 rows from 10M weights (one part of x, two), 9 to 16 and 17 to 64 (one K part, several): rows of up
# to 4096 and longer ones of skinny.hip, with a ragged N.
@pytest.mark.parametrize("dt", [hipq.Q4_K, hipq.Q5_K])
@pytest.mark.parametrize("M,N,K", [(3, 2567, 4096), (5, 5008, 2048), (8, 1601, 6656), (4, 1601, 16640), (9, 97, 2048),
                                   (16, 97, 5120), (17, 97, 2304), (40, 130, 4096), (64, 40001, 512)])
def test_infinities_as_in_f32(dev, dt, M, N, K):
    print(f"[case] infinities dt={hipq.NAMES[dt]} M={M} N={N} K={K}", flush=True)
    w = torch.from_numpy(synth.gguf_weight(dt, N, K, synth.rng(K + M))).to(dev)
    wd = hipq.dequant(w, N * K, dt).view(N, K).double()
    x = torch.randn(M, K, device=dev)
    ok = hipq.matmul_q(x, w, N, K, dt)
    x = _plant(x)
    y = hipq.matmul_q(x, w, N, K, dt)
    _same_class(y, x.double() @ wd.t())
    if M > 4:
        assert torch.equal(y[3:-1], ok[3:-1]), "other rows changed"
    if 4 < M <= 16 or K == 4096:  # (other gated calls of up to four rows quantize x to int8)
        h = hipq.matmul_q_gated(x, w, w, N, K, dt)
        a = x.double() @ wd.t()
        _same_class(h, torch.nn.functional.silu(a) * a)


@pytest.mark.parametrize("xdt", [torch.float32, torch.bfloat16, torch.float16])
@pytest.mark.parametrize("M,N,K", [(3, 3208, 4096), (8, 5000, 2688), (5, 2056, 18944), (9, 12296, 4096), (16, 4104, 8192)])
def test_int4_infinities_as_in_f32(dev, xdt, M, N, K):
    print(f"[case] infinities int4 x={xdt} M={M} N={N} K={K}", flush=True)
    codes, s, z = (torch.from_numpy(a).to(dev) for a in synth.int4_weight(N, K, 128, synth.rng(N)))
    codes, z = codes.view(torch.int32), z.round()  # (whole zeros: weights of exactly 0 come up)
    wd = hipq.int4_dequant(codes, s, z, 128).double()
    x = torch.randn(M, K, device=dev).to(xdt)
    ok = hipq.int4_matmul(x, codes, s, z, 128)
    x = _plant(x)
    y = hipq.int4_matmul(x, codes, s, z, 128)
    assert (wd == 0).any()
    _same_class(y.float(), x.double() @ wd.t())
    if M > 4:
        assert torch.equal(y[3:-1], ok[3:-1]), "other rows changed"
