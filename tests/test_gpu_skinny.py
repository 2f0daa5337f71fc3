"""The f16 MFMA product for 3 to 16 rows of x (skinny.hip) against float64 on the dequantized weight.

Bounds, relative to |w_n| |x_m| (Cauchy-Schwarz on the rounding of x; the weights are exact
integers and f32 scales): one f16 part of x is 2^-12 per element, so 2.5e-4 with the f32 sums;
two parts are 2^-22, which leaves the f32 sums' 2e-5; 16-bit x is exact in one part down to 2^-24 of
its unit's largest element, so its output rounding (bf16 2^-8, f16 2^-11 of |y| <= |w| |x|) is what shows.
"""
import pytest
import torch

from light_amd import hipq, synth

pytestmark = pytest.mark.gpu


def _x(M, K, dev, seed):
    """N(0, 1) rows; row 0 with outliers and a zero stretch, row 1 tiny, row 2 huge."""
    g = torch.Generator(device=dev).manual_seed(seed)
    x = torch.randn(M, K, device=dev, generator=g)
    x[0, ::97] *= 40.0
    x[0, 256:512] = 0.0
    x[1] *= 1e-20
    x[2] *= 1e20
    return x


def _weight(dt, N, K, dev, seed):
    w = torch.from_numpy(synth.gguf_weight(dt, N, K, synth.rng(seed))).to(dev)
    return w, hipq.dequant(w, N * K, dt).view(N, K).double()


def _big_weight(dt, N, K, dev):
    """Random quants under one small scale, made on the GPU."""
    per, size = hipq.BLOCK[dt]
    g = torch.Generator(device=dev).manual_seed(N + K)
    w = torch.randint(0, 256, (N * K // per, size), dtype=torch.uint8, device=dev, generator=g)
    w[:, 0:4] = torch.tensor([1e-4, 7e-4], dtype=torch.float16, device=dev).view(torch.uint8)
    return w


def _err(y, want, x, wd):
    scale = torch.outer(x.double().norm(dim=1), wd.norm(dim=1))
    return ((y.double() - want).abs() / scale).max().item()


# (N, K): tile and group remainders of the resident kernel (K <= 4096; 16, 15, 8 and 2 groups), then
# of the long one (17 groups: two chunks of 9 and 8; one tile, two tiles and four per workgroup).
SHAPES = [(2567, 4096), (2640, 3840), (5008, 2048), (20011, 512), (2440, 4352), (1536, 14336), (5000, 4608),
          (10000, 5120), (1600, 16640)]


@pytest.mark.parametrize("dt", [hipq.Q4_K, hipq.Q5_K])
@pytest.mark.parametrize("M", [3, 4, 5, 8, 9, 16])
@pytest.mark.parametrize("N,K", SHAPES)
def test_matmul_q(dev, dt, M, N, K):
    print(f"[case] skinny dt={hipq.NAMES[dt]} M={M} N={N} K={K}", flush=True)
    w, wd = _weight(dt, N, K, dev, seed=N + K)
    x = _x(M, K, dev, seed=M)
    y = hipq.matmul_q(x, w, N, K, dt)
    pair = M <= 8 and (K < 4096 or K > 16384)
    assert _err(y, x.double() @ wd.t(), x, wd) <= (2e-5 if pair else 2.5e-4)
    assert torch.equal(y, hipq.matmul_q(x, w, N, K, dt)), "not deterministic"


@pytest.mark.parametrize("M", [9, 16])
@pytest.mark.parametrize("N,K", [(1, 256), (17, 256), (40, 768), (100, 8192)])
def test_small_weights(dev, M, N, K):
    print(f"[case] skinny small M={M} N={N} K={K}", flush=True)
    w, wd = _weight(hipq.Q4_K, N, K, dev, seed=K)
    x = _x(M, K, dev, seed=M)
    assert _err(hipq.matmul_q(x, w, N, K, hipq.Q4_K), x.double() @ wd.t(), x, wd) <= 2.5e-4


@pytest.mark.parametrize("dt", [hipq.Q4_K, hipq.Q5_K])
@pytest.mark.parametrize("M", [17, 32, 33, 48, 49, 64])
@pytest.mark.parametrize("N,K", [(1, 256), (130, 512), (127, 768), (2567, 4096), (4000, 14336), (40001, 1024), (1000, 1280),
                                 (4096, 4864), (300, 8448), (500, 8192)])
def test_mid_rows(dev, dt, M, N, K):
    """17 to 64 rows: row-tile and column-group remainders; on 256 CUs one K part, eight even ones, two of two
    and three units, seven of two and three, eleven of three, sixteen of two."""
    print(f"[case] skinny mid dt={hipq.NAMES[dt]} M={M} N={N} K={K}", flush=True)
    w, wd = _weight(dt, N, K, dev, seed=N + K)
    x = _x(M, K, dev, seed=M)
    y = hipq.matmul_q(x, w, N, K, dt)
    assert _err(y, x.double() @ wd.t(), x, wd) <= 2.5e-4
    assert torch.equal(y, hipq.matmul_q(x, w, N, K, dt)), "not deterministic"


@pytest.mark.parametrize("dt", [hipq.Q4_K, hipq.Q5_K])
@pytest.mark.parametrize("M,N,K", [(3, 2567, 4096), (8, 5008, 2048), (16, 1000, 3840), (5, 1608, 6400), (12, 6000, 4352)])
def test_gated(dev, dt, M, N, K):
    print(f"[case] skinny gated dt={hipq.NAMES[dt]} M={M} N={N} K={K}", flush=True)
    (wg, g), (wu, u) = _weight(dt, N, K, dev, seed=N), _weight(dt, N, K, dev, seed=N + 1)
    x = torch.randn(M, K, device=dev, generator=torch.Generator(device=dev).manual_seed(M)) * 0.01
    h = hipq.matmul_q_gated(x, wg, wu, N, K, dt)
    a, b = x.double() @ g.t(), x.double() @ u.t()
    # The product rule on the plain bound (|silu'| <= 1.1), and f32's exp.
    xn, gn, un = x.double().norm(dim=1)[:, None], g.norm(dim=1)[None, :], u.norm(dim=1)[None, :]
    silu = torch.nn.functional.silu(a)
    bound = 2.5e-4 * xn * (1.1 * gn * b.abs() + un * silu.abs()) + 1e-5 * (silu * b).abs() + 1e-7 * xn * xn * gn * un
    assert ((h.double() - silu * b).abs() <= bound).all()


@pytest.mark.parametrize("M,H,I", [(3, 4096, 5120), (5, 2048, 8192), (8, 4096, 3072), (6, 8192, 2048), (4, 8192, 2048),
                                   (4, 5120, 6144)])
def test_mlp_equals_its_halves(dev, M, H, I):
    """A block is its two calls, whichever kernels those take, whatever the workspace: on F32 h where the
    gated call takes the f16 tiles, on quantized h where it takes the GEMV.  (Past I = 4096 the down half
    takes the tiles on that h, which is its F32 form to 2^-15.)"""
    print(f"[case] skinny mlp M={M} H={H} I={I}", flush=True)
    (wg, _), (wu, _), (wd, _) = (_weight(hipq.Q4_K, r, c, dev, seed=i) for i, (r, c) in enumerate(((I, H), (I, H), (H, I))))
    x = torch.randn(M, H, device=dev, generator=torch.Generator(device=dev).manual_seed(M)) * 0.01
    h = hipq.matmul_q_gated(x, wg, wu, I, H, hipq.Q4_K)
    got = hipq.mlp_q(x, wg, wu, wd, H, I, hipq.Q4_K)
    if M > 4 or H <= 4096:
        assert torch.equal(got, hipq.matmul_q(h, wd, H, I, hipq.Q4_K))
    elif I <= 4096:
        act = hipq.matmul_q_gated_act(x, wg, wu, I, H, hipq.Q4_K)
        assert torch.equal(got, hipq.matmul_q_act(act, wd, M, H, I, hipq.Q4_K))
    else:
        wdd = hipq.dequant(wd, H * I, hipq.Q4_K).view(H, I).double()
        assert _err(got, h.double() @ wdd.t(), h, wdd) <= 2.5e-4
    ws = torch.empty(hipq.mlp_q_ws_bytes(M, H, I, hipq.Q4_K), dtype=torch.uint8, device=dev)
    assert torch.equal(hipq.mlp_q(x, wg, wu, wd, H, I, hipq.Q4_K, ws=ws), got)


@pytest.mark.parametrize("dt", [hipq.Q4_K, hipq.Q5_K])
@pytest.mark.parametrize("M,N,K", [(3, 2567, 4096), (8, 1536, 14336), (5, 1700, 6144), (4, 1600, 16640)])
def test_prepared_whatever_the_workspace(dev, dt, M, N, K):
    """hq_matmul_q_act asks for no workspace at 3 to 8 rows, writes none that it is given, and gives the
    same bits with none, any, and under capture on a stream whose library workspace cannot grow."""
    print(f"[case] skinny act dt={hipq.NAMES[dt]} M={M} N={N} K={K}", flush=True)
    w, wd = _weight(dt, N, K, dev, seed=K)
    x = torch.randn(M, K, device=dev, generator=torch.Generator(device=dev).manual_seed(M))
    act = hipq.quantize_act(x)
    assert hipq.lib().hq_matmul_q_act_ws_bytes(M, N, K, dt) == 0
    y = hipq.matmul_q_act(act, w, M, N, K, dt)
    for n in (16, 1 << 20):
        ws = torch.full((n,), 171, dtype=torch.uint8, device=dev)
        assert torch.equal(hipq.matmul_q_act(act, w, M, N, K, dt, ws=ws), y)
        assert (ws == 171).all(), "the caller's buffer was written"
    out, g, s = torch.empty_like(y), torch.cuda.CUDAGraph(), torch.cuda.Stream()
    s.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(s), torch.cuda.graph(g, stream=s):
        hipq.matmul_q_act(act, w, M, N, K, dt, out=out)
    for _ in range(3):
        out.fill_(float("nan"))
        g.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, y)
    # (x by q8_1: 1e-3 from K = 4096 on where the GEMV reads one level.)
    assert _err(y, x.double() @ wd.t(), x, wd) <= 1e-3


@pytest.mark.parametrize("xdt", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("M", [3, 4, 7, 9, 15, 16])
@pytest.mark.parametrize("K", [128, 256, 384, 512, 1024, 1152, 2048])
def test_int4_short_rows(dev, xdt, M, K):
    """Rows of one to eight groups of 256, whose x the waves of a group convert together (M = 9 to 16 from
    the rule's 30M and 45M weights)."""
    N, G = (45000000 if M > 8 else 12600000) // K + 5, 128
    print(f"[case] skinny int4 short x={xdt} M={M} N={N} K={K}", flush=True)
    g = torch.Generator(device=dev).manual_seed(K)
    codes = torch.randint(-2 ** 31, 2 ** 31, (N, K // 8), dtype=torch.int64, device=dev, generator=g).to(torch.int32)
    s, z = torch.rand(N, K // G, device=dev, generator=g) * 0.01 + 1e-3, torch.randint(0, 16, (N, K // G), device=dev, generator=g).float()
    x = torch.randn(M, K, device=dev, generator=g).to(xdt)
    wd = hipq.int4_dequant(codes, s, z, G).double()
    tol = 2.0 ** -8 if xdt == torch.bfloat16 else 2.5e-4 if M > 8 else 2e-5
    assert _err(hipq.int4_matmul(x, codes, s, z, G), x.double() @ wd.t(), x, wd) <= tol


@pytest.mark.parametrize("dt", [hipq.Q4_K, hipq.Q5_K])
@pytest.mark.parametrize("M", [3, 4, 7, 8, 9, 13, 16])
@pytest.mark.parametrize("K", [256, 512, 768, 1024, 1280, 2048])
def test_short_rows(dev, dt, M, K):
    """The same for the K formats, with x of every scale."""
    N = 10000000 // K + 21
    print(f"[case] skinny short dt={hipq.NAMES[dt]} M={M} N={N} K={K}", flush=True)
    w = _big_weight(dt, N, K, dev)
    wd = hipq.dequant(w, N * K, dt).view(N, K).double()
    x = _x(M, K, dev, seed=M)
    y = hipq.matmul_q(x, w, N, K, dt)
    assert _err(y, x.double() @ wd.t(), x, wd) <= (2e-5 if M <= 8 else 2.5e-4)
    assert torch.equal(y, hipq.matmul_q(x, w, N, K, dt)), "not deterministic"


# Tiles of the long kernel: from one up to six per workgroup, ragged last workgroups and a second round.
LONG_N = [(3000, 4608), (5003, 4352), (10003, 4352), (14003, 4352), (18003, 4352), (22003, 4352), (30003, 4352)]


@pytest.mark.parametrize("dt", [hipq.Q4_K, hipq.Q5_K])
@pytest.mark.parametrize("M", [3, 8, 16])
@pytest.mark.parametrize("N,K", LONG_N)
def test_long_row_tiles(dev, dt, M, N, K):
    print(f"[case] skinny long dt={hipq.NAMES[dt]} M={M} N={N} K={K}", flush=True)
    w = _big_weight(dt, N, K, dev)
    wd = hipq.dequant(w, N * K, dt).view(N, K).double()
    x = _x(M, K, dev, seed=M)
    y = hipq.matmul_q(x, w, N, K, dt)
    assert _err(y, x.double() @ wd.t(), x, wd) <= 2.5e-4
    assert torch.equal(y, hipq.matmul_q(x, w, N, K, dt)), "not deterministic"


@pytest.mark.parametrize("xdt,tol", [(torch.float32, 2.5e-4), (torch.bfloat16, 2.0 ** -8), (torch.float16, 2.0 ** -10)])
@pytest.mark.parametrize("M", [4, 13])
@pytest.mark.parametrize("N,K", LONG_N)
def test_int4_long_row_tiles(dev, xdt, tol, M, N, K):
    print(f"[case] skinny int4 long x={xdt} M={M} N={N} K={K}", flush=True)
    g = torch.Generator(device=dev).manual_seed(N)
    codes = torch.randint(-2 ** 31, 2 ** 31, (N, K // 8), dtype=torch.int64, device=dev, generator=g).to(torch.int32)
    s, z = torch.rand(N, K // 128, device=dev, generator=g) * 0.01 + 1e-3, torch.rand(N, K // 128, device=dev, generator=g) * 15
    x = torch.randn(M, K, device=dev, generator=g).to(xdt)
    wd = hipq.int4_dequant(codes, s, z, 128).double()
    # (M > 8 below 30M weights: the bf16 GEMM for some dtypes, both operands rounded.)
    tiles = M <= 8 or N * K >= 30000000
    assert _err(hipq.int4_matmul(x, codes, s, z, 128), x.double() @ wd.t(), x, wd) <= (tol if tiles else 2.0 ** -8 + tol)


@pytest.mark.parametrize("xdt,tol", [(torch.float32, 2e-5), (torch.bfloat16, 2.0 ** -8), (torch.float16, 2.0 ** -10)])
@pytest.mark.parametrize("M", [3, 8, 9, 16])
@pytest.mark.parametrize("N,K,G", [(3208, 4096, 128), (3600, 3584, 256), (5000, 2688, 128), (4100, 4224, 128),
                                   (2056, 18944, 128), (4104, 8192, 512), (11009, 4096, 128), (16001, 3072, 256)])
def test_int4(dev, xdt, tol, M, N, K, G):
    """3 and 8 rows on the tiles; 9 and 16 too where the rule has them: F32 x from 30M weights (16M past
    K = 4096), BF16 from 45M (30M, but not 129 tiles of 18944), F16 past K = 4096 only; else the GEMMs, which
    round x and w to bf16."""
    print(f"[case] skinny int4 x={xdt} M={M} N={N} K={K} G={G}", flush=True)
    codes, s, z = (torch.from_numpy(a).to(dev) for a in synth.int4_weight(N, K, G, synth.rng(N + K)))
    z = z + 0.25  # fractional zero points
    codes = codes.view(torch.int32)
    x = torch.randn(M, K, device=dev, generator=torch.Generator(device=dev).manual_seed(M)).to(xdt)
    y = hipq.int4_matmul(x, codes, s, z, G)
    wd = hipq.int4_dequant(codes, s, z, G).double()
    least = {torch.float32: (30, 16), torch.bfloat16: (45, 30), torch.float16: (1e9, 16)}[xdt][K > 4096] * 1e6
    tiles = M <= 8 or (N * K >= least and not (xdt == torch.bfloat16 and K == 18944))
    if M > 8 and tiles and xdt == torch.float32:
        tol = 2.5e-4  # (one part of x)
    assert _err(y, x.double() @ wd.t(), x, wd) <= (tol if tiles else 2.0 ** -8 + tol)


# Which kernel serves a call shows in its bits: the int8 GEMV gives a row of four the bits it has in a call
# of two rows, the GEMM a row of nine those it has among seventeen.
@pytest.mark.parametrize("xdt,M,N,K,G,tiles", [
    (torch.float32, 4, 2048, 9984, 128, True), (torch.float32, 4, 2048, 10240, 128, False),
    (torch.float32, 4, 2560, 10240, 128, True), (torch.bfloat16, 4, 2544, 17152, 128, False),
    (torch.bfloat16, 4, 2048, 17408, 128, True), (torch.float32, 3, 12288, 14464, 128, False),
    (torch.float32, 3, 12296, 14464, 128, True), (torch.float16, 5, 2048, 14336, 128, True),
    (torch.bfloat16, 4, 24576, 8320, 128, True), (torch.bfloat16, 4, 24584, 8320, 128, False),
    (torch.bfloat16, 4, 24584, 8192, 128, True),
    (torch.bfloat16, 9, 14336, 3072, 128, False), (torch.bfloat16, 16, 11008, 4096, 128, True),
    (torch.bfloat16, 9, 3056, 18944, 256, False), (torch.bfloat16, 16, 3072, 18944, 256, True),
    (torch.float16, 9, 1024, 18944, 256, False), (torch.float16, 16, 2048, 18944, 256, True),
    (torch.float16, 9, 2048, 22528, 256, False), (torch.float16, 16, 3072, 22528, 256, True)])
def test_int4_takes_the_faster_kernel(dev, xdt, M, N, K, G, tiles):
    print(f"[case] skinny route int4 x={xdt} M={M} N={N} K={K} G={G}", flush=True)
    g = torch.Generator(device=dev).manual_seed(K)
    codes = torch.randint(-2 ** 31, 2 ** 31, (N, K // 8), dtype=torch.int64, device=dev, generator=g).to(torch.int32)
    s = torch.rand(N, K // G, device=dev, generator=g) * 0.01
    z = torch.rand(N, K // G, device=dev, generator=g) * 15
    other = 2 if M <= 8 else 17
    x = torch.randn(max(M, other), K, device=dev, generator=g).to(xdt)
    ym, yo = (hipq.int4_matmul(x[:m].contiguous(), codes, s, z, G) for m in (M, other))
    n = min(M, other)
    assert torch.equal(ym[:n], yo[:n]) != tiles


@pytest.mark.parametrize("dt,N,K,tiles", [(hipq.Q4_K, 24576, 4352, True), (hipq.Q4_K, 24592, 4352, False),
                                          (hipq.Q5_K, 28656, 4352, False), (hipq.Q5_K, 28672, 4352, True),
                                          (hipq.Q4_K, 24592, 16640, True), (hipq.Q5_K, 24592, 16640, False)])
def test_many_long_rows_of_four_take_the_faster_kernel(dev, dt, N, K, tiles):
    print(f"[case] skinny route dt={hipq.NAMES[dt]} N={N} K={K}", flush=True)
    w = _big_weight(dt, N, K, dev)
    x = torch.randn(4, K, device=dev, generator=torch.Generator(device=dev).manual_seed(K))
    y4, y2 = hipq.matmul_q(x, w, N, K, dt), hipq.matmul_q(x[:2].contiguous(), w, N, K, dt)
    assert torch.equal(y4[:2], y2) != tiles


@pytest.mark.parametrize("dt", [hipq.Q4_K, hipq.Q5_K])
@pytest.mark.parametrize("M,H,I,gemv", [(3, 2048, 8192, True), (4, 1536, 16384, True), (4, 2048, 16640, False),
                                        (4, 2304, 8192, False), (5, 2048, 8192, False)])
def test_narrow_mlp_of_four_rows_takes_the_gemv(dev, dt, M, H, I, gemv):
    print(f"[case] skinny route mlp dt={hipq.NAMES[dt]} M={M} H={H} I={I}", flush=True)
    wg, wu, wd = (_big_weight(dt, r, c, dev) for r, c in ((I, H), (I, H), (H, I)))
    x = torch.randn(M, H, device=dev, generator=torch.Generator(device=dev).manual_seed(M)) * 0.01
    want = hipq.matmul_q_act(hipq.matmul_q_gated_act(x, wg, wu, I, H, dt), wd, M, H, I, dt)
    assert torch.equal(hipq.mlp_q(x, wg, wu, wd, H, I, dt), want) == gemv
