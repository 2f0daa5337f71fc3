"""hq_dequant to BF16 is its F32 output rounded once (dtype/half.go:118-129), bit for bit, on blocks of
random bytes: scales that are NaN, infinite or subnormal come up too."""
import numpy as np
import pytest
import torch

import oracle
from light_amd import hipq, synth

pytestmark = pytest.mark.gpu

FORMATS = [hipq.Q8_0, hipq.Q4_0, hipq.Q5_0, hipq.Q4_K, hipq.Q5_K, hipq.Q6_K]


def _bf16(f32):
    """BF16FromF32: to nearest even; a NaN keeps its top bits with the quiet bit set."""
    u = f32.view(np.uint32).astype(np.uint64)
    return np.where(np.isnan(f32), (u >> 16) | 0x40, (u + 0x7FFF + ((u >> 16) & 1)) >> 16).astype(np.uint16)


@pytest.mark.parametrize("dt", FORMATS)
@pytest.mark.parametrize("n", [256, 256 * 37, 256 * 4099])
def test_bf16_is_f32_rounded_once(dev, dt, n):
    size = synth.gguf_weight(dt, 1, 256, synth.rng(0)).nbytes * (n // 256)
    raw = np.random.default_rng(n + dt).integers(0, 256, size, dtype=np.uint8)
    src = torch.from_numpy(raw).to(dev)
    f32 = hipq.dequant(src, n, dt, hipq.F32).cpu().numpy().reshape(-1)
    got = hipq.dequant(src, n, dt, hipq.BF16).view(torch.int16).cpu().numpy().view(np.uint16).reshape(-1)
    assert np.isnan(f32).any() or n == 256
    np.testing.assert_array_equal(got, _bf16(f32))
    ref = oracle.dequant(dt, raw, n).reshape(-1)
    ok = ~np.isnan(ref)
    np.testing.assert_array_equal(np.isnan(f32), ~ok)
    np.testing.assert_array_equal(f32.view(np.uint32)[ok], ref.view(np.uint32)[ok])
