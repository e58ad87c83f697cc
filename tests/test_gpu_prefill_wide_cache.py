"""The flash prefill over a cache whose K and V slabs are larger than 4 GiB:
row offsets that do not fit 32 bits. Only the first keys carry a V and a
score, so the rest of the cache (zeros) is a term of the softmax's
denominator and a float64 reference over the first keys is the whole answer."""
import math

import numpy as np
import pytest
import torch

import runtherder_amd as R
from gpu_util import DEV, int_dev, step, sync

pytestmark = pytest.mark.gpu


# keys x kv heads x 128 = 2^32 + 33 rows: the distance from the first tile to
# the end of the cache, times the row's bytes, is 2^32 and a few rows.
@pytest.mark.parametrize("hkv,rest", [(64, 33), (64, 1)])
def test_first_tile_of_a_slab_past_4_gib(hkv, rest):
    d, n = 128, 1
    total = (1 << 32) // (hkv * d) + rest
    g = torch.Generator(device=DEV)
    g.manual_seed(31 + rest)
    k = torch.zeros((total, hkv, d), dtype=torch.uint8, device=DEV)
    v = torch.zeros((total, hkv, d), dtype=torch.uint8, device=DEV)
    ks = torch.ones((total, hkv), dtype=torch.float32, device=DEV)
    vs = torch.ones((total, hkv), dtype=torch.float32, device=DEV)
    k[:64] = torch.randn((64, hkv, d), generator=g, device=DEV).to(torch.float8_e4m3fn).view(
        torch.uint8)
    v[:64] = torch.randn((64, hkv, d), generator=g, device=DEV).to(torch.float8_e4m3fn).view(
        torch.uint8)
    q = (4 * torch.randn((n, hkv, d), generator=g, device=DEV)).to(torch.bfloat16)
    out = torch.empty((n, hkv, d), dtype=torch.bfloat16, device=DEV)
    step(f"prefill over {total} keys x {hkv} kv heads")
    R.flash_prefill_bf16(out, q, k, v, ks, vs, n, int_dev(total - n), hkv, hkv, d, d ** -0.5)
    sync()
    kf = k[:64].view(torch.float8_e4m3fn).cpu().to(torch.float64).numpy()
    vf = v[:64].view(torch.float8_e4m3fn).cpu().to(torch.float64).numpy()
    s = np.einsum("hd,jhd->hj", q[0].cpu().to(torch.float64).numpy(), kf) / math.sqrt(d)
    m = np.maximum(s.max(1, keepdims=True), 0.0)
    p = np.exp(s - m)
    den = p.sum(1, keepdims=True) + (total - 64) * np.exp(-m)
    want = np.einsum("hj,jhd->hd", p / den, vf)
    got = out[0].cpu().to(torch.float64).numpy()
    # bf16 output (2^-9 of a value) and f16 p and V (2^-11 each); absolute where
    # the terms cancel.
    err = np.abs(got - want)
    assert (err <= 2.0 ** -7 * np.abs(want) + 2.0 ** -9 * np.abs(want).max()).all(), err.max()
