"""The flash prefill's packed rows (the q heads of a kv head share row blocks)
and its half-tile pipeline, at the sizes where they can go wrong: groups that
do not divide a wave's 32 rows, blocks and waves that end mid-token, one to a
few key tiles (the pipeline's first and last tile), the step from one head per
block to packed heads (64 / 65 tokens), and the one-round ordering of the
blocks on either side of one workgroup per compute unit. Against the oracle,
with the attention tolerance of the other prefill tests."""
import numpy as np
import pytest
import torch

import oracle_lib as O
import runtherder_amd as R
from gpu_util import DEV, NTHREADS, bf16_dev, bf16_host, f32_dev, int_dev, step, sync, u8_dev
from test_gpu_prefill import dynamic_range_inputs, mixed_magnitude_q

pytestmark = pytest.mark.gpu


def run(n, clen, hq, hkv, seed):
    d, total = 128, clen + n
    q = O.normal_bf16((n, hq, d), seed)
    k8, ks = O.quantize_kv_fp8(O.normal_bf16((total * hkv, d), seed + 1), d)
    v8, vs = O.quantize_kv_fp8(O.normal_bf16((total * hkv, d), seed + 2), d)
    out = torch.full((n, hq, d), float("nan"), dtype=torch.bfloat16, device=DEV)
    step(f"packed prefill n={n} clen={clen} hq={hq} hkv={hkv}")
    R.flash_prefill_bf16(out, bf16_dev(q), u8_dev(k8), u8_dev(v8), f32_dev(ks), f32_dev(vs), n,
                         int_dev(clen), hq, hkv, d, d ** -0.5)
    sync()
    got = bf16_host(out)
    rows = min(n, 48)   # the last (longest) tokens in full, and the first ones
    want = O.attention_f32(q[-rows:], k8, v8, ks, vs, rows, total - rows, hq, hkv, d, d ** -0.5,
                           NTHREADS)
    mx, mean = O.bf16_err(got[-rows:], want)
    assert mx <= 2e-2 and mean <= 2e-3, (mx, mean)
    first = min(n, 40)
    want = O.attention_f32(q[:first], k8, v8, ks, vs, first, clen, hq, hkv, d, d ** -0.5, NTHREADS)
    mx, mean = O.bf16_err(got[:first], want)
    assert mx <= 2e-2 and mean <= 2e-3, (mx, mean)
    assert np.isfinite(O.bf16_to_f32(got)).all()
    # Two tokens of every 128, the first and one inside.
    for t in [t for b in range(40, n - 48, 128) for t in (b, min(b + 77, n - 1))]:
        row = O.attention_f32(q[t:t + 1], k8, v8, ks, vs, 1, clen + t, hq, hkv, d, d ** -0.5,
                              NTHREADS)
        mx, mean = O.bf16_err(got[t:t + 1], row)
        assert mx <= 2e-2 and mean <= 2e-3, (t, mx, mean)


# (tokens, cached, q heads, kv heads): G = 7, 3, 5, 1, 32
@pytest.mark.parametrize("n,clen,hq,hkv", [
    (1, 0, 28, 4), (2, 62, 28, 4), (19, 45, 24, 8), (64, 0, 15, 3), (65, 0, 15, 3),
    (65, 127, 28, 4), (91, 37, 28, 4), (128, 64, 24, 8), (129, 63, 6, 6), (33, 300, 32, 1),
    (86, 511, 24, 8)])
def test_packed_rows_match_oracle(n, clen, hq, hkv):
    run(n, clen, hq, hkv, 7000 + n)


# Grids just below and above one 128-row workgroup per compute unit, and at the
# end of the one-round ordering (two per compute unit): 8 kv heads, G = 1. Every
# row block is checked (run), the ones on both sides of the reordering among them.
@pytest.mark.parametrize("step_blocks", [-1, 0, 1])
@pytest.mark.parametrize("rounds", [1, 2])
def test_one_round_block_order(rounds, step_blocks):
    cus = torch.cuda.get_device_properties(0).multi_processor_count
    blocks = rounds * (cus // 8) + step_blocks
    run(128 * blocks - 5, 0, 8, 8, 7300 + 10 * rounds + step_blocks)


# Key runs of few tokens (41..80 with splits that fill the chip): run minimum
# of 2 tiles and of 4 (from 65 tokens, over 2560 rows) on both sides of one run,
# ragged last runs, runs without keys for the first rows, G = 3, 4, 6, 7, and the
# split count just below the switch.
@pytest.mark.parametrize("n,clen,hq,hkv,splits", [
    (41, 0, 24, 8, 32), (48, 80, 32, 8, 16), (48, 81, 32, 8, 16), (64, 64, 32, 8, 16),
    (64, 65, 32, 8, 16), (65, 191, 32, 8, 16), (66, 191, 32, 8, 16), (80, 1000, 28, 4, 22),
    (80, 3001, 24, 8, 15), (50, 5000, 28, 4, 64), (64, 3000, 32, 8, 15),
    (80, 48, 32, 8, 16), (80, 49, 32, 8, 16), (65, 191, 48, 8, 8), (66, 191, 48, 8, 8)])
def test_few_token_key_runs_match_oracle(n, clen, hq, hkv, splits):
    d, total = 128, clen + n
    q = O.normal_bf16((n, hq, d), 7500 + n)
    k8, ks = O.quantize_kv_fp8(O.normal_bf16((total * hkv, d), 7501 + n), d)
    v8, vs = O.quantize_kv_fp8(O.normal_bf16((total * hkv, d), 7502 + n), d)
    out = torch.full((n, hq, d), float("nan"), dtype=torch.bfloat16, device=DEV)
    part = R.new_flash_split_scratch(n * hq, d, splits)
    step(f"key runs n={n} clen={clen} hq={hq} hkv={hkv} splits={splits}")
    R.flash_prefill_split_bf16(out, bf16_dev(q), u8_dev(k8), u8_dev(v8), f32_dev(ks), f32_dev(vs),
                               part, splits, n, int_dev(clen), hq, hkv, d, d ** -0.5)
    sync()
    want = O.attention_f32(q, k8, v8, ks, vs, n, clen, hq, hkv, d, d ** -0.5, NTHREADS)
    mx, mean = O.bf16_err(bf16_host(out), want)
    assert mx <= 2e-2 and mean <= 2e-3, (mx, mean)


# The merge of the runs: a whole wave per row up to 4096 rows, half a wave
# beyond, each in batches of 16 / 8 runs and maxima over 32: one run, two, the
# edges of a batch and of the maximum's first load, and rows past one pass.
@pytest.mark.parametrize("n,hq,hkv,tiles,run_tiles", [
    (42, 24, 8, 2, 2), (42, 24, 8, 4, 2), (42, 24, 8, 32, 2), (42, 24, 8, 34, 2),
    (42, 24, 8, 64, 2), (42, 24, 8, 66, 2), (64, 64, 8, 34, 2), (65, 64, 8, 8, 4),
    (65, 64, 8, 32, 4), (65, 64, 8, 36, 4), (300, 64, 8, 17, 8),
    # (rows by XCD: one and two kv heads each, groups of 1, 2 and 3; 4, 2 and 1 kv
    # heads over two, four and all XCDs; in order: 5 and 12 kv heads)
    (81, 16, 16, 12, 4), (83, 48, 16, 9, 4), (99, 16, 8, 12, 4), (137, 48, 16, 17, 8),
    (81, 28, 4, 12, 4), (45, 28, 4, 30, 2), (83, 10, 2, 9, 4), (201, 64, 2, 17, 8),
    (97, 7, 1, 12, 4), (101, 15, 5, 9, 4), (82, 24, 12, 9, 4)])
def test_key_run_merge_matches_oracle(n, hq, hkv, tiles, run_tiles):
    d, total = 128, 64 * tiles - 3
    clen, splits = total - n, max(32, tiles // run_tiles)
    q = O.normal_bf16((n, hq, d), 7600 + tiles)
    k8, ks = O.quantize_kv_fp8(O.normal_bf16((total * hkv, d), 7601 + tiles), d)
    v8, vs = O.quantize_kv_fp8(O.normal_bf16((total * hkv, d), 7602 + tiles), d)
    out = torch.full((n, hq, d), float("nan"), dtype=torch.bfloat16, device=DEV)
    part = R.new_flash_split_scratch(n * hq, d, splits)
    part.fill_(float("nan"))   # slots without a live run hold anything
    step(f"merge n={n} hq={hq} tiles={tiles} splits={splits}")
    R.flash_prefill_split_bf16(out, bf16_dev(q), u8_dev(k8), u8_dev(v8), f32_dev(ks), f32_dev(vs),
                               part, splits, n, int_dev(clen), hq, hkv, d, d ** -0.5)
    sync()
    want = O.attention_f32(q, k8, v8, ks, vs, n, clen, hq, hkv, d, d ** -0.5, NTHREADS)
    mx, mean = O.bf16_err(bf16_host(out), want)
    assert mx <= 2e-2 and mean <= 2e-3, (mx, mean)


# A key whose score is NaN (an E4M3 NaN code, a NaN scale) or infinite (an
# infinite scale) makes NaN of the rows that see it, in whichever of the runs it
# lies, and of nothing else. (A row whose score is -inf keeps its other keys,
# here and in the plain prefill; the oracle, which scales the codes first, makes
# NaN of 0 x inf.)
@pytest.mark.parametrize("what", ["k code", "k_scale nan", "k_scale inf", "v code"])
@pytest.mark.parametrize("n,clen,splits,key", [
    (48, 2000, 16, 5), (48, 2000, 16, 1000), (64, 3000, 16, 3030), (100, 3000, 16, 1500),
    (250, 5000, 8, 5100)])
def test_key_runs_propagate_nan(n, clen, splits, key, what):
    hq, hkv, d, total = 32, 8, 128, clen + n
    q = O.normal_bf16((n, hq, d), 7700 + n)
    k8, ks = O.quantize_kv_fp8(O.normal_bf16((total * hkv, d), 7701 + n), d)
    v8, vs = O.quantize_kv_fp8(O.normal_bf16((total * hkv, d), 7702 + n), d)
    at = key * hkv + 3   # kv head 3
    if what == "k code":
        k8[at, 17] = 0x7F
    elif what == "v code":
        v8[at, 17] = 0x7F
    else:
        ks[at] = np.nan if what == "k_scale nan" else np.inf
    out = torch.full((n, hq, d), 7.0, dtype=torch.bfloat16, device=DEV)
    part = R.new_flash_split_scratch(n * hq, d, splits)
    step(f"key runs with a NaN: {what} n={n} clen={clen} splits={splits} key={key}")
    R.flash_prefill_split_bf16(out, bf16_dev(q), u8_dev(k8), u8_dev(v8), f32_dev(ks), f32_dev(vs),
                               part, splits, n, int_dev(clen), hq, hkv, d, d ** -0.5)
    sync()
    got = O.bf16_to_f32(bf16_host(out))
    plain = torch.full_like(out, 7.0)
    R.flash_prefill_bf16(plain, bf16_dev(q), u8_dev(k8), u8_dev(v8), f32_dev(ks), f32_dev(vs), n,
                         int_dev(clen), hq, hkv, d, d ** -0.5)
    sync()
    plain = O.bf16_to_f32(bf16_host(plain))
    with np.errstate(invalid="ignore"):
        want = O.bf16_to_f32(O.attention_f32(q, k8, v8, ks, vs, n, clen, hq, hkv, d, d ** -0.5,
                                             NTHREADS))
    nan = np.isnan(want)
    assert nan.any() and not nan.all()
    if what == "v code":
        # P V runs in MFMAs over 32 keys: a row of the key's tile that does not
        # see it gets 0 x NaN, as in the plain prefill; rows after it all do.
        first = max(0, key - clen)
        assert np.isnan(got[first:, 12:16, 17]).all()
        assert not np.isnan(np.delete(got, 17, axis=2)).any()
        return
    assert np.array_equal(np.isnan(got), np.isnan(plain))
    if what == "k_scale inf":
        assert np.isnan(got).any() and not np.isnan(got)[~nan].any()
    else:
        assert np.array_equal(np.isnan(got), nan)
    assert np.abs(got - want)[~nan].max() <= 2e-2


# Scores that jump by hundreds between the runs and q rows whose elements span 22
# binades, through the key runs' own reference maxima and the merge.
@pytest.mark.parametrize("what", ["score range", "mixed q"])
@pytest.mark.parametrize("n,splits", [(48, 16), (100, 16), (250, 8)])
def test_key_runs_dynamic_range(n, splits, what):
    hq, hkv, d, total = 32, 8, 128, 1300
    q, k8, v8, ks, vs = dynamic_range_inputs(total, hq, hkv, d)
    q = q[-n:]
    if what == "mixed q":
        q = mixed_magnitude_q(n, hq, d, 46)
        ks = np.minimum(ks, np.float32(0.02))   # (the score range alone is the other case)
    out = torch.full((n, hq, d), float("nan"), dtype=torch.bfloat16, device=DEV)
    part = R.new_flash_split_scratch(n * hq, d, splits)
    step(f"key runs, {what} n={n} splits={splits}")
    R.flash_prefill_split_bf16(out, bf16_dev(q), u8_dev(k8), u8_dev(v8), f32_dev(ks), f32_dev(vs),
                               part, splits, n, int_dev(total - n), hq, hkv, d, d ** -0.5)
    sync()
    want = O.attention_f32(q, k8, v8, ks, vs, n, total - n, hq, hkv, d, d ** -0.5, NTHREADS)
    mx, mean = O.bf16_err(bf16_host(out), want)
    assert mx <= 2e-2 and mean <= 2e-3, (mx, mean)


# An odd row count and an odd split count: the scratch's O rows start 8 bytes
# past a 16-byte boundary. 81 tokens: key runs; 9: the decode kernel's route.
@pytest.mark.parametrize("n", [81, 9])
def test_odd_rows_and_splits_match_oracle(n):
    hq, hkv, d, clen, splits = 7, 1, 128, 1000, 3
    total = clen + n
    q = O.normal_bf16((n, hq, d), 7800 + n)
    k8, ks = O.quantize_kv_fp8(O.normal_bf16((total * hkv, d), 7801 + n), d)
    v8, vs = O.quantize_kv_fp8(O.normal_bf16((total * hkv, d), 7802 + n), d)
    out = torch.full((n, hq, d), float("nan"), dtype=torch.bfloat16, device=DEV)
    part = R.new_flash_split_scratch(n * hq, d, splits)
    assert part.data_ptr() % 16 == 0 and n * hq * splits % 2 == 1
    step(f"odd rows and splits n={n}")
    R.flash_prefill_split_bf16(out, bf16_dev(q), u8_dev(k8), u8_dev(v8), f32_dev(ks), f32_dev(vs),
                               part, splits, n, int_dev(clen), hq, hkv, d, d ** -0.5)
    sync()
    want = O.attention_f32(q, k8, v8, ks, vs, n, clen, hq, hkv, d, d ** -0.5, NTHREADS)
    mx, mean = O.bf16_err(bf16_host(out), want)
    assert mx <= 2e-2 and mean <= 2e-3, (mx, mean)


# Slabs and tensors that start 4 or 8 bytes past a 16-byte boundary (a view into
# a larger buffer): the copies and stores are 16 bytes wide.
@pytest.mark.parametrize("at", [4, 8])
@pytest.mark.parametrize("n,clen", [(70, 100), (300, 60)])
def test_slabs_off_a_16_byte_boundary(n, clen, at):
    hq, hkv, d, total = 24, 8, 128, clen + n

    def shifted(t):
        raw = torch.zeros(t.numel() * t.element_size() + 16, dtype=torch.uint8, device=DEV)
        got = raw[at:at + t.numel() * t.element_size()].view(t.dtype).view(t.shape)
        got.copy_(t)
        assert got.data_ptr() % 16 == at
        return got

    q = O.normal_bf16((n, hq, d), 7900 + n)
    k8, ks = O.quantize_kv_fp8(O.normal_bf16((total * hkv, d), 7901 + n), d)
    v8, vs = O.quantize_kv_fp8(O.normal_bf16((total * hkv, d), 7902 + n), d)
    out = torch.full((n, hq, d), float("nan"), dtype=torch.bfloat16, device=DEV)
    got = shifted(out)
    step(f"slabs {at} bytes off n={n} clen={clen}")
    args = (n, int_dev(clen), hq, hkv, d, d ** -0.5)
    kv = (u8_dev(k8), u8_dev(v8), f32_dev(ks), f32_dev(vs))
    R.flash_prefill_bf16(out, bf16_dev(q), *kv, *args)
    R.flash_prefill_bf16(got, shifted(bf16_dev(q)), *map(shifted, kv), *args)
    sync()
    assert np.array_equal(bf16_host(got), bf16_host(out))
    assert not torch.isnan(got).any()


# The most splits an entry takes, at few rows: most runs hold no key.
@pytest.mark.parametrize("n", [41, 81])
def test_most_splits(n):
    hq, hkv, d, clen, splits = 1, 1, 128, 1000, 65536
    total = clen + n
    q = O.normal_bf16((n, hq, d), 7950 + n)
    k8, ks = O.quantize_kv_fp8(O.normal_bf16((total * hkv, d), 7951 + n), d)
    v8, vs = O.quantize_kv_fp8(O.normal_bf16((total * hkv, d), 7952 + n), d)
    out = torch.full((n, hq, d), float("nan"), dtype=torch.bfloat16, device=DEV)
    part = R.new_flash_split_scratch(n * hq, d, splits)
    step(f"most splits n={n}")
    R.flash_prefill_split_bf16(out, bf16_dev(q), u8_dev(k8), u8_dev(v8), f32_dev(ks), f32_dev(vs),
                               part, splits, n, int_dev(clen), hq, hkv, d, d ** -0.5)
    sync()
    want = O.attention_f32(q, k8, v8, ks, vs, n, clen, hq, hkv, d, d ** -0.5, NTHREADS)
    mx, mean = O.bf16_err(bf16_host(out), want)
    assert mx <= 2e-2 and mean <= 2e-3, (mx, mean)


def test_few_token_key_runs_refuse_what_the_decode_route_refused():
    hq, hkv, d = 17, 1, 128   # a group the MFMA decode kernel does not serve
    out = torch.empty((64, hq, d), dtype=torch.bfloat16, device=DEV)
    kv = torch.zeros((100, hkv, d), dtype=torch.uint8, device=DEV)
    s = torch.zeros((100, hkv), dtype=torch.float32, device=DEV)
    part = R.new_flash_split_scratch(64 * hq, d, 128)
    with pytest.raises(R._ffi.RthError, match="head_dim"):
        R.flash_prefill_split_bf16(out, out, kv, kv, s, s, part, 128, 64, int_dev(0), hq, hkv, d,
                                   0.1)
