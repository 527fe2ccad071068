"""Tier 2's double-double pass (ea_refine.h): rows that tier 1 lists are certified there, or go on to
the 128-bit path; either way the bits are the oracle's."""

import numpy as np
import pytest

from exactattention_amd.formats import default_alpha_bits
from test_gpu_parity import _oracle, _rand_problem, _run

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("T,S,kind", [(300, 300, "normal"), (70, 1000, "normal"), (64, 130, "outlier"), (96, 200, "dupes"),
                                      (80, 129, "wide")])
def test_many_listed_rows(gpu, T, S, kind):
    """fp32 outputs of the int8 prefill kernel with logits 4 times the usual scale: its bounds leave
    many rows, more than the pass has chunk counters for, so blocks take whole rows. dupes: sums
    that are exact and quotients that tie."""
    rng = np.random.default_rng(T + S)
    prob = _rand_problem(rng, kind, kind, B=1, T=T, Hq=2, Hkv=1, S=S, d=128, dv=128)
    ab = int(np.float32(0.5).view(np.uint32))
    want, wflags = _oracle(prob, ab, "fp32")
    got, flags, st = _run(prob, ab, "fp32")
    assert not np.any(wflags) and not flags.any(), st
    assert np.array_equal(got, want), st
    assert st["tier2_certified"] == st["tier1_flagged"], st
    if kind == "normal":
        assert st["tier1_flagged"] > 32, st
    # decided by the double-double pass itself, but for terms a window apart (wide) or past 2^-120 (outlier)
    assert st["tier2_wide_rows"] == 0 or kind in ("wide", "outlier"), st
    assert kind != "wide" or st["tier2_wide_rows"] > 0, st


@pytest.mark.parametrize("d,dv", [(128, 128), (64, 64), (40, 6)])
@pytest.mark.parametrize("S", [1, 127, 129, 5000])
def test_few_listed_rows(gpu, d, dv, S):
    """Rows that cancel to about 2^-45 of their terms in some channels fail tier 1's bound whatever
    the kernel: few of them, so their keys are split into chunks; a chunk without keys, tree keys,
    misaligned rows. Their neighbours are certified by tier 1."""
    rng = np.random.default_rng(d + S)
    prob = _rand_problem(rng, "normal", "normal", B=2, T=1, Hq=2, Hkv=2, S=S + 60, d=d, dv=dv)
    prob["seq_len"][:] = S + 60
    prob["kv_len"][:] = S
    prob["tree_base"] = np.full(2, S, np.int32)
    prob["tree_mask"] = np.array([(1 << 59) | 5, 0], np.uint64)
    # sequence 0, head 0: q = 0, so all weights are equal; channel 0 sums to one small element
    prob["q"][0, 0, 0] = 0
    n = S + 3  # its visible keys
    col = np.zeros(n, np.uint16)
    col[0:n - 1:2], col[1:n:2] = 0x3FC0, 0xBFC0  # 1.5, -1.5, ...
    if n % 2:
        col[n - 1] = 0
    col[n // 2] = (0x2C00 if col[n // 2] == 0 else col[n // 2])
    keys = np.concatenate([np.arange(S), S + np.array([0, 2, 59])])
    prob["v"][0, 0, keys, 0] = col
    if n > 2:
        prob["v"][0, 0, keys[n - 1], 0] = 0x2C00  # about 2^-39
        if n % 2 == 0:
            prob["v"][0, 0, keys[n - 2], 0] = 0
    ab = default_alpha_bits(d)
    for out in ("bf16", "fp32"):
        want, wflags = _oracle(prob, ab, out)
        got, flags, st = _run(prob, ab, out)
        assert not np.any(wflags) and not flags.any(), st
        assert np.array_equal(got, want), st
        assert st["tier2_certified"] == st["tier1_flagged"] == 1 and st["tier2_wide_rows"] == 0, st


def test_domain_errors_among_listed_rows(gpu):
    """NaN/inf in q, K and V, an fp32 logit overflow and a row without keys, beside rows the pass
    certifies: exactly those that see a bad value are flag 2, +0."""
    rng = np.random.default_rng(9)
    T = 70
    prob = _rand_problem(rng, "normal", "normal", B=1, T=T, Hq=2, Hkv=1, S=400, d=128, dv=128)
    prob["seq_len"][:] = 400
    prob["kv_len"][:] = 200 + np.arange(T)
    prob["kv_len"][3] = 0
    ab = int(np.float32(0.5).view(np.uint32))
    want, _ = _oracle(prob, ab, "fp32")
    prob["q"][0, 3, 0, 1] = 0x7FC0   # without keys: still a domain error
    prob["q"][0, 10, 1, 0] = 0xFF80
    prob["k"][0, 0, 250, 5] = 0x7FC0  # tokens 51 ..
    prob["v"][0, 0, 260, 7] = 0x7F80  # tokens 61 ..
    prob["q"][0, 20, 0, :] = 0x7F00   # about 2^127 per element: the logit overflows
    got, flags, st = _run(prob, ab, "fp32")
    exp = np.zeros((T, 2), np.uint8)
    exp[3, 0] = exp[10, 1] = exp[20, 0] = 2
    exp[51:] = 2
    assert np.array_equal(flags.reshape(T, 2), exp), st
    ok = exp[None] == 0
    assert np.array_equal(got[ok], want[ok]) and not got[~ok].any(), st


def _spread_problem(rng, B, T, Hq, Hkv, S, d):
    """Logits of exactly +600 and -600 (alpha 1) in every row, and a few of 600.5 below the top: weights
    1200 binades apart, which tier 1 flags and the double-double pass (800 at most) leaves."""
    prob = _rand_problem(rng, "normal", "normal", B=B, T=T, Hq=Hq, Hkv=Hkv, S=S, d=d, dv=d)
    prob["seq_len"][:] = S
    prob["kv_len"][:] = np.tile(S - T + 1 + np.arange(T), B)
    prob["q"][:] = 0
    prob["q"][..., 0] = 0x3F80
    t = rng.choice(np.float32([600, 599.5, -600]), size=prob["k"].shape[:3])
    t[:, :, :2] = [600, -600]
    prob["k"][:] = 0
    hi = np.float32(np.round(t / 8) * 8)  # bf16 keeps 8 bits: t as two terms
    prob["k"][..., 0] = hi.view(np.uint32) >> 16
    prob["q"][..., 1] = 0x3F80
    prob["k"][..., 1] = np.float32(t - hi).view(np.uint32) >> 16
    return prob


@pytest.mark.parametrize("out", ["bf16", "fp32"])
@pytest.mark.parametrize("B,T,Hq,Hkv,S,d", [(1, 1, 3, 1, 5000, 64), (1, 1, 4, 1, 90, 128), (2, 5, 8, 2, 700, 64),
                                            (3, 1, 64, 4, 300, 128), (8, 1, 40, 8, 200, 64)])
def test_rows_left_to_the_128_bit_path(gpu, B, T, Hq, Hkv, S, d, out):
    """Every row past the double-double pass: few rows (their keys split into chunks), more than there
    are blocks, and more than that pass counts chunks for; the 128-bit path certifies them all."""
    rng = np.random.default_rng(S)
    prob = _spread_problem(rng, B, T, Hq, Hkv, S, d)
    ab = int(np.float32(1).view(np.uint32))
    want, wflags = _oracle(prob, ab, out)
    got, flags, st = _run(prob, ab, out)
    assert st["tier2_wide_rows"] == flags.size == st["tier1_flagged"] == st["tier2_certified"], st
    assert not flags.any() and not np.any(wflags)
    assert np.array_equal(got, want), st


def test_rows_left_are_shared_by_the_blocks(gpu):
    """64 rows past the double-double pass take little longer than on force_tier2's 32 blocks (a single block
    took 32 times as long), and so does one long row, whose keys are split."""
    import torch
    from exactattention_amd.hip import DeviceProblem, launch_hip
    rng = np.random.default_rng(1)
    ab = int(np.float32(1).view(np.uint32))
    for B, Hq, S in ((8, 8, 2000), (1, 1, 30000)):
        dp = DeviceProblem(_spread_problem(rng, B, 1, Hq, 1, S, 64))
        ms = {}
        for force in (False, True):
            for _ in range(3):
                a, b = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
                a.record()
                launch_hip(dp, ab, force_tier2=force)
                b.record()
                torch.cuda.synchronize()
                ms[force] = min(ms.get(force, 1e9), a.elapsed_time(b))
        assert not dp.flags.any()
        assert ms[False] < 4 * ms[True], (B, S, ms)


def test_reference_moves_past_the_number_range(gpu):
    """A row's reference exponent moves by 790 binades twice, each move in another pass of 128 keys (more
    rows than are split into chunks): the first pass's terms end below the smallest fp64 number. Channel
    0's quotient is an exact tie; in channels 1 and 2 those terms put it below and above, by 2^-1580."""
    from exactattention_amd.hip import attention_problem
    rng = np.random.default_rng(0)
    prob = _rand_problem(rng, "normal", "normal", B=10, T=1, Hq=4, Hkv=2, S=384, d=64, dv=64)
    prob["seq_len"][:] = prob["kv_len"][:] = 384
    prob["q"][:] = 0
    prob["q"][..., :2] = 0x3F80
    prob["k"][:] = 0
    for p, (hi, lo) in enumerate(((0, 0), (784, 6), (1576, 4))):
        keys = slice(128 * p, 128 * p + 128)
        prob["k"][:, :, keys, 0] = int(np.float32(hi).view(np.uint32)) >> 16
        prob["k"][:, :, keys, 1] = int(np.float32(lo).view(np.uint32)) >> 16
        prob["v"][:, :, keys, :3] = (0x3F80 + np.arange(128) % 2)[:, None]  # 1 and 1 + 2^-7: the mean is a tie
    prob["v"][:, :, :128, 1] = 0x3F80
    prob["v"][:, :, :128, 2] = 0x3F81
    ab = int(np.float32(1).view(np.uint32))
    want, _ = _oracle(prob, ab)
    got, flags, st = attention_problem(prob, alpha_bits=ab)
    assert st["tier1_flagged"] == flags.size, st
    assert not flags.any() and np.array_equal(got, want), st
    assert (got[..., :3] == [0x3F80, 0x3F80, 0x3F81]).all()
