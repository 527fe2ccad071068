"""The multi-row split kernel (ea_mrow.hip) at the edges of its row blocks (4, 8, 16 rows), key steps
(16 keys per wave, 64 per tile), splits and head sizes, against the oracle. Every result is
certified, so the bar is equal bits."""

import ctypes

import numpy as np
import pytest

from exactattention_amd import problem
from exactattention_amd.formats import default_alpha_bits
from gen import bf16
from test_gpu_parity import _oracle, _rand_problem, _run

pytestmark = pytest.mark.gpu


def _block_rows(prob, splits=0):
    """Rows per block of the kernel the step takes (decided by sizes; pointers here are aligned ones)."""
    from exactattention_amd import hip
    ptrs = {n: 1 << 20 for n in ("q", "k", "v", "seq_len", "kv_len", "out", "flags")}
    if prob["block_table"] is not None:
        ptrs["block_table"] = 1 << 20
    return hip.step_route(prob["geom"], ptrs, splits=splits)[3]


def _check(prob, ab, out="bf16", splits=0, mrow=True):
    want, wflags = _oracle(prob, ab, out)
    got, flags, st = _run(prob, ab, out, splits)
    assert st["decode_kernel_rows"] == flags.size and st["mrow_kernel_rows"] == (flags.size if mrow else 0), st
    assert not flags.any() and not np.any(wflags), st
    assert np.array_equal(got, want), st
    # tier 1 itself decides these rows: seen were none in bf16 and up to 8 of 2520 in fp32, whose 24 bits
    # leave a rounding undecided for one channel in some 10^5
    assert st["tier1_flagged"] <= (2 + flags.size // 50 if out == "fp32" else 1 + flags.size // 1000), st
    assert st["tier2_wide_rows"] == 0, st
    return st


@pytest.mark.parametrize("T,grp", [(1, 3), (1, 4), (5, 1), (2, 4), (3, 3), (1, 16), (17, 1), (9, 2)])
@pytest.mark.parametrize("d,dv", [(8, 4), (64, 64), (72, 40), (128, 64), (96, 96), (128, 128)])
def test_rows_and_head_sizes(gpu, T, grp, d, dv):
    """3 to 18 rows per segment (one full row block, one row more, a partial one), head sizes on both
    sides of the 64-dim variant and with dims or channels that fill a chunk only in part; one key,
    a wave's step and a tile with one key less and more, and several splits. Contiguous and paged."""
    rng = np.random.default_rng(1000 * T + 100 * grp + d + dv)
    ab = default_alpha_bits(d)
    for S, page in ((T, 0), (15 + T, 16), (16, 0), (17, 64), (63 + T, 0), (64, 16), (65 + T, 16), (777, 64)):
        prob = _rand_problem(rng, "normal", "normal", B=2, T=T, Hq=2 * grp, Hkv=2, S=max(S, T), d=d, dv=dv)
        if page:
            prob = problem.to_paged(prob, page, rng, "HND" if S & 1 else "NHD")
        _check(prob, ab, "fp32" if S & 2 else "bf16", splits=3 if S == 777 else 0)


@pytest.mark.parametrize("T,grp,rb", [(5, 1, 8), (1, 8, 8), (9, 1, 16), (1, 16, 16), (17, 1, 16), (9, 2, 16)])
@pytest.mark.parametrize("d,dv", [(8, 4), (64, 64), (72, 40), (128, 64), (96, 96), (128, 128)])
def test_wide_row_blocks(gpu, T, grp, rb, d, dv):
    """Blocks of 8 and 16 rows, which only steps of many units take: the same edges, contiguous and
    paged, one and several splits."""
    rng = np.random.default_rng(1000 * T + 100 * grp + d + dv + 1)
    ab = default_alpha_bits(d)
    for S, page, splits in ((T, 0, 0), (15 + T, 16, 0), (64, 0, 0), (65 + T, 16, 0), (200, 64, 2)):
        prob = _rand_problem(rng, "normal", "normal", B=70, T=T, Hq=2 * grp, Hkv=2, S=max(S, T), d=d, dv=dv)
        if page:
            prob = problem.to_paged(prob, page, rng, "HND" if S & 1 else "NHD")
        assert _block_rows(prob, splits) == rb
        _check(prob, ab, "fp32" if S & 2 else "bf16", splits=splits)


@pytest.mark.parametrize("rows", [4, 8, 16])
@pytest.mark.parametrize("kind", ["wide", "outlier", "dupes", "subnormal"])
def test_value_kinds(gpu, rows, kind):
    """Scores that cancel over 48 binades, exact zeros and ties, subnormals; and logits hundreds apart
    (alpha 8), so that reference exponents move by more than their headroom. Long rows of few
    segments (4-row blocks) and short rows of many (8 and 16). Every row ends with the oracle's bits,
    at most a few of them through the host tier."""
    from exactattention_amd.hip import attention_problem
    rng = np.random.default_rng(rows)
    for d, alpha in ((128, None), (64, np.float32(8.0))):
        for B, S in ((2, 1500), (70, 130)):
            prob = _rand_problem(rng, kind, kind, B=B, T=1, Hq=2 * rows, Hkv=2, S=S, d=d, dv=d)
            assert _block_rows(prob) == (rows if B == 70 else 4)
            ab = default_alpha_bits(d) if alpha is None else int(alpha.view(np.uint32))
            want, _ = _oracle(prob, ab)
            got, flags, st = attention_problem(prob, alpha_bits=ab)
            assert st["mrow_kernel_rows"] == flags.size, st
            assert not flags.any() and np.array_equal(got, want), st
            assert st["host_exact_rows"] <= 1 + flags.size // 500, st  # seen: 1 of 2240, dupes
            if kind != "wide" and d == 128:  # tier 1's own: seen 3 of 64 (outlier), 976 of 2240 (subnormal)
                assert st["tier1_flagged"] <= flags.size // 2, st


@pytest.mark.parametrize("B,S", [(2, 1000), (70, 150)])
@pytest.mark.parametrize("rows", [4, 8, 16])
def test_every_pair_waits(gpu, rows, B, S):
    """Logits exactly half way between two fp32 values for every pair (alpha 1, s = k0 + 2^-24 with k0
    in [1, 2), in the even rows): no interval decides them, so every step fills the wave's list."""
    rng = np.random.default_rng(rows)
    prob = _rand_problem(rng, "normal", "normal", B=B, T=1, Hq=2 * rows, Hkv=2, S=S, d=64, dv=64)
    prob["q"][:, :, ::2, :] = 0
    prob["q"][:, :, ::2, 0] = 0x3F80               # 1
    prob["q"][:, :, ::2, 1] = 0x3380               # 2^-24
    prob["k"][..., 0] = 0x3F80 | rng.integers(0, 128, prob["k"].shape[:3])
    prob["k"][..., 1] = 0x3F80
    st = _check(prob, 0x3F800000)
    n = int(prob["seq_len"].sum()) * rows          # half of the 2 rows query heads, each with every key
    assert st["slow_path_scores"] >= n, (st, n)
    assert _block_rows(prob) == (rows if B > 2 else 4)


@pytest.mark.parametrize("B", [3, 72])
@pytest.mark.parametrize("rows", [4, 8, 16])
def test_trees_and_bad_rows(gpu, rows, B):
    """A tree mask across a step boundary; a NaN query row and an inf key flag exactly the rows that
    see them, and a segment without keys is +0. Few segments (4-row blocks) and many."""
    rng = np.random.default_rng(50 + rows)
    T, S, d = rows // 2, 100, 64
    prob = _rand_problem(rng, "normal", "normal", B=B, T=T, Hq=4, Hkv=2, S=S, d=d, dv=d)
    prob["seq_len"][:] = np.tile([S, 0, S], B // 3)
    prob["kv_len"][:] = np.tile(np.repeat([70, 0, 0], T), B // 3)
    prob["tree_base"] = np.tile(np.array([75, 0, 60], np.int32), B // 3)
    prob["tree_mask"] = rng.integers(0, 1 << 25, size=B * T).astype(np.uint64) | np.uint64(1)
    assert _block_rows(prob) == (4 if B == 3 else rows)
    ab = default_alpha_bits(d)
    _check(prob, ab)
    prob["q"][0, T - 1, 1, 5] = 0x7FC0
    prob["q"][1, 0, 0, 9] = 0xFF80   # a row without keys is still a domain error
    prob["k"][2, 1, 60, 3] = 0x7F80  # tree key 0 of sequence 2, KV head 1: every row of heads 2, 3
    clean = {k: (v.copy() if hasattr(v, "copy") else v) for k, v in prob.items()}
    clean["q"][0, T - 1, 1, 5] = 0
    clean["q"][1, 0, 0, 9] = 0
    clean["k"][2, 1, 60, 3] = 0
    want, _ = _oracle(clean, ab)
    got, flags, st = _run(prob, ab)
    exp = np.zeros((B, T, 4), np.uint8)
    exp[0, T - 1, 1] = exp[1, 0, 0] = 2
    exp[2, :, 2:] = 2
    assert np.array_equal(flags.reshape(exp.shape), exp), (flags, st)
    assert np.array_equal(got[exp == 0], want[exp == 0])


def test_equal_share_plan(gpu):
    """Ragged lengths on the equal-share plan, with shares that cross units, against the oracle and
    one split; 200 sequences of few keys, so that most shares reach several units."""
    ab = default_alpha_bits(128)
    for B, S, Hq, T in ((200, 900, 8, 1), (16, 3000, 16, 2)):
        rng = np.random.default_rng(B)
        lens = rng.integers(T, S + 1, size=B)
        lens[:2] = [S, T]
        q, k, v = bf16(rng, (B, T, Hq, 128)), bf16(rng, (B, 2, S, 128), "outlier"), bf16(rng, (B, 2, S, 128))
        prob = problem.contiguous(q, k, v, lens[:, None] - T + 1 + np.arange(T), seq_len=lens)
        prob = problem.to_paged(prob, 16, rng)
        want, _ = _oracle(prob, ab)
        for splits in (0, 40, 1):
            got, flags, st = _run(prob, ab, splits=splits)
            assert st["mrow_kernel_rows"] == flags.size and not flags.any(), st
            assert splits != 40 or st["decode_equal_share_steps"] == 1, st
            assert np.array_equal(got, want), st


@pytest.mark.parametrize("splits", [0, 2, 3, 5])
def test_combine_of_many_rows(gpu, splits):
    """8192 rows, where the combine keeps 2 splits per load round instead of 8: one and two splits, and
    more than fit a round, with empty splits on the causal rows; then 2 rows per segment of few
    keys, on both sides of the line to the decode kernel."""
    rng = np.random.default_rng(800 + splits)
    prob = _rand_problem(rng, "normal", "normal", B=16, T=64, Hq=8, Hkv=2, S=330, d=64, dv=64)
    _check(prob, default_alpha_bits(64), splits=splits)
    for B, S in ((3, 500), (128, 128), (127, 128)):
        prob = _rand_problem(rng, "normal", "outlier", B=B, T=1, Hq=32, Hkv=16, S=S, d=128, dv=128)
        _check(prob, default_alpha_bits(128), splits=splits, mrow=B != 128)  # 128 x 16 x 2 tiles: ea_decode's


def _fma():
    f = ctypes.CDLL("libm.so.6").fma
    f.argtypes, f.restype = [ctypes.c_double] * 3, ctypes.c_double
    return f


@pytest.mark.parametrize("kind", ["normal", "wide", "cancel", "subnormal"])
def test_matrix_instructions_are_fma_chains(gpu, kind):
    """v_mfma_f64_16x16x4 and 4x4x4 give, bit for bit, chains of four single-rounding FMAs in ascending
    K order, on which the kernel's error bounds rest: random operands, exponents far apart, sums that
    cancel to their last bits, and operands and sums that are subnormal."""
    import torch
    from exactattention_amd import hip
    rng = np.random.default_rng(12)
    n = 24
    a, b, c = rng.standard_normal((n, 64)), rng.standard_normal((n, 64)), rng.standard_normal((n, 4, 64))
    if kind == "wide":
        a, b = np.ldexp(a, rng.integers(-300, 300, a.shape)), np.ldexp(b, rng.integers(-300, 300, b.shape))
        c = np.ldexp(c, rng.integers(-500, 500, c.shape))
    elif kind == "cancel":
        # K pairs (0, 1) and (2, 3) of nearly opposite products, and an accumulator near minus the rest
        a[:, 16:32], b[:, 16:32] = -a[:, :16], b[:, :16] * (1 + rng.integers(-4, 5, (n, 16)) * 2.0 ** -52)
        a[:, 48:], b[:, 48:] = -a[:, 32:48], b[:, 32:48] * (1 + rng.integers(-4, 5, (n, 16)) * 2.0 ** -52)
        c *= 2.0 ** -50
    elif kind == "subnormal":
        a, b = np.ldexp(a, rng.integers(-560, -500, a.shape)), np.ldexp(b, rng.integers(-560, -500, b.shape))
        c = np.ldexp(c, rng.integers(-1080, -1030, c.shape))
    lib = hip.load()
    dev = [torch.from_numpy(np.ascontiguousarray(x)).cuda() for x in (a, b, c)]
    o16 = torch.zeros((n, 4, 64), dtype=torch.float64, device="cuda")
    o4 = torch.zeros((n, 64), dtype=torch.float64, device="cuda")
    assert lib.ea_hip_kat_mfma_f64(n, *(t.data_ptr() for t in dev), o16.data_ptr(), o4.data_ptr(), None) == 0
    torch.cuda.synchronize()
    fma = _fma()
    w16, w4 = np.zeros((n, 4, 64)), np.zeros((n, 64))
    for w in range(n):
        A, B = a[w].reshape(4, 16), b[w].reshape(4, 16)  # [K][row or column]
        for x in range(4):
            for col in range(16):
                for i in range(4):
                    s = c[w, i, 16 * x + col]
                    for k in range(4):
                        s = fma(A[k, 4 * i + x], B[k, col], s)
                    w16[w, i, 16 * x + col] = s
                s = c[w, 0, 16 * x + col]
                for k in range(4):
                    s = fma(A[k, col // 4 * 4 + x], B[k, col], s)
                w4[w, 16 * x + col] = s
    assert np.array_equal(o16.cpu().numpy().view(np.uint64), w16.view(np.uint64))
    assert np.array_equal(o4.cpu().numpy().view(np.uint64), w4.view(np.uint64))


@pytest.mark.parametrize("page", [8, 16])
def test_merge_order_where_another_kernel_stands_in(gpu, page):
    """A merge order of the reported length on pages the multi-row kernel cannot read: the kernel that
    stands in merges 64 splits instead of 32 and leaves the order alone. Same bits either way."""
    rng = np.random.default_rng(31)
    q, k, v = bf16(rng, (1, 1, 4, 64)), bf16(rng, (1, 1, 16384, 64), "outlier"), bf16(rng, (1, 1, 16384, 64))
    prob = problem.to_paged(problem.contiguous(q, k, v, [[16000]]), page, rng)
    ab = default_alpha_bits(64)
    want, _ = _oracle(prob, ab)
    got, flags, st = _run(prob, ab, merge_order=list(range(31, -1, -1)))
    assert st["nsplit"] == 32 and st["mrow_kernel_rows"] == (flags.size if page == 16 else 0), st
    assert not flags.any() and np.array_equal(got, want), st


def test_step_near_the_allocation_free_limit(gpu):
    """58,000 units whose equal-share plan would not fit where the general kernel's arrays do: uniform
    splits, many rounds of blocks, within the limit."""
    from exactattention_amd.hip import workspace_size
    rng = np.random.default_rng(32)
    B, Hkv, S = 7250, 8, 8
    prob = _rand_problem(rng, "normal", "normal", B=B, T=1, Hq=Hkv, Hkv=Hkv, S=S, d=8, dv=96)
    assert workspace_size(prob["geom"])[0] <= 128 << 20
    st = _check(prob, default_alpha_bits(8))
    assert st["decode_equal_share_steps"] == 0, st
