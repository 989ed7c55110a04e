"""GPU parity of the blocked prefill's linear (ai_amd.prefill.matrix ->
rv12_prefill_linear: the 12-bit decode fused into an MFMA GEMM of split
activations over all tokens) against the oracle's float64 closed form: 1e-3 abs + 1e-2 rel and 4x
the fp32 forward-error bound, for store, residual add and the silu(g) * u
prologue, ragged token counts and row counts, on the golden matrices, a
matrix with exceptions in many rows, activations of very different scales,
and (at the Qwen3-8B gu shape over 2048 tokens, beyond what the float64
oracle finishes in seconds) sampled rows against the decode kernels."""
import zlib

import numpy as np
import pytest
import torch

from conftest import ref_dict
from oracle import codec, linear

pytestmark = pytest.mark.gpu


def _check(cnp, T, seed, add, mode=None, scales=None, rms=False):
    from ai_amd import prefill, wcomp
    rng = np.random.default_rng(seed)
    N, K = cnp["N"], cnp["K"]
    mode = (1 if add else 0) if mode is None else mode
    X = rng.standard_normal((T, 2 * K if mode == 2 else K)) * 2
    if scales is not None:  # MODE 2: g and u each by the square root, so that x' ~ the scale
        sc = np.asarray(scales, np.float64)[:T, None]
        X *= np.sqrt(sc) if mode == 2 else sc
    X = X.astype(np.float32)
    Y0 = rng.standard_normal((T, N)).astype(np.float32)
    lnw = lw = ln = None
    if rms:  # the RMSNorm prologue (rmsg_k fused): a bf16 weight of K entries
        lnw = codec.f32_to_bf16_rne((1.0 + 0.1 * rng.standard_normal(K)).astype(np.float32))
        lw = codec.bf16_to_f32(lnw)
        ln = torch.from_numpy(lnw.view(np.int16).copy()).view(torch.bfloat16).cuda()
    W = codec.decode_f32(cnp).astype(np.float64)
    ref = linear.linear(cnp, X, mode, Y0 if mode else None, lnw=lw, W=W)
    bound = linear.error_bound(cnp, X, mode, lnw=lw, W=W)
    c = wcomp.prepare({k: (torch.from_numpy(np.ascontiguousarray(v)) if isinstance(v, np.ndarray) else v)
                       for k, v in cnp.items()})
    y = torch.from_numpy(Y0.copy()).cuda()
    if mode == 2:
        prefill._linear(torch.from_numpy(X).cuda(), c, y, 2)
    else:
        prefill.matrix(torch.from_numpy(X).cuda(), c, y, add=add, lnw=ln)
    torch.cuda.synchronize()
    got = y.cpu().numpy().astype(np.float64)
    # outputs beyond the float32 range: the closed form rounded to float32
    # (inf), as an fp32 evaluation must produce
    with np.errstate(over="ignore"):
        ref = ref.astype(np.float32).astype(np.float64)
    fin = np.isfinite(ref)
    assert np.array_equal(np.isnan(got), np.isnan(ref))
    assert np.array_equal(got[np.isinf(ref)], ref[np.isinf(ref)])
    err = np.abs(got[fin] - ref[fin])
    assert np.all(err <= 1e-3 + 1e-2 * np.abs(ref[fin])), float(err.max())
    # plus the rounding of the final add into y (2^-23 |y|) where y is accumulated
    tight = 4 * bound[fin] + (2.0 ** -23 * np.abs(ref[fin]) if mode else 0.0) + 1e-30
    assert np.all(err <= tight), float((err - tight).max())
    return float(np.linalg.norm(err) / max(np.linalg.norm(ref[fin]), 1e-30))


@pytest.mark.parametrize("case", ["prefill_seed7", "outliers_rows_cols", "chunk128", "subnormal_heavy"])
def test_matrix_on_golden_dicts(golden, case):
    cnp = ref_dict(golden[case])
    for add in (False, True):
        _check(cnp, 300, 1, add)


def test_matrix_with_exceptions_in_many_rows():
    rng = np.random.default_rng(3)
    w = (rng.standard_normal((777, 1024)) * 0.02).astype(np.float32)
    idx = rng.choice(w.size, 400, replace=False)
    w.reshape(-1)[idx[::2]] = 3e4
    w.reshape(-1)[idx[1::2]] = -1e-30
    w[5] *= 20
    cnp = codec.compress(codec.f32_to_bf16_rne(w))
    assert cnp["er"].size > 100
    _check(cnp, 513, 2, True)


@pytest.mark.parametrize("T", [1, 17, 128, 129, 300])
def test_ragged_tokens_rows_and_modes(T):
    """Token counts around the 128-token tile, a row count that is not a
    multiple of the 256-row tile, every mode, and the RMSNorm prologue
    (store and accumulate)."""
    rng = np.random.default_rng(T)
    w = (rng.standard_normal((300, 512)) * 0.02).astype(np.float32)
    w[rng.choice(300, 2)] *= 20
    cnp = codec.compress(codec.f32_to_bf16_rne(w))
    for mode in (0, 1, 2):
        print("T", T, "mode", mode, flush=True)
        _check(cnp, T, T + mode, mode != 0, mode=mode)
    for mode in (0, 1):
        print("T", T, "mode", mode, "rms", flush=True)
        _check(cnp, T, T + 7 + mode, mode != 0, mode=mode, rms=True)


def test_rms_prologue_on_golden_dicts_and_scales(golden):
    """The fused RMSNorm (rs per token over its full row, lnw x staged) on
    the golden matrices, and over tokens scaled by 2^-60 .. 2^60: the sum of
    squares runs over (x 2^-32)^2, so no token overflows or vanishes."""
    for case in ("prefill_seed7", "outliers_rows_cols"):
        _check(ref_dict(golden[case]), 300, 5, False, rms=True)
    rng = np.random.default_rng(12)
    w = (rng.standard_normal((200, 1024)) * 0.02).astype(np.float32)
    cnp = codec.compress(codec.f32_to_bf16_rne(w))
    T = 40
    scales = [2.0 ** e for e in np.linspace(-60, 60, T)]
    _check(cnp, T, 13, False, mode=0, scales=scales, rms=True)


def test_rms_prologue_rejected_in_mode_2():
    import ctypes
    from ai_amd import _lib, wcomp
    rng = np.random.default_rng(1)
    cnp = codec.compress(codec.f32_to_bf16_rne((rng.standard_normal((32, 256)) * 0.02).astype(np.float32)))
    c = wcomp.prepare({k: (torch.from_numpy(np.ascontiguousarray(v)) if isinstance(v, np.ndarray) else v)
                       for k, v in cnp.items()})
    x = torch.zeros(4, 512, device="cuda")
    y = torch.zeros(4, 32, device="cuda")
    ln = torch.ones(256, dtype=torch.bfloat16, device="cuda")
    ws = torch.empty(1 << 20, dtype=torch.uint8, device="cuda")
    L = _lib.lib()
    rc = L.rv12_prefill_linear(ctypes.byref(wcomp._matrix(c)), ctypes.c_void_p(x.data_ptr()),
                               ctypes.c_void_p(y.data_ptr()), 4, ctypes.c_void_p(ln.data_ptr()), 1e-6, 2,
                               ctypes.c_void_p(ws.data_ptr()), ws.numel(), None)
    assert rc == _lib.RV12_E_MODE


def test_token_scales():
    """Tokens scaled by 2^-60 .. 2^60 (and one of zeros) in one prompt: each
    token's exact power-of-two scale keeps the fp32 bound."""
    rng = np.random.default_rng(9)
    w = (rng.standard_normal((200, 1024)) * 0.02).astype(np.float32)
    cnp = codec.compress(codec.f32_to_bf16_rne(w))
    T = 40
    scales = [2.0 ** e for e in np.linspace(-60, 60, T)]
    scales[7] = 0.0
    for mode in (0, 2):
        _check(cnp, T, 11 + mode, False, mode=mode, scales=scales)


def test_qwen3_8b_gu_2048_tokens_against_the_decode_kernels():
    """The 24576 x 4096 gu matrix over 2048 tokens: sampled token rows equal
    the MFMA decode-linear's (rv12_gemm at 16 tokens) within the tolerance,
    and a 64-token slice of rows equals the float64 closed form."""
    from ai_amd import prefill, wcomp
    g = torch.Generator(device="cuda").manual_seed(8)
    N, K, T = 24576, 4096, 2048
    w = (torch.randn(N, K, device="cuda", generator=g) * 0.02)
    w[torch.randperm(N, device="cuda", generator=g)[:24]] *= 20
    w = w.bfloat16()
    c = wcomp.compress(w)
    x = torch.randn(T, K, device="cuda", generator=g)
    y = torch.zeros(T, N, device="cuda")
    prefill.matrix(x, c, y)
    pick = torch.tensor([0, 1, 127, 128, 1000, 1777, 2046, 2047, 5, 6, 7, 8, 9, 10, 11, 12], device="cuda")
    xs = x[pick].contiguous()
    ys = torch.zeros(16, N, device="cuda")
    wcomp.gemvc_tc(xs, c, ys, 0, 16)
    torch.cuda.synchronize()
    ref = ys.cpu().numpy().astype(np.float64)
    got = y[pick].cpu().numpy().astype(np.float64)
    assert np.all(np.abs(got - ref) <= 1e-3 + 1e-2 * np.abs(ref)), float(np.abs(got - ref).max())
    # 64 rows against float64
    rows = slice(4096, 4160)
    W64 = w[rows].float().cpu().numpy().astype(np.float64)
    want = x[:64].cpu().numpy().astype(np.float64) @ W64.T
    mag = np.abs(x[:64].cpu().numpy().astype(np.float64)) @ np.abs(W64).T
    err = np.abs(y[:64, rows].cpu().numpy() - want)
    assert np.all(err <= 4 * (K + 8) * 2.0 ** -24 * mag + 1e-30), float(err.max())
    del c, w, x, y
    torch.cuda.empty_cache()


@pytest.mark.parametrize("K", [160, 224, 288])
def test_step_counts_off_the_ring(K):
    """K / 32 steps off the kernel's unroll and its load ring of five slots (four
    with three parts): 5, 7, 9 steps; the steps past the end load zeros
    through the 0-byte descriptors and add nothing; every mode, with and
    without the RMS prologue, exceptions in many rows."""
    rng = np.random.default_rng(K)
    w = (rng.standard_normal((300, K)) * 0.02).astype(np.float32)
    w[rng.choice(300, 3)] *= 20
    w.reshape(-1)[rng.choice(w.size, 60, replace=False)] = 1e-30
    cnp = codec.compress(codec.f32_to_bf16_rne(w), CH=32)
    assert cnp["er"].size > 30
    for T in (17, 130):
        for mode in (0, 1, 2):
            print("K", K, "T", T, "mode", mode, flush=True)
            _check(cnp, T, K + T + mode, mode != 0, mode=mode)
        _check(cnp, T, K + T + 7, False, mode=0, rms=True)


def test_random_draws_of_shapes_tokens_and_modes():
    """24 seeded draws of row count (1-600), K (128-2048 in steps of 32,
    codec chunks of 32), token count (1-400), MODE, the RMS prologue (MODES 0
    and 1), outlier rows and exceptions (3e4, -1e-30 or 1e-35 at random
    positions), each against the float64 closed form and the fp32 bound."""
    rng = np.random.default_rng(4242)
    for d in range(24):
        N = int(rng.integers(1, 601))
        K = 32 * int(rng.integers(4, 65))
        T = int(rng.integers(1, 401))
        mode = int(rng.integers(0, 3))
        rms = bool(rng.integers(0, 2)) and mode != 2
        w = (rng.standard_normal((N, K)) * 0.02).astype(np.float32)
        nout = int(rng.integers(0, 4))
        if nout:
            w[rng.choice(N, min(N, nout), replace=False)] *= 20
        nexc = int(rng.integers(0, 1 + N * K // 500))
        if nexc:
            w.reshape(-1)[rng.choice(w.size, nexc, replace=False)] = float(rng.choice([3e4, -1e-30, 1e-35]))
        cnp = codec.compress(codec.f32_to_bf16_rne(w), CH=32)
        print("draw", d, N, K, T, mode, rms, int(cnp["er"].size), flush=True)
        _check(cnp, T, 9000 + d, mode != 0, mode=mode, rms=rms)


@pytest.mark.parametrize("case", ["special_values", "all_zero"])
def test_matrix_on_golden_special_values(golden, case):
    """Golden matrices with infinities, NaNs, subnormals and zeros among the
    weights: NaN and infinite outputs where the closed form (rounded to
    float32) has them, every finite output within the tolerance.  (The
    golden matrices of weights near the top of the float32 range, huge_with_inf
    and window_hits_inf, are decode vectors only: a sum of their products
    overflows float32 part-way in an order-dependent way, so an infinite
    weight meets an overflowed partial sum of either sign.)"""
    cnp = ref_dict(golden[case])
    for add in (False, True):
        _check(cnp, 40, 3, add)


@pytest.mark.parametrize("K", [512, 544, 1056])
@pytest.mark.parametrize("T", [300, 513])
def test_unsplit_sums_over_chunks_of_steps(K, T):
    """Enough rows for unsplit workgroups whose K steps are a whole chunk of the
    fp32 sums, one step more, and two chunks and one step; rows off the vector
    store's four, one token in the last tile.  The norm of the error stays below
    4e-7 of the output's (2.2e-7 measured, 6e-5 without the second part)."""
    rng = np.random.default_rng(K + T)
    N = 22003
    w = (rng.standard_normal((N, K)) * 0.02).astype(np.float32)
    w[rng.choice(N, 20, replace=False)] *= 20
    w.reshape(-1)[rng.choice(w.size, 300, replace=False)] = 1e-30
    cnp = codec.compress(codec.f32_to_bf16_rne(w), CH=32)
    for mode, rms in ((0, True), (1, False)):
        print("K", K, "T", T, "mode", mode, "rms", rms, flush=True)
        rel = _check(cnp, T, K + T + mode, mode != 0, mode=mode, rms=rms)
        assert rel <= 4e-7, rel


@pytest.mark.parametrize("N,T", [(300, 300), (22003, 300)])
@pytest.mark.parametrize("big", [0, 20, 40])
def test_tokens_over_many_exponents(N, T, big):
    """Values 2^big above the rest in a column whose weights are zero: the
    output is the other columns' alone, and the fp32 bound of those alone holds,
    which float16 parts scaled to the huge value would miss by far.  Tiles with
    and without such a token, K split and unsplit."""
    from ai_amd import prefill, wcomp
    rng = np.random.default_rng(big)
    K = 256
    w = (rng.standard_normal((N, K)) * 0.02).astype(np.float32)
    w[:, 77] = 0
    bits = codec.f32_to_bf16_rne(w)
    x = rng.standard_normal((T, K)).astype(np.float32)
    x[[3, 5, T - 1]] *= np.float32(2.0) ** -big
    x[[3, 5, T - 1], 77] = 1.5
    c = wcomp.compress(torch.from_numpy(bits.view(np.int16)).view(torch.bfloat16).cuda())
    y = torch.zeros(T, N, device="cuda")
    prefill.matrix(torch.from_numpy(x).cuda(), c, y)
    w64 = codec.bf16_to_f32(bits).astype(np.float64)
    w64[:, 77] = 0
    want, mag = x.astype(np.float64) @ w64.T, np.abs(x.astype(np.float64)) @ np.abs(w64).T
    err = np.abs(y.cpu().numpy() - want)
    assert np.all(err <= 4 * (K + 8) * 2.0 ** -24 * mag + 1e-30), float((err / mag).max())


def _on_gpu(bits):
    return torch.from_numpy(bits.view(np.int16)).view(torch.bfloat16).cuda()


@pytest.mark.parametrize("K,low", [(32, 17), (64, 34), (480, 14), (544, 1), (544, 300), (4096, 8),
                                   (4096, 113), (4096, 200), (4096, 2200)])
@pytest.mark.parametrize("drop", [14, 20, 25, 28, 36, 60])
def test_tokens_of_two_levels(K, low, drop):
    """`low` columns 2^drop below the others, in every third token, and rows with
    weights on those columns alone (kept in the tiles where they are more than the
    zeros).  The norm of a token's error over the rows stays below
    sqrt(K) 2^-24 of its output's, the random walk of a float32 sum of K products,
    plus 2^-23 for the split of the activations, for the rows of either kind; so
    does a token of one level in the same tile."""
    from ai_amd import prefill, wcomp
    rng = np.random.default_rng(K + low + drop)
    N, T = 512, 140
    cols = rng.choice(K, low, replace=False)
    w = (rng.standard_normal((N, K)) * 0.02).astype(np.float32)
    w = np.copysign(np.maximum(np.abs(w), 1e-3), w)
    rest = np.setdiff1d(np.arange(K), cols)
    w[::2, rest] = 0
    bits = codec.f32_to_bf16_rne(w)
    x = rng.standard_normal((T, K)).astype(np.float32)
    x[::3, cols] *= np.float32(2.0) ** -drop
    y = torch.zeros(T, N, device="cuda")
    prefill.matrix(torch.from_numpy(x).cuda(), wcomp.compress(_on_gpu(bits), CH=32), y)
    want = x.astype(np.float64) @ codec.bf16_to_f32(bits).astype(np.float64).T
    err = y.cpu().numpy() - want
    for rows in (slice(0, N, 2), slice(1, N, 2)):
        rel = np.linalg.norm(err[:, rows], axis=1) / np.linalg.norm(want[:, rows], axis=1)
        print("K", K, "low", low, "drop", drop, "rel", float(rel.max()), flush=True)
        assert rel.max() <= K ** 0.5 * 2.0 ** -24 + 2.0 ** -23, (float(rel.max()), int(rel.argmax()))


@pytest.mark.parametrize("N,K,T", [(300, 256, 140), (301, 1056, 300), (22003, 160, 200)])
@pytest.mark.parametrize("mode", [0, 1])
def test_a_token_does_not_depend_on_its_neighbours(N, K, T, mode):
    """The same token rows beside tokens of many exponents and without, K split and
    unsplit, rows with exceptions, store and add: bit for bit the same outputs."""
    from ai_amd import prefill, wcomp
    rng = np.random.default_rng(N + K)
    w = (rng.standard_normal((N, K)) * 0.02).astype(np.float32)
    w.reshape(-1)[rng.choice(w.size, 200, replace=False)] = 1e-30
    c = wcomp.compress(_on_gpu(codec.f32_to_bf16_rne(w)), CH=32)
    plain = rng.standard_normal((T, K)).astype(np.float32)
    spread = plain.copy()
    spread[:, rng.permutation(K)[:K // 2]] *= np.float32(2.0 ** -40)
    rows = np.zeros(T, bool)
    rows[[3, 70, 71, 130, T - 1]] = True
    mixed = np.where(rows[:, None], spread, plain)
    y0 = torch.from_numpy(rng.standard_normal((T, N)).astype(np.float32)).cuda()
    out = []
    for x in (plain, spread, mixed):
        y = y0.clone()
        prefill.matrix(torch.from_numpy(x).cuda(), c, y, add=bool(mode))
        out.append(y)
    r = torch.from_numpy(rows).cuda()
    assert torch.equal(out[2][~r], out[0][~r]) and torch.equal(out[2][r], out[1][r])


@pytest.mark.parametrize("N", [256, 300])
def test_row_windows_at_any_four_byte_address(N):
    """rbase has the alignment of its type: the same outputs from a copy that starts
    4, 8 and 12 bytes past a 16-byte boundary."""
    from ai_amd import prefill, wcomp
    rng = np.random.default_rng(N)
    w = (rng.standard_normal((N, 256)) * 0.02 * 2.0 ** rng.integers(-9, 9, (N, 1))).astype(np.float32)
    c = wcomp.compress(_on_gpu(codec.f32_to_bf16_rne(w)))
    x = torch.from_numpy(rng.standard_normal((33, 256)).astype(np.float32)).cuda()
    y = torch.zeros(4, 33, N, device="cuda")
    rb = c["q16_rbase"]
    for off in range(4):
        room = torch.empty(N + 4, dtype=torch.int32, device="cuda")
        c["q16_rbase"] = room[off:off + N].copy_(rb)
        assert c["q16_rbase"].data_ptr() % 16 == 4 * off
        prefill.matrix(x, c, y[off], add=True)
    assert torch.equal(y[1:], y[:1].expand(3, -1, -1)) and bool(y[0].any())


def test_sums_over_chunks_keep_their_accuracy():
    """K = 4096 unsplit: the norm of the error stays below 4e-7 of the output's
    (2.3e-7 measured; 5.9e-7 without the float32 sums over chunks of steps, 5e-5
    without the activations' second part)."""
    from ai_amd import _lib, prefill, wcomp
    N, K, T = 8192, 4096, 1024
    g = torch.Generator(device="cuda").manual_seed(5)
    assert _lib.lib().rv12_prefill_workspace_bytes(N, K, T) == T * K * 10 + T * 8  # no K split
    w = (torch.randn(N, K, device="cuda", generator=g) * 0.02).bfloat16()
    x = torch.randn(T, K, device="cuda", generator=g)
    y = torch.zeros(T, N, device="cuda")
    prefill.matrix(x, wcomp.compress(w), y)
    want = x.double() @ w.double().t()
    rel = float((y.double() - want).norm() / want.norm())
    assert rel <= 4e-7, rel


def test_three_parts_hold_24_bits():
    """parts = 3: an activation of 24 significant bits times a power of two comes
    out exactly.  (Two float16 parts hold 23: half of these lose their last.)"""
    from ai_amd import prefill, wcomp
    rng = np.random.default_rng(24)
    N, K, T = 64, 96, 200
    bits = codec.f32_to_bf16_rne((2.0 ** rng.integers(-9, -3, (N, K)) * rng.choice([-1, 1], (N, K))).astype(np.float32))
    x = np.zeros((T, K), np.float32)
    at = rng.integers(0, K, T)
    x[np.arange(T), at] = (rng.integers(1 << 22, 1 << 23, T) * 2 + 1).astype(np.float32)
    v = x[np.arange(T), at] / np.float32(2.0 ** 9)
    hi = v.astype(np.float16).astype(np.float32)
    two = hi + ((v - hi) * np.float32(2048)).astype(np.float16).astype(np.float32) / np.float32(2048)
    assert np.count_nonzero(two != v) > T // 4  # two parts could not pass
    c = wcomp.compress(_on_gpu(bits), CH=32)
    y = torch.zeros(T, N, device="cuda")
    prefill.matrix(torch.from_numpy(x).cuda(), c, y, parts=3)
    want = x[np.arange(T), at][:, None] * codec.bf16_to_f32(bits).T[at]
    assert np.array_equal(y.cpu().numpy(), want)


@pytest.mark.parametrize("N,K,T,rms,crc", [(304, 96, 17, False, 0xAAA1E959), (301, 1056, 130, True, 0x9B0F214F),
                                           (22003, 512, 300, True, 0xA5022E4F)])
def test_three_parts_keep_their_order_of_sums(N, K, T, rms, crc):
    """parts = 3, K split and unsplit: the bits that every version of the linear so
    far gave, so that a layer's keys and values for an input stay the same (the
    checksums are of the library that had three parts alone)."""
    from ai_amd import prefill, wcomp
    rng = np.random.default_rng(N)
    bits = codec.f32_to_bf16_rne((rng.standard_normal((N, K)) * 0.02).astype(np.float32))
    x = rng.standard_normal((T, K)).astype(np.float32)
    lw = codec.f32_to_bf16_rne((1 + 0.1 * rng.standard_normal(K)).astype(np.float32))
    y = torch.zeros(T, N, device="cuda")
    prefill._linear(torch.from_numpy(x).cuda(), wcomp.compress(_on_gpu(bits), CH=32), y, 0, _on_gpu(lw) if rms else None,
                    1e-6, parts=3)
    assert zlib.crc32(y.cpu().numpy().tobytes()) == crc


@pytest.mark.parametrize("T,K", [(17, 160), (300, 512), (130, 1056)])
def test_three_parts_on_request(T, K):
    """parts = 3: the linear whose outputs are rounded into the caches; steps off
    the four-slot ring, split and unsplit, the RMS prologue."""
    from ai_amd import prefill, wcomp
    rng = np.random.default_rng(T)
    N = 301
    bits = codec.f32_to_bf16_rne((rng.standard_normal((N, K)) * 0.02).astype(np.float32))
    c = wcomp.compress(torch.from_numpy(bits.view(np.int16)).view(torch.bfloat16).cuda(), CH=32)
    x = rng.standard_normal((T, K)).astype(np.float32)
    lw = codec.f32_to_bf16_rne((1 + 0.1 * rng.standard_normal(K)).astype(np.float32))
    y = torch.zeros(T, N, device="cuda")
    prefill._linear(torch.from_numpy(x).cuda(), c, y, 0, torch.from_numpy(lw.view(np.int16)).view(torch.bfloat16).cuda(),
                    1e-6, parts=3)
    x64 = x.astype(np.float64)
    x64 = x64 / np.sqrt((x64 ** 2).mean(1, keepdims=True) + 1e-6) * codec.bf16_to_f32(lw).astype(np.float64)
    w64 = codec.bf16_to_f32(bits).astype(np.float64)
    err, mag = np.abs(y.cpu().numpy() - x64 @ w64.T), np.abs(x64) @ np.abs(w64).T
    assert np.all(err <= 4 * (K + 8) * 2.0 ** -24 * mag), float((err / mag).max())
    with pytest.raises(ValueError):
        prefill._linear(torch.from_numpy(x).cuda(), c, y, 0, parts=4)
