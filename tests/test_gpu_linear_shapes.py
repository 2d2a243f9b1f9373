"""Linear kernels at the edges of their tiles: each dispatch branch at the row
counts, widths and depths where it can go wrong, against the CPU oracle."""
import numpy as np
import pytest

import oracle as O
from gpu_util import act_host, assert_close, dev, empty

pytestmark = pytest.mark.gpu

ALL_FMTS = [O.W_DENSE, O.W_Q4_B32, O.W_Q4_G64, O.W_Q8_G32]


def _weights(rng, N, K, wfmt, act, std=0.02):
    wf = (rng.standard_normal((N, K)) * std).astype(np.float16).astype(np.float32)
    return (O.to_act(wf, act), None) if wfmt == O.W_DENSE else O.quantize(wf, wfmt)


def _sdev(s):
    return None if s is None else dev(s)


# --------------------------------------------------------------------------- fp32 GEMM
# Up to 256 tiles of 32 x 32: eight waves split K (steps of 256, which end in
# zeros for the K here); 70 x 6000 and 63 x 15970: 64 x 64 tiles; 300 x 3352
# and 33 x 8150: 32 x 64.  Partial tiles in M and N.
@pytest.mark.parametrize("wfmt", ALL_FMTS)
@pytest.mark.parametrize("M,N,K", [(5, 1, 64), (33, 31, 192), (64, 200, 832), (65, 64, 64), (70, 6000, 192),
                                   (33, 8150, 192), (63, 15970, 64), (300, 3352, 768)])
def test_fp32_gemm_vs_oracle(ctx, rng, wfmt, M, N, K):
    print(f"case: fp32 GEMM {wfmt} {M} x {N} x {K}", flush=True)
    x = O.to_act(rng.standard_normal((M, K)), O.F32)
    w, s = _weights(rng, N, K, wfmt, O.F32)
    y = empty((M, N), O.F32)
    ctx.linear(dev(x), dev(w), _sdev(s), y, M, N, K, wfmt, O.F32)
    ref = O.linear(x, w, s, M, N, K, wfmt, O.F32, round_dequant=1)
    # fp32 products and sums: K roundings of partial sums of a few outputs' size
    assert_close(act_host(y, O.F32), ref, O.F32, 1e-5, "fp32 gemm")


@pytest.mark.parametrize("M,N,K", [(40, 96, 32), (40, 96, 96)])
def test_fp32_gemm_dense_short_k_strides_epilogues(ctx, rng, M, N, K):
    """K of 32 and 96 (dense and group-32 only), padded rows in and out, SiLU
    and the in-place residual."""
    import lite_ssm_amd as L
    for wfmt in (O.W_DENSE, O.W_Q8_G32):
        print(f"case: fp32 GEMM strided {wfmt} {M} x {N} x {K}", flush=True)
        xp = rng.standard_normal((M, K + 4)).astype(np.float32)
        x = np.ascontiguousarray(xp[:, :K])
        w, s = _weights(rng, N, K, wfmt, O.F32)
        res = rng.standard_normal((M, N + 3)).astype(np.float32)
        y = dev(res)
        ctx.linear(dev(xp), dev(w), _sdev(s), y, M, N, K, wfmt, O.F32, epi=L.EPI_ADD, residual=y,
                   x_stride=K + 4, y_stride=N + 3)
        ref = O.linear(O.to_act(x, O.F32), w, s, M, N, K, wfmt, O.F32, epi=O.EPI_ADD,
                       residual=np.ascontiguousarray(res[:, :N]), round_dequant=1)
        got = act_host(y, O.F32)
        assert_close(np.ascontiguousarray(got[:, :N]), ref, O.F32, 1e-5, "add")
        assert np.array_equal(got[:, N:], res[:, N:])          # the padding is left alone
        y2 = empty((M, N), O.F32)
        ctx.linear(dev(x), dev(w), _sdev(s), y2, M, N, K, wfmt, O.F32, epi=L.EPI_SILU)
        ref = O.linear(O.to_act(x, O.F32), w, s, M, N, K, wfmt, O.F32, epi=O.EPI_SILU, round_dequant=1)
        assert_close(act_host(y2, O.F32), ref, O.F32, 1e-5, "silu")


# --------------------------------------------------------------------------- batched decode GEMV
def _norm_linear(ctx, x, nw, w, s, M, N, K, wfmt, act, res=None):
    import lite_ssm_amd as L
    y = dev(res) if res is not None else empty((M, N), act)
    L.check(L.lib.lssm_norm_linear_decode(ctx.h, dev(x).data_ptr(), dev(nw).data_ptr(), 1e-5, dev(w).data_ptr(),
                                          None if s is None else dev(s).data_ptr(), y.data_ptr(),
                                          y.data_ptr() if res is not None else None, M, N, K, wfmt, act,
                                          L.EPI_NONE if res is None else L.EPI_ADD))
    return act_host(y, act)


# Rows at the edges of the 16-row tiles; widths for 1, 2, 3, 4 and 5 tiles of W
# per block and for more tiles than five per CU, with a partial last tile;
# depths of one quad (seven waves idle), ten (an uneven split) and the most;
# and a dense weight wide enough for the tiled GEMM behind a norm launch.
@pytest.mark.parametrize("act", [O.F16, O.BF16])
@pytest.mark.parametrize("wfmt", ALL_FMTS)
@pytest.mark.parametrize("N,K", [(40, 128), (300, 1280), (72, 8192), (5000, 256), (9001, 128), (13000, 256),
                                 (17000, 256), (25000, 128), (32780, 2048)])
def test_decode_rows_vs_oracle(ctx, rng, act, wfmt, N, K):
    if N > 32768 and wfmt != O.W_DENSE:
        pytest.skip("dense only")
    import lite_ssm_amd as L
    nw = O.to_act(1 + 0.1 * rng.standard_normal(K), act)
    w, s = _weights(rng, N, K, wfmt, act)
    for M in (5, 16, 17, 33, 64):
        print(f"case: decode rows act {act} fmt {wfmt} {M} x {N} x {K}", flush=True)
        x = O.to_act(rng.standard_normal((M, K)), act)
        res = O.to_act(rng.standard_normal((M, N)), act) if M == 17 else None
        got = _norm_linear(ctx, x, nw, w, s, M, N, K, wfmt, act, res)
        xn = O.rmsnorm(x, nw, 1e-5, act)
        ref = O.linear(xn, w, s, M, N, K, wfmt, act, epi=O.EPI_NONE if res is None else O.EPI_ADD, residual=res)
        assert_close(got, ref, act, {O.F16: 2e-3, O.BF16: 1.6e-2}[act], "decode rows")


@pytest.mark.parametrize("act", [O.F16, O.BF16])
@pytest.mark.parametrize("M", [1, 2, 4])
def test_decode_rows_few_dense_deep(ctx, rng, act, M):
    """One to four rows of a dense weight too deep for the VALU GEMV's table."""
    N, K = 72, 8192
    nw = O.to_act(1 + 0.1 * rng.standard_normal(K), act)
    w, s = _weights(rng, N, K, O.W_DENSE, act)
    x = O.to_act(rng.standard_normal((M, K)), act)
    print(f"case: decode rows dense act {act} {M} x {N} x {K}", flush=True)
    got = _norm_linear(ctx, x, nw, w, s, M, N, K, O.W_DENSE, act)
    ref = O.linear(O.rmsnorm(x, nw, 1e-5, act), w, s, M, N, K, O.W_DENSE, act)
    assert_close(got, ref, act, {O.F16: 2e-3, O.BF16: 1.6e-2}[act], "decode rows")


@pytest.mark.parametrize("M", [1, 2, 3, 4])
@pytest.mark.parametrize("K", [768, 1536, 2560])
def test_gemv_int8_bf16(ctx, rng, M, K):
    """int8 weights against bf16 rows in the VALU GEMV (every int8 value is a
    bf16), the extreme values among them."""
    N, act = 200, O.BF16
    x = O.to_act(rng.standard_normal((M, K)), act)
    w, s = _weights(rng, N, K, O.W_Q8_G32, act)
    w.view(np.int8).reshape(-1)[:256] = np.arange(-128, 128)
    y = empty((M, N), act)
    print(f"case: int8 x bf16 GEMV {M} x {N} x {K}", flush=True)
    ctx.linear(dev(x), dev(w), dev(s), y, M, N, K, O.W_Q8_G32, act)
    ref = O.linear(x, w, s, M, N, K, O.W_Q8_G32, act)
    assert_close(act_host(y, act), ref, act, 1.6e-2, "gemv")


# --------------------------------------------------------------------------- small-tile GEMM
# Rows at the edges of the 64- and 128-row tiles, partial tiles in N, depths of
# 1, 2, 3, 5 and 13 K steps, K deep enough to be split, and enough columns for
# each of the three tiles; the largest has more tiles than CUs.  The last seven:
# the most rows of the kernel for few, with fewer K slices than row tiles too, at
# both ends of its 49 to 64 rows, and 15 and 16 slices of int8.
@pytest.mark.parametrize("act", [O.F16, O.BF16])
@pytest.mark.parametrize("wfmt", ALL_FMTS)
@pytest.mark.parametrize("M,N,K", [(33, 200, 64), (63, 72, 1088), (64, 64, 128), (65, 130, 192), (127, 500, 320),
                                   (129, 1000, 832), (300, 1100, 2560), (17, 40, 5120), (12, 300, 8192),
                                   (100, 9000, 192), (300, 6000, 128), (700, 2560, 320), (1000, 2000, 128),
                                   (37, 200, 1536), (48, 40, 2048), (40, 40, 64),
                                   (49, 200, 768), (64, 300, 1024), (5, 40, 3840), (16, 200, 4096)])
def test_small_tile_gemm_vs_oracle(ctx, rng, act, wfmt, M, N, K):
    print(f"case: small-tile GEMM act {act} fmt {wfmt} {M} x {N} x {K}", flush=True)
    x = O.to_act(rng.standard_normal((M, K)), act)
    w, s = _weights(rng, N, K, wfmt, act)
    y = empty((M, N), act)
    ctx.linear(dev(x), dev(w), _sdev(s), y, M, N, K, wfmt, act)
    ref = O.linear(x, w, s, M, N, K, wfmt, act, round_dequant=1)
    assert_close(act_host(y, act), ref, act, {O.F16: 2e-3, O.BF16: 1.6e-2}[act], "small-tile gemm")


@pytest.mark.parametrize("act", [O.F16, O.BF16])
@pytest.mark.parametrize("M,N,K", [(37, 130, 192), (70, 256, 5120), (13, 130, 4096)])
def test_small_tile_gemm_strides_epilogues(ctx, rng, act, M, N, K):
    """Padded rows (an odd y stride: element stores), SiLU and the in-place
    residual, in one pass, (K = 5120) through the slices' sum and (K = 4096) in
    the kernel for few rows."""
    import lite_ssm_amd as L
    for wfmt in (O.W_DENSE, O.W_Q4_G64, O.W_Q8_G32):
        w, s = _weights(rng, N, K, wfmt, act)
        xp = O.to_act(rng.standard_normal((M, K + 8)), act)
        x = np.ascontiguousarray(xp[:, :K])
        for pad in (8, 3):
            res = O.to_act(rng.standard_normal((M, N + pad)), act)
            for epi in (L.EPI_NONE, L.EPI_SILU, L.EPI_ADD):
                print(f"case: small-tile GEMM strided act {act} fmt {wfmt} {M} x {N} x {K} pad {pad} epi {epi}", flush=True)
                y = dev(res)
                ctx.linear(dev(xp), dev(w), _sdev(s), y, M, N, K, wfmt, act, epi=epi,
                           residual=y if epi == L.EPI_ADD else None, x_stride=K + 8, y_stride=N + pad)
                ref = O.linear(x, w, s, M, N, K, wfmt, act, epi=epi, round_dequant=1,
                               residual=np.ascontiguousarray(res[:, :N]) if epi == L.EPI_ADD else None)
                got = act_host(y, act)
                assert_close(np.ascontiguousarray(got[:, :N]), ref, act, {O.F16: 2e-3, O.BF16: 1.6e-2}[act], "epilogue")
                assert np.array_equal(got[:, N:], res[:, N:])


# --------------------------------------------------------------------------- infinities, threads
# One shape for each kernel: fp32 with a K step wider than K, few rows, small
# tiles in one pass and split, and the batched decode GEMV.
@pytest.mark.parametrize("act,wfmt,M,N,K", [(O.F32, O.W_Q8_G32, 40, 96, 96), (O.F32, O.W_DENSE, 40, 96, 96),
                                            (O.F16, O.W_Q8_G32, 40, 70, 768), (O.BF16, O.W_DENSE, 100, 300, 320),
                                            (O.F16, O.W_Q4_B32, 100, 300, 320), (O.BF16, O.W_Q4_G64, 70, 256, 5120)])
def test_gemm_rows_with_infinities_leave_the_others(ctx, rng, act, wfmt, M, N, K):
    """A row with an infinity or a NaN (at both ends of K) is non-finite; the
    other rows keep their bits."""
    print(f"case: infinities act {act} fmt {wfmt} {M} x {N} x {K}", flush=True)
    x = rng.standard_normal((M, K))
    w, s = _weights(rng, N, K, wfmt, act)
    wd, sd = dev(w), _sdev(s)
    out = []
    for bad in (False, True):
        if bad:
            x[5, 0], x[17, K - 1], x[M - 1, 0] = np.inf, -np.inf, np.nan
        y = empty((M, N), act)
        ctx.linear(dev(O.to_act(x, act)), wd, sd, y, M, N, K, wfmt, act)
        out.append(act_host(y, act))
    hit = np.array([5, 17, M - 1])
    assert not np.isfinite(O.from_act(out[1][hit], act)).any()
    assert np.array_equal(np.delete(out[0], hit, 0), np.delete(out[1], hit, 0))


@pytest.mark.parametrize("act,wfmt,M", [(O.BF16, O.W_Q8_G32, 24), (O.F16, O.W_Q4_B32, 33), (O.BF16, O.W_DENSE, 64)])
def test_decode_rows_with_infinities_leave_the_others(ctx, rng, act, wfmt, M):
    N, K = 300, 1280
    print(f"case: infinities in decode rows act {act} fmt {wfmt} {M} x {N} x {K}", flush=True)
    x = rng.standard_normal((M, K))
    nw = O.to_act(1 + 0.1 * rng.standard_normal(K), act)
    w, s = _weights(rng, N, K, wfmt, act)
    clean = _norm_linear(ctx, O.to_act(x, act), nw, w, s, M, N, K, wfmt, act)
    x[3, 0], x[18, K - 1], x[M - 1, 640] = np.inf, -np.inf, np.nan
    got = _norm_linear(ctx, O.to_act(x, act), nw, w, s, M, N, K, wfmt, act)
    hit = np.array([3, 18, M - 1])
    assert not np.isfinite(O.from_act(got[hit], act)).any()
    assert np.array_equal(np.delete(clean, hit, 0), np.delete(got, hit, 0))


def test_two_threads_share_a_context(ctx, rng):
    """Calls that pass data on in the context's scratch, from two threads: packed
    rows in one, split K in the other."""
    import threading
    import lite_ssm_amd as L
    print("case: two threads on one context", flush=True)
    M, N, K, act = 24, 300, 2560, O.BF16
    nw = dev(O.to_act(1 + 0.1 * rng.standard_normal(K), act))
    w, s = (dev(a) for a in _weights(rng, N, K, O.W_Q8_G32, act))
    x, y = dev(O.to_act(rng.standard_normal((M, K)), act)), empty((M, N), act)
    M2, N2, K2 = 70, 256, 5120
    w2, s2 = (dev(a) for a in _weights(rng, N2, K2, O.W_Q4_G64, act))
    x2, y2 = dev(O.to_act(rng.standard_normal((M2, K2)), act)), empty((M2, N2), act)

    def rows():
        L.check(L.lib.lssm_norm_linear_decode(ctx.h, x.data_ptr(), nw.data_ptr(), 1e-5, w.data_ptr(), s.data_ptr(),
                                              y.data_ptr(), None, M, N, K, O.W_Q8_G32, act, L.EPI_NONE))

    def split():
        ctx.linear(x2, w2, s2, y2, M2, N2, K2, O.W_Q4_G64, act)

    rows()
    split()
    want = act_host(y, act).copy(), act_host(y2, act).copy()
    wrong = []

    def loop(call, out, ref):
        # (numpy copies of the outputs: the calls themselves return when done)
        for _ in range(50):
            call()
        if not np.array_equal(act_host(out, act), ref):
            wrong.append(call.__name__)

    both = [threading.Thread(target=loop, args=a) for a in ((rows, y, want[0]), (split, y2, want[1]))]
    for t in both:
        t.start()
    for t in both:
        t.join(30)
    assert not wrong and not any(t.is_alive() for t in both)
