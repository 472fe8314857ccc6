"""Kernel-level parity (-m gpu) of gemv_reg.hip -- decode linears of at most 8 rows on int4 / int8 weights -- against the oracle's
matmul, through mi_op_gemv_reg (include/mi355_ops.h).  Tolerances as in test_gpu_kernels.py."""
import numpy as np
import pytest
import torch

from oracle import ref_model, ref_quant
from oracle.numerics import matmul_nt, round_to

pytestmark = pytest.mark.gpu

from mlx_parallm_amd import _lib as L  # noqa: E402
from gpu_helpers import dev, dev_u32, gemv_reg, host, op_linear, to_tiled  # noqa: E402
from test_gpu_kernels import _assert_close  # noqa: E402
from test_gpu_skinny import KINDS, _weight  # noqa: E402

QUANT = [k for k in KINDS if k[1].startswith("q")]


# K in blocks of 128 (int4): fewer than the 8 waves (two of them, one wave with work), not a multiple of 8, each register size's last
# K and the first of the next, the register path's last K and the first beyond, the long path's steps, its last K
@pytest.mark.parametrize("act,kind", QUANT)
@pytest.mark.parametrize("M,N,K", [(1, 16, 128), (8, 80, 256), (3, 64, 1152), (5, 48, 2048), (8, 32, 2176), (7, 32, 4096), (2, 32, 4224),
                                   (8, 48, 5120), (8, 32, 5248), (6, 48, 8192), (4, 16, 11264), (8, 16, 14336), (1, 32, 17408),
                                   (8, 16 * 515, 256)])      # (more tiles than two rounds of workgroups)
def test_matches_oracle(act, kind, M, N, K):
    if kind.startswith("q8") and K > 5120:
        pytest.skip("int8: K in registers only")
    rng = np.random.default_rng(M * 1000003 + N * 1009 + K)
    ol, wdense, keep = _weight(kind, N, K, rng)
    x = round_to(rng.standard_normal((M, K)).astype(np.float32), act)
    h = round_to(rng.standard_normal((M, N)).astype(np.float32) * 4.0, act)
    xd, hd = dev(np.concatenate([x, np.full((1, K), np.nan, np.float32)]), act), dev(np.concatenate([h, h[:1]]), act)
    y = round_to(matmul_nt(x, wdense), act)
    outs = []
    for _ in range(2):
        out = torch.full((M + 1, N), 7.0, dtype=xd.dtype, device="cuda")
        gemv_reg(ol, xd, M, act, epi=L.EPI_STORE, out=out, ldo=N)
        outs.append(host(out))
    assert np.array_equal(outs[0], outs[1]) and np.all(outs[0][M:] == 7.0)
    _assert_close(outs[0][:M], y, act)
    out = torch.full((M + 1, N), 7.0, dtype=torch.float32, device="cuda")
    gemv_reg(ol, xd, M, act, epi=L.EPI_STORE_F32, out=out, ldo=N)
    assert np.array_equal(host(out), outs[0])
    gemv_reg(ol, xd, M, act, epi=L.EPI_RESID, resid=hd, ldo=N)
    got = host(hd)
    assert np.array_equal(got[:M], round_to(h + outs[0][:M], act)) and np.array_equal(got[M:], h[:1])


@pytest.mark.parametrize("act,kind", QUANT)
@pytest.mark.parametrize("M,N,K", [(1, 16, 128), (8, 80, 1152), (5, 4128, 2048), (3, 32, 4096), (8, 48, 5120)])
def test_norm_and_swiglu(act, kind, M, N, K):
    rng = np.random.default_rng(M * 1000003 + N * 1009 + K + 1)
    ol, wdense, keep = _weight(kind, 2 * N, K, rng)
    x = round_to(rng.standard_normal((M, K)).astype(np.float32) * 0.5, act)
    nw = round_to(1.0 + 0.1 * rng.standard_normal(K).astype(np.float32), act)
    xd, nwd = dev(x, act), dev(nw, act)
    xn = ref_model.rms_norm(x, act, nw, act, 1e-5)[0]
    y = round_to(matmul_nt(xn, wdense), act)
    out = torch.zeros((M, 2 * N), dtype=torch.float32, device="cuda")
    gemv_reg(ol, xd, M, act, epi=L.EPI_STORE_F32, out=out, ldo=2 * N, norm_w=nwd)
    _assert_close(host(out), y, act)
    if kind.startswith("q8"):
        return                                          # (int8 SwiGLU and normed 16-bit stores: gemm_skinny.hip)
    out2 = torch.zeros((M, 2 * N), dtype=xd.dtype, device="cuda")
    gemv_reg(ol, xd, M, act, epi=L.EPI_STORE, out=out2, ldo=2 * N, norm_w=nwd)
    assert np.array_equal(host(out2), host(out))
    sig = round_to(1.0 / (1.0 + np.exp(-y[:, :N].astype(np.float64))), act)
    out = torch.zeros((M, N), dtype=xd.dtype, device="cuda")
    gemv_reg(ol, xd, M, act, epi=L.EPI_SWIGLU, out=out, ldo=N, pair_offset=N, norm_w=nwd)
    _assert_close(host(out), round_to(round_to(y[:, :N] * sig, act) * y[:, N:], act), act, scale=4.0)


@pytest.mark.parametrize("kind,M,K,epi,norm", [("q4_bf16", 9, 256, L.EPI_STORE, False), ("q4_bf16", 8, 17536, L.EPI_STORE, False),
                                               ("q4_bf16", 8, 5248, L.EPI_STORE, True), ("q4_bf16", 8, 256, L.EPI_SWIGLU, False),
                                               ("q8_bf16", 8, 5248, L.EPI_STORE, False), ("q8_bf16", 8, 256, L.EPI_STORE, True)])
def test_refuses_what_it_does_not_take(kind, M, K, epi, norm):
    ol, _, keep = _weight(kind, 32, K)
    xd = torch.zeros((M, K), dtype=torch.bfloat16, device="cuda")
    out = torch.zeros((M, 32), dtype=torch.bfloat16, device="cuda")
    with pytest.raises(Exception, match="gemv_reg"):
        gemv_reg(ol, xd, M, "bfloat16", epi=epi, out=out, ldo=32, pair_offset=16, norm_w=xd[0] if norm else None)


DENSE = [("bfloat16", "bf16"), ("float16", "f16"), ("float32", "bf16")]


# K in pairs of 64: one (seven idle waves), not a multiple of 8, each register size's last K and the first of the next
@pytest.mark.parametrize("act,kind", DENSE)
@pytest.mark.parametrize("M,N,K", [(1, 16, 64), (8, 80, 576), (3, 48, 2048), (5, 32, 2112), (7, 32, 4096), (2, 32, 4160), (8, 48, 5120),
                                   (8, 16 * 515, 128)])
def test_dense_matches_oracle(act, kind, M, N, K):
    rng = np.random.default_rng(M * 1000003 + N * 1009 + K + 2)
    ol, w, keep = _weight(kind, N, K, rng)
    x = rng.standard_normal((M, K)).astype(np.float32)
    h = rng.standard_normal((M, N)).astype(np.float32) * 4.0
    nw = 1.0 + 0.1 * rng.standard_normal(K).astype(np.float32)
    if act != "float32":
        x, h, nw = round_to(x, act), round_to(h, act), round_to(nw, act)
    xd, hd, nwd = dev(np.concatenate([x, np.full((1, K), np.nan, np.float32)]), act), dev(np.concatenate([h, h[:1]]), act), dev(nw, act)
    for norm in (None, nwd):
        xn = x if norm is None else ref_model.rms_norm(x, act, nw, act, 1e-5)[0]
        want = matmul_nt(xn, w)
        outs = []
        for _ in range(2):
            out = torch.full((M + 1, N), 7.0, dtype=xd.dtype, device="cuda")
            gemv_reg(ol, xd, M, act, epi=L.EPI_STORE, out=out, ldo=N, norm_w=norm)
            outs.append(host(out))
        assert np.array_equal(outs[0], outs[1]) and np.all(outs[0][M:] == 7.0)
        _assert_close(outs[0][:M], want if act == "float32" else round_to(want, act), act, scale=float(np.sqrt(K)) if act == "float32" else None)
        out = torch.full((M + 1, N), 7.0, dtype=torch.float32, device="cuda")
        gemv_reg(ol, xd, M, act, epi=L.EPI_STORE_F32, out=out, ldo=N, norm_w=norm)
        assert np.array_equal(host(out), outs[0])
    gemv_reg(ol, xd, M, act, epi=L.EPI_RESID, resid=hd, ldo=N, norm_w=nwd)
    got = host(hd)
    want = h + outs[0][:M]
    assert np.array_equal(got[:M], want if act == "float32" else round_to(want, act)) and np.array_equal(got[M:], h[:1])


@pytest.mark.parametrize("M,I,K", [(1, 16, 64), (8, 48, 576), (5, 4128, 2048), (8, 48, 5120)])
def test_dense_swiglu_on_interleaved_rows(M, I, K):
    rng = np.random.default_rng(M * 1000003 + I * 1009 + K + 3)
    w = round_to(rng.standard_normal((2 * I, K)).astype(np.float32) * 0.05, "bfloat16")
    order = np.concatenate([np.r_[8 * t:8 * t + 8, I + 8 * t:I + 8 * t + 8] for t in range(I // 8)])
    wd = dev(w[order], "bfloat16")
    ol, keep = op_linear("bf16", 2 * I, K, wd), [wd]
    assert to_tiled(ol, keep)
    x = rng.standard_normal((M, K)).astype(np.float32)
    nw = 1.0 + 0.1 * rng.standard_normal(K).astype(np.float32)
    xd, nwd = dev(x, "float32"), dev(nw, "float32")
    y = matmul_nt(ref_model.rms_norm(x, "float32", nw, "float32", 1e-5)[0], w).astype(np.float64)
    out = torch.full((M + 1, I), 7.0, dtype=torch.float32, device="cuda")
    gemv_reg(ol, xd, M, "float32", epi=4, out=out, ldo=I, pair_offset=I, norm_w=nwd)
    want = y[:, :I] / (1.0 + np.exp(-y[:, :I])) * y[:, I:]
    assert np.all(host(out)[M:] == 7.0)
    _assert_close(host(out)[:M], want, "float32", scale=float(np.abs(y).max()) ** 2)


@pytest.mark.parametrize("act,kind", [("bfloat16", "bf16"), ("float16", "f16"), ("bfloat16", "q4_bf16"), ("bfloat16", "q8_bf16")])
@pytest.mark.parametrize("K", [256, 1152, 2048, 2176])      # waves without a block, with one less than others, with fewer than registers, full
def test_an_infinite_weight_stays_in_its_own_products(act, kind, K):
    """A wave with fewer blocks than its registers hold loads its last one again: that copy must not enter the sums, where zero times
    infinity is NaN.  One infinite weight (quantised: bias, i.e. a group of them) in every block of one output row in turn: the row's
    outputs are infinite with the sign of x there (of the sum of x over the group), the others finite."""
    rng = np.random.default_rng(K)
    for at in range(7, K, 64):
        if kind.startswith("q"):
            packed, scales, biases = ref_quant.quantize(round_to(rng.standard_normal((32, K)).astype(np.float32), act), 64, int(kind[1]), act)
            biases[5, at // 64] = np.inf
            keep = [dev_u32(packed), dev(scales, act), dev(biases, act)]
        else:
            w = round_to(rng.standard_normal((32, K)).astype(np.float32), act)
            w[5, at] = np.inf
            keep = [dev(w, act)]
        ol = op_linear(kind, 32, K, *keep)
        assert to_tiled(ol, keep)
        x = round_to(np.abs(rng.standard_normal((3, K))).astype(np.float32) + 0.5, act)
        x[1] *= -1.0
        xd = dev(x, act)
        out = torch.zeros((3, 32), dtype=torch.float32, device="cuda")
        gemv_reg(ol, xd, 3, act, epi=L.EPI_STORE_F32, out=out, ldo=32)
        got = host(out)
        assert np.array_equal(got[:, 5], [np.inf, -np.inf, np.inf]), (at, got[:, 5])
        assert np.isfinite(np.delete(got, 5, 1)).all(), at
