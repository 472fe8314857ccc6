"""gemm_q4.hip (-m gpu) where its loops turn: more than 16 blocks of 128 k per K lane (the biases' products run twice), lanes with unequal numbers of
blocks, three row tiles, slices of K, tiles that end inside a workgroup's ten.  Against the oracle's matmul over the dequantised weights."""
import numpy as np
import pytest
import torch

from oracle import ref_model
from oracle.numerics import matmul_nt, round_to

pytestmark = pytest.mark.gpu

from mlx_parallm_amd import _lib as L  # noqa: E402
from gpu_helpers import dev, gemm_skinny, host, op_linear, q4_force, to_tiled  # noqa: E402
from test_gpu_gemm_codes import _weight  # noqa: E402
from test_gpu_kernels import _assert_close  # noqa: E402


@pytest.mark.parametrize("act", ["bfloat16", "float16"])
@pytest.mark.parametrize("M,N,K,mt,ks", [
    (33, 176, 128 * 67, 3, 1),       # 17, 17, 17 and 16 blocks a lane
    (64, 160, 128 * 129, 4, 2),      # two slices of 64 and 65
    (17, 336, 128 * 2, 2, 1),        # two of four lanes without a block
    (128, 96, 128 * 5, 4, 3),        # two slabs, slices of one and two blocks
])
def test_block_counts_and_slices(act, M, N, K, mt, ks):
    rng = np.random.default_rng(K + M)
    ol, w, keep = _weight(4, act, N, K, rng)
    x = round_to(rng.standard_normal((M, K)).astype(np.float32), act)
    xd = dev(x, act)
    outs = []
    for _ in range(2):
        out = torch.full((M + 2, N), 7.0, dtype=xd.dtype, device="cuda")
        gemm_skinny(ol, xd, M, act, epi=L.EPI_STORE, out=out, ldo=N, ksplit=q4_force(mt=mt, ksplit=ks))
        outs.append(host(out))
    assert np.array_equal(outs[0], outs[1]) and np.all(outs[0][M:] == 7.0)
    _assert_close(outs[0][:M], round_to(matmul_nt(x, w), act), act)


def test_every_forced_plan_and_every_norm_in_front_of_a_wide_matrix_is_taken():
    """ksplit < 0 forces the kernel also where only fields are set that it ignores; a norm in front of >= 1024 column tiles is applied at any row count and K."""
    act, M, N, K = "bfloat16", 20, 16384, 256
    rng = np.random.default_rng(5)
    ol, w, keep = _weight(4, act, N, K, rng)
    x = round_to(rng.standard_normal((M, K)).astype(np.float32), act)
    nw = round_to(1.0 + 0.1 * rng.standard_normal(K).astype(np.float32), act)
    xd, nwd = dev(x, act), dev(nw, act)
    out = torch.full((M + 2, N), 7.0, dtype=xd.dtype, device="cuda")
    gemm_skinny(ol, xd, M, act, epi=L.EPI_STORE, out=out, ldo=N, norm_w=nwd, eps=1e-5)
    assert np.all(host(out)[M:] == 7.0)
    _assert_close(host(out)[:M], round_to(matmul_nt(ref_model.rms_norm(x, act, nw, act, 1e-5)[0], w), act), act)
    ol.N = 208                                                   # (its first rows alone)
    want = round_to(matmul_nt(x, w[:208]), act)
    for code in (4 << 3, 2 << 7, 2 << 15):                       # tile units, K lanes, staging waves
        out = torch.full((M + 2, 208), 7.0, dtype=xd.dtype, device="cuda")
        gemm_skinny(ol, xd, M, act, epi=L.EPI_STORE, out=out, ldo=208, ksplit=-code)
        assert np.all(host(out)[M:] == 7.0)
        _assert_close(host(out)[:M], want, act)


@pytest.mark.parametrize("act", ["bfloat16", "float16"])
@pytest.mark.parametrize("M,N,K,epi", [
    (17, 48, 128, "store"),          # one block of K: seven waves without one; an odd number of column tiles
    (33, 176, 128 * 9, "resid"),     # three row tiles; one wave with two blocks
    (64, 4112, 128 * 17, "f32"),     # 129 units (the other CUs read ahead), blocks that differ by wave
    (100, 96, 128 * 5, "norm"),      # two slabs
    (128, 8224, 128 * 2, "store"),   # two slabs, more workgroups than CUs
    (33, 7376, 128 * 3, "store"),    # 231 units: too few other CUs to read ahead
    (40, 2 * 80, 128 * 8, "swiglu"),
    (97, 2 * 48, 128 * 7, "swiglu"),
])
def test_narrow_matrices(act, M, N, K, epi):
    """q4_rows_kernel: partial waves, units, slabs and row tiles, every epilogue and the norm in front."""
    rng = np.random.default_rng(K + M)
    ol, w, keep = _weight(4, act, N, K, rng)
    x = round_to(rng.standard_normal((M, K)).astype(np.float32), act)
    h = round_to(rng.standard_normal((M, N)).astype(np.float32), act)
    nw = round_to(1.0 + 0.1 * rng.standard_normal(K).astype(np.float32), act)
    xd, nwd = dev(x, act), dev(nw, act)
    y = matmul_nt(ref_model.rms_norm(x, act, nw, act, 1e-5)[0] if epi == "norm" else x, w)
    cols = N // 2 if epi == "swiglu" else N
    outs = []
    for _ in range(2):
        out = torch.full((M + 2, cols), 7.0, dtype=torch.float32 if epi == "f32" else xd.dtype, device="cuda")
        if epi == "resid":
            out[:M] = dev(h, act)
        kw = {"store": {}, "resid": dict(resid=out), "f32": {}, "norm": dict(norm_w=nwd, eps=1e-5), "swiglu": dict(pair_offset=N // 2)}[epi]
        code = {"resid": L.EPI_RESID, "f32": L.EPI_STORE_F32, "swiglu": L.EPI_SWIGLU}.get(epi, L.EPI_STORE)
        gemm_skinny(ol, xd, M, act, epi=code, out=out, ldo=cols, ksplit=q4_force(rows=1), **kw)
        outs.append(host(out))
    assert np.array_equal(outs[0], outs[1]) and np.all(outs[0][M:] == 7.0)
    want = round_to(y, act)
    if epi == "resid":
        want = round_to(h + want, act)
    if epi == "swiglu":
        g, u = want[:, :cols], want[:, cols:]
        want = round_to(round_to(g * round_to(1.0 / (1.0 + np.exp(-g.astype(np.float64))), act), act) * u, act)
    _assert_close(outs[0][:M], want, act)


def test_a_few_spare_cus_do_not_hold_the_launch_up():
    """252 and 256 units of two column tiles: nearly the same work, so nearly the same time (15 us each; 98 and 15 where four CUs read ahead for 252 units)."""
    M, K, us = 32, 8192, []
    x = torch.randn((M, K), device="cuda").to(torch.bfloat16)
    for N in (8064, 8192):
        keep = [torch.randint(-2 ** 31, 2 ** 31 - 1, (N, K // 8), device="cuda", dtype=torch.int32)] + [torch.full((N, K // 64), 0.01, device="cuda", dtype=torch.bfloat16)] * 2
        ol = op_linear("q4_bf16", N, K, *keep)
        assert to_tiled(ol, keep)
        out = torch.zeros((M, N), dtype=torch.bfloat16, device="cuda")
        us.append(min(gemm_skinny(ol, x, M, "bfloat16", epi=L.EPI_STORE, out=out, ldo=N, ksplit=q4_force(rows=1), iters=20)[1] * 1e3 for _ in range(4)))
    assert us[0] <= 2.0 * us[1], us


@pytest.mark.parametrize("act", ["bfloat16", "float16"])
@pytest.mark.parametrize("M,K", [(17, 128), (128, 2048), (33, 2176), (64, 4224), (48, 8192), (20, 8320)])
def test_norm_in_front_by_pieces_of_the_row(act, M, K):
    """The preparation with a norm: one to four pieces of a row a thread, the last ones partly filled, and the loop above 8192 columns."""
    rng = np.random.default_rng(K)
    ol, w, keep = _weight(4, act, 48, K, rng)
    x = round_to(rng.standard_normal((M, K)).astype(np.float32), act)
    nw = round_to(1.0 + 0.1 * rng.standard_normal(K).astype(np.float32), act)
    xd, nwd = dev(x, act), dev(nw, act)
    out = torch.full((M + 2, 48), 7.0, dtype=xd.dtype, device="cuda")
    gemm_skinny(ol, xd, M, act, epi=L.EPI_STORE, out=out, ldo=48, norm_w=nwd, eps=1e-5, ksplit=q4_force(rows=1))
    assert np.all(host(out)[M:] == 7.0)
    _assert_close(host(out)[:M], round_to(matmul_nt(ref_model.rms_norm(x, act, nw, act, 1e-5)[0], w), act), act)


@pytest.mark.parametrize("K,narrow", [(384, False), (512, True)])
def test_where_the_narrow_kernel_begins_without_a_norm(K, narrow):
    """By the bits: of half a million results the two kernels round some hundred differently."""
    act, M, N = "bfloat16", 128, 4096
    keep = [torch.randint(-2 ** 31, 2 ** 31 - 1, (N, K // 8), device="cuda", dtype=torch.int32), (0.01 + 0.01 * torch.rand((N, K // 64), device="cuda")).to(torch.bfloat16),
            (-0.1 * torch.rand((N, K // 64), device="cuda")).to(torch.bfloat16)]
    ol = op_linear("q4_bf16", N, K, *keep)
    assert to_tiled(ol, keep)
    x = torch.randn((M, K), device="cuda").to(torch.bfloat16)

    def bits(ksplit):
        out = torch.zeros((M, N), dtype=torch.bfloat16, device="cuda")
        used = gemm_skinny(ol, x, M, act, epi=L.EPI_STORE, out=out, ldo=N, ksplit=ksplit)[0]
        return host(out), used
    chosen, used = bits(0)
    rows, streaming = bits(q4_force(rows=1))[0], bits(used)[0]
    assert not np.array_equal(rows, streaming)
    assert np.array_equal(chosen, rows if narrow else streaming)
