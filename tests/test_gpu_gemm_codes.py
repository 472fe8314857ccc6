"""Kernel-level parity (-m gpu) of the tile GEMM on int4 / int8 codes (gemm_prefill.hip: gemm_codes256_kernel, the nn.QuantizedLinear of
the prefill call, utils.py:243-262,679-690) through mi_op_gemm_codes: against the oracle's matmul over the dequantised weights on
sampled rows, for every epilogue, at the edges of tiles and runs.  The codes kernel is forced: below some 4e9 products the call alone would run on the
[hi | lo] copy."""
import ctypes as C
import time

import numpy as np
import pytest
import torch

from oracle import ref_quant
from oracle.numerics import matmul_nt, round_to

pytestmark = pytest.mark.gpu

from mlx_parallm_amd import _lib as L  # noqa: E402
from gpu_helpers import dev, dev_u32, gemm_skinny, gemv_args, host, op_linear, to_tiled  # noqa: E402
from test_gpu_gemm_prefill import _rows  # noqa: E402
from test_gpu_kernels import _assert_close  # noqa: E402


def _weight(bits, sdt, N, K, rng):
    """groups whose mean is up to four of their own deviations: the bias term is no small one"""
    w = (rng.standard_normal((N, K // 64, 64)) + 4 * rng.standard_normal((N, K // 64, 1))).astype(np.float32) * 0.05
    packed, s, b = ref_quant.quantize(round_to(w.reshape(N, K), sdt), 64, bits, sdt)
    kind = f"q{bits}_" + {"bfloat16": "bf16", "float16": "f16"}[sdt]
    keep = [dev_u32(packed), dev(s, sdt), dev(b, sdt)]
    ol = op_linear(kind, N, K, *keep)
    assert to_tiled(ol, keep)
    return ol, ref_quant.dequantize(packed, s, b, 64, bits), keep


def _run(ol, x, M, act, rnd=0, force=False, **kw):
    """force: the codes kernel at any size, or an error"""
    a = gemv_args(x, M, act, **kw)
    a.rnd = rnd
    torch.cuda.synchronize()
    L.check(L.lib().mi_op_gemm_codes(C.byref(ol), C.byref(a), -1 if force else 0, None))
    torch.cuda.synchronize()


@pytest.mark.parametrize("act", ["bfloat16", "float16"])
@pytest.mark.parametrize("bits", [4, 8])
@pytest.mark.parametrize("M,N,K", [
    (256, 2048, 1024),       # one row tile, K split: slices that end inside the groups
    (300, 2064, 1152),       # ragged rows, a column tile of 16, 18 groups (the bias columns end inside a K tile)
    (2085, 6144, 128),       # two groups: a run that is all prologue, unsplit
    (2304, 5632, 640),       # an even number of groups, unsplit
    (129, 4096, 4096),       # fewer rows than half a tile, eight slices
])
def test_store_logits_and_residual(act, bits, M, N, K):
    rng = np.random.default_rng(1000 * bits + M)
    ol, w, keep = _weight(bits, act, N, K, rng)
    x = round_to(rng.standard_normal((M, K)).astype(np.float32), act)
    h0 = round_to(rng.standard_normal((M, N)).astype(np.float32), act)
    xd, rows = dev(x, act), _rows(M)
    y = round_to(matmul_nt(x[rows], w), act)
    out = torch.full((M + 3, N), 7.0, dtype=xd.dtype, device="cuda")
    _run(ol, xd, M, act, force=True, epi=L.EPI_STORE, out=out, ldo=N)
    o = host(out)
    assert np.all(o[M:] == 7.0), "rows past M were written"
    _assert_close(o[:M][rows], y, act)
    lg = torch.full((M + 3, N), 7.0, dtype=torch.float32, device="cuda")          # logits: the same values as float32
    _run(ol, xd, M, act, force=True, epi=L.EPI_STORE_F32, out=lg, ldo=N)
    assert np.array_equal(host(lg)[:M], o[:M]) and np.all(host(lg)[M:] == 7.0)
    h = dev(h0, act)
    _run(ol, xd, M, act, force=True, epi=L.EPI_RESID, resid=h, out=h, ldo=N)
    _assert_close(host(h)[rows], round_to(h0[rows] + y, act), act)
    odd = torch.full((M + 1, N + 2), 7.0, dtype=xd.dtype, device="cuda")          # rows that are no whole 16-byte pieces
    _run(ol, xd, M, act, force=True, epi=L.EPI_STORE, out=odd, ldo=N + 2)
    assert np.array_equal(host(odd)[:M, :N], o[:M]) and np.all(host(odd)[M:] == 7.0) and np.all(host(odd)[:, N:] == 7.0)
    odd[:M, :N] = dev(h0, act)
    _run(ol, xd, M, act, force=True, epi=L.EPI_RESID, resid=odd, out=odd, ldo=N + 2)
    assert np.array_equal(host(odd)[:M, :N], host(h)) and np.all(host(odd)[M:] == 7.0) and np.all(host(odd)[:, N:] == 7.0)


@pytest.mark.parametrize("act", ["bfloat16", "float16"])
@pytest.mark.parametrize("bits,M,I,K", [(4, 2085, 3072, 512), (8, 517, 8208, 192), (4, 2048, 3200, 256), (8, 130, 144, 64)])
def test_swiglu(act, bits, M, I, K):
    rng = np.random.default_rng(M)
    ol, w, keep = _weight(bits, act, 2 * I, K, rng)
    x = round_to(rng.standard_normal((M, K)).astype(np.float32) * 0.3, act)
    xd, rows = dev(x, act), _rows(M)
    y = round_to(matmul_nt(x[rows], w), act)
    gt, up = y[:, :I].astype(np.float64), y[:, I:]
    sig = round_to((1.0 / (1.0 + np.exp(-gt))).astype(np.float32), act)
    want = round_to(round_to(gt.astype(np.float32) * sig, act) * up, act)
    out = torch.full((M + 1, I), 7.0, dtype=xd.dtype, device="cuda")
    _run(ol, xd, M, act, force=True, epi=L.EPI_SWIGLU, out=out, ldo=I, pair_offset=I)
    o = host(out)
    assert np.all(o[M:] == 7.0)
    _assert_close(o[:M][rows], want, act, scale=float(np.abs(y).max()))
    odd = torch.full((M + 1, I + 2), 7.0, dtype=xd.dtype, device="cuda")
    _run(ol, xd, M, act, force=True, epi=L.EPI_SWIGLU, out=odd, ldo=I + 2, pair_offset=I)
    assert np.array_equal(host(odd)[:M, :I], o[:M]) and np.all(host(odd)[M:] == 7.0) and np.all(host(odd)[:, I:] == 7.0)


@pytest.mark.parametrize("bits", [4, 8])
@pytest.mark.parametrize("M,N,K,rnd", [(300, 2048, 1024, 0), (2085, 6144, 256, 0), (64, 2768, 4096, 0), (131, 48, 4096, 0), (1024, 6144, 640, L.RND_BF16)])
def test_float32_rows(bits, M, N, K, rnd):
    """three bf16 terms of x (a run over the codes per term), every epilogue; rnd: layer 0's rounded call, x is one term"""
    if bits == 8 and M <= 128:
        M += 128                                                 # (up to there int8 keeps the streaming kernel)
    rng = np.random.default_rng(K)
    ol, w, keep = _weight(bits, "bfloat16", N, K, rng)
    x = rng.standard_normal((M, K)).astype(np.float32)
    if rnd:
        x = round_to(x, "bfloat16")
    rows, xd = _rows(M), dev(x)
    want = matmul_nt(x[rows], w)
    # exact products; K / 64 + 2 float32 additions of a group's sums and the biases', of up to 16 scales x |x| each
    tol = 2.0 ** -24 * (K / 64 + 8) * 4 * np.abs(x[rows]).sum(1).max() * np.abs(w).max()

    def call(epi, cols, fill=None, pad=0):
        out = torch.full((M + 1, cols + pad), 7.0, dtype=torch.float32, device="cuda")
        if fill is not None:
            out[:M, :cols] = dev(fill)
        _run(ol, xd, M, "float32", rnd=rnd, force=True, epi=epi, out=out, resid=out if epi == L.EPI_RESID else None, ldo=cols + pad, pair_offset=cols if epi == L.EPI_SWIGLU else 0)
        o = host(out)
        assert np.all(o[M:] == 7.0) and np.all(o[:, cols:] == 7.0)
        return o[:M, :cols]
    got = call(L.EPI_STORE, N)
    assert np.array_equal(call(L.EPI_STORE, N, pad=2), got)      # (rows that are no whole 16-byte pieces)
    if rnd:
        _assert_close(got[rows], round_to(want, "bfloat16"), "bfloat16")
        return
    assert np.max(np.abs(got[rows] - want)) <= tol
    assert np.array_equal(call(L.EPI_STORE_F32, N), got)
    h = rng.standard_normal((M, N)).astype(np.float32)
    for pad in (0, 2):
        assert np.array_equal(call(L.EPI_RESID, N, fill=h, pad=pad), h + got)
    I = N // 32 * 16
    gt, up = want[:, :I].astype(np.float64), want[:, I:2 * I].astype(np.float64)
    unit = gt / (1 + np.exp(-gt))
    for pad in (0, 2):                                           # |silu'| <= 1.1; its expf, quotient and two products: 2^-21 of the result
        y = call(L.EPI_SWIGLU, I, pad=pad)[rows]
        assert np.all(np.abs(y - unit * up) <= tol * (1.1 * np.abs(up) + np.abs(unit) + tol) + 2.0 ** -21 * np.abs(unit * up))


@pytest.mark.parametrize("M,N,K,epi", [(129, 1024, 1024, "STORE"), (300, 208, 704, "STORE"), (1365, 1024, 1024, "RESID"), (200, 2048, 1024, "SWIGLU"), (160, 48, 64, "STORE"),
                                       (256, 16, 1024, "STORE_F32")])
def test_int8_on_float32_rows_is_as_close_as_float32_sums(M, N, K, epi):
    """Small matrices, groups whose mean is twelve of their deviations: a [hi | lo] pair of the weight is 1.9e-6 off in 2-norm.  Here the products are exact,
    and a result takes one rounding per group of 64 and one per 32 of the 6 K / 64 bias columns, each of at most half an ulp of the partial sum: in 2-norm
    some 2^-24 sqrt(K / 64 + 6 K / 2048 + 2), the residual's and the unit's own roundings among the last two."""
    rng = np.random.default_rng(M)
    w = (rng.standard_normal((N, K // 64, 64)) + 12 * rng.standard_normal((N, K // 64, 1))).astype(np.float32) * 0.05
    packed, s, b = ref_quant.quantize(w.reshape(N, K), 64, 8, "bfloat16")
    keep = [dev_u32(packed), dev(s, "bfloat16"), dev(b, "bfloat16")]
    ol = op_linear("q8_bf16", N, K, *keep)
    assert to_tiled(ol, keep)
    codes = packed.view(np.uint8).reshape(N, K).astype(np.float64)
    w = codes * np.repeat(s, 64, 1).astype(np.float64) + np.repeat(b, 64, 1)
    x = rng.standard_normal((M, K)).astype(np.float32)
    want = x.astype(np.float64) @ w.T
    cols = N
    if epi == "SWIGLU":
        cols = N // 2
        gt, up = want[:, :cols], want[:, cols:]
        want = gt / (1 + np.exp(-np.clip(gt, -700, None))) * up
    h = rng.standard_normal((M, cols)).astype(np.float32) if epi == "RESID" else np.zeros((M, cols), np.float32)
    out = dev(h)
    _run(ol, dev(x), M, "float32", epi=getattr(L, "EPI_" + epi), out=out, ldo=cols, resid=out if epi == "RESID" else None, pair_offset=cols if epi == "SWIGLU" else 0)
    got = host(out).astype(np.float64)
    off = np.linalg.norm(got - (want + h)) / np.linalg.norm(want + h)
    # (SwiGLU: two such factors, and the sigmoid's expf and quotient, 3 ulp)
    n = K / 64 + 6 * K / 2048 + 2
    assert off <= 2.0 ** -24 * np.sqrt(n if epi != "SWIGLU" else 2 * n + 12), off


@pytest.mark.parametrize("bits,M,N,K", [(4, 64, 256, 8192), (8, 160, 512, 8192), (8, 192, 256, 14336), (4, 96, 512, 2048)])
@pytest.mark.parametrize("mean", [0, 4, 12])
def test_float32_rows_are_no_further_off_than_the_streaming_kernel(bits, M, N, K, mean):
    """The codes kernel takes float32 rows from the streaming kernel: its 2-norm from 64 bits is no larger, whatever the biases' share of the result."""
    rng = np.random.default_rng(K + mean)
    w = (rng.standard_normal((N, K // 64, 64)) + mean * rng.standard_normal((N, K // 64, 1))).astype(np.float32) * 0.05
    packed, s, b = ref_quant.quantize(w.reshape(N, K), 64, bits, "bfloat16")
    keep = [dev_u32(packed), dev(s, "bfloat16"), dev(b, "bfloat16")]
    ol = op_linear(f"q{bits}_bf16", N, K, *keep)
    assert to_tiled(ol, keep)
    codes = np.stack([packed >> np.uint32(bits * i) & np.uint32((1 << bits) - 1) for i in range(32 // bits)], -1).reshape(N, K).astype(np.float64)
    x = rng.standard_normal((M, K)).astype(np.float32)
    want = x.astype(np.float64) @ (codes * np.repeat(s, 64, 1).astype(np.float64) + np.repeat(b, 64, 1)).T
    xd, out = dev(x), torch.zeros((M, N), dtype=torch.float32, device="cuda")
    _run(ol, xd, M, "float32", force=True, epi=L.EPI_STORE, out=out, ldo=N)
    off = np.linalg.norm(host(out) - want)
    out.zero_()
    for r in range(0, M, 32):
        gemm_skinny(ol, xd[r:r + 32], 32, "float32", epi=L.EPI_STORE, out=out[r:r + 32], ldo=N)
    ref = np.linalg.norm(host(out) - want)
    assert off <= ref, (off / np.linalg.norm(want), ref / np.linalg.norm(want))


@pytest.mark.parametrize("kv", ["float32", "model"])
def test_the_last_piece_of_wide_logits_is_no_other_kernel(kv):
    """Logits of many positions are made 32768 columns at a time.  The last sixteen of these have the weights of the first sixteen: the same numbers, up to
    the sums' roundings (two results, each as above) -- with a [hi | lo] copy for them it is 5.1e-7 (int4 groups, means of 100 of their deviations)."""
    from mlx_parallm_amd.engine import Engine

    H, V, K = 1024, 32784, 1024
    cfg = dict(model_type="llama", hidden_size=H, num_hidden_layers=1, num_attention_heads=8, num_key_value_heads=8, head_dim=128, intermediate_size=1024,
               vocab_size=V, rms_norm_eps=1e-5, rope_theta=10000.0, tie_word_embeddings=False, max_position_embeddings=1024, quantization={"bits": 4, "group_size": 64})
    eng = Engine(cfg, device=0, max_positions=512, act_dtype="bfloat16")
    rng = np.random.default_rng(7)

    def put(name, n, mean=0.0, repeat=0):
        w = ((rng.standard_normal((n, K // 64, 64)) + mean * rng.standard_normal((n, K // 64, 1))) * 0.03).astype(np.float32).reshape(n, K)
        if repeat:
            w[-repeat:] = w[:repeat]
        packed, s, b = ref_quant.quantize(w, 64, 4, "bfloat16")
        for part, t in ((".weight", dev_u32(packed)), (".scales", dev(s, "bfloat16")), (".biases", dev(b, "bfloat16"))):
            eng.set_tensor(name + part, t)
    put("model.embed_tokens", V)
    p = "model.layers.0."
    for n in ("self_attn.q_proj", "self_attn.k_proj", "self_attn.v_proj", "self_attn.o_proj", "mlp.gate_proj", "mlp.up_proj", "mlp.down_proj"):
        put(p + n, H)
    for n in (p + "input_layernorm", p + "post_attention_layernorm", "model.norm"):
        eng.set_tensor(n + ".weight", torch.ones(H, dtype=torch.bfloat16, device="cuda"))
    put("lm_head", V, mean=100.0, repeat=16)
    eng.finalize()
    got = np.array(eng.forward(rng.integers(0, V, (1, 256)).astype(np.int32), eng.new_kv(1, capacity=300, kv_dtype=kv), all_positions=True), dtype=np.float64)[0]
    eng.close()
    first, last = got[:, :16], got[:, -16:]
    assert np.all(np.isfinite(got)) and np.linalg.norm(first) > 0
    off = np.linalg.norm(first - last) / np.linalg.norm(first)
    if kv == "model":                                            # (bfloat16 logits: at most some that fall to the other neighbour)
        assert np.mean(first != last) <= 0.01 and off <= 2.0 ** -8
    else:
        assert off <= 2.0 ** -24 * np.sqrt(2 * (K / 64 + 6 * K / 2048 + 2)), off


@pytest.mark.parametrize("act", ["bfloat16", "float16"])
@pytest.mark.parametrize("bits", [4, 8])
@pytest.mark.parametrize("kv_dtype", ["model", "float32"])
def test_kept_codes_and_codes_per_call_give_the_same_bits(bits, act, kv_dtype):
    """The copy that an engine makes of its quantised weights and the one made in front of a product hold the same: prompts' logits, and the logits of every position
    in pieces of 32768 columns, with and without it (float32 caches: the other order of the biases).  1500 rows: q|k|v, gate|up, down and the logits run on the codes.
    The copies take what codes_bytes says, are given back and made again; memory asked for in earnest comes before them; set in time, the option makes none."""
    from mlx_parallm_amd.engine import Engine, SampleArgs

    H, F, V = 1024, 2816, 33024
    cfg = dict(model_type="llama", hidden_size=H, num_hidden_layers=2, num_attention_heads=8, num_key_value_heads=8, head_dim=128, intermediate_size=F, vocab_size=V,
               rms_norm_eps=1e-5, rope_theta=10000.0, tie_word_embeddings=False, max_position_embeddings=1024, quantization={"bits": bits, "group_size": 64})
    dt = getattr(torch, act)
    g = torch.Generator(device="cuda").manual_seed(bits)

    def put(e, name, n, k):
        e.set_tensor(name + ".weight", torch.randint(-2 ** 31, 2 ** 31 - 1, (n, k * bits // 32), generator=g, device="cuda", dtype=torch.int32))
        scale = 2.0 / (2 ** bits - 1) / k ** 0.5
        e.set_tensor(name + ".scales", (scale * (1.0 + torch.rand((n, k // 64), generator=g, device="cuda"))).to(dt))
        e.set_tensor(name + ".biases", (-1.5 / k ** 0.5 * (1.0 + 0.3 * torch.randn((n, k // 64), generator=g, device="cuda"))).to(dt))

    def engine(kept):
        e = Engine(cfg, device=0, max_positions=1024, act_dtype=act)
        if not kept:
            e.set_option("prefill_codes_copy", 0)
        g.manual_seed(bits)
        put(e, "model.embed_tokens", V, H)
        put(e, "lm_head", V, H)
        for i in range(2):
            p = f"model.layers.{i}."
            for n, rows, cols in (("self_attn.q_proj", H, H), ("self_attn.k_proj", H, H), ("self_attn.v_proj", H, H), ("self_attn.o_proj", H, H), ("mlp.gate_proj", F, H),
                                  ("mlp.up_proj", F, H), ("mlp.down_proj", H, F)):
                put(e, p + n, rows, cols)
            for n in ("input_layernorm", "post_attention_layernorm"):
                e.set_tensor(p + n + ".weight", torch.ones(H, device="cuda", dtype=dt))
        e.set_tensor("model.norm.weight", torch.ones(H, device="cuda", dtype=dt))
        e.finalize()
        return e
    toks = np.random.default_rng(3).integers(0, V, (3, 500)).astype(np.int32)

    def results(e, kv):
        kv.reset()
        logits = np.asarray(e.forward(toks, kv)).copy()
        kv.reset()
        r = e.score_tokens(kv, toks, toks, SampleArgs(top_logprobs=3))
        return logits, np.asarray(r["logprobs"]).copy(), np.asarray(r["top_logprobs"]).copy()

    def bias_columns(k):                                         # (six products of a group's sum and its bias, whole K tiles)
        return -(-6 * (k // 64) // 64) * 64
    linears = [(V, H)] + [(3 * H, H), (H, H), (2 * F, H), (H, F)] * 2
    want = sum(n * (2 * k + k // 64 * 4 + 2 * bias_columns(k) * (2 if act == "bfloat16" else 1)) for n, k in linears)
    e = engine(True)
    kv, out = e.new_kv(3, capacity=512, kv_dtype=kv_dtype), []
    assert e.codes_bytes() == want
    out.append(results(e, kv))
    e.sync()
    free = torch.cuda.mem_get_info()[0]
    e.set_option("prefill_codes_copy", 0)
    assert e.codes_bytes() == 0 and torch.cuda.mem_get_info()[0] - free >= 0.9 * want
    out.append(results(e, kv))
    e.set_option("prefill_codes_copy", 1)
    assert e.codes_bytes() == want
    with pytest.raises(RuntimeError, match="out of device memory"):
        e.new_paged_kv(2, block_tokens=64, n_blocks=1 << 25, max_tokens_per_row=512, kv_dtype=kv_dtype)       # (17 TB)
    assert e.codes_bytes() == 0
    out.append(results(e, kv))
    e.close()
    e = engine(False)
    assert e.codes_bytes() == 0
    out.append(results(e, e.new_kv(3, capacity=512, kv_dtype=kv_dtype)))
    e.close()
    assert np.all(np.isfinite(out[0][0]))
    for other in out[1:]:
        for a, b in zip(out[0], other):
            assert np.array_equal(a, b)


@pytest.mark.parametrize("what", ["slices", "splits"])
def test_the_kept_codes_go_for_a_workspace_in_the_middle_of_a_call(what):
    """A workspace does not fit beside the copies: they go in the middle of the call that asks for it.  slices: a prompt's, for slices of K (128 MiB, of the first call below 4096
    rows), and the call then makes its own copy of the codes in a scratch of that size; splits: the decode attention's, for 2048 slots.  The same logits as with room for all."""
    from mlx_parallm_amd.engine import Engine

    H, F, V = 1024, 2816, 65792
    cfg = dict(model_type="llama", hidden_size=H, num_hidden_layers=1, num_attention_heads=8, num_key_value_heads=8, head_dim=128, intermediate_size=F, vocab_size=V,
               rms_norm_eps=1e-5, rope_theta=10000.0, tie_word_embeddings=False, max_position_embeddings=2048, quantization={"bits": 4, "group_size": 64})
    p, rng, out, MiB = "model.layers.0.", np.random.default_rng(3), [], 1 << 20

    def settled():                                                # what has been freed is told of some time later
        seen = [torch.cuda.mem_get_info()[0]]
        while len(seen) < 40 and (len(seen) < 4 or len(set(seen[-4:])) > 1):
            time.sleep(0.05)
            seen.append(torch.cuda.mem_get_info()[0])
        return seen[-1]
    long, short = rng.integers(0, V, (3, 1400)).astype(np.int32), rng.integers(0, V, (3, 500)).astype(np.int32)
    for full in (False, True):
        e = Engine(cfg, device=0, max_positions=2048, act_dtype="bfloat16")
        g = torch.Generator(device="cuda").manual_seed(1)
        for name, n, k in (("model.embed_tokens", V, H), ("lm_head", V, H), (p + "self_attn.q_proj", H, H), (p + "self_attn.k_proj", H, H), (p + "self_attn.v_proj", H, H),
                           (p + "self_attn.o_proj", H, H), (p + "mlp.gate_proj", F, H), (p + "mlp.up_proj", F, H), (p + "mlp.down_proj", H, F)):
            e.set_tensor(name + ".weight", torch.randint(-2 ** 31, 2 ** 31 - 1, (n, k // 8), generator=g, device="cuda", dtype=torch.int32))
            e.set_tensor(name + ".scales", (2.0 / 15 / k ** 0.5 * (1.0 + torch.rand((n, k // 64), generator=g, device="cuda"))).bfloat16())
            e.set_tensor(name + ".biases", (-1.5 / k ** 0.5 * (1.0 + 0.3 * torch.randn((n, k // 64), generator=g, device="cuda"))).bfloat16())
        for n in (p + "input_layernorm", p + "post_attention_layernorm", "model.norm"):
            e.set_tensor(n + ".weight", torch.ones(H, device="cuda", dtype=torch.bfloat16))
        e.finalize()
        if what == "slices":
            kv = e.new_kv(3, capacity=1408)
            e.forward(long, kv)                                  # (4200 rows: everything but that workspace)
            kv.reset()
        else:
            kv = e.new_paged_kv(2048, block_tokens=64, n_blocks=64, max_tokens_per_row=1536)
            e.forward_segments(kv, [7], [long[0]], want=[1399])
        e.sync()
        torch.cuda.empty_cache()
        held = []
        while full and len(held) < 8 and settled() > 120 * MiB:      # (what is free is told to within a few parts in a thousand)
            held.append(torch.empty(settled() - 108 * MiB, dtype=torch.uint8, device="cuda"))
        assert not full or 64 * MiB < settled() < 128 * MiB
        assert e.codes_bytes() > 128 * MiB
        out.append(np.array(e.forward(short, kv) if what == "slices" else e.forward_segments(kv, [7], [short[0, :1]], want=[0])))
        assert (e.codes_bytes() == 0) == full
        e.close()
        del held
        torch.cuda.empty_cache()
    assert np.all(np.isfinite(out[0])) and np.array_equal(out[0], out[1])


@pytest.mark.parametrize("rows", [256, 97])
def test_float32_prompts_take_one_route_with_and_without_kept_codes(rows):
    """The streaming kernel and the codes differ in their last bits: which of them a prompt takes is no matter of the memory that was free at load time (gate|up at 256 rows
    and the logits of 97 positions lie where the copy's price would decide)."""
    from mlx_parallm_amd.engine import Engine

    H, F, V = 2048, 6400, 32000
    cfg = dict(model_type="llama", hidden_size=H, num_hidden_layers=1, num_attention_heads=16, num_key_value_heads=4, head_dim=128, intermediate_size=F, vocab_size=V,
               rms_norm_eps=1e-5, rope_theta=10000.0, tie_word_embeddings=False, max_position_embeddings=512, quantization={"bits": 4, "group_size": 64})
    out = []
    for kept in (1, 0):
        e = Engine(cfg, device=0, max_positions=512, act_dtype="bfloat16")
        e.set_option("prefill_codes_copy", kept)
        g = torch.Generator(device="cuda").manual_seed(1)
        p = "model.layers.0."
        for name, n, k in (("model.embed_tokens", V, H), ("lm_head", V, H), (p + "self_attn.q_proj", H, H), (p + "self_attn.k_proj", 512, H), (p + "self_attn.v_proj", 512, H),
                           (p + "self_attn.o_proj", H, H), (p + "mlp.gate_proj", F, H), (p + "mlp.up_proj", F, H), (p + "mlp.down_proj", H, F)):
            e.set_tensor(name + ".weight", torch.randint(-2 ** 31, 2 ** 31 - 1, (n, k // 8), generator=g, device="cuda", dtype=torch.int32))
            e.set_tensor(name + ".scales", (2.0 / 15 / k ** 0.5 * (1.0 + torch.rand((n, k // 64), generator=g, device="cuda"))).bfloat16())
            e.set_tensor(name + ".biases", (-1.5 / k ** 0.5 * (1.0 + 0.3 * torch.randn((n, k // 64), generator=g, device="cuda"))).bfloat16())
        for n in (p + "input_layernorm", p + "post_attention_layernorm", "model.norm"):
            e.set_tensor(n + ".weight", torch.ones(H, device="cuda", dtype=torch.bfloat16))
        e.finalize()
        assert (e.codes_bytes() > 0) == bool(kept)
        toks = np.random.default_rng(3).integers(0, V, (1, rows)).astype(np.int32)
        out.append(np.array(e.forward(toks, e.new_kv(1, capacity=300, kv_dtype="float32"), all_positions=True)))
        e.close()
    assert np.all(np.isfinite(out[0])) and np.array_equal(out[0], out[1])


@pytest.mark.parametrize("act", ["bfloat16", "float16"])
@pytest.mark.parametrize("bits,M,N,K,epi", [
    (4, 700, 2 * 11520, 1024, "swiglu"),     # 270 tiles: one round, and 15 in K slices
    (8, 300, 2 * 1040, 1088, "swiglu"),      # fewer tiles than CUs, the last ones ragged: all in slices
    (4, 700, 24016, 1024, "f32"),            # 282 tiles; the last column of tiles holds 208 columns
    (8, 601, 22032, 1024, "resid"),
    (8, 1270, 13216, 1024, "resid"),         # whole slices do not fit the workspace: 5 of 260 tiles in slices
])
def test_tiles_of_a_last_round_in_slices(act, bits, M, N, K, epi):
    """Against the oracle; every row of a call has one order of sums, whatever its place: a row's copy at the end gives the same bits."""
    rng = np.random.default_rng(M + N)
    ol, w, keep = _weight(bits, act, N, K, rng)
    x = round_to(rng.standard_normal((M, K)).astype(np.float32) * 0.3, act)
    h0 = round_to(rng.standard_normal((M, N)).astype(np.float32), act)
    x[M - 1], h0[M - 1] = x[5], h0[5]
    xd, rows = dev(x, act), _rows(M)
    y = want = round_to(matmul_nt(x[rows], w), act)
    cols, kw, code = N, {}, L.EPI_STORE_F32
    if epi == "swiglu":
        cols, code = N // 2, L.EPI_SWIGLU
        kw = dict(pair_offset=cols)
        sig = round_to((1.0 / (1.0 + np.exp(-y[:, :cols].astype(np.float64)))).astype(np.float32), act)
        want = round_to(round_to(y[:, :cols] * sig, act) * y[:, cols:], act)
    out = torch.full((M + 1, cols), 7.0, dtype=torch.float32 if epi == "f32" else xd.dtype, device="cuda")
    if epi == "resid":
        out[:M] = dev(h0, act)
        code, kw, want = L.EPI_RESID, dict(resid=out), round_to(h0[rows] + y, act)
    _run(ol, xd, M, act, force=True, epi=code, out=out, ldo=cols, **kw)
    o = host(out)
    assert np.all(o[M:] == 7.0) and np.array_equal(o[M - 1], o[5])
    _assert_close(o[:M][rows], want, act, scale=float(np.abs(y).max()))


def test_a_round_of_more_than_half_of_the_tiles_is_not_sliced():
    """By the bits of 5632 x 4096 SwiGLU: 700 rows (132 tiles) have those of the same rows among 1025 (220 tiles), 300 rows (88 tiles, two slices) differ in some."""
    h, K = 5632, 4096
    g = torch.Generator(device="cuda").manual_seed(7)
    keep = [torch.randint(-2 ** 31, 2 ** 31 - 1, (2 * h, K // 8), generator=g, device="cuda", dtype=torch.int32)]
    keep += [(0.002 * (1 + torch.rand((2 * h, K // 64), generator=g, device="cuda"))).bfloat16(), (-0.02 * (1 + 0.3 * torch.randn((2 * h, K // 64), generator=g, device="cuda"))).bfloat16()]
    ol = op_linear("q4_bf16", 2 * h, K, *keep)
    assert to_tiled(ol, keep)
    x = torch.randn((1025, K), generator=g, device="cuda").bfloat16()

    def rows(M):
        out = torch.zeros((M, h), dtype=torch.bfloat16, device="cuda")
        _run(ol, x, M, "bfloat16", force=True, epi=L.EPI_SWIGLU, out=out, ldo=h, pair_offset=h)
        return host(out)
    all_rows = rows(1025)
    assert np.all(np.isfinite(all_rows)) and np.array_equal(rows(700), all_rows[:700]) and not np.array_equal(rows(300), all_rows[:300])


@pytest.mark.parametrize("M,N,K,swiglu,most", [
    (700, 6144, 4096, False, 1.4e-7),         # 72 tiles: seven slices of K 1.22e-7, three 1.80e-7
    (300, 2 * 6400, 2048, True, 1.85e-7),     # 100 tiles: five slices 1.62e-7, two 2.10e-7, none 2.07e-7
])
def test_float32_rows_stay_as_close_to_64_bits(M, N, K, swiglu, most):
    """How K is split decides how far float32 rows are from 64 bits: 2-norms as measured for the slices named, the bound between them."""
    rng = np.random.default_rng(0)
    w = rng.standard_normal((N, K)).astype(np.float32) * 0.05
    lo, hi = w.reshape(N, K // 64, 64).min(-1), w.reshape(N, K // 64, 64).max(-1)
    s, b = round_to((hi - lo) / 15, "bfloat16"), round_to(lo, "bfloat16")
    q = np.clip(np.rint((w.reshape(N, K // 64, 64) - b[..., None]) / s[..., None]), 0, 15).astype(np.uint32)
    packed = np.bitwise_or.reduce(q.reshape(N, K // 8, 8) << (np.arange(8, dtype=np.uint32) * 4), axis=-1).astype(np.uint32)
    keep = [dev_u32(packed), dev(s, "bfloat16"), dev(b, "bfloat16")]
    ol = op_linear("q4_bf16", N, K, *keep)
    assert to_tiled(ol, keep)
    x, rows = rng.standard_normal((M, K)).astype(np.float32), _rows(M)
    y = x[rows].astype(np.float64) @ (q * s[..., None].astype(np.float64) + b[..., None]).reshape(N, K).T
    cols = N // 2 if swiglu else N
    want = y[:, :cols] / (1.0 + np.exp(-y[:, :cols])) * y[:, cols:] if swiglu else y
    out = torch.zeros((M, cols), dtype=torch.float32, device="cuda")
    _run(ol, dev(x), M, "float32", force=True, epi=L.EPI_SWIGLU if swiglu else L.EPI_STORE, out=out, ldo=cols, pair_offset=cols if swiglu else 0)
    off = np.linalg.norm(host(out)[rows].astype(np.float64) - want) / np.linalg.norm(want)
    assert off <= most, off


@pytest.mark.parametrize("bits,act,H,V", [(4, "bfloat16", 384, 36864), (8, "float16", 2112, 6656), (4, "float16", 4224, 1680), (8, "bfloat16", 8192, 832), (4, "bfloat16", 8320, 832)])
def test_norm_and_group_sums_in_one_launch(bits, act, H, V):
    """The norm in front of a product on codes leaves the sums of its groups (one to four pieces of a row a thread, the last ones partly filled; above 8192 columns a launch
    of its own; logits in two pieces of columns).  Layers that add nothing, so the logits of every position are W_hat . norm(embedding): two roundings to 16 bits (the
    logits' and the embedding's own) of 2^-9 (2^-12) in root mean square at most; a sum that went astray is off by the groups' means, four deviations."""
    from mlx_parallm_amd.engine import Engine

    cfg = dict(model_type="llama", hidden_size=H, num_hidden_layers=1, num_attention_heads=2, num_key_value_heads=2, head_dim=64, intermediate_size=128, vocab_size=V,
               rms_norm_eps=1e-5, rope_theta=10000.0, tie_word_embeddings=False, max_position_embeddings=512, quantization={"bits": bits, "group_size": 64})
    e = Engine(cfg, device=0, max_positions=512, act_dtype=act)
    rng = np.random.default_rng(H)

    def put(name, n, k, zero=False):
        w = (rng.standard_normal((n, k // 64, 64)) + 4 * rng.standard_normal((n, k // 64, 1))).astype(np.float32).reshape(n, k) * 0.05
        packed, s, b = ref_quant.quantize(round_to(w, act), 64, bits, act)
        if zero:
            s, b = np.zeros_like(s), np.zeros_like(b)
        for part, t in ((".weight", dev_u32(packed)), (".scales", dev(s, act)), (".biases", dev(b, act))):
            e.set_tensor(name + part, t)
        return ref_quant.dequantize(packed, s, b, 64, bits)
    emb = put("model.embed_tokens", V, H)
    head = put("lm_head", V, H)
    p = "model.layers.0."
    for n, rows, cols in (("self_attn.q_proj", 128, H), ("self_attn.k_proj", 128, H), ("self_attn.v_proj", 128, H), ("mlp.gate_proj", 128, H), ("mlp.up_proj", 128, H)):
        put(p + n, rows, cols)
    put(p + "self_attn.o_proj", H, 128, zero=True)
    put(p + "mlp.down_proj", H, 128, zero=True)
    nw = round_to(1.0 + 0.2 * rng.standard_normal(H).astype(np.float32), act)
    for n in (p + "input_layernorm", p + "post_attention_layernorm", "model.norm"):
        e.set_tensor(n + ".weight", dev(nw, act))
    e.finalize()
    toks = rng.integers(0, V, (1, 320)).astype(np.int32)
    got = np.array(e.forward(toks, e.new_kv(1, capacity=384), all_positions=True), dtype=np.float64)[0]
    e.close()
    x = np.asarray(round_to(emb[toks[0]], act), dtype=np.float64)
    xn = round_to((x / np.sqrt((x * x).mean(-1, keepdims=True) + 1e-5)).astype(np.float32), act)
    xn = round_to(np.asarray(xn, dtype=np.float32) * np.asarray(nw, dtype=np.float32), act)
    want = (torch.from_numpy(np.asarray(xn, dtype=np.float64)) @ torch.from_numpy(np.asarray(head, dtype=np.float64)).T).numpy()
    off = np.linalg.norm(got - want) / np.linalg.norm(want)
    assert off <= 2.0 * 2.0 ** (-9 if act == "bfloat16" else -12), off
