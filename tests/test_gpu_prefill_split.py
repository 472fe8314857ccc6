"""Float32-cache prefill (-m gpu): gate|up stores its SwiGLU as the two bf16 terms that the down projection multiplies.  The terms are those of the pass
that split the float32 row, so the logits are the same bits (ragged rows, a gated width that is no multiple of the tile, chunks behind a cache)."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

from mlx_parallm_amd.engine import Engine  # noqa: E402


@pytest.mark.parametrize("B,lengths", [(2, (1024,)), (3, (700, 683)), (1, (2011,))])
@pytest.mark.parametrize("ff", [3072, 3152])
def test_same_bits_as_the_separate_pass(B, lengths, ff):
    H, V = 256, 512
    cfg = dict(model_type="llama", hidden_size=H, num_hidden_layers=2, num_attention_heads=4, num_key_value_heads=2, head_dim=64, intermediate_size=ff,
               vocab_size=V, rms_norm_eps=1e-5, rope_theta=10000.0, tie_word_embeddings=False, max_position_embeddings=4096)
    eng = Engine(cfg, device=0, max_positions=4096, act_dtype="bfloat16")
    gen = torch.Generator(device="cuda").manual_seed(ff + B)

    def put(name, *shape, std=0.08):
        t = torch.randn(shape, generator=gen, device="cuda") * std
        eng.set_tensor(name, (t + 1.0 if len(shape) == 1 else t).to(torch.bfloat16))
    put("model.embed_tokens.weight", V, H, std=1.0)
    for i in range(2):
        p = f"model.layers.{i}."
        for n, rows, cols in (("self_attn.q_proj", H, H), ("self_attn.k_proj", 128, H), ("self_attn.v_proj", 128, H), ("self_attn.o_proj", H, H),
                              ("mlp.gate_proj", ff, H), ("mlp.up_proj", ff, H), ("mlp.down_proj", H, ff)):
            put(p + n + ".weight", rows, cols)
        put(p + "input_layernorm.weight", H, std=0.1)
        put(p + "post_attention_layernorm.weight", H, std=0.1)
    put("model.norm.weight", H, std=0.1)
    put("lm_head.weight", V, H)
    eng.finalize()
    rng = np.random.default_rng(B)
    chunks = [rng.integers(0, V, (B, n)).astype(np.int32) for n in lengths]
    got = []
    for split in (1, 0):
        eng.set_option("prefill_split_act", split)
        kv = eng.new_kv(B, capacity=sum(lengths) + 2, kv_dtype="float32")
        got.append([np.array(eng.forward(c, kv)) for c in chunks])
    for a, b in zip(*got):
        assert np.all(np.isfinite(a)) and np.array_equal(a, b)
    eng.close()


@pytest.mark.parametrize("epi", ["store", "resid", "swiglu", "logits"])
@pytest.mark.parametrize("M,N", [(2085, 6160), (2304, 5632)])
def test_rows_in_pieces_and_by_elements_store_the_same(epi, M, N):
    """The 256 x 256 tile takes 16-byte pieces of rows where stride and base allow it, single elements elsewhere: the same bits, nothing beside them."""
    from gpu_helpers import dev, gemm_prefill, host, op_linear, to_tiled
    from mlx_parallm_amd import _lib as L

    rng = np.random.default_rng(N)
    K = 192
    wd = dev(rng.standard_normal((N, K)).astype(np.float32) * 0.05, "bfloat16")
    ol, keep = op_linear("bf16", N, K, wd), [wd]
    assert to_tiled(ol, keep)
    xd = dev(rng.standard_normal((M, K)).astype(np.float32), "bfloat16")
    cols = N // 2 if epi == "swiglu" else N
    h = rng.standard_normal((M, cols)).astype(np.float32)
    dt = torch.float32 if epi == "logits" else torch.bfloat16
    got = []
    for pad, shift in ((8, 0), (2, 0), (8, 2)):                   # strides and bases of whole pieces; a stride that is none; a base that is none
        buf = torch.full(((M + 1) * (cols + pad) + 8,), 7.0, dtype=dt, device="cuda")
        out = buf[shift:shift + (M + 1) * (cols + pad)].view(M + 1, cols + pad)
        if epi == "resid":
            out[:M, :cols] = dev(h, "bfloat16")
        kw = {"store": dict(epi=L.EPI_STORE), "resid": dict(epi=L.EPI_RESID, resid=out), "logits": dict(epi=L.EPI_STORE_F32),
              "swiglu": dict(epi=L.EPI_SWIGLU, pair_offset=cols)}[epi]
        gemm_prefill(ol, xd, M, "bfloat16", out=out, ldo=cols + pad, **kw)
        torch.cuda.synchronize()
        o = host(out)
        assert np.all(o[M:] == 7.0) and np.all(o[:, cols:] == 7.0)
        got.append(o[:M, :cols])
    assert np.array_equal(got[0], got[1]) and np.array_equal(got[0], got[2])
