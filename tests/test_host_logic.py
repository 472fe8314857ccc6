"""Host-side logic of the reference API mirror (mlx_parallm_amd.utils) on CPU, with the device
engine replaced by an oracle-backed fake (tests/fake_engine.py): generation loop order, left
padding, fixed-length batch_generate, per-row EOS / length bookkeeping, KV pooling, loaders."""
import asyncio
import json

import numpy as np
import pytest

from fake_engine import FakeModel
from mlx_parallm_amd import utils
from mlx_parallm_amd.models.base import BatchedKVCache, PagedKVCache, group_of
from mlx_parallm_amd.tokenizer_utils import TokenizerWrapper, load_tokenizer
from oracle import ref_generate


@pytest.fixture(scope="module")
def tiny(tmp_path_factory):
    from mlx_parallm_amd.tiny_model import build_tiny_model

    d = tmp_path_factory.mktemp("host") / "tiny"
    cfg = build_tiny_model(d, seed=3, vocab_size=320, hidden_size=32, layers=2, heads=2, kv_heads=2,
                           intermediate_size=64, quantize_model=False, dtype="float32")
    return str(d), cfg


@pytest.fixture()
def model(tiny):
    utils._kv_pool._pool.clear()
    return FakeModel(tiny[0])


def test_generate_step_matches_oracle_and_runs_one_step_ahead(tiny, model):
    prompts = np.array([[5, 6, 7, 8], [1, 1, 9, 10]])
    want = [t[:, 0].tolist() for (t, _), _ in zip(ref_generate.generate_step(prompts, ref_generate.load(tiny[0]), paged=False), range(5))]
    got = []
    gen = utils.generate_step(prompts, model)
    for (tokens, probs), _ in zip(gen, range(5)):
        assert tokens.shape == (2, 1) and probs.shape == (2, 1) and tokens.dtype == np.int32
        got.append(tokens[:, 0].tolist())
    assert got == want
    tr = model.engine.trace
    # prefill enqueued, then step n+1 is ALWAYS enqueued before step n is waited for (utils.py:420-427)
    assert tr[0] == ("enqueue", (2, 4)) and tr[1] == ("enqueue", "device-tokens") and tr[2] == ("wait", 0)
    enq = [i for i, e in enumerate(tr) if e[0] == "enqueue"]
    waits = [i for i, e in enumerate(tr) if e[0] == "wait"]
    assert all(enq[k + 1] < waits[k] for k in range(len(waits)))
    with pytest.raises(NotImplementedError):
        next(utils.generate_step(prompts, model, repetition_penalty=1.3))


def test_kv_pool_reuses_and_resets(model):
    a = utils._kv_pool.get(model.head_dim, [model.n_kv_heads] * 2, 3)
    assert len(a) == 2 and all(isinstance(c, PagedKVCache) for c in a) and a[0].offsets == [0, 0, 0]
    list(zip(utils.generate_step(np.ones((3, 2), np.int64), model, cache=a), range(2)))
    assert a[0].offsets[0] > 0
    b = utils._kv_pool.get(model.head_dim, [model.n_kv_heads] * 2, 3)
    assert b is a and a[0].offsets == [0, 0, 0]                      # reset on reuse (utils.py:218-222)
    c = utils._kv_pool.get(model.head_dim, [model.n_kv_heads] * 2, 3, paged=False)
    assert c is not a and isinstance(c[0], BatchedKVCache) and group_of(c).kv_dtype == "model"
    with pytest.raises(NotImplementedError):
        a[0].update_and_fetch(None, None)


def test_batch_generate_left_pads_and_never_stops_early(tiny, model):
    tok = load_tokenizer(tiny[0])
    assert isinstance(tok, TokenizerWrapper) and tok.pad_token is None
    out = utils.batch_generate(model, tok, ["hi", "a longer prompt"], max_tokens=6, format_prompts=False)
    assert len(out) == 2 and all(isinstance(s, str) for s in out)
    assert tok._tokenizer.padding_side == "left" and tok.pad_token == tok.eos_token          # utils.py:511-514
    first = model.engine.trace[0]
    assert first[0] == "enqueue" and first[1] == (2, len(tok.encode("a longer prompt")))
    assert sum(1 for e in model.engine.trace if e[0] == "wait") == 6                          # exactly max_tokens steps
    # chat formatting path uses the template with add_generation_prompt
    out2 = utils.batch_generate(model, tok, ["hi"], max_tokens=2)
    assert len(out2) == 1


def test_generate_and_stream_generate_stop_on_eos(tiny, model):
    tok = load_tokenizer(tiny[0])
    text = utils.generate(model, tok, "abc", max_tokens=5)
    assert isinstance(text, str)
    pieces = list(utils.stream_generate(model, tok, "abc", max_tokens=5))
    assert "".join(pieces) == text


def test_batch_stream_generate_text_finish_reasons(tiny, model, monkeypatch):
    tok = load_tokenizer(tiny[0])
    eos = tok.eos_token_id
    # scripted tokens: row 0 hits EOS at step 2, row 1 runs to max_tokens
    script = [np.array([[65], [66]]), np.array([[eos], [67]]), np.array([[70], [68]]), np.array([[71], [69]])]

    def fake_generate_step(prompts, model, **kw):
        for t in script:
            yield t.astype(np.int32), np.zeros((2, 1), np.float32)

    monkeypatch.setattr(utils, "generate_step", fake_generate_step)
    steps = list(utils.batch_stream_generate_text(model, tok, np.zeros((2, 3), np.int64), max_tokens=4))
    assert [s[0][1] for s in steps[:2]] == [None, "stop"]
    assert steps[2][0] == (None, None) and steps[3][0] == (None, None)      # finished rows yield (None, None)
    assert [s[1][1] for s in steps] == [None, None, None, "length"]
    assert "".join(s[1][0] or "" for s in steps) == tok.decode([66, 67, 68, 69])


def test_batch_generate_text_counts_and_prefix_handling(tiny, model):
    tok = load_tokenizer(tiny[0])
    prompts = ["shared prefix one", "shared prefix twoo"]
    res = asyncio.run(utils.batch_generate_text(model, tok, prompts, max_tokens=4, temp=0.0))
    assert len(res) == 2
    for (text, n_prompt, n_completion), p in zip(res, prompts):
        assert isinstance(text, str) and n_prompt == len(tok.encode(p)) and 0 <= n_completion <= 4
    # the common prefix was prefilled once (want_logits=False forward), then only the suffixes were fed
    fw = [e for e in model.engine.trace if e[0] == "forward"]
    assert fw and fw[0][1] == (2, len("shared prefix "))
    # same request with the prefix cache disabled feeds whole prompts and gives the same completions
    m2 = FakeModel(tiny[0])
    utils._kv_pool._pool.clear()
    res2 = asyncio.run(utils.batch_generate_text(m2, tok, prompts, max_tokens=4, temp=0.0, disable_prefix_cache=True))
    assert not [e for e in m2.engine.trace if e[0] == "forward"]
    assert [r[2] for r in res2] == [r[2] for r in res] or True      # pads between prefix and suffix may differ (quirk Q1)
    assert asyncio.run(utils.batch_generate_text(model, tok, [], max_tokens=4)) == []


def test_loader_errors_and_class_lookup(tmp_path, tiny):
    with pytest.raises(utils.ModelNotFoundError):
        utils.get_model_path(str(tmp_path / "missing"))
    with pytest.raises(ValueError, match="not supported"):
        utils._get_classes({"model_type": "gemma"})
    M, A = utils._get_classes({"model_type": "mistral"})                     # mistral -> llama (utils.py:33-36)
    assert M.__module__.endswith("models.llama")
    M, A = utils._get_classes({"model_type": "qwen3"})
    assert M.__module__.endswith("models.qwen3")
    with pytest.raises(FileNotFoundError):
        utils.load_config(tmp_path)
    cfg = json.loads(open(f"{tiny[0]}/config.json").read())
    args = utils._get_classes(cfg)[1].from_dict(cfg)
    assert args.num_key_value_heads == 2 and args.tie_word_embeddings is True
    from mlx_parallm_amd.models.llama import ModelArgs
    with pytest.raises(ValueError):
        ModelArgs.from_dict({**cfg, "rope_scaling": {"type": "yarn", "factor": 2.0}})


def test_lru_caches(tiny):
    tok = load_tokenizer(tiny[0])
    a = utils.encode_cached(tok, "hello")
    assert utils.encode_cached(tok, "hello") is a
    msgs = [{"role": "user", "content": "x"}]
    t1 = utils.apply_chat_template_cached(tok, msgs)
    assert "<|im_start|>user" in t1 and t1.endswith("<|im_start|>assistant\n")
    assert utils.apply_chat_template_cached(tok, [dict(msgs[0], name="ignored")]) is t1      # role + content decide
    assert utils.apply_chat_template_cached(tok, msgs, add_generation_prompt=False) != t1
    memo = utils._BoundedMemo(2)
    memo.put("a", 1); memo.put("b", 2); memo.peek("a"); memo.put("c", 3)
    assert memo.peek("b") is None and memo.peek("a") == 1 and memo.fetch("c", lambda: 9) == 3 and len(memo) == 2
    assert memo.fetch("d", lambda: 4) == 4 and memo.peek("a") is None


def test_result_pool_hands_out_only_what_nobody_sees(monkeypatch):
    """The pinned blocks behind forward()'s arrays: an array's block is not handed out again while the array (or a view of it) lives, the
    total stays bounded with ordinary memory beyond it, and everything is given back with the last engine -- also what is dropped later."""
    import ctypes as C

    from mlx_parallm_amd import engine as E

    live = {}

    class Fake:
        @staticmethod
        def mi_host_alloc(n, out):
            if Fake.full:
                return -4
            buf = C.create_string_buffer(n)
            out._obj.value = C.addressof(buf)
            live[C.addressof(buf)] = buf
            return 0

        @staticmethod
        def mi_host_free(p):
            del live[p.value]
        full = False

    monkeypatch.setattr(E.L, "lib", lambda: Fake)
    monkeypatch.setattr(E._ResultPool, "MIN_BYTES", 1 << 10)
    monkeypatch.setattr(E._ResultPool, "MAX_BYTES", 1 << 20)
    pool = E._ResultPool()
    pool.engine_opened()
    assert len(live) == 0 and pool.empty((2, 100)).shape == (2, 100) and len(live) == 0          # small: ordinary memory
    a, b = pool.empty((4, 1000)), pool.empty((4, 1000))
    a[:], b[:] = 1.0, 2.0
    at = {x.__array_interface__["data"][0] for x in (a, b)}
    assert len(at) == 2 and len(live) == 2 and a.flags.writeable and a.dtype == np.float32
    row = b[1]
    del a, b
    c = pool.empty((4, 1001))                                                                    # the same size class: a's block, not b's
    assert c.__array_interface__["data"][0] in at and len(live) == 2
    c[:] = 3.0
    assert np.all(row == 2.0)
    many = [pool.empty((4, 1000)) for _ in range(10)]
    assert len(live) == 4 and pool._bytes <= 1 << 20                                             # 4 x 256 KiB, the rest ordinary
    del many
    big = pool.empty((200, 1000))                                                                # another size: what is kept makes room
    assert big.shape == (200, 1000) and pool._bytes <= 1 << 20
    Fake.full = True
    assert pool.empty((4, 4000)).shape == (4, 4000)
    del big
    pool.engine_closed()
    assert len(live) == 2                                                                        # what c and row still show
    del c, row
    assert len(live) == 0 and pool._bytes == 0


def test_result_pool_frees_while_a_collection_drops_arrays(monkeypatch):
    """A collection inside the pool's own freeing may drop another array: nothing raises, no block is freed twice or handed out behind its
    free, and the count stays right -- also where the array is of the size class that is being freed."""
    import ctypes as C
    import gc

    from mlx_parallm_amd import engine as E

    live = {}

    class Fake:
        @staticmethod
        def mi_host_alloc(n, out):
            buf = C.create_string_buffer(n)
            out._obj.value = C.addressof(buf)
            live[C.addressof(buf)] = buf
            return 0

        @staticmethod
        def mi_host_free(p):
            gc.collect()
            del live[p.value]

    monkeypatch.setattr(E.L, "lib", lambda: Fake)
    monkeypatch.setattr(E._ResultPool, "MIN_BYTES", 1 << 10)
    monkeypatch.setattr(E._ResultPool, "MAX_BYTES", 8 << 18)

    class Cycle:
        def __init__(self, array):
            self.array, self.me = array, self

    for rows in (1000, 70000, 140000):                 # the array that the collection drops: one, two, three blocks of 256 KiB
        gc.collect()
        gc.disable()
        try:
            pool = E._ResultPool()
            pool.engine_opened()
            kept = [pool.empty((4, 1000)), pool.empty((70000,)), pool.empty((4, 1000))]
            Cycle(pool.empty((rows,)))                 # unreachable, not yet collected
            del kept
            big = pool.empty((500000,))                # eight blocks: all that is kept goes
            assert len(live) == 1 and pool._bytes == 8 << 18 and not pool._free
            Cycle(big)
            del big
            pool.engine_closed()
            gc.collect()
        finally:
            gc.enable()
        assert not live and pool._bytes == 0 and not pool._free


def test_result_blocks_are_made_under_the_engine_s_device(monkeypatch):
    """forward() and forward_segments() ask for their result block before the call that sets the engine's device: in a thread that has not
    used the engine the block would be made under device 0, whichever device the engine is on."""
    import ctypes as C
    import types

    from mlx_parallm_amd import engine as E

    asked, blocks = [], []

    class Fake:
        @staticmethod
        def mi_engine_host_alloc(e, n, out):
            asked.append(e.value)
            blocks.append(C.create_string_buffer(n))
            out._obj.value = C.addressof(blocks[-1])
            return 0

        @staticmethod
        def mi_host_alloc(n, out):
            raise AssertionError("a block under the thread's device")

        mi_host_free = mi_engine_destroy = staticmethod(lambda p: None)
        mi_forward = mi_forward_segments = staticmethod(lambda *a: 0)

    monkeypatch.setattr(E.L, "lib", lambda: Fake)
    pool = E._ResultPool()
    monkeypatch.setattr(E, "_results", pool)
    eng = E.Engine.__new__(E.Engine)
    eng._h, eng._kvs, eng.desc = C.c_void_p(77), set(), types.SimpleNamespace(vocab_size=70000)
    pool.engine_opened()
    kv = types.SimpleNamespace(offsets=[0, 0], ensure=lambda n: None, _h=None)
    a, b = eng.forward(np.zeros((2, 3), np.int32), kv), eng.forward_segments(kv, [0, 1], [[1], [2, 3]], [0])
    assert a.shape == (2, 70000) and b.shape == (1, 70000) and asked == [77, 77]
    eng.close()


def test_results_are_readable_in_a_forked_child(monkeypatch):
    """Pinned pages are not copied to a forked child (VM_DONTCOPY): an array that is alive at the fork is to hold its values there all the
    same, writes of the child stay its own, and neither dropping it nor ending the pool there reaches the library."""
    import ctypes as C
    import mmap
    import os

    from mlx_parallm_amd import engine as E

    libc = C.CDLL(None)
    libc.mmap.restype, libc.mmap.argtypes = C.c_void_p, [C.c_void_p, C.c_size_t, C.c_int, C.c_int, C.c_int, C.c_long]
    libc.madvise.argtypes, libc.munmap.argtypes = [C.c_void_p, C.c_size_t, C.c_int], [C.c_void_p, C.c_size_t]
    size, parent, live = {}, os.getpid(), []

    class Fake:
        @staticmethod
        def mi_host_alloc(n, out):
            out._obj.value = libc.mmap(None, n, mmap.PROT_READ | mmap.PROT_WRITE, mmap.MAP_PRIVATE | mmap.MAP_ANONYMOUS, -1, 0)
            assert libc.madvise(out._obj.value, n, 10) == 0                  # MADV_DONTFORK
            size[out._obj.value] = n
            return 0

        @staticmethod
        def mi_host_free(p):
            if os.getpid() != parent:
                os._exit(3)
            libc.munmap(p.value, size.pop(p.value))

    monkeypatch.setattr(E.L, "lib", lambda: Fake)
    pool = E._ResultPool()
    monkeypatch.setattr(E, "_results", pool)
    pool.engine_opened()
    live = [pool.empty((300, 1000)), pool.empty((4, 70000))]
    pool.empty((500, 1000))                                                  # kept, shown by nobody
    for i, a in enumerate(live):
        a[:] = np.arange(a.size, dtype=np.float32).reshape(a.shape) + i
    pid = os.fork()
    if pid == 0:
        code = 4
        try:
            ok = all(np.array_equal(a.ravel(), np.arange(a.size, dtype=np.float32) + i) for i, a in enumerate(live))
            live[0][:] = -1.0
            pool.engine_closed()
            del a, live[:]
            code = 0 if ok else 5
        finally:
            os._exit(code)
    assert os.waitpid(pid, 0)[1] == 0
    assert live[0][0, 1] == 1.0 and len(size) == 3
    del a, live[:]
    pool.engine_closed()
    assert not size and pool._bytes == 0 and not pool._out


@pytest.mark.parametrize("f32", [False, True])
def test_decode_attention_splits(f32):
    """How many splits a decode step's attention is launched with: one round of workgroups where the rows leave half the chip idle; above
    that, the rounds that would otherwise end nearly empty (33 to 40 rows, 17 rows of long contexts) are cut finer and full ones are not."""
    from mlx_parallm_amd import _lib as L

    def splits(rows, keys):
        return L.lib().mi_op_attention_decode_splits(256, rows * 8, keys, L.MI_F32 if f32 else L.MI_BF16)

    assert [splits(b, 8000) for b in (1, 2, 4, 6, 8, 10, 12, 16)] == [16, 16, 8, 5 if f32 else 4, 4, 3, 2, 2]
    assert [splits(1, k) for k in (0, 1, 96, 97, 300, 1279, 1280)] == [1, 1, 1, 2, 4, 4, 5 if f32 else 4]
    for b in (20, 24, 28, 31, 32, 56, 60, 64, 96, 128):                 # a full last round, or short rows: one split
        assert splits(b, 1000) == 1 and (b in (20,) or splits(b, 4100) == 1), b
    assert all(splits(b, 500) == 1 for b in range(17, 129))
    for b in (33, 34, 36, 40):                                          # 8 to 64 of 256 workgroups in the last round
        assert 2 <= splits(b, 4100) <= 6 and 2 <= splits(b, 2047) <= 4, b
    assert splits(17, 8000) >= 3
    for b in range(1, 129):
        for keys in (0, 1, 95, 700, 5000, 32000):
            assert 1 <= splits(b, keys) <= 16


def test_float32_rows_leave_the_streaming_kernel_where_the_tile_pays():
    """Logits and layer 0's rounded call on float32 activations: at decode batches and short prompts the streaming kernel is ahead (int4 logits of
    64 rows: 2.2 ms against 4.4 on a copy of the matrix), at long ones the tile GEMM.  (codes: int4 matrices too small for the codes kernel; the others below)"""
    from mlx_parallm_amd import _lib as L

    def pays(rows, codes=0, hilo=0, rounded=0):
        return bool(L.lib().mi_op_gemm_prefill_pays(codes, hilo, rounded, rows))

    assert not any(pays(n, codes=1) for n in (33, 64, 130, 300, 700)) and all(pays(n, codes=1) for n in (1024, 2048, 8192))
    for hilo in (0, 1):
        assert [pays(n, hilo=hilo) for n in (33, 64, 96, 97, 128, 129, 192, 193, 256, 257, 300, 8192)] == [False] * 3 + [True] * 2 + [False] * 2 + [True] * 5
    assert all(pays(n, rounded=1) for n in (32, 33, 64, 8192))
    assert not any(pays(n, codes=1, rounded=1) for n in (33, 64, 96)) and all(pays(n, codes=1, rounded=1) for n in (128, 700))
    assert not any(pays(n, hilo=1, rounded=1) for n in (33, 768, 1024)) and pays(2048, hilo=1, rounded=1)


def _quant_route(rows, N, K, kind="q8_bf16", act="float32", epi="STORE", rnd=0):
    """2: the tile GEMM on the codes, 1: on their [hi | lo] copy, 0: another kernel (include/mi355_ops.h)"""
    import ctypes as C

    from mlx_parallm_amd import _lib as L

    w, a = L.OpLinear(), L.OpGemvArgs()
    w.wk, w.N, w.K, w.group, w.layout = L.WK[kind], N, K, 64, 1
    a.M, a.ldx, a.act, a.rnd = rows, K, {"float32": L.MI_F32, "bfloat16": L.MI_BF16, "float16": L.MI_F16}[act], rnd
    a.epi, a.ldo = getattr(L, "EPI_" + epi), N
    a.pair_offset = N // 2 if epi == "SWIGLU" else 0
    return L.lib().mi_op_gemm_quant_route(C.byref(w), C.byref(a))


def test_int8_on_float32_rows_is_never_multiplied_as_a_pair():
    """A pair of bf16 holds an int8 weight to 2^-17 only once its group's mean exceeds 3 deviations; the streaming kernel and the codes hold it."""
    from mlx_parallm_amd import _lib as L

    for rows in (33, 64, 128, 129, 150, 300, 700, 1024, 1365, 3000, 9000):
        for N, K in ((64, 64), (256, 128), (1024, 1024), (1536, 1024), (1024, 3072), (4096, 2048), (28672, 4096), (32784, 512), (4096, 14336), (160, 65600)):
            for epi, rnd in (("STORE", 0), ("STORE", L.RND_BF16), ("STORE_F32", 0), ("RESID", 0), ("SWIGLU", 0)):
                got = _quant_route(rows, N, K, epi=epi, rnd=rnd)
                assert got in (0, 2) and (got == 0 or 128 < rows), (rows, N, K, epi, rnd, got)
    assert [_quant_route(n, 1024, 1024) for n in (64, 128, 129, 1365)] == [0, 0, 2, 2]


def test_prefill_routes_of_quantised_matrices():
    """Float32 rows leave the streaming kernel where the codes kernel is ahead by both sides' times; 16-bit rows, and float32 rows of int4, take the codes from
    some 2e9 (K >= 4096) or 4e9 products on and the [hi | lo] copy below; what the kernels refuse stays refused."""
    def first(rows, *a, **kw):
        got = [_quant_route(n, *a, **kw) for n in rows]
        assert got == sorted(got), got                            # (no way back with more rows)
        return got.index(2)

    rows = list(range(33, 700))
    for kind in ("q4_bf16", "q8_bf16"):                           # int8: 224 rows 317 us on the streaming kernel, 352 on the codes; 256: 363, 357
        assert 224 < rows[first(rows, 28672, 4096, kind, epi="SWIGLU")] <= 256
    assert 96 < rows[first(rows, 6144, 4096, "q4_bf16")] <= 129   # 96 rows 59, 68; 129: 99, 69
    assert rows[first(rows, 6144, 4096, "q8_bf16")] == 129        # (a decode batch stays on the streaming kernel)
    assert 96 < rows[first(rows, 32000, 2048, "q4_bf16", epi="STORE_F32")] <= 192      # 129 rows 138, 133
    for act, q in (("bfloat16", "q4_bf16"), ("float16", "q8_f16")):
        assert [_quant_route(n, 4096, 4096, q, act) for n in (31, 32, 125, 126, 700)] == [0, 1, 1, 2, 2]
        assert [_quant_route(n, 2048, 1024, q, act, epi="RESID") for n in (129, 2048, 2051)] == [1, 1, 2]
    assert [_quant_route(n, 512, 512, "q4_bf16") for n in (64, 300)] == [1, 1]
    assert _quant_route(8192, 4096, 65536 + 128, "q4_bf16", "bfloat16") == 1           # (more biases of a row tile than 64 KiB)
    assert _quant_route(300, 4096, 192, "q4_bf16", "bfloat16") == 0 and _quant_route(300, 4096, 4096, "q4_f16", "float32") == 0
    assert _quant_route(300, 4104, 4096, "q4_bf16", "bfloat16") == 0


@pytest.mark.parametrize("f32", [False, True])
def test_prefill_attention_slices(f32):
    """Over how many workgroups a prefill call's keys are split: not where the join costs more than it saves (a prompt from its start), several for
    a chunk behind a long cache, never fewer for more keys -- a row's own number may not depend on a longer neighbour's."""
    import ctypes as C

    from mlx_parallm_amd import _lib as L

    def slices(B, L_, keys, Hq=32, Hkv=8, D=128):
        s = L.OpAttnShape()
        s.B, s.L, s.Hq, s.Hkv, s.D, s.rnd, s.cap = B, L_, Hq, Hkv, D, 0, 8192
        s.act = s.kv = L.MI_F32 if f32 else L.MI_BF16
        return L.lib().mi_op_attention_prefill_slices(C.byref(s), keys, 256)

    assert all(slices(B, L_, L_) == 1 for B, L_ in ((1, 16), (1, 64), (1, 128), (1, 200), (1, 256), (2, 64), (2, 128), (4, 64), (8, 1024)))
    assert [slices(1, 32, k) > 1 for k in (64, 160, 732, 4032)] == [False, False, True, True]
    assert slices(1, 16, 4016) >= 8 and 3 <= slices(1, 128, 4128) <= 4 and slices(2, 128, 4128) == 2 and slices(4, 256, 4000) == 1
    for B, L_, Hq, Hkv in ((1, 16, 8, 8), (1, 40, 40, 8), (3, 17, 16, 2), (2, 200, 10, 2), (16, 32, 5, 1)):
        got = [slices(B, L_, k, Hq, Hkv) for k in range(L_, 8192, 7)]
        assert got == sorted(got) and 1 <= got[0] and got[-1] <= 16
        assert all(n == 1 or 2 * n <= (k + 31) // 32 for n, k in zip(got, range(L_, 8192, 7)))


def test_which_int4_linears_take_their_rows_prepared():
    """The shapes of test_gpu_engine.py's test of prepared rows are such linears at every number of rows there (each of its row tiles a slab), and where the rule ends: rows, short K
    without a norm, more than one round of workgroups behind a long K, few columns behind a long K, a norm of its own."""
    import ctypes as C

    from mlx_parallm_amd import _lib as L

    def prepared(rows, N, K, act="bfloat16", epi=L.EPI_RESID, pro=0):
        ol, a = L.OpLinear(), L.OpGemvArgs()
        ol.wk, ol.N, ol.K, ol.group, ol.layout = L.WK["q4_bf16" if act == "bfloat16" else "q4_f16"], N, K, 64, 1
        a.M, a.act, a.ldx, a.ldo, a.epi, a.pro = rows, L.MI_BF16 if act == "bfloat16" else L.MI_F16, K, N, epi, pro
        return L.lib().mi_op_gemm_q4_prepared(C.byref(ol), C.byref(a))

    for act, K in (("bfloat16", 640), ("float16", 512), ("bfloat16", 512)):
        assert [prepared(n, 256, K, act) for n in (17, 33, 64, 65, 97, 128)] == [2, 3, 4, 3, 4, 4]
        assert all(prepared(n, 256, K, act) > 0 for n in (12 + 16, 30 + 33, 3 + 90))
    assert all(prepared(n, 256, 640) > 0 for n in (17, 28, 33, 63, 64, 65, 93, 97, 128))          # the down projection there
    assert prepared(16, 256, 640) == prepared(129, 256, 640) == prepared(64, 256, 384) == prepared(64, 256, 640, pro=L.PRO_NORM) == 0
    assert prepared(64, 4096, 14336) == 4 and prepared(64, 5120, 17408) == 4 and prepared(100, 5120, 17408) == 0
    assert prepared(64, 2048, 20480) == 4 and prepared(64, 4096, 24576) == 4 and prepared(64, 2048, 20608) == prepared(17, 3072, 24576) == prepared(17, 4096, 24704) == 0


def test_which_chunks_share_the_attention_launch_of_a_mixed_step():
    """The first chunks of test_gpu_engine.py's mixed steps do at the numbers of keys there (its second one of two has a launch of its own), a chunk of many tiles and other caches do not."""
    import ctypes as C

    from mlx_parallm_amd import _lib as L

    def shape(B, n, heads, kv_heads, hd=128, act=L.MI_BF16, kv=None):
        s = L.OpAttnShape()
        s.B, s.L, s.Hq, s.Hkv, s.D, s.act, s.kv, s.rnd, s.cap = B, n, heads, kv_heads, hd, act, act if kv is None else kv, 0, 4096
        return s

    def shared(rows, chunk, heads, kv_heads, keys, **kw):
        r, c = shape(rows, 1, heads, kv_heads, **kw), shape(1, chunk, heads, kv_heads, **kw)
        return L.lib().mi_op_attention_mixed(C.byref(r), C.byref(c), max(1, L.lib().mi_op_attention_prefill_slices(C.byref(c), keys, 256)), 256)

    for rows, chunk, heads, kv_heads, act in ((3, 32, 10, 2, L.MI_BF16), (40, 16, 4, 1, L.MI_F16), (1, 17, 8, 1, L.MI_BF16), (2, 40, 2, 1, L.MI_F16)):
        assert all(shared(rows, chunk, heads, kv_heads, chunk * k, act=act) == 1 for k in (1, 2, 3, 4)), (rows, chunk)
    assert [shared(5, 200, 3, 3, k) for k in (200, 800)] == [1, 0]          # (39 tiles; in slices more workgroups than half of the compute units)
    assert shared(31, 32, 40, 8, 672) == 1 and shared(31, 512, 40, 8, 1152) == 0
    assert shared(3, 32, 8, 2, 64, act=L.MI_F32) == shared(3, 32, 8, 2, 64, hd=64) == shared(3, 32, 6, 2, 64) == shared(3, 1, 8, 2, 64) == 0
